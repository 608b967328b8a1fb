"""A point whose cavity outgrows the lists and which needs exact predicates on the far side of it, in a
run that evaluates its exact predicates on the device: each try alone meets the next of them."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def shell(dim, n, rng):
    """points on a sphere around 0, and for each of its facets the point opposite 0 on the sphere through
    the facet and 0: the facet's outer simplex has 0 on its sphere, up to rounding"""
    if dim == 2:
        a = 2 * np.pi * (np.arange(n) + 0.3 * rng.random(n)) / n
        S = np.stack([np.cos(a), np.sin(a)], axis=1)
        F = np.stack([np.arange(n), (np.arange(n) + 1) % n], axis=1)
    else:
        from scipy.spatial import ConvexHull
        S = rng.normal(size=(n, 3))
        S /= np.linalg.norm(S, axis=1)[:, None]
        F = ConvexHull(S).simplices
    # the center c of the sphere through 0 and the facet: 2 c . v = |v|^2
    far = np.array([np.linalg.solve(S[f], np.sum(S[f] ** 2, axis=1)) for f in F])
    return np.vstack([S, far])


@pytest.mark.parametrize("boot", [0, 256])
@pytest.mark.parametrize("dim,n", [(2, 150), (3, 300)])
def test_large_cavity_with_exact_predicates_behind_it(dim, n, boot):
    import voronoids_amd as vo
    rng = np.random.default_rng(dim)
    A = shell(dim, n, rng)
    B = 0.25 * shell(dim, 12, rng) + 10.0          # a small one, whose center needs exact predicates at once
    P = np.vstack([A, B, 20 + rng.random((100, dim))])
    Q = np.vstack([np.zeros((1, dim)), np.full((1, dim), 10.0), 22 + rng.random((6, dim))])
    t = vo.DelaunayTree(np.vstack([P, Q]))
    t.config("small_run", 0)
    t.config("boot_window", boot)
    t.add_points_to_tree(P)
    before = t.stats()
    t.add_points_to_tree(Q, seed=1)
    s = t.stats()
    print(dim, boot, "rounds", s["rounds"] - before["rounds"], "solo", s["solo_runs"] - before["solo_runs"],
          "exact", s["exact_evaluated"] - before["exact_evaluated"], flush=True)
    assert s["points_inserted"] == len(P) + len(Q) and s["solo_runs"] > before["solo_runs"]
    assert t.violations() == 0
