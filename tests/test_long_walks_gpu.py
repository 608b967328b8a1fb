"""Points whose walks are far longer than a round's budget: points along a line, whose hint cells
hold thousands of them, on a hint grid sized by a tiny first load."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def line(n, dim, seed, lo=0.0, hi=1.0):
    rng = np.random.default_rng(seed)
    P = np.empty((n, dim))
    P[:, 0] = rng.uniform(lo, hi, n)
    P[:, 1:] = 0.5 + 1e-4 * rng.uniform(-1, 1, (n, dim - 1))
    return P


@pytest.mark.parametrize("pipelined", [1, 0])
@pytest.mark.parametrize("budget", [1, 16])
@pytest.mark.parametrize("dim", [3, 2])
def test_a_load_thousands_of_simplices_from_every_hint(dim, budget, pipelined):
    import voronoids_amd as vo
    P = np.vstack([line(20000, dim, 1), line(4, dim, 3, 0.52, 0.53), line(100, dim, 2, 0.95, 0.951)])
    t = vo.DelaunayTree(P)
    t.config("walk_budget", budget)
    t.config("pipelined", pipelined)
    t.add_points_to_tree(P[:16])
    t.add_points_to_tree(P[16:20000])
    for k in range(20000, 20004):            # the hints of the line's upper half: all near 0.52
        t.add_points_to_tree(P[k:k + 1])
    rounds = t.stats()["rounds"]
    t.add_points_to_tree(P[20004:])          # thousands of simplices from there, in one short stretch
    assert t.stats()["rounds"] - rounds < 200
    assert t.violations() == 0 and t.stats()["points_inserted"] == len(P)
    other = vo.delaunay(P[::-1], seed=4)
    T, E = other.canonical()
    Tt, Et = t.canonical()
    assert len(T) == len(Tt) and len(E) == len(Et)
    assert np.array_equal(np.unique(np.sort(len(P) - 1 - T, axis=1), axis=0), Tt)
