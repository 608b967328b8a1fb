"""The first points of an empty tree, inserted by one workgroup in LDS: sizes around where the phase
takes a whole set (96 points in 3D, 128 in 2D) and where it hands over, against the oracle."""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu


def check(P, seed=3):
    import voronoids_amd as vo
    t = vo.DelaunayTree(P)
    t.add_points_to_tree(P, seed=seed)
    if P.shape[0] > 1:                 # (the oracle has no super simplex around a single point)
        ref = O.Tree.delaunay(P, O.MODE_EXACT).canonical()
        T, E = t.canonical()
        assert np.array_equal(T, ref.T) and np.array_equal(E, ref.E)
    assert t.violations() == 0
    st = t.stats()
    assert st["points_inserted"] == st["winners_total"] == P.shape[0]
    assert t.counts()[1] == t.export()[0].shape[0] == 1 + st["created"] - st["killed"]
    return t


@pytest.mark.parametrize("dim,n", [(3, 1), (3, 2), (3, 7), (3, 8), (3, 9), (3, 47), (3, 48), (3, 49), (3, 95), (3, 96),
                                   (3, 97), (3, 105), (2, 1), (2, 31), (2, 32), (2, 33), (2, 127), (2, 128), (2, 129)])
def test_sizes(dim, n):
    for k in range(3):
        check(np.random.default_rng(100 * n + k).random((n, dim)))


@pytest.mark.parametrize("dim", [2, 3])
def test_near_cospherical_points_and_large_cavities_hand_over(dim):
    # every simplex's sphere holds nearly all points: queued exact predicates, cavities beyond the
    # lists, and in 3D (points along a curve) more simplices than LDS holds
    rng = np.random.default_rng(7)
    u = rng.normal(size=(90, dim))
    check(np.vstack([0.5 + 0.3 * u / np.linalg.norm(u, axis=1)[:, None], 0.5 + 0.05 * rng.random((5, dim))]))
    s = np.sort(rng.random(90))
    check(np.stack([s, s ** 2, s ** 3], axis=1)[:, :dim])


@pytest.mark.parametrize("dim", [2, 3])
def test_duplicates_among_the_first_points(dim):
    import voronoids_amd as vo
    P = np.random.default_rng(9).random((40, dim))
    Q = np.vstack([P, P[:7]])
    t = vo.DelaunayTree(Q)
    with pytest.raises(vo.VoError) as e:
        t.add_points_to_tree(Q, seed=1)
    assert e.value.code == -4
    st = t.stats()
    assert st["points_inserted"] == 40 and st["points_duplicate"] == 7 and t.violations() == 0
    t.reset(P)                                         # the handle goes on as a fresh one
    t.add_points_to_tree(P[:20])
    t.add_points_to_tree(P[20:])
    ref = O.Tree.delaunay(P, O.MODE_EXACT).canonical()
    T, E = t.canonical()
    assert np.array_equal(T, ref.T) and np.array_equal(E, ref.E)
