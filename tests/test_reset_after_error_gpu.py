"""A handle whose run failed (a point outside the super simplex) is a fresh tree after a reset: no
record of the failed run is left."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("pipelined", [1, 0])
@pytest.mark.parametrize("n", [20, 60, 90, 125, 400, 5000])
@pytest.mark.parametrize("dim", [2, 3])
def test_reset_after_a_point_outside(dim, n, pipelined):
    import voronoids_amd as vo
    rng = np.random.default_rng(n)
    P = rng.random((n, dim))
    Q = P.copy()
    Q[n // 2] = 1e6                          # far outside the super simplex of P
    t = vo.DelaunayTree(P)
    t.config("pipelined", pipelined)
    for k, m in enumerate((n, n // 2, 10, 3 * n)):
        with pytest.raises(vo.VoError) as e:
            t.add_points_to_tree(Q, seed=k)
        assert e.value.code == -1
        if k % 2:
            with pytest.raises(vo.VoError):  # the error stays until the reset
                t.add_points_to_tree(P[:k])
        R = rng.random((m, dim))
        t.reset(R)
        t.add_points_to_tree(R, seed=k)
        s, nb = t.export()
        f = vo.delaunay(R, seed=k)
        assert len(s) == t.counts()[1] == f.counts()[1] and t.violations() == 0
        for a, b in zip(t.canonical(), f.canonical()):
            assert np.array_equal(a, b)
        t.reset(P)
