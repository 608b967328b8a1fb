"""vo_tri_set_vertex finds its vertex among the ids of the first, the last and any point, staged or
inserted, and no other."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim", [2, 3])
@pytest.mark.parametrize("n", [1, 255, 256, 257, 70000])
def test_vertex_ids(dim, n):
    import voronoids_amd as vo
    P = np.random.default_rng(n).random((n + 3, dim))
    t = vo.DelaunayTree(P)
    t.add_points_to_tree(P[:n], seed=2)
    t.stage(P[n:], seed=3)
    X = t.coordinates()
    for k in {0, n // 3, n - 1, n, n + 2}:
        vid = 2 * t.M + k
        t.set_vertex(vid, X[vid] * 0.5, records=False)
        X[vid] *= 0.5
        assert np.array_equal(t.coordinates(), X)
    for vid in (-1, 0, 2 * t.M - 1, 2 * t.M + n + 3, 2**31, 2**40):
        with pytest.raises(vo.VoError) as e:
            t.set_vertex(vid, P[0])
        assert e.value.code == -1
    assert np.array_equal(t.coordinates(), X)
