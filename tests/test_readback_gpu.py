"""Large results on their way to the host, at the sizes where the pinned slots take over (8 MB),
where a last slot is partly filled, and where slots are used again (twelve of 2 MB)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim,n", [(2, 524287), (2, 524288), (2, 524289), (3, 349525), (3, 349526),
                                   (2, 1572863), (2, 1572864), (2, 1572865), (3, 1048576), (3, 1048577), (2, 3400001)])
def test_coordinates_come_back(dim, n):
    import voronoids_amd as vo
    P = np.random.default_rng(n).random((n, dim))
    t = vo.DelaunayTree(P)
    t.stage(P)
    for _ in range(2):                            # the second time through slots used before
        assert np.array_equal(t.coordinates()[2 * t.M:], P)


@pytest.mark.parametrize("dim,n", [(2, 90001), (3, 20011), (3, 150007)])
def test_export_and_canonical_hold_the_same_simplices(dim, n):
    import voronoids_amd as vo
    from voronoids_amd.batch import canonical_from_simplices
    P = np.random.default_rng(n).random((n, dim))
    t = vo.delaunay(P)
    s, nb = t.export()
    T, E = t.canonical()
    Th, Eh = canonical_from_simplices(s, dim)
    assert np.array_equal(T, Th) and np.array_equal(E, Eh)
    i, k = np.nonzero(nb >= 0)                    # adjacency is mutual
    assert np.all(np.any(nb[nb[i, k]] == i[:, None], axis=1))
