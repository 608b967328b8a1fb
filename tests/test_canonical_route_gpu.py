"""Which way canonical forms are sorted, at the sizes where it changes (vo_canonical_route): what
compares a device's sort with the host's has to have been sorted on the device."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
BUCKETS, RADIX, HOST = 1, 2, 3


def star(dim, n, seed=5):
    rng = np.random.default_rng(seed)
    u = rng.normal(size=(n, dim))
    u *= (1 + 1e-10 * rng.random((n, 1))) / np.linalg.norm(u, axis=1, keepdims=True)
    return np.vstack([np.zeros((1, dim)), u])


def route():
    from voronoids_amd import _lib
    return _lib.lib().vo_canonical_route()


@pytest.mark.parametrize("dim,n,way", [(2, 3, BUCKETS), (2, 64, BUCKETS), (2, 65, BUCKETS), (2, 4096, BUCKETS), (2, 4097, RADIX),
                                       (3, 4, BUCKETS), (3, 35, BUCKETS), (3, 2050, BUCKETS), (3, 2051, RADIX)])
def test_trees(dim, n, way):
    import voronoids_amd as vo
    t = vo.delaunay(star(dim, n))
    t.canonical()
    assert route() == way
    empty = vo.DelaunayTree(np.zeros((0, dim)))
    T, E = empty.canonical()
    assert route() == 0 and len(T) == len(E) == 0


@pytest.mark.parametrize("dim", [2, 3])
def test_results_of_an_engine(dim):
    import voronoids_amd as vo
    from voronoids_amd import datasets
    from voronoids_amd.batch import canonical_from_simplices
    e = vo.Engine(dim, max_points=1 << 16)
    small, large, hub = e.batch([datasets.uniform(20, dim, seed=1), datasets.uniform(4096, dim, seed=2),
                                 star(dim, 4500 if dim == 2 else 2100)])
    assert len(small.simplices) < 1024 <= len(large.simplices)
    for r, way in ((small, HOST), (large, BUCKETS), (hub, RADIX)):
        T, E = r.canonical()
        assert route() == way
        Th, Eh = canonical_from_simplices(r.simplices, dim)
        assert route() == HOST and np.array_equal(T, Th) and np.array_equal(E, Eh)
    large.n_points -= 1                        # the last point's index is then past the end
    large.canonical()
    assert route() == HOST
    large.n_points += 1
    e.close()
    large.canonical()
    assert route() == HOST
