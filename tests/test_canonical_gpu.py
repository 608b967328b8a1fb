"""The canonical form sorted on the device, at the sizes where its buckets change hands: 64 entries
(lane groups), 4,096 (one block in LDS), above that (radix sort)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def star(dim, n, seed=5):
    """point 0 with every other point around it on a circle or sphere, so that all of them are its
    neighbors (2D: n simplices at point 0, 3D: 2 n - 4)"""
    rng = np.random.default_rng(seed)
    u = rng.normal(size=(n, dim))
    u *= (1 + 1e-10 * rng.random((n, 1))) / np.linalg.norm(u, axis=1, keepdims=True)
    return np.vstack([np.zeros((1, dim)), u])


@pytest.mark.parametrize("dim,n", [(2, 3), (2, 63), (2, 64), (2, 65), (2, 4095), (2, 4096), (2, 4097),
                                   (3, 4), (3, 34), (3, 35), (3, 2050), (3, 2051)])
def test_bucket_sizes(dim, n):
    import voronoids_amd as vo
    from voronoids_amd.batch import canonical_from_simplices
    t = vo.delaunay(star(dim, n))
    T, E = t.canonical()
    Th, Eh = canonical_from_simplices(t.export()[0], dim)
    assert np.array_equal(T, Th) and np.array_equal(E, Eh)
    assert np.sum(E[:, 0] == 0) == n


@pytest.mark.parametrize("dim", [2, 3])
@pytest.mark.parametrize("n", [0, 1, 2, 3, 4, 5, 255, 1025])
def test_small_trees_and_edited_ones(dim, n):
    import voronoids_amd as vo
    from voronoids_amd import datasets
    from voronoids_amd.batch import canonical_from_simplices
    P = datasets.uniform(n, dim, seed=21)
    t = vo.DelaunayTree(P)
    t.add_points_to_tree(P)
    for swap in (False, True):
        if swap:                                  # vertices swapped, adjacency not: the same edges
            t.swap_simplex_vertices(0, 0, 1)
        T, E = t.canonical()
        Th, Eh = canonical_from_simplices(t.export()[0], dim)
        assert np.array_equal(T, Th) and np.array_equal(E, Eh)


@pytest.mark.parametrize("dim,n", [(2, 30), (3, 100), (3, 150), (2, 700), (3, 4096)])
def test_engine_results_sorted_on_the_device_equal_the_hosts(dim, n):
    import voronoids_amd as vo
    from voronoids_amd import datasets
    from voronoids_amd.batch import canonical_from_simplices
    e = vo.Engine(dim, max_points=1 << 16)
    sets = [datasets.uniform(n, dim, seed=41), star(dim, 70), datasets.uniform(n + 1, dim, seed=42)]
    res = e.batch(sets)
    for closed in (False, True):                  # a closed engine's results are sorted on the host
        if closed:
            e.close()
        for r in res:
            T, E = r.canonical()
            Th, Eh = canonical_from_simplices(r.simplices, dim)
            assert np.array_equal(T, Th) and np.array_equal(E, Eh)
