"""The canonical form with vertices of more than 4,096 simplices or edges: hubs as the first, a middle
and the last point, two of them beside uniform points, and none of them a simplex of points only."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def hub(dim, n, seed, at=0):
    rng = np.random.default_rng(seed)
    u = rng.normal(size=(n, dim))
    u *= (1 + (1e-3 if dim == 3 else 1e-10) * rng.random((n, 1))) / np.linalg.norm(u, axis=1, keepdims=True)
    return np.insert(u, at, 0.0, axis=0)


def sets(dim):
    n = 3000 if dim == 3 else 4500
    yield hub(dim, n, 1)
    yield hub(dim, n, 2, at=n // 2)
    yield hub(dim, n, 3, at=n)
    far = 10 + np.random.default_rng(4).random((5000, dim))
    yield np.vstack([hub(dim, n, 5), far, 4 + hub(dim, n, 6, at=n)])


@pytest.mark.parametrize("dim", [2, 3])
def test_hubs(dim):
    import voronoids_amd as vo
    from voronoids_amd.batch import canonical_from_simplices
    e = vo.Engine(dim, max_points=1 << 16)
    for P in sets(dim):
        t = vo.delaunay(P)
        for swap in (False, True):                 # (an edited tree gives every edge of every simplex)
            if swap:
                t.swap_simplex_vertices(0, 0, 1)
            s = t.export()[0]
            for _ in range(2):
                T, E = t.canonical()
                Th, Eh = canonical_from_simplices(s, dim)
                assert np.array_equal(T, Th) and np.array_equal(E, Eh)
        assert np.bincount(E.ravel()).max() > (4096 if dim == 2 else 2500)
        r = e.batch([P])[0]
        for twice in (False, True):
            if twice:
                r.simplices = np.vstack([r.simplices, r.simplices[::5]])
            T, E = r.canonical()
            Th, Eh = canonical_from_simplices(r.simplices, dim)
            assert np.array_equal(T, Th) and np.array_equal(E, Eh)


@pytest.mark.parametrize("dim", [2, 3])
def test_edges_without_a_simplex_of_points(dim):
    import voronoids_amd as vo
    from voronoids_amd.batch import canonical_from_simplices
    e = vo.Engine(dim, max_points=1 << 16)
    r = e.batch([np.random.default_rng(1).random((6000, dim))])[0]
    M = dim + 1
    rows = np.zeros((5000, M), np.int32)           # (super vertex, point 0, any point)
    rows[:, 1], rows[:, 2] = 2 * M, 2 * M + 1 + np.arange(5000)
    rows[:, M - 1], rows[:, 2 if dim == 2 else 2] = rows[:, 2], rows[:, 2]
    if dim == 3:
        rows[:, 3] = 1
    r.simplices = rows
    T, E = r.canonical()
    Th, Eh = canonical_from_simplices(rows, dim)
    assert len(T) == 0 and len(E) == 5000 and np.array_equal(E, Eh) and T.shape == Th.shape
