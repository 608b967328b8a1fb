"""vo_engine_canonical on lists that a caller made: rows given twice come out twice, as the host
sorts them (buckets of lane groups and of one block)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim,n", [(2, 700), (2, 3000), (3, 300), (3, 3000)])
def test_rows_given_twice(dim, n):
    import voronoids_amd as vo
    from voronoids_amd import datasets
    from voronoids_amd.batch import canonical_from_simplices
    e = vo.Engine(dim, max_points=1 << 16)
    star = np.random.default_rng(n).normal(size=(200, dim))
    star = np.vstack([np.zeros((1, dim)), star / np.linalg.norm(star, axis=1)[:, None]])
    for r in e.batch([datasets.uniform(n, dim, seed=43), np.vstack([star, 2 + datasets.uniform(n, dim, seed=44)])]):
        s = r.simplices
        rng = np.random.default_rng(1)
        r.simplices = rng.permuted(np.vstack([s, s[::3], s[::7]])[rng.permutation(len(s) + len(s[::3]) + len(s[::7]))], axis=1)
        T, E = r.canonical()
        Th, Eh = canonical_from_simplices(r.simplices, dim)
        assert np.array_equal(T, Th) and np.array_equal(E, Eh) and len(T) > len(canonical_from_simplices(s, dim)[0])
