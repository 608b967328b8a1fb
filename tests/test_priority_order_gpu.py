"""The insertion order made on the device is the Fisher-Yates shuffle over splitmix64(seed).  It
shows in which of two equal points is kept: the one that comes first."""
import numpy as np
import pytest

MASK = (1 << 64) - 1


def fisher_yates(n, seed):
    perm, s = list(range(n)), seed
    for i in range(n - 1, 0, -1):
        s = (s + 0x9E3779B97F4A7C15) & MASK
        z = ((s ^ (s >> 30)) * 0xBF58476D1CE4E5B9) & MASK
        z = ((z ^ (z >> 27)) * 0x94D049BB133111EB) & MASK
        j = ((z ^ (z >> 31)) * (i + 1)) >> 64
        perm[i], perm[j] = perm[j], perm[i]
    return np.array(perm)


@pytest.mark.gpu
@pytest.mark.parametrize("dim", [2, 3])
@pytest.mark.parametrize("pairs,seed", [(4, 0), (31, 1), (33, 2), (500, MASK), (4095, 7), (4096, 8), (4097, 9), (20000, 10)])
def test_the_first_of_two_equal_points_is_kept(dim, pairs, seed):
    import voronoids_amd as vo
    from voronoids_amd import datasets
    P = datasets.uniform(pairs, dim, seed=31)
    P = np.vstack([P, P])
    t = vo.DelaunayTree(P)
    with pytest.raises(vo.VoError) as e:
        t.add_points_to_tree(P, seed=seed)
    assert e.value.code == -4
    place = np.empty(2 * pairs, np.int64)
    place[fisher_yates(2 * pairs, seed)] = np.arange(2 * pairs)
    first = np.where(place[:pairs] < place[pairs:], np.arange(pairs), np.arange(pairs) + pairs)
    kept = np.unique(t.export()[0])
    M = dim + 1
    assert np.array_equal(kept[kept >= 2 * M] - 2 * M, np.sort(first))
    assert np.array_equal(t.coordinates()[2 * M:], P)
