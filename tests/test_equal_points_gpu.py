"""Of equal points the first in the insertion order is kept, also where its walk pauses and a later one
arrives before it."""
import numpy as np
import pytest

from test_priority_order_gpu import fisher_yates

pytestmark = pytest.mark.gpu


def points(kind, n, dim, rng):
    if kind == "uniform":
        return rng.random((n, dim))
    if kind == "cauchy":
        return rng.standard_cauchy((n, dim))
    P = np.empty((n, dim))
    P[:, 0] = rng.random(n)
    P[:, 1:] = 1e-4 * rng.uniform(-1, 1, (n, dim - 1))
    return P


@pytest.mark.parametrize("pipelined", [1, 0])
@pytest.mark.parametrize("budget", [1, 16])
@pytest.mark.parametrize("kind,n,copies", [("uniform", 3000, 2), ("uniform", 20000, 5), ("line", 4000, 3), ("cauchy", 12000, 2)])
@pytest.mark.parametrize("dim", [2, 3])
def test_the_first_is_kept(dim, kind, n, copies, budget, pipelined):
    import voronoids_amd as vo
    rng = np.random.default_rng(n + budget)
    U = points(kind, n, dim, rng)
    which = np.concatenate([np.arange(n)] + [rng.integers(0, n, n // 2) for _ in range(copies - 1)])
    which = which[rng.permutation(len(which))]
    P = U[which]
    # zeros of either sign are equal
    P[which < 20, 1] = np.where(rng.random((which < 20).sum()) < 0.5, 0.0, -0.0)
    t = vo.DelaunayTree(P)
    t.config("walk_budget", budget)
    t.config("pipelined", pipelined)
    M = t.M
    perm = fisher_yates(len(P), 5)
    w, at = np.unique(which[perm], return_index=True)      # the first place of each point in the order
    first = np.sort(perm[at])
    for load in range(2):
        with pytest.raises(vo.VoError) as e:
            t.add_points_to_tree(P, seed=5)
        assert e.value.code == -4
        kept = np.unique(t.export()[0])
        assert np.array_equal(kept[kept >= 2 * M] - 2 * M, first)
        X = t.coordinates()[2 * M:]
        assert np.array_equal(X.view(np.int64), np.vstack([P] * (load + 1)).view(np.int64))
        assert t.violations() == 0 and t.stats()["points_inserted"] == n
