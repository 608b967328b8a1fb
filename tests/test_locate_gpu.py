"""vo_tri_locate at the sizes where its lists change hands: one pass (64 pairs), several, and more
killed simplices than LDS holds (2,048); the insertion of the same point gives the counts."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim,n", [(2, 3), (2, 40), (2, 3000), (3, 4), (3, 12), (3, 40), (3, 700), (3, 1400)])
def test_cavity_of_the_center_of_a_shell(dim, n):
    import voronoids_amd as vo
    u = np.random.default_rng(n).normal(size=(n, dim))
    P = u * (1 + 1e-9 * np.arange(n)[:, None]) / np.linalg.norm(u, axis=1)[:, None]
    q = np.full((1, dim), 1e-3)
    t = vo.DelaunayTree(np.vstack([P, q]))
    t.add_points_to_tree(P)
    s, nb = t.export()
    killed, facets = t.locate(q[0])
    assert np.array_equal(killed, np.unique(killed)) and killed[0] >= 0 and killed[-1] < s.shape[0]
    # the facets are the faces between the cavity and the rest, each with its own vertices
    inside = np.zeros(s.shape[0] + 1, bool)
    inside[killed] = True
    rows = {(int(i), int(nb[i, f]) if nb[i, f] >= 0 else -1, tuple(sorted(np.delete(s[i], f).tolist())))
            for i in killed for f in range(dim + 1) if not inside[nb[i, f]]}
    assert {(int(r[0]), int(r[1]), tuple(sorted(r[2:].tolist()))) for r in facets} == rows and len(rows) == len(facets)
    before = t.stats()
    t.add_points_to_tree(q)
    after = t.stats()
    assert after["killed"] - before["killed"] == len(killed) and after["created"] - before["created"] == len(facets)


@pytest.mark.parametrize("reuse", [0, 1])
@pytest.mark.parametrize("dim,n", [(2, 1), (2, 160), (2, 171), (3, 37), (3, 38), (2, 40000), (3, 9000)])
def test_positions_of_queries_all_over(dim, n, reuse):
    """export positions from the first record that a query meets on: records within one tile of
    1,024, just past one, many tiles; near the super simplex (the oldest records) and inside"""
    import voronoids_amd as vo
    rng = np.random.default_rng(n)
    P = rng.random((n, dim))
    t = vo.DelaunayTree(P)
    t.config("reuse", reuse)
    t.add_points_to_tree(P)
    s, nb = t.export()
    X = t.coordinates()
    Q = np.vstack([rng.random((6, dim)), 3 * rng.random((3, dim)) - 1, 0.5 * P[:1] + 0.5 * X[:1], X[:dim + 1] * 0.7 + 0.15])
    for q in Q:
        killed, facets = t.locate(q)
        assert np.array_equal(killed, np.unique(killed)) and killed[0] >= 0 and killed[-1] < s.shape[0]
        inside = np.zeros(s.shape[0] + 1, bool)
        inside[killed] = True
        rows = {(int(i), int(nb[i, f]) if nb[i, f] >= 0 else -1, tuple(sorted(np.delete(s[i], f).tolist())))
                for i in killed for f in range(dim + 1) if nb[i, f] < 0 or not inside[nb[i, f]]}
        assert {(int(r[0]), int(r[1]), tuple(sorted(r[2:].tolist()))) for r in facets} == rows and len(rows) == len(facets)
