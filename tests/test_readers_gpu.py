"""Reading calls of one tree from several threads at once: each gets what it gets alone (large
enough for the pinned slots and small)."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim,n", [(2, 3000), (2, 530000), (3, 360000)])
def test_readers_beside_each_other(dim, n):
    import voronoids_amd as vo
    P = np.random.default_rng(n).random((n, dim))
    t = vo.delaunay(P)
    q = np.full(dim, 0.37)
    calls = {"coordinates": lambda: (t.coordinates(),), "canonical": t.canonical, "export": t.export,
             "locate": lambda: (t.locate(q)[0],), "violations": lambda: (np.array(t.violations()),)}
    alone = {k: f() for k, f in calls.items()}
    bad = []

    def read(name, f):
        try:
            for _ in range(6):
                if not all(np.array_equal(a, b) for a, b in zip(f(), alone[name])):
                    bad.append(name)
        except Exception as e:
            bad.append((name, repr(e)))

    threads = [threading.Thread(target=read, args=kf) for kf in calls.items()]
    for th in threads:
        th.start()
    for th in threads:
        th.join()
    assert not bad
