"""Results over the library's own memory (no GPU: the host's canonical form)."""
import copy
import dataclasses
import os
import pickle
import subprocess
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

_AT_EXIT = """
import atexit
kept = []
atexit.register(lambda: print("sum", int(kept[0].sum(dtype="int64")), int(kept[1].sum(dtype="int64")), flush=True))
import numpy as np
from voronoids_amd.batch import canonical_from_simplices
T, E = canonical_from_simplices(np.random.default_rng(0).integers(8, 10**6, (10**6, 4)), 3)
kept += [T, E]
print("sum", int(T.sum(dtype="int64")), int(E.sum(dtype="int64")), flush=True)
"""


def test_an_engines_result_is_a_plain_record():
    import numpy as np
    from voronoids_amd.batch import Engine, SetResult
    s = np.array([[8, 9, 10, 11], [0, 8, 9, 12]], np.int32)
    e = Engine.__new__(Engine)                 # (stands for the engine it came from)
    r = e._mine([SetResult(7, 3, 0, 5, 0, s, 0.0, 0.25, 0.5, 3)])[0]
    names = ["tag", "dim", "status", "n_points", "points_duplicate", "simplices", "t_submit", "t_admit", "t_done", "rounds"]
    assert [f.name for f in dataclasses.fields(r)] == names
    d = pickle.loads(pickle.dumps(dataclasses.asdict(r)))
    assert list(d) == names and np.array_equal(d["simplices"], s) and len(dataclasses.astuple(r)) == len(names)
    for q in (pickle.loads(pickle.dumps(r)), copy.copy(r), copy.deepcopy(r), dataclasses.replace(r, tag=7)):
        T, E = q.canonical()                   # sorted on the host: a copy knows no engine
        assert q.tag == 7 and T.tolist() == [[0, 1, 2, 3]] and len(E) == 8


def test_arrays_are_there_for_exit_handlers():
    r = subprocess.run([sys.executable, "-c", _AT_EXIT], capture_output=True, text=True, cwd=ROOT, timeout=120)
    assert r.returncode == 0, r.stderr
    alive, at_exit = r.stdout.strip().splitlines()
    assert alive == at_exit and alive.startswith("sum")
