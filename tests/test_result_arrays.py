"""Result arrays over the library's own memory (no GPU: the host's canonical form)."""
import os
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


def test_arrays_are_there_for_exit_handlers():
    r = subprocess.run([sys.executable, "-c", _AT_EXIT], capture_output=True, text=True, cwd=ROOT, timeout=120)
    assert r.returncode == 0, r.stderr
    alive, at_exit = r.stdout.strip().splitlines()
    assert alive == at_exit and alive.startswith("sum")
