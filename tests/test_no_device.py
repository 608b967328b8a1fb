"""Without a device vo_tri_create names the call that failed; bad points are refused before it."""
import os
import subprocess
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_create_without_a_device():
    code = """
import os
os.environ["HIP_VISIBLE_DEVICES"] = "-1"
import numpy as np, voronoids_amd as vo
for P in (np.zeros((3, 2)), np.full((9000, 3), np.nan)):
    try:
        vo.DelaunayTree(P)
    except vo.VoError as e:
        print(e.code, e)
"""
    r = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, cwd=ROOT, timeout=120)
    assert r.returncode == 0, r.stderr
    hip, bad = r.stdout.strip().splitlines()
    assert hip.startswith("-3 ") and "hipGetDeviceCount" in hip
    assert bad.startswith("-1 ") and "non-finite" in bad
