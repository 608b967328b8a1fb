"""The 3D commit's ridge match (csrc/ridges.hpp) on the CPU: closed boundaries pair up, and on
broken ones (a tree edited by hand) the search ends and leaves ridges unpaired."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


def test_ridge_match(tmp_path):
    cxx = shutil.which("g++")
    if cxx is None:
        pytest.skip("g++ not found")
    exe = tmp_path / "ridges"
    r = subprocess.run([cxx, "-std=c++17", "-O1", "-Wall", "-Wextra", "-Werror", "-o", str(exe),
                        os.path.join(HERE, "cpp", "test_ridges.cpp")], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=20)
    assert r.returncode == 0 and "ridges: ok" in r.stdout, r.stdout + r.stderr
