"""Calls that meet the end of the device's memory (tests/cpp/test_limited_memory.cpp, built by
tests/cpp/Makefile: a hipMalloc of its own refuses what would pass a limit)."""
import os
import subprocess

import pytest

BIN = os.path.join(os.path.dirname(os.path.abspath(__file__)), "cpp", "_bin", "test_limited_memory")


@pytest.mark.gpu
@pytest.mark.parametrize("what", ["points", "copies", "equal", "compact"])
def test_limited_memory(what):
    r = subprocess.run([BIN, what], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0 and f"{what}: ok" in r.stdout, r.stdout + r.stderr
