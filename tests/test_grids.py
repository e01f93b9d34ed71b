"""Calls of more events than one launch holds: their parts, on the host
(tests/cpp/test_grids.cpp)."""
import os
import subprocess

BIN = os.path.join(os.path.dirname(os.path.abspath(__file__)), "cpp", "bin", "test_grids")


def test_parts_of_large_calls():
    r = subprocess.run([BIN], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr
