"""What the makefile builds with and without torch (dry runs: nothing is
compiled)."""

import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "sglang-mlx_amd", "csrc")


@pytest.mark.parametrize("python,native", [("python3", True), ("python3 -S", False), ("/nonexistent/python3", False)])
def test_c_library_builds_without_torch(python, native):
    r = subprocess.run(["make", "-C", CSRC, "-n", "-B", "PYTHON=" + python], capture_output=True, text=True)
    assert r.returncode == 0 and not r.stderr, r.stderr
    assert "libpagedkv_gfx950.so" in r.stdout
    assert ("_native.so" in r.stdout) == native
