"""What the makefile builds with and without torch (dry runs: nothing is
compiled), and what the package does when a library is missing."""

import os
import shutil
import subprocess
import sys

import pytest

PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "sglang-mlx_amd")
CSRC = os.path.join(PKG, "csrc")


@pytest.mark.parametrize("python,native", [("python3", True), ("python3 -S", False), ("/nonexistent/python3", False)])
def test_c_library_builds_without_torch(python, native):
    r = subprocess.run(["make", "-C", CSRC, "-n", "-B", "PYTHON=" + python], capture_output=True, text=True)
    assert r.returncode == 0 and not r.stderr, r.stderr
    assert "libpagedkv_gfx950.so" in r.stdout
    assert ("_native.so" in r.stdout) == native


@pytest.mark.parametrize("missing", ["libpagedkv_gfx950.so", "_native.so"])
def test_package_imports_without_a_library_and_calls_raise(tmp_path, missing):
    shutil.copytree(os.path.join(PKG, "sglang_mlx_amd"), tmp_path / "sglang_mlx_amd",
                    ignore=shutil.ignore_patterns(missing, "__pycache__"))
    code = ("import sglang_mlx_amd._ext as e, sglang_mlx_amd._lib as l\n"
            "try:\n    l.lib()\nexcept ImportError as x:\n    print('raised', x)\n")
    r = subprocess.run([sys.executable, "-c", code], cwd=tmp_path, capture_output=True, text=True,
                       env={**os.environ, "PYTHONPATH": str(tmp_path)})
    assert r.returncode == 0, r.stderr
    assert "raised" in r.stdout and missing in r.stdout
