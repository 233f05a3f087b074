"""The library and its C programs build where Python has no torch: the native call path of the
wrappers is left out."""
import os
import shutil
import subprocess

import pytest

import kami_amd

CSRC = os.path.join(os.path.dirname(kami_amd.__file__), "csrc")


@pytest.mark.skipif(shutil.which("make") is None, reason="needs make")
@pytest.mark.parametrize("python,built", [("python3", True), ("false", False)])
def test_what_is_built(python, built):
    r = subprocess.run(["make", "-n", "-B", "-C", CSRC, f"PYTHON={python}"], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    assert "libkami.so" in r.stdout and "kami_bench" in r.stdout
    assert ("fast_calls.cpp" in r.stdout) == built
