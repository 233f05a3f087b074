"""The wave units that a batched launch reads, from the library's own host code: every 16 x 16
atom of every queue entry once, at every wave tile size (tests/sanitize/units_check.cpp)."""
import os
import shutil
import subprocess

import pytest

import kami_amd

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SRC = os.path.join(ROOT, "tests", "sanitize", "units_check.cpp")
LIB = os.path.dirname(kami_amd.__file__)


@pytest.mark.skipif(not os.path.exists(SRC) or not os.path.exists("/opt/rocm/bin/hipcc") or
                    shutil.which("make") is None, reason="needs hipcc and the check's source")
def test_units_cover_every_entry_once(tmp_path):
    exe = str(tmp_path / "units_check")
    subprocess.run(["/opt/rocm/bin/hipcc", "--offload-arch=gfx950", "-O1", "-std=c++17", "-w",
                    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops", "-I" + os.path.join(LIB, "csrc"),
                    "-x", "hip", SRC, "-o", exe, "-L" + LIB, "-lkami", "-Wl,-rpath," + LIB], check=True, timeout=600)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0 and " 0 faults" in r.stdout, r.stdout + r.stderr
