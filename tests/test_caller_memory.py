"""Which caller memory the kernels may touch themselves (tests/caller_memory_check.cpp)."""
from __future__ import annotations

import os
import shutil
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_ranges_lie_in_one_allocation(tmp_path):
    exe = str(tmp_path / "caller_memory_check")
    cxx = os.environ.get("CXX", shutil.which("g++") or "g++")
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    subprocess.run([cxx, "-std=c++17", "-O1", "-D__HIP_PLATFORM_AMD__", "-I", os.path.join(rocm, "include"),
                    "-I", os.path.join(ROOT, "relearn_amd", "csrc"),
                    os.path.join(ROOT, "tests", "caller_memory_check.cpp"), "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=20)
    assert r.returncode == 0, r.stdout
