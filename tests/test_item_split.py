"""The work split of a launch over its workgroups (make_split in launch.h), host
code only, built with g++ (tests/item_split.cc)."""

from __future__ import annotations

import shutil
import subprocess
from pathlib import Path

import pytest

HERE = Path(__file__).resolve().parent
CSRC = HERE.parent / "arthip_amd" / "csrc"


def test_split_covers_every_item_and_never_lengthens_the_longest_range(tmp_path):
    gxx = shutil.which("g++")
    if gxx is None or not Path("/opt/rocm/include/hip/hip_runtime.h").exists():
        pytest.skip("g++ or the HIP headers are not available")
    exe = tmp_path / "item_split"
    subprocess.run([gxx, "-std=c++17", "-O1", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-I", str(CSRC),
                    str(HERE / "item_split.cc"), "-o", str(exe)], check=True, capture_output=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
