"""The chunked download of a frame (host_copy.cc) on a simulated HIP runtime
(tests/chunked_download.cc, host code only, built with g++): the bytes arrive,
a failure is reported only when nothing can still write the staging, and helper
threads do not busy-wait for the GPU."""

from __future__ import annotations

import shutil
import subprocess
from pathlib import Path

import pytest

HERE = Path(__file__).resolve().parent
CSRC = HERE.parent / "arthip_amd" / "csrc"


@pytest.fixture(scope="module")
def download(tmp_path_factory):
    gxx = shutil.which("g++")
    if gxx is None or not Path("/opt/rocm/include/hip/hip_runtime.h").exists():
        pytest.skip("g++ or the HIP headers are not available")
    exe = tmp_path_factory.mktemp("download") / "chunked_download"
    subprocess.run([gxx, "-std=c++17", "-O1", "-pthread", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    "-I", str(CSRC), str(HERE / "chunked_download.cc"), str(CSRC / "host_copy.cc"),
                    "-o", str(exe)], check=True, capture_output=True)
    return exe


# Exit status 0: copied; 2: refused, with every chunk that was sent landed.
# "slow": while the frame's first chunk is not there, the caller alone waits (a
# wait for an event keeps a core busy).
@pytest.mark.parametrize("scenario,status", [("ok", 0), ("slow", 0), ("copy", 2), ("first_wait", 2), ("last_wait", 2),
                                             ("device", 2)])
def test_download(download, scenario, status):
    r = subprocess.run([str(download), scenario], capture_output=True, text=True, timeout=60)
    assert r.returncode == status, (scenario, r.returncode, r.stdout, r.stderr)
