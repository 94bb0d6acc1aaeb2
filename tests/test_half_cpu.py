"""Host fp32 -> fp16 rounding (half.h) against numpy's, at every place where it
can go wrong: each half, the middle to its neighbour and one float either side
of both, of both signs, the ends of the normal and subnormal ranges, infinities
and NaN."""

from __future__ import annotations

import shutil
import subprocess
from pathlib import Path

import numpy as np
import pytest

HERE = Path(__file__).resolve().parent
CSRC = HERE.parent / "arthip_amd" / "csrc"


def test_f32_to_f16(tmp_path):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ is not available")
    exe = tmp_path / "half_convert"
    subprocess.run([gxx, "-std=c++17", "-O2", "-I", str(CSRC), str(HERE / "half_convert.cc"), "-o", str(exe)],
                   check=True, capture_output=True)
    halfs = np.arange(0x7c01, dtype=np.uint16).view(np.float16).astype(np.float32)
    halfs[-1] = 65536.0  # past the largest half, as the middle above it needs it
    mid = (halfs[:-1] + halfs[1:]) / 2  # exact in fp32
    base = np.concatenate([halfs, mid]).view(np.uint32)
    bits = np.concatenate([base, base + 1, np.maximum(base, 1) - 1,
                           np.array([0x7f800000, 0x7f7fffff, 0x7fc00000, 0x7f800001, 1], np.uint32)])
    f = np.concatenate([bits, bits | 0x80000000]).view(np.float32)
    r = subprocess.run([str(exe)], input=f.tobytes(), capture_output=True, check=True, timeout=60)
    got = np.frombuffer(r.stdout, np.float16)
    with np.errstate(over="ignore"):
        want = f.astype(np.float16)
    nan = np.isnan(f)
    assert np.isnan(got[nan]).all() and got.size == f.size
    np.testing.assert_array_equal(got[~nan].view(np.uint16), want[~nan].view(np.uint16))
