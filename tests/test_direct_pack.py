"""Layout of the direct taps of narrow layers (arthip_conv3x3_pack): the products
that the kernels in direct.hip issue reproduce a direct correlation."""

from __future__ import annotations

import ctypes

import numpy as np
import pytest

from arthip_amd import _lib


def _packed(w):
    lib = _lib.lib()
    m, c = w.shape[:2]
    u = np.zeros(lib.arthip_conv3x3_packed_halfs(m, c), np.uint16)
    b = np.zeros(lib.arthip_conv3x3_bias_len(m), np.float32)
    u16, f32 = ctypes.POINTER(ctypes.c_uint16), ctypes.POINTER(ctypes.c_float)
    rc = lib.arthip_conv3x3_pack(w.view(np.uint16).ctypes.data_as(u16), None, m, c, u.ctypes.data_as(u16), u.size,
                                 b.ctypes.data_as(f32), b.size)
    assert rc == 0
    return u.view(np.float16).astype(np.float64)


@pytest.mark.parametrize("c,m", [(2, 32), (3, 64), (4, 96), (16, 16), (24, 8), (32, 32), (40, 40), (48, 24), (48, 48)])
def test_direct_taps_reproduce_the_conv(c, m):
    rng = np.random.default_rng(c * 100 + m)
    w = (rng.standard_normal((m, c, 3, 3)) * 0.2).astype(np.float16)
    x = rng.standard_normal((3, 5, c)).astype(np.float16).astype(np.float64)  # rows, pixels, channels
    n_ob, kr = (m + 15) // 16, (3 * c + 31) // 32
    head = c <= 4
    n = n_ob * 64 * 16 if head else 3 * kr * n_ob * 64 * 8
    taps = _packed(w)[-n:]
    # Output pixels 0 .. 2 read pixels p .. p + 2: 3 C contiguous values per row.
    rows = np.zeros((3, 3, 64 * kr))
    for p in range(3):
        rows[:, p, :3 * c] = x[:, p:p + 3].reshape(3, -1)
    got = np.zeros((n_ob, 16, 3))
    for q in range(4):
        for i in range(16):
            lane = 16 * q + i
            for b in range(n_ob):
                if head:
                    if q < 3:
                        got[b, i] += rows[q, :, :16] @ taps.reshape(n_ob, 64, 16)[b, lane]
                    else:
                        assert not taps.reshape(n_ob, 64, 16)[b, lane].any()
                else:
                    for dy in range(3):
                        for kc in range(kr):
                            k = 32 * kc + 8 * q
                            got[b, i] += rows[dy, :, k:k + 8] @ taps.reshape(3, kr, n_ob, 64, 8)[dy, kc, b, lane]
    want = np.einsum("mcyx,ypxc->mp", w.astype(np.float64),
                     np.stack([x[:, p:p + 3] for p in range(3)], 1))
    for ch in range(m):
        b, i = ch % (4 * n_ob) // 4, ch // (4 * n_ob) * 4 + ch % 4
        np.testing.assert_allclose(got[b, i], want[ch], rtol=1e-12, atol=1e-12)
    if not head:  # rows of A past M are zero
        dead = [(ch % (4 * n_ob) // 4, ch // (4 * n_ob) * 4 + ch % 4) for ch in range(m, 16 * n_ob)]
        assert not any(got[b, i].any() for b, i in dead)
