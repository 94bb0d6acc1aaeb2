"""Direct convs of narrow layers (direct.hip) against the CPU oracle at the edges
of their tiles, and the dispatch rules that route a conv there."""

from __future__ import annotations

import ctypes

import numpy as np
import pytest

from arthip_amd import _lib
from tests.test_conv_kernel_gpu import (check, make_case, oracle_conv, pack, run_conv, to_padded)

pytestmark = pytest.mark.gpu

# Segments are 64 pixels (16 per wave) in the head: single pixels, one less and
# one more than a block or segment, odd heights, many rows per workgroup.
HEAD_SIZES = [(1, 1, 1), (1, 2, 15), (2, 3, 17), (1, 5, 63), (1, 1, 64), (2, 4, 65), (1, 300, 129), (1, 7, 1921)]


@pytest.mark.parametrize("n,h,w", HEAD_SIZES)
@pytest.mark.parametrize("c,m", [(2, 32), (2, 96), (3, 64), (3, 96), (4, 32), (4, 64)])
def test_head(c, m, n, h, w):
    x, wt, b = make_case(50, n, c, m, h, w)
    check(run_conv(x, wt, b, 1), oracle_conv(x, wt, b, 1), f"head c{c}m{m} {n}x{h}x{w}")


@pytest.mark.parametrize("act", [0, 2])
@pytest.mark.parametrize("c", [2, 3, 4])
def test_head_act(c, act):
    x, wt, b = make_case(51, 1, c, 64, 19, 70)
    check(run_conv(x, wt, b, act), oracle_conv(x, wt, b, act), f"head c{c} act{act}")


def _nonfinite_stays_local(c, m, h, w, skips=()):
    """An infinite pixel reaches its 3x3 neighbourhood and nothing else (no value
    of another pixel is multiplied by a padding zero of the filters)."""
    x, wt, b = make_case(52, 1, c, m, h, w)
    clean = run_conv(x, wt, b, 0, skips)
    bad = x.copy()
    ys, xs = [0, h // 2, h - 1], [0, w // 2, w - 1]
    near = np.zeros((h, w), bool)
    for y, xx in zip(ys, xs):
        bad[0, :, y, xx] = np.inf
        near[max(0, y - 1):y + 2, max(0, xx - 1):xx + 2] = True
    got = run_conv(bad, wt, b, 0, skips)
    np.testing.assert_array_equal(got[0][:, ~near], clean[0][:, ~near])
    assert not np.isfinite(got[0][:, near]).all(axis=0).any()


@pytest.mark.parametrize("c", [2, 3, 4])
def test_head_nonfinite(c):
    _nonfinite_stays_local(c, 64, 9, 131)


def _run_offset(x, wt, b, skip, off):
    """run_conv with every activation buffer `off` bytes into its allocation."""
    import torch
    lib = _lib.lib()
    n, c, h, w = x.shape
    m = wt.shape[0]
    u, bias = pack(wt, b)

    def buf(a):
        t = torch.zeros(a.size + 64, dtype=torch.float16, device="cuda")
        v = t[off // 2:off // 2 + a.size]
        v.copy_(torch.from_numpy(a.reshape(-1)))
        return v

    xin = buf(to_padded(x))
    hp, wp = to_padded(x).shape[1:3]
    sk = None if skip is None else buf(to_padded(skip))
    out = buf(np.zeros((n, hp, wp, m), np.float16))
    ut, bt = torch.from_numpy(u.view(np.float16)).cuda(), torch.from_numpy(bias).cuda()
    ptr = lambda t: None if t is None else ctypes.c_void_p(t.data_ptr())
    rc = lib.arthip_conv3x3_f16_nhwc(ptr(xin), ptr(ut), ptr(bt), 1, ptr(sk), None, ptr(out), n, h, w, c, m, None)
    assert rc == 0, _lib.last_error()
    torch.cuda.synchronize()
    o = out.cpu().numpy().reshape(n, hp, wp, m)
    return o[:, 1:h + 1, 1:w + 1].astype(np.float32).transpose(0, 3, 1, 2)


@pytest.mark.parametrize("c,m", [(3, 64)])
def test_unaligned_buffers(c, m):
    """Buffers on 8 bytes only: accepted, by the general kernel."""
    x, wt, b = make_case(53, 1, c, m, 21, 67)
    check(_run_offset(x, wt, b, None, 8), oracle_conv(x, wt, b, 1), f"offset c{c}m{m}")
