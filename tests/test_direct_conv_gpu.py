"""Direct convs of narrow layers (direct.hip) against the CPU oracle at the edges
of their tiles, and the dispatch rules that route a conv there."""

from __future__ import annotations

import ctypes

import numpy as np
import pytest

from arthip_amd import _lib, models
from arthip_amd.engine import Engine
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


# conv3x3_rows: one wave per segment of up to 62 pixels (four 16-pixel tiles), one
# output row per step, input rows two steps ahead: runs of one, two and three
# rows, segment edges, many rows per wave, several runs per wave (many segments,
# few rows).
ROWS_SIZES = [(1, 1, 1), (2, 2, 15), (1, 3, 17), (3, 5, 61), (1, 2, 62), (1, 1, 63), (2, 4, 125), (1, 700, 130),
              (1, 3, 4001), (2, 67, 1921)]


def _skips(seed, k, n, m, h, w):
    rng = np.random.default_rng(seed)
    return [rng.standard_normal((n, m, h, w)).astype(np.float16) for _ in range(k)]


@pytest.mark.parametrize("n,h,w", ROWS_SIZES)
@pytest.mark.parametrize("c,m,k", [(16, 16, 1), (24, 24, 2), (32, 32, 0), (48, 48, 1)])
def test_rows(c, m, k, n, h, w):
    x, wt, b = make_case(60, n, c, m, h, w)
    sk = _skips(61, k, n, m, h, w)
    check(run_conv(x, wt, b, 1, sk), oracle_conv(x, wt, b, 1, sk), f"rows c{c}m{m} skip{k} {n}x{h}x{w}")


@pytest.mark.parametrize("c", [16, 24, 32, 40, 48])
@pytest.mark.parametrize("m", [8, 16, 24, 32, 40, 48])
def test_rows_channels(c, m):
    k = (c + m) // 8 % 3
    x, wt, b = make_case(62, 1, c, m, 13, 70)
    sk = _skips(63, k, 1, m, 13, 70)
    check(run_conv(x, wt, b, 0, sk), oracle_conv(x, wt, b, 0, sk), f"rows c{c}m{m} skip{k}")


@pytest.mark.parametrize("act", [0, 1, 2])
@pytest.mark.parametrize("k", [0, 1, 2])
def test_rows_epilogue(act, k):
    x, wt, b = make_case(64, 1, 48, 48, 19, 66)
    sk = _skips(65, k, 1, 48, 19, 66)
    check(run_conv(x, wt, b, act, sk), oracle_conv(x, wt, b, act, sk), f"rows act{act} skip{k}")


@pytest.mark.parametrize("c", [16, 24, 32, 40, 48])
def test_rows_nonfinite(c):
    _nonfinite_stays_local(c, 16, 9, 131, _skips(66, 1, 1, 16, 9, 131))


# conv3x3_head_pair and conv3x3_tail_pair (the 32-channel model in two launches)
# against every conv launched alone, on frames above the 4096 pixels from which
# they run: one segment, many segments, a single row or column, run boundaries, a
# batch, fp16 and fp32 boundaries. The head pair has the two kernels' bits; the
# tail's 288 products are summed in another order in fp32: 288 half-ulp roundings
# of partial sums, bounded here by the largest output, and one final rounding.
PAIR_SIZES = [(1, 69, 61), (2, 33, 125), (1, 1, 4500), (1, 4500, 1), (1, 271, 480), (1, 90, 57)]


@pytest.mark.parametrize("n,h,w", PAIR_SIZES)
@pytest.mark.parametrize("fp32", [False, True])
def test_pairs(n, h, w, fp32):
    spec = models.c4f32(seed=3)
    x = models.synthetic_input((n, 1, h, w), seed=5)
    x = x.astype(np.float32) if fp32 else x
    model = models.widen_to_fp32(spec) if fp32 else spec
    with Engine(0) as e, Engine(0) as alone:
        alone.set_debug(Engine.DEBUG_UNFUSED)
        got, want = e.build(model).run(x), alone.build(model).run(x)
        assert "2 launches" in e.describe() and "4 launches" in alone.describe()
    got, want = got.astype(np.float64), want.astype(np.float64)
    bound = 288 * 2.0 ** -24 * np.abs(want).max() + (0 if fp32 else 2.0 ** -10) * np.abs(want) + 1e-7
    assert np.all(np.abs(got - want) <= bound), float(np.abs(got - want).max())


@pytest.mark.parametrize("fp32", [False, True])
def test_pair_output_alignment(fp32):
    """An output on one element only: stored element by element, the same bits."""
    import torch
    spec = models.c4f32(seed=3)
    model = models.widen_to_fp32(spec) if fp32 else spec
    dt = torch.float32 if fp32 else torch.float16
    x = torch.from_numpy(models.synthetic_input((1, 1, 70, 66), seed=5)).to(dt).cuda()
    with Engine(0) as e:
        e.build(model)
        outs = []
        for off in (0, 1):
            buf = torch.full((140 * 132 + 2,), 7.0, dtype=dt, device="cuda")
            out = buf[off:off + 140 * 132].view(1, 1, 140, 132)
            e.run_device(x, out)
            torch.cuda.synchronize()
            assert float(buf[-1]) == 7.0 and (off == 0 or float(buf[0]) == 7.0)
            outs.append(out.cpu().numpy())
    np.testing.assert_array_equal(outs[0], outs[1])


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


@pytest.mark.parametrize("c,m,k", [(3, 64, 0), (32, 32, 1), (48, 24, 1)])
def test_unaligned_buffers(c, m, k):
    """Buffers on 8 bytes only: accepted, by the general kernel."""
    x, wt, b = make_case(53, 1, c, m, 21, 67)
    sk = _skips(54, k, 1, m, 21, 67)
    got = _run_offset(x, wt, b, sk[0] if k else None, 8)
    check(got, oracle_conv(x, wt, b, 1, sk), f"offset c{c}m{m}")
