"""Direct convs of narrow layers (direct.hip) against the CPU oracle at the edges
of their tiles, and the dispatch rules that route a conv there."""

from __future__ import annotations

import ctypes

import numpy as np
import pytest

from arthip_amd import _lib, models
from arthip_amd import onnx_proto as op
from arthip_amd.engine import Engine
from oracle.model import run_model
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


# conv3x3_rows: one wave per segment of up to 30 pixels (C = 16, 32, 48: two
# 16-pixel tiles) or 62 (C = 24, 40: four; but two for more than 32 outputs on up to
# 2^15 pixels, and at C = 40 without a residual input on any), one output row per
# step, input rows two steps ahead: runs of one, two and three rows, one pixel less
# and more than a tile and than a segment of either length, many rows per wave,
# several runs per wave (many segments, few rows).
ROWS_SIZES = [(1, 1, 1), (2, 2, 15), (1, 3, 17), (1, 2, 29), (1, 4, 30), (2, 3, 31), (1, 5, 32), (3, 5, 61),
              (1, 2, 62), (1, 1, 63), (2, 4, 91), (2, 4, 125), (1, 700, 130), (1, 3, 4001), (2, 67, 1921)]


def _skips(seed, k, n, m, h, w):
    rng = np.random.default_rng(seed)
    return [rng.standard_normal((n, m, h, w)).astype(np.float16) for _ in range(k)]


@pytest.mark.parametrize("n,h,w", ROWS_SIZES)
@pytest.mark.parametrize("c,m,k", [(16, 16, 1), (24, 24, 2), (32, 32, 0), (48, 48, 1), (24, 48, 2), (40, 40, 0),
                                   (40, 40, 1)])
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
@pytest.mark.parametrize("c", [32, 48])
def test_rows_epilogue(c, act, k):
    x, wt, b = make_case(64, 1, c, c, 19, 66)
    sk = _skips(65, k, 1, c, 19, 66)
    check(run_conv(x, wt, b, act, sk), oracle_conv(x, wt, b, act, sk), f"rows c{c} act{act} skip{k}")


# Outputs above 96 MiB are stored with the non-temporal hint: 1082 x 1502 padded
# pixels of 32 channels are 99 MiB. Checked against the oracle on windows at the
# corners and in the middle (with the conv's own zero padding only where the window
# ends at the image's edge: one pixel more is computed and dropped elsewhere).
@pytest.mark.parametrize("k", [0, 1])
def test_rows_large_output(k):
    h, w = 1080, 1499
    x, wt, b = make_case(67, 1, 32, 32, h, w)
    sk = _skips(68, k, 1, 32, h, w)
    got = run_conv(x, wt, b, 1, sk)
    for r0, r1, c0, c1 in ((0, 12, 0, 70), (533, 545, 700, 800), (h - 12, h, w - 70, w)):
        a0, a1, b0, b1 = max(0, r0 - 1), min(h, r1 + 1), max(0, c0 - 1), min(w, c1 + 1)
        want = oracle_conv(x[:, :, a0:a1, b0:b1], wt, b, 1, [t[:, :, a0:a1, b0:b1] for t in sk])
        check(got[:, :, r0:r1, c0:c1], want[:, :, r0 - a0:r1 - a0, c0 - b0:c1 - b0], f"rows large skip{k} {r0},{c0}")


@pytest.mark.parametrize("c", [16, 24, 32, 40, 48])
def test_rows_nonfinite(c):
    _nonfinite_stays_local(c, 16, 9, 131, _skips(66, 1, 1, 16, 9, 131))


# conv3x3_head_pair and conv3x3_tail_pair (the 32-channel model in two launches)
# against every conv launched alone: single pixels, one segment (30 output pixels
# in the head pair, 28 in the tail pair) and one pixel less and more, many
# segments, a single row or column, run boundaries, a batch, fp16 and fp32
# boundaries. The head pair has the two kernels' bits; the tail's 288 products are
# summed in another order in fp32: 288 half-ulp roundings of partial sums (of
# order one, as the inputs and the tensors between the layers are, or the size of
# the largest output), and one final rounding.
PAIR_SIZES = [(1, 1, 1), (1, 2, 3), (3, 5, 27), (1, 4, 28), (1, 3, 29), (2, 6, 30), (1, 5, 31), (1, 69, 61),
              (2, 33, 125), (1, 1, 4500), (1, 4500, 1), (1, 271, 480), (1, 90, 57)]


def _pair_engines(spec, fp32, x, debug=0):
    """Outputs of the model with and without the pairs, and the fused plan."""
    model = models.widen_to_fp32(spec) if fp32 else spec
    x = x.astype(np.float32) if fp32 else x
    with Engine(0) as e, Engine(0) as alone:
        if debug:
            e.set_debug(debug)
        alone.set_debug(Engine.DEBUG_UNFUSED)
        got, want = e.build(model).run(x), alone.build(model).run(x)
        assert "2 launches, 1 activation buffers" in e.describe() and "4 launches" in alone.describe()
    return got.astype(np.float64), want.astype(np.float64)


def _check_pair(got, want, fp32, slope=1.0):
    order = 288 * 2.0 ** -24 * max(1.0, np.abs(want).max())
    bound = slope * order + (0 if fp32 else 2.0 ** -10) * np.abs(want) + 1e-7
    assert np.all(np.abs(got - want) <= bound), float(np.abs(got - want).max())


def _check_model(got, ref, label):
    """Four layers of at most two fp16 nodes each, rounded once in the engine and
    per node in the oracle: eight independent roundings of at most 2^-11 (rms
    2^-11 / sqrt 3), carried through the He-normal convs at their size, are 8e-4
    of the rms; twice that is allowed in all, ten times it in one value."""
    ref = ref.astype(np.float64)
    rms = np.sqrt(np.mean(ref ** 2))
    err = np.abs(got - ref)
    assert np.all(err <= 2.0 ** -9 * np.abs(ref) + 8e-3 * rms), (label, float(err.max()), float(rms))
    assert np.sqrt(np.mean(err ** 2)) <= 1.6e-3 * rms, (label, float(np.sqrt(np.mean(err ** 2)) / rms))


@pytest.mark.parametrize("n,h,w", PAIR_SIZES)
@pytest.mark.parametrize("fp32", [False, True])
def test_pairs(n, h, w, fp32):
    x = models.synthetic_input((n, 1, h, w), seed=5)
    _check_pair(*_pair_engines(models.c4f32(seed=3), fp32, x), fp32)


def _pair_spec(acts, tail_act=None, clip=None):
    """c4f32 with other activations, biases, and optionally a Clip at its end."""
    b = models._Builder(9, "uniform")
    t = "x"
    for cin, act in zip((1, 32, 32), acts):
        t = b.conv(t, cin, 32, act)
    t = b.conv(t, 32, 4, tail_act)
    b.nodes.append(op.node("DepthToSpace", [t], ["d2s"], blocksize=2, mode="DCR"))
    t = "d2s"
    if clip:
        b.inits += [op.tensor(f"clip_{k}", np.array(v, np.float16)) for k, v in zip(("lo", "hi"), clip)]
        b.nodes.append(op.node("Clip", [t, "clip_lo", "clip_hi"], ["clipped"]))
        t = "clipped"
    return models.ModelSpec(b.finish("x", t, 1, 1), "pairs", 1, 1, 2, b.convs, b.skips, b.conv_in, b.skip_names)


# Every instance: the head pair's first activation is the template's, its second a
# branch; the tail pair's likewise, then the tail's activation and Clip. Against
# the convs alone, and against the oracle (SiLU's derivative stays below 1.1, so
# it widens the bound by that).
@pytest.mark.parametrize("acts", [("relu", None, "silu"), ("silu", "relu", None), (None, "silu", "relu"),
                                  (None, None, None), ("silu", "silu", "silu")])
@pytest.mark.parametrize("tail_act,clip", [(None, None), ("relu", (0.1, 0.4)), ("silu", (-0.05, 0.3))])
@pytest.mark.parametrize("fp32", [False, True])
def test_pair_epilogues(acts, tail_act, clip, fp32):
    spec = _pair_spec(acts, tail_act, clip)
    x = models.synthetic_input((1, 1, 45, 67), seed=6)
    got, want = _pair_engines(spec, fp32, x)
    assert np.unique(got).size > 100  # (not clipped away)
    _check_pair(got, want, fp32, 1.1)
    _check_model(got, run_model(spec.model, x), f"pairs {acts} {tail_act} {clip} fp32 {fp32}")


@pytest.mark.parametrize("fp32", [False, True])
def test_pairs_large(fp32):
    """The tensor between the pairs above 96 MiB: non-temporal stores, in the convs
    alone as well, so both are also compared with the oracle on windows (nine
    pixels from any edge that is not the image's, the receptive field's four and
    more)."""
    spec = models.c4f32(seed=3)
    h, w = 1080, 1499
    x = models.synthetic_input((1, 1, h, w), seed=5)
    got, want = _pair_engines(spec, fp32, x)
    _check_pair(got, want, fp32)
    for r0, r1, c0, c1 in ((0, 16, 0, 70), (533, 545, 700, 800), (h - 16, h, w - 70, w)):
        a0, a1, b0, b1 = max(0, r0 - 9), min(h, r1 + 9), max(0, c0 - 9), min(w, c1 + 9)
        ref = run_model(spec.model, x[:, :, a0:a1, b0:b1])
        ref = ref[:, :, 2 * (r0 - a0):2 * (r1 - a0), 2 * (c0 - b0):2 * (c1 - b0)]
        _check_model(got[:, :, 2 * r0:2 * r1, 2 * c0:2 * c1], ref, f"pairs large {r0},{c0}")


def test_pairs_nonfinite():
    """An infinite pixel reaches the same outputs as through the convs alone, all
    within four pixels (four 3x3 convs), and nothing else changes."""
    spec = _pair_spec((None, None, None))
    x = models.synthetic_input((1, 1, 40, 131), seed=7)
    clean, _ = _pair_engines(spec, False, x)
    near = np.zeros((40, 131), bool)
    for y, xx in ((0, 0), (17, 30), (39, 130), (20, 62)):
        x[0, 0, y, xx] = np.inf
        near[max(0, y - 4):y + 5, max(0, xx - 4):xx + 5] = True
    near = near.repeat(2, 0).repeat(2, 1)
    got, want = _pair_engines(spec, False, x)
    np.testing.assert_array_equal(np.isfinite(got), np.isfinite(want))
    np.testing.assert_array_equal(got[0, 0][~near], clean[0, 0][~near])
    assert not np.isfinite(got[0, 0][near]).all()


@pytest.mark.parametrize("fp32", [False, True])
def test_pairs_poisoned(fp32):
    """With every activation filled with NaN before the run: nothing that the run
    did not write is read."""
    x = models.synthetic_input((1, 1, 37, 70), seed=2)
    got, want = _pair_engines(models.c4f32(seed=3), fp32, x, Engine.DEBUG_POISON)
    _check_pair(got, want, fp32)


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


def _run_offset(x, wt, b, act, skips, off):
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
    sk = [buf(to_padded(t)) for t in skips] + [None, None]
    out = buf(np.zeros((n, hp, wp, m), np.float16))
    ut, bt = torch.from_numpy(u.view(np.float16)).cuda(), torch.from_numpy(bias).cuda()
    ptr = lambda t: None if t is None else ctypes.c_void_p(t.data_ptr())
    rc = lib.arthip_conv3x3_f16_nhwc(ptr(xin), ptr(ut), ptr(bt), act, ptr(sk[0]), ptr(sk[1]), ptr(out), n, h, w, c, m,
                                     None)
    assert rc == 0, _lib.last_error()
    torch.cuda.synchronize()
    o = out.cpu().numpy().reshape(n, hp, wp, m)
    return o[:, 1:h + 1, 1:w + 1].astype(np.float32).transpose(0, 3, 1, 2)


@pytest.mark.parametrize("c,m,k", [(3, 64, 0), (48, 24, 1)])
def test_unaligned_buffers(c, m, k):
    """Buffers on 8 bytes only: accepted, by the general kernel."""
    x, wt, b = make_case(53, 1, c, m, 21, 67)
    sk = _skips(54, k, 1, m, 21, 67)
    got = _run_offset(x, wt, b, 1, sk, 8)
    check(got, oracle_conv(x, wt, b, 1, sk), f"offset c{c}m{m}")


# 32 -> 32 off 16 bytes runs winograd_strip: 16-tile strips, odd heights, ranges
# that cross strips, each epilogue.
@pytest.mark.parametrize("act,k,h,w", [(0, 0, 8, 31), (1, 1, 21, 67), (2, 2, 19, 35), (1, 0, 1, 1), (2, 1, 90, 333)])
def test_unaligned_buffers_c32(act, k, h, w):
    x, wt, b = make_case(55, 1, 32, 32, h, w)
    sk = _skips(56, k, 1, 32, h, w)
    got = _run_offset(x, wt, b, act, sk, 8)
    check(got, oracle_conv(x, wt, b, act, sk), f"offset c32 act{act} skip{k} {h}x{w}")
