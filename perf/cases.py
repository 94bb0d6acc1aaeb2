"""The work that a program using this engine has it do, as timed and checked cases.

Whole calls: frames already in HBM through ``Engine.run_device``, a small picture
through ``Engine.run`` (host memory to host memory) and video frames through the
VapourSynth filter core (host planes in and out). Single layers: the kernel-level
entry points on the padded NHWC buffers that they document, and a one-conv model
with the engine's NCHW boundary on both sides.

Weights are the package's own synthetic He-normal models and layers; frames are
smooth pictures in [0, 1] with grain, activations are N(0, 0.5) like the body of
such a network. A pass runs on one launch stream kept by the program.
"""

import ctypes
import math

import numpy as np
import torch

from arthip_amd import _lib, models, vs
from arthip_amd.engine import Engine

ACTS = {"none": 0, "relu": 1, "silu": 2}
MODELS = {"c4f32": models.c4f32, "r8f64": models.r8f64, "r16f96": models.r16f96,
          "shipped_like": models.shipped_like, "single64": models.single64}
MODEL_SEED = 7


def _spec(model):
    """The model as a program loads it. The shipped architecture's last two convs are
    scaled so that most pixels lie inside its output Clip [0, 1], as a trained
    network's do (He-normal ones put nearly every pixel outside it)."""
    spec = MODELS[model](seed=MODEL_SEED)
    if model == "shipped_like":
        init = {t.name: t for t in spec.model.graph.initializers}
        last = len(spec.convs) - 1
        for i, scale in ((last - 1, 1 / 64), (last, 1 / 8)):
            w, b = init[f"w{i}"].to_numpy(), init[f"b{i}"].to_numpy()
            b = b * np.float16(scale) if i < last else np.full_like(b, 0.5)
            for name, value in ((f"w{i}", w * np.float16(scale)), (f"b{i}", b)):
                init[name].raw_data = np.ascontiguousarray(value, np.float16).tobytes()
    return spec


def listed():
    return [
        # One small picture, host to host: a patch or thumbnail, where latency and
        # launches count (the size of the repository's smoke run).
        {"name": "host_r8f64_64x96", "kind": "host", "model": "r8f64", "n": 1, "h": 64, "w": 96},
        # The flagship frame: 1080p luma to 4K, resident in HBM.
        {"name": "frame_r8f64_1080p", "kind": "frame", "model": "r8f64", "n": 1, "h": 1080, "w": 1920},
        # The largest configuration: two 4K frames in one call.
        {"name": "frame_r8f64_4k_x2", "kind": "frame", "model": "r8f64", "n": 2, "h": 2160, "w": 3840},
        # Standard-definition video with an odd width, the shipped architecture
        # (SiLU, three convs per block, a conv with a residual input, Clip).
        {"name": "frame_shipped_480x853", "kind": "frame", "model": "shipped_like", "n": 1, "h": 480, "w": 853},
        # The small real-time model on quarter-HD frames: head, two 32-channel
        # layers and tail, all bound by memory.
        {"name": "frame_c4f32_540x960", "kind": "frame", "model": "c4f32", "n": 1, "h": 540, "w": 960},
        # A 64-channel layer alone with NCHW tensors on both sides, as an
        # execution provider gets it when it is handed one conv.
        {"name": "layer_single64_1080p", "kind": "frame", "model": "single64", "n": 1, "h": 1080, "w": 1920},
        # The head of a three-channel (RGB or 4:4:4) model.
        {"name": "conv_3_64_720p", "kind": "conv", "c": 3, "m": 64, "act": "none", "skips": 0, "n": 1, "h": 720, "w": 1280},
        # A body layer of a width without kernels of its own, at an odd size.
        {"name": "conv_48_48_relu_541x963", "kind": "conv", "c": 48, "m": 48, "act": "relu", "skips": 0, "n": 1, "h": 541, "w": 963},
        # A residual layer that cannot be fused with the one before it.
        {"name": "conv_64_64_skip_720p", "kind": "conv", "c": 64, "m": 64, "act": "none", "skips": 1, "n": 1, "h": 720, "w": 1280},
        # The wide model's residual layer (half of that model's work).
        {"name": "conv_96_96_skip_1080p", "kind": "conv", "c": 96, "m": 96, "act": "none", "skips": 1, "n": 1, "h": 1080, "w": 1920},
        # A residual block with SiLU at a PAL frame cropped by one row and column.
        {"name": "block_64_silu_575x719", "kind": "block", "act": "silu", "skips": 1, "n": 1, "h": 575, "w": 719},
        # A video frame through the filter: 8-bit plane in, fp16 plane out.
        {"name": "clip_shipped_gray8_720p", "kind": "clip", "model": "shipped_like", "format": "GRAY8", "n": 1, "h": 720, "w": 1280},
    ]


def _size(rng, lo, hi):
    """A size spread over the logarithm of its range, odd as often as even."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["host", "frame", "frame", "conv", "conv", "block", "clip"])
    if kind == "host":
        return {"kind": "host", "model": rng.choice(["c4f32", "r8f64", "shipped_like"]), "n": rng.choice([1, 1, 2]),
                "h": _size(rng, 16, 270), "w": _size(rng, 16, 480)}
    if kind == "frame":
        model = rng.choice(["c4f32", "r8f64", "r16f96", "shipped_like", "single64"])
        return {"kind": "frame", "model": model, "n": rng.choice([1, 1, 2]),
                "h": _size(rng, 64, 1080), "w": _size(rng, 64, 1920)}
    if kind == "conv":
        c, m = rng.choice([(1, 64), (3, 64), (4, 64), (16, 16), (24, 24), (32, 32), (48, 24), (48, 48),
                           (64, 64), (96, 96)])
        skips = 0 if c == 1 or c != m else rng.choice([0, 1, 1, 2])
        return {"kind": "conv", "c": c, "m": m, "act": rng.choice(["none", "relu", "silu"]), "skips": skips,
                "n": rng.choice([1, 1, 2]), "h": _size(rng, 16, 1080), "w": _size(rng, 16, 1920)}
    if kind == "block":
        return {"kind": "block", "act": rng.choice(["none", "relu", "silu"]), "skips": rng.choice([0, 1, 2]),
                "n": rng.choice([1, 1, 2]), "h": _size(rng, 16, 1080), "w": _size(rng, 16, 1920)}
    return {"kind": "clip", "model": rng.choice(["c4f32", "r8f64", "shipped_like"]), "format": rng.choice(["GRAY8", "GRAY16", "GRAYH"]),
            "n": 1, "h": _size(rng, 64, 1080), "w": _size(rng, 64, 1920)}


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------

_stream = None


def launch_stream():
    """The program's one launch stream (Engine.run_device takes the legacy default
    stream for "none given", so a program that orders its frames keeps one)."""
    global _stream
    if _stream is None:
        _stream = torch.cuda.Stream()
    return _stream


def _generator(seed, salt):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) * 1000003 + salt)
    return g


def _picture(case, seed, channels=1):
    """Smooth frames in [0, 1] with grain, [n][channels][h][w] fp32."""
    g = _generator(seed, 1)
    n, h, w = case["n"], case["h"], case["w"]
    low = torch.rand((n, channels, h // 12 + 2, w // 12 + 2), generator=g, device="cuda")
    x = torch.nn.functional.interpolate(low, size=(h, w), mode="bilinear", align_corners=False)
    x += 0.03 * torch.randn((n, channels, h, w), generator=g, device="cuda")
    return x.clamp_(0.0, 1.0)


def _activations(case, seed, channels, salt):
    """N(0, 0.5) activations in the padded NHWC layout, zero border."""
    n, h, w = case["n"], case["h"], case["w"]
    hp, wp = 2 * ((h + 1) // 2) + 2, 2 * ((w + 1) // 2) + 2
    x = torch.zeros((n, hp, wp, channels), dtype=torch.float16, device="cuda")
    x[:, 1:h + 1, 1:w + 1] = (0.5 * torch.randn((n, h, w, channels), generator=_generator(seed, salt), device="cuda")).half()
    return x


def _layer_weights(case, salt, c, m):
    """One layer's fp16 weights (OIHW) and bias: part of the program, like a model's."""
    rng = np.random.default_rng(MODEL_SEED * 100 + salt)
    return models.he_normal(rng, m, c), rng.uniform(-0.1, 0.1, m).astype(np.float16)


def _packed(weights, bias):
    """The layer's packed filters and bias on the GPU, laid out once."""
    lib = _lib.lib()
    m, c = weights.shape[:2]
    u = np.zeros(lib.arthip_conv3x3_packed_halfs(m, c), np.uint16)
    b = np.zeros(lib.arthip_conv3x3_bias_len(m), np.float32)
    u16, f32 = ctypes.POINTER(ctypes.c_uint16), ctypes.POINTER(ctypes.c_float)
    w16, b16 = np.ascontiguousarray(weights).view(np.uint16), np.ascontiguousarray(bias).view(np.uint16)
    rc = lib.arthip_conv3x3_pack(w16.ctypes.data_as(u16), b16.ctypes.data_as(u16), m, c, u.ctypes.data_as(u16), u.size,
                                 b.ctypes.data_as(f32), b.size)
    if rc != 0:
        raise RuntimeError(_lib.last_error())
    return torch.from_numpy(u.view(np.float16)).cuda(), torch.from_numpy(b).cuda()


def _layer_inputs(case, seed):
    if case["kind"] == "block":
        c = m = 64
        layers = [_layer_weights(case, 1, 64, 64), _layer_weights(case, 2, 64, 64)]
    else:
        c, m = case["c"], case["m"]
        layers = [_layer_weights(case, 1, c, m)]
    x = _activations(case, seed, c, 2)
    skips = [_activations(case, seed, m, 3 + k) for k in range(case["skips"])]
    return x, skips, layers


def _plane(case, seed):
    """One frame's luma plane in the clip's sample format (host memory)."""
    x = _picture(case, seed)[0, 0]
    if case["format"] == "GRAY8":
        return (x * 255).round().to(torch.uint8).cpu().numpy()
    if case["format"] == "GRAY16":
        return (x * 65535).round().to(torch.int32).cpu().numpy().astype(np.uint16)
    return x.half().cpu().numpy()


def _frame_input(case, seed):
    if case["model"] == "single64":
        n, h, w = case["n"], case["h"], case["w"]
        return (0.5 * torch.randn((n, 64, h, w), generator=_generator(seed, 1), device="cuda")).half()
    return _picture(case, seed).half()


# ---------------------------------------------------------------------------
# What a program has in hand, and one pass
# ---------------------------------------------------------------------------

def prepare(case, seed):
    kind = case["kind"]
    state = {"case": case}
    if kind in ("conv", "block"):
        x, skips, layers = _layer_inputs(case, seed)
        state.update(x=x, skips=skips, layers=[_packed(*layer) for layer in layers])
        state["out"] = torch.zeros(x.shape[:3] + (64 if kind == "block" else case["m"],), dtype=torch.float16, device="cuda")
        launch_stream()
    elif kind == "clip":
        state["plane"] = _plane(case, seed)
        state["filter"] = vs.Model(case["format"], case["w"], case["h"], _spec(case["model"]).bytes())
    else:
        state["engine"] = Engine(0).build(_spec(case["model"]))
        x = _frame_input(case, seed)
        if kind == "host":
            state["x"] = x.cpu().numpy()
        else:
            state["x"] = x
            state["out"] = torch.empty(state["engine"].output_shape(x.shape), dtype=torch.float16, device="cuda")
            launch_stream()
    torch.cuda.synchronize()
    return state


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "host":
        return state["engine"].run(state["x"])
    if kind == "clip":
        return state["filter"].get_frame([state["plane"]])
    stream = launch_stream().cuda_stream
    if kind == "frame":
        state["engine"].run_device(state["x"], state["out"], stream=stream)
        return state["out"]

    def ptr(t):
        return ctypes.c_void_p(t.data_ptr())

    lib = _lib.lib()
    skips = [ptr(t) for t in state["skips"]] + [None, None]
    n, h, w = case["n"], case["h"], case["w"]
    if kind == "conv":
        u, b = state["layers"][0]
        rc = lib.arthip_conv3x3_f16_nhwc(ptr(state["x"]), ptr(u), ptr(b), ACTS[case["act"]], skips[0], skips[1], ptr(state["out"]),
                                         n, h, w, case["c"], case["m"], ctypes.c_void_p(stream))
    else:
        (u1, b1), (u2, b2) = state["layers"]
        rc = lib.arthip_conv3x3_block_f16_nhwc(ptr(state["x"]), ptr(u1), ptr(b1), ACTS[case["act"]], ptr(u2), ptr(b2), skips[0], skips[1],
                                               ptr(state["out"]), n, h, w, 64, ctypes.c_void_p(stream))
    if rc != 0:
        raise RuntimeError(_lib.last_error())
    return state["out"]


# ---------------------------------------------------------------------------
# What a pass cannot do without, how close results have to be
# ---------------------------------------------------------------------------

def _convs(case):
    if case["kind"] == "conv":
        return [(case["c"], case["m"])]
    if case["kind"] == "block":
        return [(64, 64), (64, 64)]
    return _spec(case["model"]).convs


def work(case):
    """Inputs, weights and outputs once, in the types that the caller hands over;
    2 * 9 * C * M per pixel and conv (the sum that a 3x3 conv is; a fast algorithm
    multiplies less)."""
    pixels = case["n"] * case["h"] * case["w"]
    convs = _convs(case)
    flops = sum(18.0 * c * m for c, m in convs) * pixels
    weights = sum(18.0 * c * m + 4 * m for c, m in convs)
    if case["kind"] in ("conv", "block"):
        values = convs[0][0] + convs[-1][1] * (1 + case["skips"])
    else:  # a 64-channel layer, or one luma value in and four out
        values = 128 if case["model"] == "single64" else 5
    nbytes = 2.0 * values * pixels + weights
    if case.get("format") == "GRAY8":
        nbytes -= pixels
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    """About four times the distance to 64-bit results that the engine shows: fp16
    tensors between layers, fp16 transformed filters and inputs, fp32 sums."""
    kind = case["kind"]
    if kind in ("conv", "block"):
        return {"rel": 2.5e-3, "max": 2.5e-2}
    return {"single64": {"rel": 1.7e-3, "max": 1.3e-2}, "c4f32": {"rel": 3.3e-3, "max": 2.4e-2},
            "r8f64": {"rel": 6.5e-3, "max": 5e-2}, "shipped_like": {"rel": 4e-3, "max": 3e-2},
            "r16f96": {"rel": 1e-2, "max": 8e-2}}[case["model"]]


# ---------------------------------------------------------------------------
# 64-bit results
# ---------------------------------------------------------------------------

def _conv64(x, w, b):
    """3x3 SAME conv in fp64: x [n][h][w][c], w OIHW fp16 values."""
    n, h, wd, c = x.shape
    p = torch.nn.functional.pad(x, (0, 0, 1, 1, 1, 1))
    w = torch.from_numpy(w.astype(np.float64)).cuda()
    y = torch.zeros((n * h * wd, w.shape[0]), dtype=torch.float64, device="cuda")
    y += torch.from_numpy(b.astype(np.float64)).cuda()
    for dy in range(3):
        for dx in range(3):
            y += p[:, dy:dy + h, dx:dx + wd].reshape(-1, c) @ w[:, :, dy, dx].t().contiguous()
    return y.view(n, h, wd, -1)


def _act64(y, act):
    return y.clamp(min=0) if act == "relu" else y * torch.sigmoid(y) if act == "silu" else y


def _graph64(spec, x):
    """The model's graph on x (NCHW, fp64), channels last inside."""
    graph = spec.model.graph
    const = {t.name: t.to_numpy() for t in graph.initializers}
    last = {}
    for i, node in enumerate(graph.nodes):
        for name in node.inputs:
            last[name] = i
    value = {"x": x.permute(0, 2, 3, 1).contiguous()}
    for i, node in enumerate(graph.nodes):
        a = value[node.inputs[0]]
        op = node.op_type
        if op == "Conv":
            y = _conv64(a, const[node.inputs[1]], const[node.inputs[2]])
        elif op == "Relu":
            y = a.clamp(min=0)
        elif op == "Sigmoid":
            y = torch.sigmoid(a)
        elif op == "Add":
            y = a + value[node.inputs[1]]
        elif op == "Mul":
            y = a * value[node.inputs[1]]
        elif op == "Clip":
            y = a.clamp(float(const[node.inputs[1]]), float(const[node.inputs[2]]))
        elif op == "DepthToSpace":  # block 2, depth-column-row order
            n, h, w, k = a.shape
            y = a.view(n, h, w, 2, 2, k // 4).permute(0, 1, 3, 2, 4, 5).reshape(n, 2 * h, 2 * w, k // 4)
        else:
            raise ValueError(op)
        value[node.outputs[0]] = y
        for name in node.inputs:
            if last.get(name) == i:
                value.pop(name, None)
    return value[graph.outputs[0].name].permute(0, 3, 1, 2).contiguous()


def exact(case, seed):
    kind = case["kind"]
    if kind in ("conv", "block"):
        x, skips, layers = _layer_inputs(case, seed)
        h, w = case["h"], case["w"]

        def inner(t):
            return t[:, 1:h + 1, 1:w + 1].double()

        y = inner(x)
        if kind == "block":
            y = _conv64(_act64(_conv64(y, *layers[0]), case["act"]), *layers[1])
        else:
            y = _act64(_conv64(y, *layers[0]), case["act"])
        for s in skips:
            y = y + inner(s)
        out = torch.zeros(x.shape[:3] + (y.shape[3],), dtype=torch.float64, device="cuda")
        out[:, 1:h + 1, 1:w + 1] = y
        return out
    spec = _spec(case["model"])
    if kind == "clip":
        p = _plane(case, seed)
        scale = {"GRAY8": 255.0, "GRAY16": 65535.0}.get(case["format"], 1.0)
        x = torch.from_numpy(p.astype(np.float64) / scale).cuda()[None, None]
        return [_graph64(spec, x)[0, 0].cpu().numpy()]
    y = _graph64(spec, _frame_input(case, seed).double())
    return y.cpu().numpy() if kind == "host" else y
