"""LDS ordering at every workgroup barrier, checked without a GPU.

Mirrors the reference's kernel memory-ordering gate (tests/correctness/
test_kernel.py): an `s_barrier` orders control flow but does not retire
outstanding LDS stores, so a wave could pass a barrier with its stores still in
flight and another wave read stale shared memory (the corruption the reference's
NOTES.md describes). Every barrier in the HIP sources (kernels.hip, block.hip)
goes through `lds_sync` (wino_dev.h), which emits `s_waitcnt lgkmcnt(0)` itself
instead of relying on the compiler's waitcnt pass. Checked two ways:
- in the source: `__syncthreads` appears only inside `lds_sync`;
- in the gfx950 assembly hipcc emits for each HIP source: in every kernel, walking
  back from each `s_barrier` inside its basic block, an `s_waitcnt lgkmcnt(0)`
  comes before any LDS instruction (the compiler may schedule ALU work between
  the drain and the barrier, which is harmless).
"""

from __future__ import annotations

import hashlib
import re
import shutil
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parents[1] / "arthip_amd" / "csrc"
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
HIP_SOURCES = sorted(p.name for p in CSRC.glob("*.hip"))
DEVICE_SOURCES = HIP_SOURCES + ["wino_dev.h"]


def _strip_comments(text: str) -> str:
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return re.sub(r"//[^\n]*", "", text)


def test_barriers_only_through_lds_sync():
    assert "kernels.hip" in HIP_SOURCES and "block.hip" in HIP_SOURCES
    found = 0
    for name in DEVICE_SOURCES:
        src = _strip_comments((CSRC / name).read_text())
        m = re.search(r"void lds_sync\(\)\s*\{(.*?)\n\}", src, flags=re.S)
        if m:
            found += 1
            body = m.group(1)
            assert "lgkmcnt(0)" in body and "__syncthreads" in body
            src = src[:m.start()] + src[m.end():]
        assert "__syncthreads" not in src, f"{name}: a barrier outside lds_sync"
        assert "s_barrier" not in src, f"{name}: a raw s_barrier outside lds_sync"
    assert found == 1, f"lds_sync defined {found} times"


@pytest.fixture(scope="session")
def kernel_asm(tmp_path_factory) -> str:
    """The gfx950 assembly of every HIP source, concatenated."""
    if not Path(HIPCC).exists():
        pytest.skip("hipcc not available")
    tmp = tmp_path_factory.mktemp("asm")
    text = []
    for name in HIP_SOURCES:
        src = CSRC / name
        digest = hashlib.sha1(src.read_bytes()).hexdigest()[:12]
        out = tmp / f"{src.stem}_{digest}.s"
        cmd = [HIPCC, "--offload-arch=gfx950", "-O3", "-std=c++17", "-Xclang", "-target-feature",
               "-Xclang", "-packed-fp32-ops", "--cuda-device-only", "-S", "-o", str(out),
               str(src)]
        subprocess.run(cmd, check=True, cwd=CSRC, capture_output=True)
        text.append(out.read_text())
    return "\n".join(text)


def _kernels(asm: str):
    """(symbol, instruction list) for every kernel in the assembly."""
    lines = asm.splitlines()
    i = 0
    while i < len(lines):
        m = re.match(r"^(_Z\S+):\s*(;.*)?$", lines[i])
        if m and ".amdhsa" not in lines[i]:
            name = m.group(1)
            body = []
            i += 1
            while i < len(lines) and not lines[i].startswith(".Lfunc_end"):
                t = lines[i].split(";", 1)[0].strip()
                if t.endswith(":"):
                    body.append(":label")  # a basic block starts: other paths join here
                elif t and not t.startswith("."):
                    body.append(t)
                i += 1
            yield name, body
        i += 1


def _drained(ins, k) -> bool:
    """Walking back from instruction k in its basic block: a drain before any
    LDS instruction (ds_*) or the block's start."""
    for t in reversed(ins[:k]):
        if t.startswith("s_waitcnt") and "lgkmcnt(0)" in t:
            return True
        if t.startswith("ds_") or t == ":label":
            return False
    return False


def test_every_barrier_is_preceded_by_an_lds_drain(kernel_asm):
    checked = 0
    for name, ins in _kernels(kernel_asm):
        for k, t in enumerate(ins):
            if t.startswith("s_barrier"):
                assert _drained(ins, k), (
                    f"{name}: barrier at instruction {k} is reached with LDS work not drained: "
                    f"{ins[max(0, k - 8):k]}")
                checked += 1
    assert checked > 100, f"only {checked} barriers found; the assembly parse looks wrong"


def test_drain_check_catches_a_missing_drain():
    """The checker itself: a store, then a barrier, fails; a drain in between,
    or only ALU work after the drain, passes."""
    assert not _drained(["ds_write_b128 v1, v[2:5]", "s_barrier"], 1)
    assert _drained(["ds_write_b128 v1, v[2:5]", "s_waitcnt lgkmcnt(0)", "v_add_u32 v1, v2, v3",
                     "s_barrier"], 3)
    assert not _drained([":label", "v_add_u32 v1, v2, v3", "s_barrier"], 2)


def _regs(operand):
    m = re.fullmatch(r"([va])(?:\[(\d+):(\d+)\]|(\d+))", operand.strip())
    if not m:
        return set()
    lo = int(m.group(2) or m.group(4))
    return {(m.group(1), r) for r in range(lo, int(m.group(3) or lo) + 1)}


def _mixed_accumulators(ins):
    """Matrix products that accumulate onto the result of one of another shape in
    their basic block."""
    shape = {}  # register -> shape of the product that wrote it last
    bad = []
    for t in ins:
        if t == ":label":
            shape.clear()
            continue
        op, _, rest = t.partition(" ")
        args = [a for a in re.split(r",\s*(?![^\[]*\])", rest.strip())]
        mfma = re.match(r"v_mfma_\w+?_(\d+x\d+x\d+)", op)
        if mfma and any(shape.get(r, mfma.group(1)) != mfma.group(1) for r in _regs(args[3].split()[0])):
            bad.append(t)
        for r in _regs(args[0].split()[0] if args[0] else ""):
            if mfma:
                shape[r] = mfma.group(1)
            elif not op.startswith(("ds_write", "global_store", "buffer_store")):
                shape.pop(r, None)
    return bad


def test_no_product_accumulates_onto_another_shape(kernel_asm):
    """hipcc issues v_mfma_f32_16x16x16_f16 right behind the v_mfma_f32_16x16x32_f16
    whose result it adds to, with no wait states, as it does for products of one
    shape; on the GPU the first two registers of the sum were wrong then. No kernel
    may hold such a pair."""
    products = 0
    for name, ins in _kernels(kernel_asm):
        products += sum(t.startswith("v_mfma") for t in ins)
        assert not _mixed_accumulators(ins), (name, _mixed_accumulators(ins)[:3])
    assert products > 1000
    first = "v_mfma_f32_16x16x32_f16 v[0:3], v[2:5], v[10:13], v[6:9]"
    assert _mixed_accumulators([first, "v_mfma_f32_16x16x16_f16 v[0:3], v[14:15], v[4:5], v[0:3]"])
    assert not _mixed_accumulators([first, "v_mfma_f32_16x16x32_f16 v[0:3], v[2:5], v[4:7], v[0:3]"])
    assert not _mixed_accumulators([first, "v_add_f32_e32 v0, v0, v8", "v_add_f32_e32 v1, v1, v8", "v_mov_b32_e32 v2, 0",
                                    "v_mov_b32_e32 v3, 0", "v_mfma_f32_16x16x16_f16 v[0:3], v[4:5], v[4:5], v[0:3]"])
