"""The 256 x 256 tiles on the 16x16 MFMA shapes use every register of their waves in the K loop: whatever an epilogue keeps live
across the loop, and every address the compiler hoists in front of it, is spilled, and a reload inside the loop waits for the
stages in flight (bf16 8192 x 4096 x 1024 took 8 % longer).  Read off the assembly of two instantiations (hipcc, device pass
only, no GPU needed)."""
import os
import re
import subprocess
import tempfile

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "zluda_amd", "csrc")
HIPCC = "/opt/rocm/bin/hipcc"
pytestmark = pytest.mark.skipif(not os.path.exists(HIPCC), reason="needs hipcc")


def kernels(instances, *flags):
    """the instruction lines of the kernels instantiated in `instances`, in their order"""
    with tempfile.TemporaryDirectory() as tmp:
        src, out = os.path.join(tmp, "k.hip"), os.path.join(tmp, "k.s")
        with open(src, "w") as f:
            f.write('#include "mfma_launch.hpp"\nnamespace zluda_amd {\n%s\n}\n' % "\n".join("template __global__ void %s(MfmaParams);" % i for i in instances))
        cmd = [HIPCC, "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC", "-fvisibility=hidden", "-Xclang", "-target-feature", "-Xclang",
               "-packed-fp32-ops", *flags, "--cuda-device-only", "-S", "-I" + CSRC, src, "-o", out]
        res = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
        assert res.returncode == 0, res.stdout[-2000:]
        text = open(out).read()
    found = [[l.strip() for l in m.group(1).split("\n")]
             for m in re.finditer(r"^_ZN9zluda_amd\S*gemm_mfma_pipe16\S*:\s*;.*?\n(.*?)^\.Lfunc_end", text, re.S | re.M)]
    assert len(found) == len(instances)
    return found


def k_loop(lines, first=False):
    """the loop with the most MFMAs, or the first one that has any"""
    labels = {m.group(1): i for i, l in enumerate(lines) for m in [re.match(r"(\.LBB\d+_\d+):", l)] if m}
    loops = []
    for i, l in enumerate(lines):
        m = re.match(r"s_c?branch\S*\s+(\.LBB\d+_\d+)", l)
        if m and labels.get(m.group(1), i) < i:
            loops.append(lines[labels[m.group(1)]:i])
    if first:
        return next(b for b in loops if any(x.startswith("v_mfma") for x in b))
    return max(loops, key=lambda b: sum(x.startswith("v_mfma") for x in b))


def test_no_reload_in_the_loop_of_a_256x256_tile():
    kinds = ["KIND_I8", "KIND_BF16"]
    for kind, lines in zip(kinds, kernels(["gemm_mfma_pipe16_kernel<%s, 0, 0, 256, 256, 2, 4>" % k for k in kinds])):
        body = k_loop(lines)
        assert sum(x.startswith("v_mfma") for x in body) == 128, kind
        assert not [x for x in body if x.startswith("scratch_")], kind


# (bf16, A:N B:T and one operand K-contiguous; the flag is that of the units which hold these kernels)
@pytest.mark.parametrize("tile,stages,turn", [(64, 6, 6), (64, 3, 6), (128, 4, 4)])
def test_turns_of_a_deep_ring_address_nothing_at_run_time(tile, stages, turn):
    names = ["gemm_mfma_pipe16_kernel<KIND_BF16, 0, 0, %d, %d, 2, 2, %s, %d>" % (tile, tile, mc, stages) for mc in ("true, true", "true, false")]
    for lines in kernels(names, "-mllvm", "-amdgpu-mfma-vgpr-form=1"):
        body = k_loop(lines, first=True)
        mfmas = (tile // 32) ** 2 * 2
        assert sum(x.startswith("v_mfma") for x in body) == turn * mfmas
        assert sum(x.startswith("s_barrier") for x in body) == turn
        assert not [x for x in body if x.startswith("scratch_")]
        # beside the MFMAs: with a slot in a register and the masks of the last stages 13 to 29 vector instructions a stage
        assert len([x for x in body if x.startswith("v_") and not x.startswith("v_mfma")]) <= turn
        # the scalar ones: offsets, M0 and its wait states of each DMA instruction, the barrier (38 to 65 a stage before)
        loads = sum(x.startswith("buffer_load") for x in body)
        scalar = [x for x in body if x.startswith("s_") and not x.startswith(("s_waitcnt", "s_barrier"))]
        assert len(scalar) <= 3.5 * loads + 4 * turn


def test_epilogues_with_an_aux_matrix_have_kernels_of_their_own():
    plain, aux = kernels(["gemm_mfma_pipe16_kernel<KIND_BF16, 0, 0, 128, 128, 2, 2, true, true, 2%s>" % more for more in ("", ", true")],
                         "-mllvm", "-amdgpu-mfma-vgpr-form=1")
    # the gradient's aux matrix: dwordx4 loads that do not go to LDS, one for each pair of the 4 x 4 tiles of a wave
    to_registers = lambda lines: sum(x.startswith("buffer_load_dwordx4") and " lds" not in x for x in lines)
    assert to_registers(aux) == 8 and to_registers(plain) == 0
    # and one exponential per element and epilogue: GELU, its gradient
    assert sum(x.startswith("v_exp_f32") for x in aux) == 2 * 4 * 4 * 4


def test_aux_epilogues_store_whole_lines():
    # 256 x 256 tiles: D's and aux's stores run along a column's rows, 64 bytes further on with each (the gradient's first, then GELU's)
    lines = kernels(["gemm_mfma_pipe16_kernel<KIND_BF16, 0, 0, 256, 256, 2, 4, false, false, 2, true>"])[0]
    assert not [x for x in k_loop(lines) if x.startswith("scratch_")]
    offsets = {}   # window -> the scalar offsets of its stores
    for x in lines:
        m = re.match(r"buffer_store_dwordx4 v\[\d+:\d+\], v\d+, (s\[\d+:\d+\]), (\S+) offen", x)
        if m:
            offsets.setdefault(m.group(1), []).append(m.group(2))
    assert sorted(len(v) for v in offsets.values()) == [16, 16, 16]
    assert all(v[:2] == ["0", "64"] for v in offsets.values())
