"""The MFMA epilogues drop the lanes past the end of D's unit-stride dimension by an offset that no store window reaches.
tests/host_c/store_window_check.cpp replays the offsets of wave tiles of matrices up to 64 GiB with the kernels' own arithmetic
(kernels/store_window.hpp); here it is built and run, and run again against a window of 4 GiB.  On the GPU: a D of a little
over 2 GiB whose rows no tile divides, on every kernel that stores from the accumulators."""
import ctypes as C
import os
import re
import shutil
import subprocess

import pytest

from zluda_amd import abi as K
from zluda_amd.cublaslt import MatmulCall

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
KERNELS = os.path.join(ROOT, "zluda_amd", "csrc", "kernels")
HEADER = "zluda_amd/csrc/kernels/store_window.hpp"
CHECK = "tests/host_c/store_window_check.cpp"
needs_gxx = pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")


def build_and_run(tree, exe):
    subprocess.run(["g++", "-O1", "-std=c++17", os.path.join(tree, CHECK), "-o", str(exe)], check=True)
    return subprocess.run([str(exe)], capture_output=True, text=True)


@needs_gxx
def test_windows_hold_what_exists_and_nothing_else(tmp_path):
    res = build_and_run(ROOT, tmp_path / "check")
    assert res.returncode == 0, res.stdout
    assert int(res.stdout.split()[0]) > 50000


@needs_gxx
def test_a_window_beyond_the_masked_offset_is_caught(tmp_path):
    for rel in (HEADER, CHECK):
        (tmp_path / rel).parent.mkdir(parents=True, exist_ok=True)
        shutil.copy(os.path.join(ROOT, rel), tmp_path / rel)
    text = (tmp_path / HEADER).read_text()
    old = "left > (int64_t)kWindowEnd ? kWindowEnd :"
    assert text.count(old) == 1
    (tmp_path / HEADER).write_text(text.replace(old, "left > 0xFFFFFFFFll ? 0xFFFFFFFFu :"))
    res = build_and_run(str(tmp_path), tmp_path / "check")
    assert res.returncode != 0 and "does not exist is stored" in res.stdout


def test_every_window_of_d_comes_from_the_checked_header():
    for name in sorted(os.listdir(KERNELS)):
        src = open(os.path.join(KERNELS, name)).read()
        if name != "store_window.hpp":
            assert "tile_window_bytes(int64_t" not in src and not re.search(r"kStoreNowhere\s*=", src), name
        # descriptors over D take their size from it (mfma_store_tile_raw writes whole tiles of scratch, nothing is dropped)
        src = src.replace("const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc((void *)Dw, 0, 0xFFFFFFFF, 0x00020000);", "", 1)
        for m in re.finditer(r"make_buffer_rsrc\(\(void \*\)Dw, 0, ([^,]*\([^)]*\)|[^,]*),", src):
            assert m.group(1).startswith("tile_window_bytes("), (name, m.group(0))


GIB2 = 1 << 31
CASES = [   # (operand type, D, family, variants)
    ("bf16", K.CUDA_R_16BF, K.ZLUDA_KERNEL_MFMA_H16, (0, 3, 6, 8, 9, 11), 1),
    ("bf16", K.CUDA_R_16BF, K.ZLUDA_KERNEL_MFMA_TR16, (1, 3), 0),
    ("bf16", K.CUDA_R_32F, K.ZLUDA_KERNEL_MFMA_H16, (2, 8, 11), 1),
    ("i8", K.CUDA_R_32I, K.ZLUDA_KERNEL_MFMA_I8, (5, 8, 11), 1),
]


@pytest.mark.gpu
@pytest.mark.parametrize("case", range(len(CASES)))
def test_a_ragged_d_of_more_than_2_gib(gpu_api, case):
    """Operands of -1, 0 and 1, K = 64: every sum is exact in every type of D.  The whole of D's storage is compared: elements,
    and the padding between the rows and the pitch, which keeps what was there."""
    import torch
    typ, d_type, family, variants, ta = CASES[case]
    k, esz = 64, 2 if d_type == K.CUDA_R_16BF else 4
    m = 32003 if esz == 4 else 50257
    ldd = (m + 15) // 16 * 16
    n = (GIB2 + (40 << 20)) // (ldd * esz)   # the last tile's columns in the first 40 MiB have more than 2 GiB behind them
    ints = typ == "i8"
    gen = torch.Generator(device="cuda:0")
    gen.manual_seed(k + case)
    op = torch.int8 if ints else torch.bfloat16
    a = torch.randint(-1, 2, (ldd if not ta else m, k) if ta else (k, ldd), device="cuda:0", generator=gen).to(op)
    b = torch.randint(-1, 2, (n, k), device="cuda:0", generator=gen).to(op)
    rows = (a if ta else a.t()[:m]).float().contiguous()
    t, dt = (K.CUDA_R_8I, torch.int32) if ints else (K.CUDA_R_16BF, torch.bfloat16 if esz == 2 else torch.float32)
    spec = dict(a_type=t, b_type=t, d_type=d_type, compute_type=K.CUBLAS_COMPUTE_32I if ints else K.CUBLAS_COMPUTE_32F,
                scale_type=K.CUDA_R_32I if ints else K.CUDA_R_32F, m=m, n=n, k=k, transa=ta, transb=0, lda=k if ta else ldd, ldd=ldd, ldc=ldd)
    scalar = C.c_int32 if ints else C.c_float
    d = torch.empty((n, ldd), dtype=dt, device="cuda:0")
    assert d.numel() * esz > GIB2
    for v in variants:
        print("case", spec, "family", family, "variant", v, flush=True)
        d.fill_(99)
        call = MatmulCall(gpu_api, spec, forced_kernel=family, forced_variant=v)
        try:
            st = call.run(scalar(1), a.data_ptr(), b.data_ptr(), scalar(0), None, d.data_ptr(), None, 0, torch.cuda.current_stream().cuda_stream)
        finally:
            call.close()
        assert st == 0
        torch.cuda.synchronize()
        for j in range(0, n, 1024):
            want = b[j:j + 1024].float() @ rows.t()
            assert bool((d[j:j + 1024, :m].float() == want).all()), (v, j)
        assert bool((d[:, m:] == 99).all()), v
