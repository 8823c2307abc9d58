"""K-contiguous operands whose rows end inside a 16-byte piece, on the transposing MFMA kernel: what lies between the end of K and
the pitch -- here NaNs, or the largest int8 -- takes no part.  8-bit rows that end inside a dword, both fp8 formats, 16- and
32-bit rows; the 64 x 64, 128 x 128 and 256 x 256 tiles, asserted from the plan."""
import ctypes as C

import numpy as np
import pytest

from oracle.cases import Case
from zluda_amd import abi as K

pytestmark = pytest.mark.gpu
GEN = K.ZLUDA_KERNEL_GENERIC
NAN = {K.CUDA_R_8I: 0x7F, K.CUDA_R_8F_E4M3: 0x7F, K.CUDA_R_8F_E5M2: 0x7F, K.CUDA_R_16BF: 0x7FC0, K.CUDA_R_16F: 0x7E00, K.CUDA_R_32F: np.nan}
FLOAT = dict(compute_type=K.CUBLAS_COMPUTE_32F, scale_type=K.CUDA_R_32F)
PAIRS = {
    "int8": dict(a_type=K.CUDA_R_8I, b_type=K.CUDA_R_8I, d_type=K.CUDA_R_32I, compute_type=K.CUBLAS_COMPUTE_32I, scale_type=K.CUDA_R_32I),
    "e4m3": dict(FLOAT, a_type=K.CUDA_R_8F_E4M3, b_type=K.CUDA_R_8F_E4M3, d_type=K.CUDA_R_16BF),
    "e5m2_e4m3": dict(FLOAT, a_type=K.CUDA_R_8F_E5M2, b_type=K.CUDA_R_8F_E4M3, d_type=K.CUDA_R_16BF),
    "e4m3_e5m2": dict(FLOAT, a_type=K.CUDA_R_8F_E4M3, b_type=K.CUDA_R_8F_E5M2, d_type=K.CUDA_R_32F),
    "bf16": dict(FLOAT, a_type=K.CUDA_R_16BF, b_type=K.CUDA_R_16BF, d_type=K.CUDA_R_16BF),
    "f16": dict(FLOAT, a_type=K.CUDA_R_16F, b_type=K.CUDA_R_16F, d_type=K.CUDA_R_16F),
    "f32": dict(FLOAT, a_type=K.CUDA_R_32F, b_type=K.CUDA_R_32F, d_type=K.CUDA_R_32F),
}


def run(gpu_api, pair, m, n, k, pitch, want_variant, tol=None):
    spec = dict(PAIRS[pair], m=m, n=n, k=k, transa=1, transb=0, lda=pitch, ldb=pitch)
    print("case", spec, flush=True)
    case = Case(spec, 9700 + k)
    for data, rows, t in ((case.A, m, spec["a_type"]), (case.B, n, spec["b_type"])):
        data[:rows * pitch].reshape(rows, pitch)[:, k:] = NAN[t]
    ref = case.run_oracle()
    st, got, plan = case.run_gpu_plan(gpu_api, 0)
    assert st == 0 and (plan.kernel, plan.variant) == (GEN, want_variant), (st, plan.kernel, plan.variant)
    case.compare(got, ref, tol=tol)


@pytest.mark.parametrize("pair", ["int8", "e4m3", "e5m2_e4m3", "e4m3_e5m2"])
@pytest.mark.parametrize("k", [1, 5, 15, 63, 66, 131, 203])
def test_8_bit_rows(gpu_api, pair, k):
    run(gpu_api, pair, 70, 36, k, (k + 3) // 4 * 4 + 4, 3)


@pytest.mark.parametrize("pair,k", [(p, k) for p in ("bf16", "f16", "f32") for k in (1, 7, 15, 31, 33, 65, 101)])
def test_16_and_32_bit_rows(gpu_api, pair, k):
    run(gpu_api, pair, 70, 37, k, k + 3, 3, tol=1e-3 if pair == "f32" else None)


@pytest.mark.parametrize("pair,m,n,k,variant", [("bf16", 2047, 2047, 41, 2), ("bf16", 2047, 2045, 67, 2), ("f32", 2047, 2047, 19, 2), ("f32", 2045, 2047, 35, 2),
                                                ("int8", 2047, 2047, 70, 2), ("bf16", 3590, 3500, 37, 4), ("f32", 3590, 3500, 21, 1)])
def test_larger_tiles(gpu_api, pair, m, n, k, variant):
    run(gpu_api, pair, m, n, k, (k + 3) // 4 * 4 + (4 if pair == "int8" else 1), variant, tol=1e-3 if pair == "f32" else None)
