"""Operands that only their alignment, or a K-contiguous row that ends inside a 16-byte piece, keeps from every MFMA family:
reported as the generic family, run on the transposing MFMA kernel.  Odd pitches, odd K around the 32-element (16-bit) and
16-element (f32) stage, one element, ends inside a lane's piece, every layout, the smallest and the largest tile, a
split along K, batches at odd strides, C read."""
import pytest

from oracle.cases import Case
from zluda_amd import abi as K

pytestmark = pytest.mark.gpu
GEN = K.ZLUDA_KERNEL_GENERIC
LAYOUTS = [(1, 0), (0, 0), (0, 1), (1, 1)]


def spec_of(t, m, n, k, ta, tb, pad=1, **more):
    f = dict(a_type=t, b_type=t, d_type=t, compute_type=K.CUBLAS_COMPUTE_32F, scale_type=K.CUDA_R_32F, m=m, n=n, k=k, transa=ta, transb=tb)
    # an odd pitch wherever the operand's own extent does not give one already
    f["lda"] = ((k if ta else m) + pad) | 1
    f["ldb"] = ((n if tb else k) + pad) | 1
    return dict(f, **more)


def check(gpu_api, spec, seed, tol, ws=0, want_ws=False):
    print("case", spec, flush=True)
    case = Case(spec, seed)
    ref = case.run_oracle()
    st, got, kernel, _ = case.run_gpu(gpu_api, workspace_bytes=ws)
    assert st == 0 and kernel == GEN, (st, kernel)
    assert (case.last_workspace_needed > 0) == want_ws
    case.compare(got, ref, tol=tol)


@pytest.mark.parametrize("ta,tb", LAYOUTS)
@pytest.mark.parametrize("k", [1, 2, 31, 32, 33, 63, 64, 65, 127, 129, 161, 200])
def test_16_bit_odd_pitches(gpu_api, k, ta, tb):
    for i, (m, n) in enumerate([(1, 1), (63, 65), (130, 17)]):
        check(gpu_api, spec_of(K.CUDA_R_16BF if k & 1 else K.CUDA_R_16F, m, n, k, ta, tb), 7600 + i, None)


@pytest.mark.parametrize("ta,tb", [(1, 0), (0, 0), (1, 1)])
@pytest.mark.parametrize("k", [1, 15, 17, 31, 33, 49, 63, 101])
def test_f32_rows_that_end_inside_a_piece(gpu_api, k, ta, tb):
    for i, (m, n) in enumerate([(1, 1), (65, 33), (150, 90)]):
        check(gpu_api, spec_of(K.CUDA_R_32F, m, n, k, ta, tb, epilogue=K.CUBLASLT_EPILOGUE_BIAS), 7700 + i, 1e-3)


@pytest.mark.parametrize("k", [4, 12, 60, 68, 100, 132])
def test_int8_rows_that_end_inside_a_piece(gpu_api, k):
    spec = dict(a_type=K.CUDA_R_8I, b_type=K.CUDA_R_8I, d_type=K.CUDA_R_32I, compute_type=K.CUBLAS_COMPUTE_32I, scale_type=K.CUDA_R_32I,
                m=100, n=72, k=k, transa=1, transb=0)
    check(gpu_api, spec, 7800, None)
    check(gpu_api, dict(spec, transa=0, n=68, with_c=True, batch=2), 7801, None)


@pytest.mark.parametrize("ta,tb", LAYOUTS)
@pytest.mark.parametrize("t", [K.CUDA_R_16BF, K.CUDA_R_32F])
def test_larger_tiles_batches_and_c(gpu_api, t, ta, tb):
    tol = 1e-3 if t == K.CUDA_R_32F else None
    k = 71 if t == K.CUDA_R_16BF else 39
    if t == K.CUDA_R_32F and (ta, tb) == (0, 1):
        return   # (neither operand K-contiguous: the TR32 family itself)
    check(gpu_api, spec_of(t, 1030, 1030, k, ta, tb), 7900, tol)              # many 64 x 64 tiles
    check(gpu_api, spec_of(t, 3600, 3500, k, ta, tb), 7901, tol)              # 256 x 256 tiles
    m, n = 97, 61
    s = spec_of(t, m, n, k, ta, tb, batch=3, with_c=True)
    s["stride_a"] = s["lda"] * (m if ta else k) + 1
    s["stride_b"] = s["ldb"] * (k if tb else n) + 3
    check(gpu_api, s, 7902, tol)


@pytest.mark.parametrize("ta,tb", LAYOUTS)
def test_split_along_k(gpu_api, ta, tb):
    check(gpu_api, spec_of(K.CUDA_R_16BF, 150, 70, 4001, ta, tb), 8000, None, ws=16 << 20, want_ws=True)
