"""The epilogues that store straight from the accumulators, on tiles that hang over the end of D's unit-stride dimension (the
end inside a pair, a group of four and a group of eight elements, and between tiles) and on a D of odd pitch: every tile
variant of the kernels with the 32x32 and the 16x16 accumulator layout, every output type."""
import pytest

from oracle.cases import Case
from zluda_amd import abi as K

pytestmark = pytest.mark.gpu

BF = dict(a_type=K.CUDA_R_16BF, b_type=K.CUDA_R_16BF, compute_type=K.CUBLAS_COMPUTE_32F, scale_type=K.CUDA_R_32F, transa=1)
I8 = dict(a_type=K.CUDA_R_8I, b_type=K.CUDA_R_8I, compute_type=K.CUBLAS_COMPUTE_32I, transa=1)
TOKEN = dict(pointer_mode=K.CUBLASLT_POINTER_MODE_ALPHA_DEVICE_VECTOR_BETA_ZERO, b_scale_mode=K.CUBLASLT_MATMUL_MATRIX_SCALE_OUTER_VEC_32F,
             alpha_range=(0.001, 0.002), scale_range=(0.5, 1.5), bias_type=K.CUDA_R_16BF)
SPECS = [
    dict(BF, d_type=K.CUDA_R_16BF, epilogue=K.CUBLASLT_EPILOGUE_GELU_BIAS),
    dict(BF, d_type=K.CUDA_R_16F, epilogue=K.CUBLASLT_EPILOGUE_RELU_BIAS),
    dict(BF, d_type=K.CUDA_R_32F, epilogue=K.CUBLASLT_EPILOGUE_BIAS),
    dict(I8, d_type=K.CUDA_R_16BF, scale_type=K.CUDA_R_32F, epilogue=K.CUBLASLT_EPILOGUE_BIAS, **TOKEN),
    dict(I8, d_type=K.CUDA_R_32I, scale_type=K.CUDA_R_32I),
]
# (rows of D, its leading dimension): the last element, pair, four, eight of the last tile; odd pitches; an exact fit
ENDS = [(257, 264), (258, 259), (259, 267), (300, 304), (319, 321), (512, 513)]


@pytest.mark.parametrize("spec", range(len(SPECS)))
@pytest.mark.parametrize("m,ldd", ENDS)
def test_ragged_end_of_d(gpu_api, spec, m, ldd):
    base = dict(SPECS[spec], m=m, n=150, k=256, ldd=ldd, ldc=ldd)
    family = K.ZLUDA_KERNEL_MFMA_H16 if base["a_type"] == K.CUDA_R_16BF else K.ZLUDA_KERNEL_MFMA_I8
    print("case", base, flush=True)
    case = Case(base, 7300 + m)
    ref = case.run_oracle()
    for v in range(12):
        if v == 11:
            continue   # (the four-wave kernel: below, where D is aligned as it wants it)
        st, got, k, used = case.run_gpu(gpu_api, forced_kernel=family, forced_variant=v)
        assert st == 0 and (k, used) == (family, v)
        case.compare(got, ref)


@pytest.mark.parametrize("spec", range(len(SPECS)))
@pytest.mark.parametrize("m", [257, 258, 263, 300, 511])
def test_ragged_end_of_d_on_the_four_wave_kernel(gpu_api, spec, m):
    base = dict(SPECS[spec], m=m, n=270, k=512, ldd=(m + 15) // 16 * 16, ldc=(m + 15) // 16 * 16)
    family = K.ZLUDA_KERNEL_MFMA_H16 if base["a_type"] == K.CUDA_R_16BF else K.ZLUDA_KERNEL_MFMA_I8
    print("case", base, flush=True)
    case = Case(base, 7400 + m)
    ref = case.run_oracle()
    st, got, k, v = case.run_gpu(gpu_api, forced_kernel=family, forced_variant=11)
    assert st == 0 and (k, v) == (family, 11)
    case.compare(got, ref)


@pytest.mark.parametrize("d_type", [K.CUDA_R_16BF, K.CUDA_R_32F])
def test_row_major_d_with_a_bias_along_its_rows(gpu_api, d_type):
    """a row-major D: the bias and the per-row scales run along the other dimension"""
    base = dict(BF, d_type=d_type, m=150, n=301, k=256, order_c=1, order_d=1, ldd=303, ldc=303, epilogue=K.CUBLASLT_EPILOGUE_GELU_BIAS)
    print("case", base, flush=True)
    case = Case(base, 7500)
    ref = case.run_oracle()
    for v in range(11):
        st, got, k, used = case.run_gpu(gpu_api, forced_kernel=K.ZLUDA_KERNEL_MFMA_H16, forced_variant=v)
        assert st == 0 and used == v
        case.compare(got, ref)
