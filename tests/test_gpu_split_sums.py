"""The sums of 2 to 8 shares of K (one instantiation each): integers exactly, floats behind the whole epilogue, with extents that end
inside a thread's four elements and columns of D that are and are not aligned for one store of them."""
import pytest

from oracle.cases import Case
from zluda_amd import abi as K

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shares", range(2, 9))
def test_shares(gpu_api, shares):
    i8 = dict(a_type=K.CUDA_R_8I, b_type=K.CUDA_R_8I, d_type=K.CUDA_R_32I, compute_type=K.CUBLAS_COMPUTE_32I, scale_type=K.CUDA_R_32I, transa=1)
    per = 192 * 64 * 4
    for spec in (dict(i8, m=130, n=61, k=8192, alpha=3), dict(i8, m=129, n=33, k=8192, ldd=131, scale_type=K.CUDA_R_32F, d_type=K.CUDA_R_32F),
                 dict(i8, m=131, n=50, k=8192, ldd=132, scale_type=K.CUDA_R_32F, d_type=K.CUDA_R_16BF, epilogue=K.CUBLASLT_EPILOGUE_RELU_BIAS,
                      bias_type=K.CUDA_R_16BF, alpha_range=(0.001, 0.002))):
        print("case", spec, shares, flush=True)
        case = Case(spec, 8800 + shares)
        st, got, kernel, variant = case.run_gpu(gpu_api, forced_kernel=K.ZLUDA_KERNEL_MFMA_I8, forced_variant=6, workspace_bytes=shares * per)
        assert st == 0 and (kernel, variant) == (K.ZLUDA_KERNEL_MFMA_I8, 6)
        case.compare(got, case.run_oracle())
