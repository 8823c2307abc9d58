"""The two forms of the 256 x 128 tile, eight waves with three stages and four with two: the same integers."""
import pytest

from oracle.cases import Case
from zluda_amd import abi as K

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [500, 2080])   # 64 tiles: eight waves; 544: four
def test_both_forms_of_the_256x128_tile(gpu_api, n):
    s = dict(a_type=K.CUDA_R_8I, b_type=K.CUDA_R_8I, d_type=K.CUDA_R_32I, compute_type=K.CUBLAS_COMPUTE_32I, scale_type=K.CUDA_R_32I, transa=1,
             m=8190, n=n, k=144)
    print("case", s, flush=True)
    case = Case(s, 6900)
    st, got, kernel, variant = case.run_gpu(gpu_api, forced_kernel=K.ZLUDA_KERNEL_MFMA_I8, forced_variant=2)
    assert st == 0 and variant == 2
    case.compare(got, case.run_oracle())
