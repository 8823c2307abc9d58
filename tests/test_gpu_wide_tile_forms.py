"""The two forms of the 256 x 128 tile, eight waves with three stages and four with two, and the rings of all tiles with a form of their own:
short and long K."""
import pytest

from oracle.cases import Case
from zluda_amd import abi as K

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,block", [(500, 512), (2080, 256)])   # 128 tiles: eight waves; 544: four
def test_both_forms_of_the_256x128_tile(gpu_api, n, block):
    s = dict(a_type=K.CUDA_R_8I, b_type=K.CUDA_R_8I, d_type=K.CUDA_R_32I, compute_type=K.CUBLAS_COMPUTE_32I, scale_type=K.CUDA_R_32I, transa=1,
             m=8190, n=n, k=144)
    print("case", s, flush=True)
    case = Case(s, 6900)
    st, got, plan = case.run_gpu_plan(gpu_api, K.ZLUDA_KERNEL_MFMA_I8, 2)
    assert st == 0 and (plan.variant, plan.block) == (2, block)
    case.compare(got, case.run_oracle())


FLOAT = dict(compute_type=K.CUBLAS_COMPUTE_32F, scale_type=K.CUDA_R_32F, transa=1)
KINDS = {  # operands and D, the family, elements of K in a stage, and their least multiple in a row
    "int8": (K.CUDA_R_8I, K.CUDA_R_32I, K.ZLUDA_KERNEL_MFMA_I8, 128, 16), "fp8": (K.CUDA_R_8F_E4M3, K.CUDA_R_16BF, K.ZLUDA_KERNEL_MFMA_F8, 128, 16),
    "bf16": (K.CUDA_R_16BF, K.CUDA_R_16BF, K.ZLUDA_KERNEL_MFMA_H16, 64, 8), "f16": (K.CUDA_R_16F, K.CUDA_R_32F, K.ZLUDA_KERNEL_MFMA_H16, 64, 8),
    "f32": (K.CUDA_R_32F, K.CUDA_R_32F, K.ZLUDA_KERNEL_MFMA_F32, 32, 4), "mxfp4": (K.CUDA_R_4F_E2M1, K.CUDA_R_16BF, K.ZLUDA_KERNEL_MFMA_MXF4, 256, 256)}


FORMS = [(kind, v, b) for kind in KINDS for v, b in ((2, 256), (2, 512), (4, 256), (5, 256), (6, 256), (10, 256))
         if (kind not in ("mxfp4", "f32") or v < 10) and (kind != "mxfp4" or b == 256)]


@pytest.mark.parametrize("kind,variant,block", FORMS)
def test_rings_that_turn_over(gpu_api, kind, variant, block):
    """one to eight stages of K, the last one whole and not: rings of two, three and six slots that are filled again, fragments fetched one
    sub-step and a whole stage ahead"""
    t, d, family, stage, least = KINDS[kind]
    for stages in (1, 2, 3, 4, 5, 8):
        for k in {stages * stage, stages * stage - least} - {0}:
            s = dict(FLOAT, a_type=t, b_type=t, d_type=d, c_type=d, m=300, n=200, k=k)
            if kind == "int8":
                s.update(compute_type=K.CUBLAS_COMPUTE_32I, scale_type=K.CUDA_R_32I)
            if kind == "mxfp4":
                s.update(a_scale_mode=K.CUBLASLT_MATMUL_MATRIX_SCALE_VEC32_UE8M0, b_scale_mode=K.CUBLASLT_MATMUL_MATRIX_SCALE_VEC32_UE8M0)
            print("case", s, variant, block, flush=True)
            case = Case(s, 6950 + k)

            def four_or_eight_waves(plan):
                plan.block = block
            st, got, plan = case.run_gpu_plan(gpu_api, family, variant, edit=four_or_eight_waves)
            assert st == 0 and plan.grid_z == 1
            case.compare(got, case.run_oracle(), tol=None if kind in ("int8", "fp8") else 1e-2)   # one rounding to 16 bits of sums in another order
