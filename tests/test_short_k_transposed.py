"""16-bit operands with unit stride along their row index on 128 x 128 tiles: a short K is transposed in registers, a long one by
the LDS reads, which cost more in front of and behind the loop and less in it.  The plan's waves tell the forms apart (four and
two workgroups fit a CU, one with the deep ring of a grid that has no more); on the GPU both sides of the change-over run with ends of K and of the
rows inside pieces."""
import ctypes as C

import pytest

from oracle.cases import Case
from zluda_amd import abi as K

TR16 = K.ZLUDA_KERNEL_MFMA_TR16
BF = dict(a_type=K.CUDA_R_16BF, b_type=K.CUDA_R_16BF, d_type=K.CUDA_R_16BF, c_type=K.CUDA_R_16BF, compute_type=K.CUBLAS_COMPUTE_32F,
          scale_type=K.CUDA_R_32F)


def waves(api, m, n, k, ta=0, tb=1, variant=1, cus=256):
    p, plan = K.zluda_gemm_problem(), K.zluda_gemm_plan()
    for dst, rows, cols in ((p.a, k if ta else m, m if ta else k), (p.b, n if tb else k, k if tb else n), (p.c, m, n), (p.d, m, n)):
        dst.type, dst.order, dst.rows, dst.cols, dst.ld, dst.batch_count = K.CUDA_R_16BF, K.CUBLASLT_ORDER_COL, rows, cols, rows, 1
    p.op.compute_type, p.op.scale_type = K.CUBLAS_COMPUTE_32F, K.CUDA_R_32F
    p.op.transa, p.op.transb, p.op.epilogue, p.op.bias_type, p.op.epilogue_aux_type = ta, tb, K.CUBLASLT_EPILOGUE_DEFAULT, -1, -1
    assert api.zluda_gemm_plan_problem(C.byref(p), TR16, variant, cus, C.byref(plan)) == 0
    return plan.waves * cus / (plan.grid_x * plan.grid_y * plan.grid_z)   # 1 / workgroups on a CU


def test_the_form_follows_k_and_the_number_of_tiles(api):
    registers, lds, alone = 0.25, 0.5, 1.0
    for k, want in ((32, registers), (128, registers), (512, registers), (768, alone), (4096, alone)):
        assert waves(api, 2048, 2048, k) == want, k      # one tile on a CU
    for k, want in ((256, registers), (512, lds), (2048, lds)):
        assert waves(api, 8192, 1024, k) == want, k      # two
    for k, want in ((1024, registers), (1536, lds)):
        assert waves(api, 4096, 3072, k) == want, k      # three: a second round for the LDS form
    assert waves(api, 2048, 2048, 4096, cus=128) == lds and waves(api, 2048, 2048, 512, cus=128) == lds
    # pitches that are no multiples of 16 bytes keep the register form, the 256 x 256 tile always reads transposed
    assert waves(api, 2044, 2048, 4096) == registers
    assert waves(api, 2048, 2048, 32, variant=3) == 1.0


@pytest.mark.gpu
@pytest.mark.parametrize("ta,tb,ks", [(0, 0, (688, 696, 720, 776, 1032)), (0, 1, (639, 690, 705, 727, 833, 1001)), (1, 1, (688, 704, 712, 904))])
def test_both_forms(gpu_api, ta, tb, ks):
    up8 = lambda x: (x + 7) // 8 * 8
    for i, k in enumerate(ks):
        m, n = (260, 250) if i & 1 else (130, 393)
        spec = dict(BF, m=m, n=n, k=k, transa=ta, transb=tb, lda=up8(k if ta else m), ldb=up8(n if tb else k))
        if i == 2:
            spec.update(batch=3, epilogue=K.CUBLASLT_EPILOGUE_GELU_BIAS)
        print("case", spec, flush=True)
        case = Case(spec, 9500 + k)
        ref = case.run_oracle()
        st, got, kernel, variant = case.run_gpu(gpu_api, forced_kernel=TR16, forced_variant=1)
        assert st == 0 and (kernel, variant) == (TR16, 1)
        case.compare(got, ref, tol=1e-2)   # one rounding to 16 bits of sums in another order
