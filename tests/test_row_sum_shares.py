"""The shares of a bias gradient's sums follow the number of CUs a plan is made for: about four workgroups on each."""
import ctypes as C

import pytest

from zluda_amd import abi as K


@pytest.mark.parametrize("cus,shares", [(64, 4), (128, 8), (256, 16), (304, 19)])
def test_shares_follow_the_cus(api, cus, shares):
    m, n, k = 64, 4096, 8192   # 4096 sums of 8192 terms: 64 groups of 64 rows
    p, plan = K.zluda_gemm_problem(), K.zluda_gemm_plan()
    for dst, rows, cols in ((p.a, m, k), (p.b, n, k), (p.c, m, n), (p.d, m, n)):
        dst.type, dst.order, dst.rows, dst.cols, dst.ld, dst.batch_count = K.CUDA_R_16BF, K.CUBLASLT_ORDER_COL, rows, cols, rows, 1
    p.op.compute_type, p.op.scale_type, p.op.transb = K.CUBLAS_COMPUTE_32F, K.CUDA_R_32F, 1
    p.op.epilogue, p.op.bias_type, p.op.epilogue_aux_type = K.CUBLASLT_EPILOGUE_BGRADB, -1, -1
    p.workspace_size = 1 << 30
    # (the variant of the matmul that splits K least: its own scratch does not hide the sums')
    assert api.zluda_gemm_plan_problem(C.byref(p), K.ZLUDA_KERNEL_GENERIC, -1, cus, C.byref(plan)) == 0
    assert plan.workspace == shares * n * 4
