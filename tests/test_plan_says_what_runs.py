"""A plan of the generic family names the kernel that the launch will run: variant 0 the scalar kernel with its grid, variant 1 + v
the transposing kernel's variant v with the grid, the shares of K and the waves that it has.  The token an application keeps
holds no variant: the family chooses for each call from the pointers it is given."""
import ctypes as C

import pytest

from oracle.cases import Case
from zluda_amd import abi as K
from zluda_amd.cublaslt import MatmulCall

GEN = K.ZLUDA_KERNEL_GENERIC
TILE = {1: 256, 2: 128, 3: 64, 4: 256}   # plan.variant -> rows of the square tile


def problem(t, m, n, k, ta, tb, lda, ldb, workspace=0):
    p = K.zluda_gemm_problem()
    for dst, rows, cols, ld in ((p.a, k if ta else m, m if ta else k, lda), (p.b, n if tb else k, k if tb else n, ldb), (p.c, m, n, m), (p.d, m, n, m)):
        dst.type, dst.order, dst.rows, dst.cols, dst.ld, dst.batch_count = t, K.CUBLASLT_ORDER_COL, rows, cols, ld, 1
    p.op.compute_type, p.op.scale_type = K.CUBLAS_COMPUTE_32F, K.CUDA_R_32F
    p.op.transa, p.op.transb, p.op.epilogue, p.op.bias_type, p.op.epilogue_aux_type = ta, tb, K.CUBLASLT_EPILOGUE_DEFAULT, -1, -1
    p.workspace_size = workspace
    return p


def plan_of(api, *args, forced=0, **more):
    plan = K.zluda_gemm_plan()
    p = problem(*args, **more)
    assert api.zluda_gemm_plan_problem(C.byref(p), forced, -1, 256, C.byref(plan)) == 0
    return plan


@pytest.mark.parametrize("m,n,k,variant", [(100, 100, 101, 3), (2047, 2047, 65, 2), (3600, 3500, 71, 1)])
@pytest.mark.parametrize("t", [K.CUDA_R_16BF, K.CUDA_R_32F])
def test_odd_pitches(api, t, m, n, k, variant):
    if variant == 1 and t == K.CUDA_R_16BF:
        variant = 4   # the same tile on the 16x16 MFMA shape, which f32 does not have
    plan = plan_of(api, t, m, n, k, 1, 0, k | 1, (k | 1) + 2)
    tile = TILE[variant]
    assert (plan.kernel, plan.variant) == (GEN, variant)
    assert plan.grid_x == -(-m // tile) * -(-n // tile) and plan.grid_y == plan.grid_z == 1
    assert plan.block == (512 if tile == 256 else 256) and plan.workspace == 0


def test_shares_of_k_and_the_scalar_kernel(api):
    plan = plan_of(api, K.CUDA_R_16BF, 150, 70, 4001, 1, 0, 4001, 4001, workspace=16 << 20)
    assert (plan.kernel, plan.variant) == (GEN, 3)
    assert plan.grid_z > 1 and plan.workspace == plan.grid_z * 192 * 128 * 4
    # what another family takes, forced here; and what none takes
    for forced, args in ((GEN, (K.CUDA_R_16BF, 512, 256, 1024, 1, 0, 1024, 1024)), (0, (K.CUDA_R_8F_E5M2, 512, 256, 1024, 1, 0, 1024, 1024))):
        t = args[0]
        p = problem(*args)
        if t == K.CUDA_R_8F_E5M2:
            p.c.type = p.d.type = K.CUDA_R_16BF
        plan = K.zluda_gemm_plan()
        assert api.zluda_gemm_plan_problem(C.byref(p), forced, -1, 256, C.byref(plan)) == 0
        assert (plan.kernel, plan.variant, plan.grid_x, plan.grid_y, plan.grid_z, plan.block) == (GEN, 0, 8, 4, 1, 256)


def test_the_token_holds_no_variant(api):
    spec = dict(a_type=K.CUDA_R_16BF, b_type=K.CUDA_R_16BF, d_type=K.CUDA_R_16BF, compute_type=K.CUBLAS_COMPUTE_32F, scale_type=K.CUDA_R_32F,
                m=100, n=100, k=101, transa=1, lda=101, ldb=103)
    call = MatmulCall(api, spec)
    assert (call.kernel, call.variant) == (GEN, 0)
    call.close()


@pytest.mark.gpu
def test_a_plan_that_meets_pointers_it_does_not_take(gpu_api):
    """planned from the layouts alone (1 + the 64 x 64 tile), launched on f32 operands two bytes off a dword: the scalar kernel"""
    import torch
    spec = dict(a_type=K.CUDA_R_32F, b_type=K.CUDA_R_32F, d_type=K.CUDA_R_32F, c_type=K.CUDA_R_32F, compute_type=K.CUBLAS_COMPUTE_32F,
                scale_type=K.CUDA_R_32F, m=150, n=90, k=77, transa=1)
    for offset, want in ((0, 3), (2, 3)):
        case = Case(spec, 9600)
        ref = case.run_oracle()
        keep, ptr, dt = case.upload(offset)
        p = case.problem(dict(ptr, A=None, B=None, alpha=case.alpha.ctypes.data, beta=case.beta.ctypes.data))
        plan = K.zluda_gemm_plan()
        assert gpu_api.zluda_gemm_plan_problem(C.byref(p), 0, -1, gpu_api.zluda_gemm_device_cu_count(), C.byref(plan)) == 0
        assert (plan.kernel, plan.variant) == (GEN, want)
        p.A, p.B = ptr["A"], ptr["B"]
        print("case", spec, "offset", offset, flush=True)
        assert gpu_api.zluda_gemm_launch(C.byref(p), C.byref(plan), torch.cuda.current_stream().cuda_stream) == 0
        torch.cuda.synchronize()
        case.compare(case.download(dt), ref, tol=1e-3)
