"""Workgroups whose waves share K in two groups (16-bit operands that are not K-contiguous, unaligned ones), with shares of one
length and not, ends of K inside a stage, and shares of K over workgroups on top."""
import ctypes as C

import pytest

from oracle.cases import Case
from zluda_amd import abi as K

pytestmark = pytest.mark.gpu


def bf(m, n, k, ta, tb, **more):
    t = K.CUDA_R_16BF
    return dict(dict(a_type=t, b_type=t, d_type=t, c_type=t, compute_type=K.CUBLAS_COMPUTE_32F, scale_type=K.CUDA_R_32F, m=m, n=n, k=k,
                     transa=ta, transb=tb), **more)


@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 1), (1, 0)])
@pytest.mark.parametrize("k", [768, 769, 799, 800, 801, 832, 1537])   # 24, 25 and 26 stages of 32, whole and not, and 49
def test_two_groups(gpu_api, ta, tb, k):
    for m, n in ((130, 131), (65, 70)):   # (64 x 64 tiles, as few as there are)
        s = bf(m, n, k, ta, tb, lda=(k if ta else m) + 3, ldb=(n if tb else k) + 1)
        print("case", s, flush=True)
        case = Case(s, 6600 + k)
        ref = case.run_oracle()
        st, got, kernel, v = case.run_gpu(gpu_api)
        assert st == 0
        case.compare(got, ref, tol=1e-2)   # one rounding to 16 bits of sums in another order
    s = bf(72, 136, k + 1 & ~1, 0, 1)
    case = Case(s, 6700 + k)
    ref = case.run_oracle()
    for v in (1, 2):
        st, got, kernel, variant = case.run_gpu(gpu_api, forced_kernel=K.ZLUDA_KERNEL_MFMA_TR16, forced_variant=v)
        assert st == 0 and variant == v
        case.compare(got, ref, tol=1e-2)


def plan_of(api, s, workspace=0, forced=K.ZLUDA_KERNEL_AUTO):
    case = Case.__new__(Case)
    case.spec, case.batch = dict(s), 1
    p = case.problem({"A": 0, "B": 0, "D": 0, "alpha": 0, "beta": 0})
    p.workspace_size = workspace
    plan = K.zluda_gemm_plan()
    assert api.zluda_gemm_plan_problem(C.byref(p), forced, -1, 256, C.byref(plan)) == 0
    return plan


@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 1), (1, 0)])
@pytest.mark.parametrize("shares", [1, 3])
def test_two_groups_on_128x128(gpu_api, ta, tb, shares):
    """odd pitches; the plan's tile, form and shares of K set by hand: shares of one length (768: eight stages of 32) and not (803: nine,
    nine, eight), a second group without a stage (160: shares of two and one) and a share without any (33)"""
    for m, n in ((130, 131), (257, 70)):
        for k in (33, 160, 768, 799, 803, 1537):
            s = bf(m, n, k, ta, tb, lda=(k if ta else m) | 1, ldb=(n if tb else k) | 1)
            print("case", s, shares, flush=True)
            case = Case(s, 6900 + k)

            def two_groups(plan):
                assert plan.kernel == K.ZLUDA_KERNEL_GENERIC
                plan.variant, plan.block, plan.grid_x, plan.grid_z = 1 + 1, 512, -(-m // 128) * -(-n // 128), shares
                plan.workspace = shares * plan.grid_x * 128 * 128 * 4 if shares > 1 else 0
            st, got, plan = case.run_gpu_plan(gpu_api, K.ZLUDA_KERNEL_GENERIC, edit=two_groups, workspace_bytes=4 << 20)
            assert st == 0
            case.compare(got, case.run_oracle(), tol=1e-2)


def test_what_the_planner_gives_two_groups(gpu_api):
    """the shapes that the form was made for, from the descriptors alone, and one of them with a shorter K run"""
    for s, workspace, variant, shares in ((bf(1024, 512, 32003, 0, 0, ldb=32003), 32 << 20, 2, 8), (bf(130, 131, 801, 1, 0, lda=805, ldb=801), 0, 3, 1),
                                          (bf(150, 70, 8003, 1, 0, lda=8003, ldb=8003), 16 << 20, 3, 8)):
        plan = plan_of(gpu_api, s, workspace)
        assert (plan.kernel, plan.variant, plan.grid_z, plan.block) == (K.ZLUDA_KERNEL_GENERIC, variant, shares, 512), s
    s = bf(1024, 512, 8003, 0, 0, ldb=8003)
    print("case", s, flush=True)
    case = Case(s, 6850)
    st, got, kernel, variant = case.run_gpu(gpu_api, workspace_bytes=32 << 20)
    assert st == 0 and kernel == K.ZLUDA_KERNEL_GENERIC
    case.compare(got, case.run_oracle(), tol=1e-2)


def test_two_groups_and_shares(gpu_api):
    for s in (bf(150, 70, 8003, 1, 0, lda=8003, ldb=8003), bf(70, 150, 8002, 0, 1, epilogue=K.CUBLASLT_EPILOGUE_GELU_BIAS)):
        print("case", s, flush=True)
        case = Case(s, 6800)
        st, got, kernel, variant = case.run_gpu(gpu_api, workspace_bytes=16 << 20)
        assert st == 0 and case.last_workspace_needed
        case.compare(got, case.run_oracle(), tol=1e-2)
