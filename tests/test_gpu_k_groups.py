"""Workgroups whose waves share K in two groups (16-bit operands that are not K-contiguous, unaligned ones), with shares of one
length and not, ends of K inside a stage, and shares of K over workgroups on top."""
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
    for variant, m, n in ((1, 130, 131), (2, 65, 70)):
        s = bf(m, n, k, ta, tb, lda=(k if ta else m) + 3, ldb=(n if tb else k) + 1)
        print("case", s, variant, flush=True)
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


def test_two_groups_and_shares(gpu_api):
    for s in (bf(150, 70, 8003, 1, 0, lda=8003, ldb=8003), bf(70, 150, 8002, 0, 1, epilogue=K.CUBLASLT_EPILOGUE_GELU_BIAS)):
        print("case", s, flush=True)
        case = Case(s, 6800)
        st, got, kernel, variant = case.run_gpu(gpu_api, workspace_bytes=16 << 20)
        assert st == 0 and case.last_workspace_needed
        case.compare(got, case.run_oracle(), tol=1e-2)
