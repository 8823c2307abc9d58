"""The rings of the 128 x 128 and 64 x 64 tiles whose LDS reads transpose, deeper ones where fewer workgroups share a CU: every position of
the ring that K can end at, K tails inside a stage, shares of K of unequal length."""
import pytest

from oracle.cases import Case
from zluda_amd import abi as K

pytestmark = pytest.mark.gpu
BF = dict(a_type=K.CUDA_R_16BF, b_type=K.CUDA_R_16BF, d_type=K.CUDA_R_16BF, compute_type=K.CUBLAS_COMPUTE_32F, scale_type=K.CUDA_R_32F, alpha=0.05)
# (a stage is 64 elements of K; the form is taken from 11 stages on with one tile to a CU, from 7 on with two)
SHORT, LONG = [704, 712, 768, 824, 832, 888, 896, 952], [448, 456, 512, 520]


@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 1)])
@pytest.mark.parametrize("k,batch", [(k, 1) for k in SHORT] + [(k, 66) for k in LONG])   # 4 and 264 tiles
def test_every_end_of_the_ring(gpu_api, k, batch, ta, tb):
    spec = dict(BF, m=200, n=136, k=k, transa=ta, transb=tb, batch=batch)
    print("case", spec, flush=True)
    case = Case(spec, 9900 + k)
    st, got, kernel, variant = case.run_gpu(gpu_api, forced_kernel=K.ZLUDA_KERNEL_MFMA_TR16, forced_variant=1)
    assert st == 0 and variant == 1
    case.compare(got, case.run_oracle(), tol=1e-2)   # one rounding to bf16 of sums in another order


@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 1)])
@pytest.mark.parametrize("k", [5632, 5704, 6152])   # eight shares of 11 to 13 stages, the last of 11, 6 and 6
def test_shares_of_k(gpu_api, k, ta, tb):
    spec = dict(BF, m=136, n=200, k=k, transa=ta, transb=tb, d_type=K.CUDA_R_32F)
    print("case", spec, flush=True)
    case = Case(spec, 9950 + k)
    st, got, plan = case.run_gpu_plan(gpu_api, K.ZLUDA_KERNEL_MFMA_TR16, 1, workspace_bytes=16 << 20)
    assert st == 0 and (plan.variant, plan.grid_z) == (1, 8)
    case.compare(got, case.run_oracle(), tol=1e-3)   # 32-bit sums in another order


@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 1)])
@pytest.mark.parametrize("batch", [1, 44, 130])   # 6, 264 and 780 tiles of 64 x 64: rings of six, three and two stages
def test_small_tiles(gpu_api, batch, ta, tb):
    for k in (8, 64, 72, 128, 192, 200, 256, 320, 384, 392, 448, 512) if batch < 130 else (8, 64, 72, 128, 192, 200):
        spec = dict(BF, m=136, n=72, k=k, transa=ta, transb=tb, batch=batch)
        print("case", spec, flush=True)
        case = Case(spec, 9970 + k)
        st, got, kernel, variant = case.run_gpu(gpu_api, forced_kernel=K.ZLUDA_KERNEL_MFMA_TR16, forced_variant=2)
        assert st == 0 and variant == 2
        case.compare(got, case.run_oracle(), tol=1e-2)


# whole turns of the ring and what is left of K behind them, at every number of stages that can be left
@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 1)])
@pytest.mark.parametrize("variant,batch,least,turn", [(2, 1, 13, 6), (2, 44, 10, 6), (1, 1, 9, 4)])
def test_turns(gpu_api, variant, batch, least, turn, ta, tb):
    for stages in range(least - 1, least + 2 * turn + 1):
        for k in (64 * stages, 64 * stages - 56):
            if variant == 1 and k < 704:
                continue   # (transposed in registers)
            spec = dict(BF, m=136, n=72, k=k, transa=ta, transb=tb, batch=batch)
            print("case", spec, flush=True)
            case = Case(spec, 10000 + k)
            st, got, kernel, chosen = case.run_gpu(gpu_api, forced_kernel=K.ZLUDA_KERNEL_MFMA_TR16, forced_variant=variant)
            assert st == 0 and chosen == variant
            case.compare(got, case.run_oracle(), tol=1e-2)


@pytest.mark.parametrize("m,n,ta,tb", [(50000, 16, 0, 0), (49160, 1, 0, 0), (16, 50000, 1, 1)])
def test_a_long_operand_along_its_row_index(gpu_api, m, n, ta, tb):
    for k in (120, 128, 136, 264):   # by the LDS reads, then in registers
        spec = dict(BF, m=m, n=n, k=k, transa=ta, transb=tb)
        print("case", spec, flush=True)
        case = Case(spec, 10300 + k)
        st, got, kernel, variant = case.run_gpu(gpu_api, forced_kernel=K.ZLUDA_KERNEL_MFMA_TR16, forced_variant=2)
        assert st == 0 and variant == 2
        case.compare(got, case.run_oracle(), tol=1e-2)
