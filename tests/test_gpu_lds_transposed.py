"""16-bit operands with unit stride along their row index whose addresses and pitches are multiples of 16 bytes: the tiles that
copy them into LDS as they lie and transpose in the LDS reads.  Ends of K inside a stage, a block of K rows and a group of four;
one, two and three stages; ends of the rows inside a 16-byte piece and between tiles; every pair of layouts; shares of K."""
import pytest

from oracle.cases import Case
from zluda_amd import abi as K

pytestmark = pytest.mark.gpu

LAYOUTS = [(0, 0), (0, 1), (1, 1)]   # (transa, transb): A, both, B with unit stride along the row index


def spec(typ, m, n, k, ta, tb, **more):
    t = {"bf16": K.CUDA_R_16BF, "f16": K.CUDA_R_16F}[typ]
    up8 = lambda x: (x + 7) // 8 * 8
    base = dict(a_type=t, b_type=t, d_type=t, c_type=t, compute_type=K.CUBLAS_COMPUTE_32F, scale_type=K.CUDA_R_32F, m=m, n=n, k=k,
                transa=ta, transb=tb, lda=up8(k if ta else m), ldb=up8(n if tb else k))
    base.update(more)
    return base


def check(gpu_api, s, seed, ws=0):
    print("case", s, flush=True)
    case = Case(s, seed)
    ref = case.run_oracle()
    for v in (1, 2, 3):
        st, got, kernel, variant = case.run_gpu(gpu_api, forced_kernel=K.ZLUDA_KERNEL_MFMA_TR16, forced_variant=v, workspace_bytes=ws)
        assert st == 0 and (kernel, variant) == (K.ZLUDA_KERNEL_MFMA_TR16, v)
        case.compare(got, ref, tol=1e-2)   # one rounding to 16 bits of sums in another order


@pytest.mark.parametrize("typ", ["bf16", "f16"])
@pytest.mark.parametrize("layout", range(3))
@pytest.mark.parametrize("m,n,k", [(128, 128, 64), (257, 264, 8), (136, 300, 72), (511, 129, 192), (264, 40, 136), (300, 520, 1000)])
def test_edges(gpu_api, typ, layout, m, n, k):
    check(gpu_api, spec(typ, m, n, k, *LAYOUTS[layout]), 9100 + m)


@pytest.mark.parametrize("k", [2, 61, 65, 101, 133, 199, 259])
def test_odd_ends_of_k_where_neither_operand_is_k_contiguous(gpu_api, k):
    check(gpu_api, spec("bf16", 260, 250, k, 0, 1), 9200 + k)


@pytest.mark.parametrize("layout", range(3))
def test_batches_and_shares_of_k(gpu_api, layout):
    check(gpu_api, spec("bf16", 200, 136, 200, *LAYOUTS[layout], batch=3), 9300)
    check(gpu_api, spec("bf16", 264, 136, 2184, *LAYOUTS[layout], epilogue=K.CUBLASLT_EPILOGUE_GELU_BIAS), 9310, ws=8 << 20)
    check(gpu_api, spec("bf16", 136, 264, 1000, *LAYOUTS[layout], order_c=1, order_d=1, ldc=272, ldd=272), 9320)
