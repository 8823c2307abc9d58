"""The row sums behind the bias-gradient epilogues with and without scratch for their shares: whole 16-byte pieces and odd
pitches, ends inside a piece, fewer terms than a share, every operand type.  Sums of few thousand terms in fp32; int8 exact."""
import pytest

from oracle.cases import Case
from zluda_amd import abi as K

pytestmark = pytest.mark.gpu
TYPES = {"f32": K.CUDA_R_32F, "f16": K.CUDA_R_16F, "bf16": K.CUDA_R_16BF, "i8": K.CUDA_R_8I, "f8": K.CUDA_R_8F_E4M3}


def run(gpu_api, spec, seed, ws, want_ws):
    print("case", spec, "workspace", ws, flush=True)
    case = Case(spec, seed)
    ref = case.run_oracle()
    st, got, _, _ = case.run_gpu(gpu_api, workspace_bytes=ws)
    assert st == 0
    assert (case.last_workspace_needed > 0) == want_ws
    return case, got, ref


@pytest.mark.parametrize("ws", [0, 8 << 20])
@pytest.mark.parametrize("n,k,ldb", [(1, 130, 16), (63, 200, 64), (257, 1000, 272), (260, 333, 261)])
@pytest.mark.parametrize("t", sorted(TYPES))
def test_sums_of_an_operand_along_its_pitch(gpu_api, t, n, k, ldb, ws):
    typ = TYPES[t]
    if t in ("i8", "f8"):
        n, ldb = (n + 3) // 4 * 4, (ldb + 3) // 4 * 4
    spec = dict(a_type=typ, b_type=typ, d_type=typ if t not in ("i8", "f8") else K.CUDA_R_16BF, m=64, n=n, k=k, transa=0, transb=1, ldb=ldb,
                compute_type=K.CUBLAS_COMPUTE_32I if t == "i8" else K.CUBLAS_COMPUTE_32F, scale_type=K.CUDA_R_32F, alpha=0.01,
                epilogue=K.CUBLASLT_EPILOGUE_BGRADB, bias_type=K.CUDA_R_32F)
    case, got, ref = run(gpu_api, spec, 8100 + n, ws, ws > 0)
    case.compare_bgrad(case.bgrad_got, case.bgrad_ref, exact=t == "i8")


@pytest.mark.parametrize("ws", [0, 8 << 20])
@pytest.mark.parametrize("m,n,ldd", [(8, 200, 8), (257, 333, 264), (300, 150, 301)])
@pytest.mark.parametrize("t", ["f32", "bf16"])
def test_sums_of_a_gelu_gradient(gpu_api, t, m, n, ldd, ws):
    typ = TYPES[t]
    spec = dict(a_type=typ, b_type=typ, d_type=typ, m=m, n=n, k=64, transa=1, transb=0, ldd=ldd, ldc=ldd, aux_ld=ldd + 8, alpha=0.05,
                compute_type=K.CUBLAS_COMPUTE_32F, scale_type=K.CUDA_R_32F, epilogue=K.CUBLASLT_EPILOGUE_DGELU_BGRAD)
    case, got, ref = run(gpu_api, spec, 8200 + m, ws, ws > 0)
    case.compare(got, ref, tol=1.6e-2 if t == "bf16" else None)   # one more rounding of D's type than a single pass
    case.compare_bgrad(case.bgrad_got, case.bgrad_ref, floor_frac=1.0)
