"""A plan determines the scratch that its launch writes and the shares its sums are taken in: a bias-gradient plan that counts no
workspace writes none, one that counts some writes no byte behind it, and the gradient's bits are the same whatever the buffer
handed over at the launch holds."""
import ctypes as C

import numpy as np
import pytest

from oracle.cases import Case
from zluda_amd import abi as K

pytestmark = pytest.mark.gpu
BF = dict(a_type=K.CUDA_R_16BF, b_type=K.CUDA_R_16BF, d_type=K.CUDA_R_16BF, compute_type=K.CUBLAS_COMPUTE_32F, scale_type=K.CUDA_R_32F,
          bias_type=K.CUDA_R_32F)
SPECS = [dict(BF, m=96, n=264, k=2000, transb=1, epilogue=K.CUBLASLT_EPILOGUE_BGRADB),
         dict(BF, m=264, n=96, k=2000, transb=1, epilogue=K.CUBLASLT_EPILOGUE_BGRADA),
         dict(BF, m=264, n=2000, k=64, transa=1, epilogue=K.CUBLASLT_EPILOGUE_DGELU_BGRAD)]
BUFFER = 8 << 20


def launch(api, spec, planned, buffer, noalloc=False):
    """(bits of the gradient, the plan's workspace, the buffer behind it is as it was)"""
    import torch
    case = Case(spec, 9400)
    ref = case.run_oracle()
    keep, ptr, dt = case.upload()
    ptrs = dict(ptr, alpha=case.alpha.ctypes.data, beta=case.beta.ctypes.data)
    p = case.problem(ptrs)
    p.workspace_size = planned
    plan = K.zluda_gemm_plan()
    assert api.zluda_gemm_plan_problem(C.byref(p), 0, -1, api.zluda_gemm_device_cu_count(), C.byref(plan)) == 0
    ws = torch.full((max(buffer, 16),), 0xCD, dtype=torch.uint8, device="cuda:0")
    p.workspace, p.workspace_size = (ws.data_ptr() if buffer else None), buffer
    print("case", spec, "planned for", planned, "buffer", buffer, "plan asks for", plan.workspace, flush=True)
    run = api.zluda_gemm_launch_noalloc if noalloc else api.zluda_gemm_launch
    assert run(C.byref(p), C.byref(plan), torch.cuda.current_stream().cuda_stream) == 0
    torch.cuda.synchronize()
    case.compare(case.download(dt), ref, tol=1.6e-2)
    got = keep[3][:case.bias.nbytes].cpu().numpy().view(case.bias.dtype).copy()
    case.compare_bgrad(got, case.bgrad_ref, floor_frac=1.0)
    return got.view(np.uint32), plan.workspace, bool((ws[plan.workspace:] == 0xCD).all())


@pytest.mark.parametrize("index", range(len(SPECS)))
def test_the_plan_bounds_the_scratch_and_fixes_the_sums(gpu_api, index):
    spec = SPECS[index]
    none, need, _ = launch(gpu_api, spec, 0, 0)
    assert need == 0
    for noalloc in (False, True):
        got, need, untouched = launch(gpu_api, spec, 0, BUFFER, noalloc)
        assert need == 0 and untouched and np.array_equal(got, none)
    small, need, untouched = launch(gpu_api, spec, 4 * 264 * 4, 4 * 264 * 4)   # four shares at the most
    assert 0 < need <= 4 * 264 * 4 and untouched
    got, _, untouched = launch(gpu_api, spec, 4 * 264 * 4, BUFFER)
    assert untouched and np.array_equal(got, small)
