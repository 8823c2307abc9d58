"""GELU with its input kept and GELU's gradient in the epilogues of the 16-bit tile kernels: every accumulator layout, tiles that hang over
either end of D, pitches and batch strides of aux of their own, and what keeps a problem on the pass behind the matmul.  Which of the two ways
a problem goes is asked of the planner's own rule and read off the scratch that the sums of a gradient leave."""
import ctypes as C

import pytest

import planner_probe
from oracle.cases import Case
from zluda_amd import abi as K

pytestmark = pytest.mark.gpu
AUX, AUX_BIAS, DG, DG_SUMS = (K.CUBLASLT_EPILOGUE_GELU_AUX, K.CUBLASLT_EPILOGUE_GELU_AUX_BIAS, K.CUBLASLT_EPILOGUE_DGELU, K.CUBLASLT_EPILOGUE_DGELU_BGRAD)
H16, TR16 = K.ZLUDA_KERNEL_MFMA_H16, K.ZLUDA_KERNEL_MFMA_TR16
BF = dict(a_type=K.CUDA_R_16BF, b_type=K.CUDA_R_16BF, d_type=K.CUDA_R_16BF, compute_type=K.CUBLAS_COMPUTE_32F, scale_type=K.CUDA_R_32F, alpha=0.05)
# One rounding of D to its type (2^-9 bf16, 2^-12 f16) of sums in another order than the oracle's, and the fast exponential and reciprocal.
# (The aux matrix is rounded once; the gradient is taken at its stored elements, as the oracle takes it.)
TOL = {K.CUDA_R_16BF: 1e-2, K.CUDA_R_16F: 2e-3}
# Behind the matmul GELU sees its input x rounded to bf16: an error of 2^-9 |x gelu'(x)|, at most 0.2 * 2^-9 where x < 0 (it is relative to the
# result elsewhere).  Compared with a floor of a tenth of D's root mean square (0.2 or more here) that is 10 * 2^-9, and D's own rounding.
TOL_BEHIND, FLOOR_BEHIND = 12 / 512, 1e-1


def run(api, spec, seed, family, variant, ws=4 << 20, block=None, in_epilogue=True, lds=None, one_rounding=None):
    """the case, its plan; `in_epilogue`: the kernel does it all, else there is a pass behind it; `lds`: transposed by the LDS reads;
    `one_rounding`: held to the bounds of a single rounding, which these inputs meet behind some plans as well"""
    import torch
    print("case", spec, "family", family, "variant", variant, flush=True)
    one_rounding = in_epilogue if one_rounding is None else one_rounding
    case = Case(spec, seed)
    ref = case.run_oracle()
    keep, ptr, dt = case.upload()
    p = case.problem(dict(ptr, alpha=case.alpha.ctypes.data, beta=case.beta.ctypes.data))
    scratch = torch.full((max(ws, 16),), 0xFF, dtype=torch.uint8, device="cuda:0")   # (NaN: a sum that is read without being written)
    p.workspace, p.workspace_size = (scratch.data_ptr() if ws else None), ws
    plan = K.zluda_gemm_plan()
    assert api.zluda_gemm_plan_problem(C.byref(p), family, variant, api.zluda_gemm_device_cu_count(), C.byref(plan)) == 0
    if block:
        plan.block = block
    sums = planner_probe.aux_sum_bytes(p, plan) if case.bgrad else 0
    assert (planner_probe.aux_in_epilogue(p, plan) == 1 and sums <= plan.workspace) == in_epilogue
    if lds is not None:
        assert planner_probe.lds_reads(p, plan, api.zluda_gemm_device_cu_count()) == lds
    assert api.zluda_gemm_launch(C.byref(p), C.byref(plan), torch.cuda.current_stream().cuda_stream) == 0
    torch.cuda.synchronize()
    case.compare(case.download(dt), ref, tol=TOL[spec["d_type"]] if one_rounding else TOL_BEHIND,
                 floor_frac=None if one_rounding else FLOOR_BEHIND)
    if case.aux_mode == 1:
        case.compare_aux(keep[10][:case.aux.nbytes].cpu().numpy().view(case.aux.dtype).copy(), case.aux_ref)
    if case.bgrad:
        case.compare_bgrad(keep[3][:case.bias.nbytes].cpu().numpy().view(case.bias.dtype).copy(), case.bgrad_ref, floor_frac=1.0)
        assert bool((scratch[plan.workspace:] == 0xFF).all())
        if in_epilogue:   # one sum per wave and row, each of them written, and nothing else
            import torch
            assert bool((scratch[:sums].view(torch.int32) != -1).all()) and bool((scratch[sums:] == 0xFF).all())
    return case, plan


# family, variant, block: 32x32 tiles of every wave shape, 16x16 tiles, the four-wave kernel; the layouts of the transposing kernels (the 64 x 64 tile
# by the LDS reads whatever the block, the 128 x 128 tile in registers: K is short)
FORMS = [(H16, v, b, 1, 0) for v, b in ((0, 0), (2, 256), (2, 512), (4, 0), (5, 0), (6, 0), (7, 0), (8, 0), (9, 0), (10, 0), (11, 0))] + \
        [(TR16, v, b, ta, tb) for v, b in ((0, 0), (1, 256), (1, 512), (2, 256), (2, 512), (3, 0)) for ta, tb in ((0, 0), (0, 1), (1, 1))]


@pytest.mark.parametrize("epi", [AUX, AUX_BIAS, DG, DG_SUMS])
@pytest.mark.parametrize("family,variant,block,ta,tb", FORMS)
def test_every_form(gpu_api, family, variant, block, ta, tb, epi):
    # (tiles that hang over both ends, at both types of D; K rows of 16-byte pieces)
    for i, (m, n, k) in enumerate(((264, 131, 128), (520, 300, 200), (8, 1, 72))):
        spec = dict(BF, m=m, n=n, k=k, transa=ta, transb=tb, epilogue=epi)
        if i == 1:
            spec.update(a_type=K.CUDA_R_16F, b_type=K.CUDA_R_16F, d_type=K.CUDA_R_16F, bias_type=K.CUDA_R_32F)
        if (ta, tb) != (1, 0) and tb:   # (the columns of B lie side by side: a whole number of 16-byte pieces for the LDS reads)
            spec["ldb"] = (n + 7) // 8 * 8
        behind = variant == 0 or (family == H16 and block == 256)   # (wave tiles of 128 x 64 on the 32x32 shapes)
        no_gradient = family == H16 and variant == 11 and epi in (DG, DG_SUMS)   # (the four-wave kernel keeps GELU's input)
        run(gpu_api, spec, 9700 + 10 * epi + i, family, variant, block=block, in_epilogue=not behind and not no_gradient,
            lds=None if family == H16 else int(variant in (2, 3)), one_rounding=not behind)


# Operands off 16 bytes (pitches of whole dwords) are transposed in registers: 64 x 64 tiles with one group of waves and with two that share K,
# the 256 x 256 tile of the 16x16 shapes
@pytest.mark.parametrize("epi", [AUX_BIAS, DG, DG_SUMS])
@pytest.mark.parametrize("variant,block", [(2, 256), (2, 512), (3, 512)])
@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 1), (1, 0)])
def test_forms_in_registers(gpu_api, ta, tb, variant, block, epi):
    for i, (m, n, k) in enumerate(((264, 131, 264), (72, 65, 800), (8, 1, 72))):
        off = lambda x: x + (2 if x % 4 == 0 else 3 if x % 2 else 4)   # (a multiple of 2, of 4 at the most)
        spec = dict(BF, m=m, n=n, k=k, transa=ta, transb=tb, epilogue=epi, lda=off(k if ta else m), ldb=off(n if tb else k))
        run(gpu_api, spec, 9820 + i, TR16, variant, block=block, lds=0)


# ... and by the LDS reads: the 128 x 128 tile on its ring of four stages (6 tiles) and of two (264), the 64 x 64 tile on three (660) and two (990)
@pytest.mark.parametrize("epi", [AUX_BIAS, DG, DG_SUMS])
@pytest.mark.parametrize("variant,k,batch", [(1, 712, 1), (1, 1016, 1), (1, 456, 44), (2, 832, 1), (2, 136, 44), (2, 136, 66)])
@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 1)])
def test_forms_by_the_lds_reads(gpu_api, ta, tb, variant, k, batch, epi):
    spec = dict(BF, m=264, n=131, k=k, transa=ta, transb=tb, batch=batch, epilogue=epi)
    if tb:
        spec["ldb"] = 136
    if batch > 1:
        spec["bias_batch_stride"] = 264
    run(gpu_api, spec, 9840, TR16, variant, ws=16 << 20, lds=1)


@pytest.mark.parametrize("family,variant,ta,tb", [(H16, 4, 1, 0), (H16, 8, 1, 0), (H16, 11, 1, 0), (TR16, 1, 0, 0), (TR16, 2, 0, 1)])
def test_batches_pitches_scales(gpu_api, family, variant, ta, tb):
    base = dict(BF, m=200, n=136, k=264, batch=3, transa=ta, transb=tb, ldd=208, ldc=208, aux_ld=224, aux_batch_stride=224 * 136 + 40)
    run(gpu_api, dict(base, epilogue=AUX_BIAS, bias_type=K.CUDA_R_32F, bias_batch_stride=203), 9801, family, variant)
    run(gpu_api, dict(base, epilogue=AUX_BIAS, bias_batch_stride=203), 9802, family, variant)     # (a bias at odd addresses)
    run(gpu_api, dict(base, epilogue=DG_SUMS, bias_batch_stride=208), 9803, family, variant, in_epilogue=variant != 11, one_rounding=True)


@pytest.mark.parametrize("change", [dict(m=260), dict(ldd=268, ldc=268), dict(aux_ld=268), dict(order_c=1, order_d=1, aux_ld=136), dict(with_c=True),
                                    dict(d_type=K.CUDA_R_32F), dict(ws=0), dict(k=4096, m=64, n=64)])
@pytest.mark.parametrize("epi,ta", [(AUX_BIAS, 1), (DG_SUMS, 0)])
def test_what_keeps_the_pass_behind_the_matmul(gpu_api, epi, ta, change):
    change = dict(change)
    ws = change.pop("ws", 4 << 20)
    spec = dict(BF, m=264, n=136, k=256, transa=ta, epilogue=epi)
    spec.update(change)
    if spec["d_type"] == K.CUDA_R_32F:
        spec["c_type"] = K.CUDA_R_32F
    if spec.get("with_c") and epi == AUX_BIAS:
        spec["beta"] = 0.5
    # (without scratch only the sums of a gradient want the pass)
    run(gpu_api, spec, 9850, H16 if ta else TR16, -1, ws=ws, in_epilogue=ws == 0 and epi == AUX_BIAS)


@pytest.mark.parametrize("epi", [AUX, DG, DG_SUMS])
def test_walked_tiles_with_a_grid_of_one_batch(gpu_api, epi):
    # (512 tiles of 128 x 128 in each of two batches: as many workgroups walk them all on 256 CUs)
    case, plan = run(gpu_api, dict(BF, m=1928, n=3969, k=16, transa=1, batch=2, epilogue=epi, bias_batch_stride=1928 if epi == DG_SUMS else 0),
                     9870, H16, -1, ws=32 << 20, in_epilogue=False)
    assert (plan.variant, plan.grid_x, plan.grid_y) == (3, 512, 1)


@pytest.mark.parametrize("family,ta", [(H16, 1), (TR16, 0)])
def test_a_plan_for_fewer_batches_is_refused(gpu_api, family, ta):
    import torch
    case = Case(dict(BF, m=200, n=136, k=264, transa=ta, batch=3), 9880)
    keep, ptr, dt = case.upload()
    p = case.problem(dict(ptr, alpha=case.alpha.ctypes.data, beta=case.beta.ctypes.data))
    plan = K.zluda_gemm_plan()
    assert gpu_api.zluda_gemm_plan_problem(C.byref(p), family, -1, 256, C.byref(plan)) == 0 and plan.grid_y == 3
    plan.grid_y = 1
    assert gpu_api.zluda_gemm_launch(C.byref(p), C.byref(plan), torch.cuda.current_stream().cuda_stream) == K.CUBLAS_STATUS_INVALID_VALUE
    torch.cuda.synchronize()
    assert bool((case.download(dt) == case.new_d()).all())


@pytest.mark.parametrize("m,n,batch", [(72, 2048, 1), (72, 2049, 1), (8, 9000, 2), (200, 9000, 1)])
@pytest.mark.parametrize("bias_type", [-1, K.CUDA_R_32F])
def test_sums_of_many_waves(gpu_api, m, n, batch, bias_type):
    # (64 x 64 tiles, two waves along D's columns: 64 partial sums of a row by four threads, 66 and 282 by 64)
    run(gpu_api, dict(BF, m=m, n=n, k=72, transa=1, batch=batch, epilogue=DG_SUMS, bias_type=bias_type, bias_batch_stride=m if batch > 1 else 0),
        9890, H16, 6, ws=1 << 20)


@pytest.mark.parametrize("family,variant,ta", [(H16, 11, 1), (H16, 8, 1), (H16, 6, 1), (TR16, 3, 0), (TR16, 2, 0)])
def test_a_scale_of_zero(gpu_api, family, variant, ta):
    # (inputs of GELU well beyond where its exponential is zero)
    import torch
    case = Case(dict(BF, m=264, n=136, k=512, transa=ta, epilogue=AUX, alpha=1, with_cd_scales=True), 9895)
    case.d_scale[:] = 0
    case.run_oracle()
    keep, ptr, dt = case.upload()
    p = case.problem(dict(ptr, alpha=case.alpha.ctypes.data, beta=case.beta.ctypes.data))
    plan = K.zluda_gemm_plan()
    print("variant", family, variant, flush=True)
    assert gpu_api.zluda_gemm_plan_problem(C.byref(p), family, variant, gpu_api.zluda_gemm_device_cu_count(), C.byref(plan)) == 0
    assert gpu_api.zluda_gemm_launch(C.byref(p), C.byref(plan), torch.cuda.current_stream().cuda_stream) == 0
    torch.cuda.synchronize()
    assert bool(((case.download(dt) & 0x7FFF) == 0).all())
    case.compare_aux(keep[10][:case.aux.nbytes].cpu().numpy().view(case.aux.dtype).copy(), case.aux_ref)
