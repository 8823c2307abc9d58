"""Many tiles of a short K (at most 128 elements of f16 / bf16): workgroups that walk the tiles with both operands of a tile in LDS
at once.  Ends of K inside and between its two chunks; ends of both extents inside a tile, in runs of one to a few tiles per
workgroup that turn over within a run; every output type; a row-major D; and what runs on other kernels all the same: a beta that
is not zero, columns of D at odd 16-bit addresses."""
import pytest

from oracle.cases import Case
from zluda_amd import abi as K

pytestmark = pytest.mark.gpu


def run(gpu_api, m, n, k, batch, t=K.CUDA_R_16BF, d=None, **more):
    s = dict(a_type=t, b_type=t, d_type=d if d is not None else t, c_type=d if d is not None else t, compute_type=K.CUBLAS_COMPUTE_32F,
             scale_type=K.CUDA_R_32F, m=m, n=n, k=k, transa=1, batch=batch)
    s.update(more)
    print("case", s, flush=True)
    case = Case(s, 7700 + m + k)
    st, got, kernel, variant = case.run_gpu(gpu_api)
    assert st == 0 and kernel == K.ZLUDA_KERNEL_MFMA_H16
    case.compare(got, case.run_oracle(), tol=1e-2)   # one rounding to 16 bits of sums in another order


@pytest.mark.parametrize("m,n,k,batch", [(130, 130, 8, 130), (128, 256, 64, 260), (300, 70, 72, 175), (66, 65, 128, 520), (256, 384, 120, 90), (1026, 200, 104, 40)])
def test_edges(gpu_api, m, n, k, batch):
    run(gpu_api, m, n, k, batch)


@pytest.mark.parametrize("t,d", [(K.CUDA_R_16F, K.CUDA_R_16F), (K.CUDA_R_16BF, K.CUDA_R_32F), (K.CUDA_R_16F, K.CUDA_R_32F), (K.CUDA_R_16BF, K.CUDA_R_16F)])
def test_output_types(gpu_api, t, d):
    run(gpu_api, 202, 130, 96, 133, t, d, alpha=0.125)
    run(gpu_api, 131, 129, 64, 133, t, K.CUDA_R_32F, ldd=133)


def test_row_major_scales_and_other_roads(gpu_api):
    run(gpu_api, 130, 202, 96, 133, order_c=1, order_d=1, ldc=208, ldd=208)
    run(gpu_api, 130, 130, 80, 133, with_scalar_scales=True, scale_range=(0.5, 1.5))
    run(gpu_api, 130, 130, 80, 133, with_c=True, beta=0.5)       # a tile per workgroup
    run(gpu_api, 131, 130, 80, 133, ldd=131)
    run(gpu_api, 130, 130, 80, 133, epilogue=K.CUBLASLT_EPILOGUE_GELU_BIAS)


def test_a_plan_for_another_number_of_cus(gpu_api):
    """64 elements of K in 60 tiles: a plan for 8 CUs has the form (16 workgroups), one for this device would not"""
    import ctypes as C
    import torch
    t = K.CUDA_R_16BF
    case = Case(dict(a_type=t, b_type=t, d_type=t, c_type=t, compute_type=K.CUBLAS_COMPUTE_32F, scale_type=K.CUDA_R_32F, m=300, n=200, k=64, transa=1, batch=10), 7800)
    print("case", case.spec, flush=True)
    keep, ptr, dt = case.upload()
    p = case.problem(dict(ptr, alpha=case.alpha.ctypes.data, beta=case.beta.ctypes.data))
    plan = K.zluda_gemm_plan()
    assert gpu_api.zluda_gemm_plan_problem(C.byref(p), K.ZLUDA_KERNEL_MFMA_H16, 3, 8, C.byref(plan)) == 0
    assert (plan.variant, plan.grid_x, plan.grid_y, plan.grid_z) == (3, 16, 1, 1)
    assert gpu_api.zluda_gemm_launch(C.byref(p), C.byref(plan), torch.cuda.current_stream().cuda_stream) == 0
    torch.cuda.synchronize()
    case.compare(case.download(dt), case.run_oracle(), tol=1e-2)


@pytest.mark.parametrize("ldd,aux_ld", [(132, 131), (131, 132)])
def test_a_kept_gelu_input_with_a_pitch_of_its_own(gpu_api, ldd, aux_ld):
    """the kernel writes the GELU input: the pitch of that matrix decides, not D's"""
    t = K.CUDA_R_16F   # (D is the GELU of a rounded input u: |u gelu'(u) / gelu(u)| < 16 down to u = -4, times half an ulp of f16: 4e-3)
    s = dict(a_type=t, b_type=t, d_type=t, c_type=t, compute_type=K.CUBLAS_COMPUTE_32F, scale_type=K.CUDA_R_32F,
             m=130, n=130, k=72, transa=1, batch=133, ldc=ldd, ldd=ldd, aux_ld=aux_ld, epilogue=K.CUBLASLT_EPILOGUE_GELU_AUX)
    print("case", s, flush=True)
    case = Case(s, 7900)
    ref = case.run_oracle()
    st, got, kernel, variant = case.run_gpu(gpu_api)
    assert st == 0 and kernel == K.ZLUDA_KERNEL_MFMA_H16
    case.compare(got, ref, tol=1e-2)
    case.compare_aux(case.aux_got, case.aux_ref)


@pytest.mark.parametrize("d", [K.CUDA_R_16BF, K.CUDA_R_32F])
def test_zeros_have_the_sign_that_the_tile_kernels_give_them(gpu_api, d):
    """a row of zeros in A, alpha -1"""
    t = K.CUDA_R_16BF
    case = Case(dict(a_type=t, b_type=t, d_type=d, c_type=d, compute_type=K.CUBLAS_COMPUTE_32F, scale_type=K.CUDA_R_32F, m=130, n=130, k=72, transa=1,
                     batch=133, alpha=-1.0), 7950)
    case.A.reshape(-1, 72)[::3] = 0
    print("case", case.spec, flush=True)
    bits = []
    for v in (3, 6):
        st, got, kernel, variant = case.run_gpu(gpu_api, forced_kernel=K.ZLUDA_KERNEL_MFMA_H16, forced_variant=v)
        assert st == 0 and variant == v
        bits.append(got.view("u4" if d == K.CUDA_R_32F else "u2").reshape(-1, 130))
    zero = [(i % 130, b) for b in range(133) for i in range(130) if (b * 130 + i) % 3 == 0]
    for i, b in zero:
        assert (bits[0][b * 130:(b + 1) * 130, i] == bits[1][b * 130:(b + 1) * 130, i]).all()


@pytest.mark.parametrize("k,d,m,n,batch", [(64, K.CUDA_R_16BF, 512, 640, 3), (128, K.CUDA_R_16BF, 512, 640, 3), (128, K.CUDA_R_32F, 384, 1300, 2), (72, K.CUDA_R_16BF, 500, 1300, 2),
                                           (40, K.CUDA_R_32F, 300, 1100, 3), (128, K.CUDA_R_16F, 130, 4000, 1)])
def test_runs_of_many_tiles(gpu_api, k, d, m, n, batch):
    """eight and sixteen workgroups: runs of four to eight tiles, whole ones in a row and turns of P between them, so that every wait is reached"""
    t = K.CUDA_R_16F if d == K.CUDA_R_16F else K.CUDA_R_16BF
    s = dict(a_type=t, b_type=t, d_type=d, c_type=d, compute_type=K.CUBLAS_COMPUTE_32F, scale_type=K.CUDA_R_32F, m=m, n=n, k=k, transa=1, batch=batch)
    case = Case(s, 7960 + k)
    ref = case.run_oracle()
    tiles = -(-m // 128) * -(-n // 128)
    for groups in (8, 16):
        print("case", s, groups, flush=True)

        def short_form(plan):
            plan.grid_x, plan.grid_y, plan.grid_z = groups, 1, 1
        st, got, plan = case.run_gpu_plan(gpu_api, K.ZLUDA_KERNEL_MFMA_H16, 3, edit=short_form)
        assert st == 0 and plan.variant == 3 and groups < tiles * batch
        case.compare(got, ref, tol=1e-2)


def test_the_planner_gives_the_form(gpu_api):
    """the problems of test_edges and test_output_types have more tiles than two workgroups per CU take in one go"""
    for m, n, k, batch in [(130, 130, 8, 130), (128, 256, 64, 260), (300, 70, 72, 175), (66, 65, 128, 520), (256, 384, 120, 90), (1026, 200, 104, 40), (202, 130, 96, 133)]:
        t = K.CUDA_R_16BF
        case = Case(dict(a_type=t, b_type=t, d_type=t, c_type=t, compute_type=K.CUBLAS_COMPUTE_32F, scale_type=K.CUDA_R_32F, m=m, n=n, k=k, transa=1, batch=batch), 7970)
        st, got, plan = case.run_gpu_plan(gpu_api, K.ZLUDA_KERNEL_AUTO)
        assert st == 0 and (plan.kernel, plan.variant, plan.grid_y, plan.grid_z) == (K.ZLUDA_KERNEL_MFMA_H16, 3, 1, 1)
        assert plan.grid_x == max(2 * gpu_api.zluda_gemm_device_cu_count() // 8 * 8, 8)
