"""MXFP4 weights with few tokens on the slab decode kernel: every shape of it, K that ends inside a wave's share, inside a unit and
leaves units and waves without any, one token and ragged second blocks, rows that leave a short last block, batches, outputs that
are and are not stored packed; a NaN scale of one row stays in that row."""
import numpy as np
import pytest

from oracle.cases import Case
from zluda_amd import abi as K

pytestmark = pytest.mark.gpu
MX = dict(a_type=K.CUDA_R_4F_E2M1, b_type=K.CUDA_R_4F_E2M1, d_type=K.CUDA_R_16BF, compute_type=K.CUBLAS_COMPUTE_32F, scale_type=K.CUDA_R_32F,
          transa=1, a_scale_mode=K.CUBLASLT_MATMUL_MATRIX_SCALE_VEC32_UE8M0, b_scale_mode=K.CUBLASLT_MATMUL_MATRIX_SCALE_VEC32_UE8M0)


def run(gpu_api, **spec):
    s = dict(MX, **spec)
    print("case", s, flush=True)
    case = Case(s, 4400 + s["k"])
    st, got, kernel, variant = case.run_gpu(gpu_api)
    assert st == 0 and kernel == K.ZLUDA_KERNEL_DECODE_W8A8
    case.compare(got, case.run_oracle())
    return variant


@pytest.mark.parametrize("k,n,variant", [(8192, 16, 16), (4352, 3, 16), (6400, 1, 16), (7936, 9, 16),        # 4 waves, one unit of 1 KiB
                                         (8192, 32, 20), (4352, 17, 20), (6912, 25, 20),                      # 8 waves, one unit, two token blocks
                                         (16384, 16, 17), (8448, 5, 17), (12544, 1, 17), (16384, 7, 17), (16640, 16, 18), (20736, 11, 18), (24576, 2, 18)])
def test_shapes(gpu_api, k, n, variant):
    assert run(gpu_api, m=300, n=n, k=k) == variant
    assert run(gpu_api, m=16 * 256 + 36, n=n, k=k, epilogue=K.CUBLASLT_EPILOGUE_GELU_BIAS) == variant


def test_outputs_orders_and_batches(gpu_api):
    run(gpu_api, m=333, n=5, k=8192, d_type=K.CUDA_R_32F, c_type=K.CUDA_R_32F)
    run(gpu_api, m=128, n=6, k=5120, batch=3)
    run(gpu_api, m=6, n=132, k=5120, order_c=1, order_d=1)
    run(gpu_api, m=6, n=132, k=9216)
    run(gpu_api, m=128, n=20, k=5120, batch=2, with_c=True, beta=0.5)


def test_a_nan_scale_stays_in_its_row(gpu_api):
    """row 37's scales are all NaN; K ends inside a unit, where the bytes behind row 36's scales are row 37's"""
    for k, n in ((4352, 4), (9472, 4), (17152, 4), (5120, 20)):
        s = dict(MX, m=128, n=n, k=k, d_type=K.CUDA_R_32F, c_type=K.CUDA_R_32F)
        print("case", s, flush=True)
        case = Case(s, 4500 + k)
        plain = case.run_oracle().copy()
        case.a_scale.reshape(128, k // 32)[37] = 255
        st, got, kernel, variant = case.run_gpu(gpu_api)
        assert st == 0 and kernel == K.ZLUDA_KERNEL_DECODE_W8A8
        got = got.view(np.float32).reshape(n, 128)
        assert np.isnan(got[:, 37]).all()
        want = plain.view(np.float32).reshape(n, 128)
        got[:, 37] = want[:, 37]
        case.compare(got.reshape(-1).view(plain.dtype), plain)


@pytest.mark.parametrize("k,n,variant", [(8192, 16, 16), (4352, 3, 16), (7936, 9, 16), (8192, 32, 20), (4352, 17, 20), (6912, 25, 20), (8448, 5, 17), (16384, 16, 17),
                                         (16640, 16, 18), (20736, 11, 18)])
def test_three_and_four_blocks_a_workgroup(gpu_api, k, n, variant):
    """two workgroups: slots of weights and scales that are filled again and read again, with whole blocks and a short last one"""
    for m in (96, 116, 128):
        s = dict(MX, m=m, n=n, k=k)
        print("case", s, variant, flush=True)
        case = Case(s, 4600 + k + m)
        st, got, plan = case.run_gpu_plan(gpu_api, K.ZLUDA_KERNEL_DECODE_W8A8, variant, grid_x=2)
        assert st == 0 and plan.variant == variant
        case.compare(got, case.run_oracle())


def test_many_rows(gpu_api):
    """beyond 64 rows per CU: the planner's own grid, four blocks in each workgroup"""
    assert run(gpu_api, m=28672, n=3, k=6144) == 16
    assert run(gpu_api, m=28672, n=17, k=8192) == 20
