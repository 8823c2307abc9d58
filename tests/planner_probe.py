"""Builds and loads tests/host_c/planner_probe.cpp: decisions of the planner that a plan does not name."""
import ctypes as C
import functools
import os
import shutil
import subprocess
import tempfile

import pytest

from zluda_amd import abi as K

BASE = 1 << 40   # (an aligned address; nothing is read from it)
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@functools.lru_cache(None)
def load():
    if shutil.which("g++") is None:
        pytest.skip("needs g++")
    with tempfile.TemporaryDirectory() as d:
        so = os.path.join(d, "planner_probe.so")
        subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-fvisibility=hidden", "-Wl,-Bsymbolic",
                        os.path.join(ROOT, "tests", "host_c", "planner_probe.cpp"), "-o", so], check=True)
        lib = C.CDLL(so)
    lib.probe_aux_sum_bytes.restype = C.c_uint64
    return lib


def aux_in_epilogue(problem, plan):
    return load().probe_aux_in_epilogue(C.byref(problem), C.byref(plan))


def aux_sum_bytes(problem, plan):
    return load().probe_aux_sum_bytes(C.byref(problem), C.byref(plan))


def lds_reads(problem, plan, cus):
    return load().probe_lds_reads(C.byref(problem), C.byref(plan), cus)


def planned(api, m, n, k, batch=1, epi=K.CUBLASLT_EPILOGUE_DEFAULT, ta=1, tb=0, workspace=32 << 20, family=0, variant=-1, cus=256):
    """bf16 matrices without padding at aligned addresses: status, problem, plan, what the problem points to"""
    p, plan, one, zero = K.zluda_gemm_problem(), K.zluda_gemm_plan(), C.c_float(1), C.c_float(0)
    for dst, rows, cols in ((p.a, k if ta else m, m if ta else k), (p.b, n if tb else k, k if tb else n), (p.c, m, n), (p.d, m, n)):
        dst.type, dst.order, dst.rows, dst.cols, dst.ld, dst.batch_count, dst.batch_stride = K.CUDA_R_16BF, K.CUBLASLT_ORDER_COL, rows, cols, rows, batch, rows * cols
    o = p.op
    o.compute_type, o.scale_type, o.transa, o.transb = K.CUBLAS_COMPUTE_32F, K.CUDA_R_32F, ta, tb
    o.epilogue, o.bias_type, o.epilogue_aux_type = epi, -1, -1
    o.epilogue_aux, o.epilogue_aux_ld, o.epilogue_aux_batch_stride, o.bias, o.bias_batch_stride = BASE, m, m * n, BASE, m
    p.A = p.B = p.C = p.D = BASE
    p.workspace, p.workspace_size = BASE, workspace
    status = api.zluda_gemm_plan_problem(C.byref(p), family, variant, cus, C.byref(plan))
    p.alpha, p.beta = C.addressof(one), C.addressof(zero)
    return status, p, plan, (one, zero)
