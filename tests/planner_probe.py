"""Builds and loads tests/host_c/planner_probe.cpp: decisions of the planner that a plan does not name."""
import ctypes as C
import functools
import os
import shutil
import subprocess
import tempfile

import pytest

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
