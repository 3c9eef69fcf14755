"""The tiled GEMM's plan (csrc/gemm_plan.cpp), compiled for the host: which path a shape takes."""
import ctypes
import os
import shutil
import subprocess
import tempfile
from collections import namedtuple

import pytest

from supersonic_amd import build as B

Plan = namedtuple("Plan", "bm bn ks split_tiles tail bytes us")
SHIM = r"""
#include "gemm_plan.hpp"
extern "C" void plan_of(int m, int k, int nseg, const int* n, int batch, size_t room, double* o) {
    const ssa::GemmPlan p = ssa::gemm_plan(m, k, nseg, n, batch, room);
    o[0] = p.bm; o[1] = p.bn; o[2] = p.ks; o[3] = p.split_tiles; o[4] = p.tail; o[5] = static_cast<double>(p.bytes); o[6] = p.us;
}
extern "C" double stream_of(int m, int k, long ncb, int staged) { return ssa::stream_us(m, k, ncb, staged != 0); }
"""
_lib = None


def _load():
    global _lib
    if _lib is None:
        cxx = shutil.which("g++") or shutil.which("c++")
        if not cxx:
            pytest.skip("no host C++ compiler")
        d = tempfile.mkdtemp()
        try:
            src, so = os.path.join(d, "shim.cpp"), os.path.join(d, "shim.so")
            with open(src, "w") as f:
                f.write(SHIM)
            subprocess.run([cxx, "-std=c++17", "-O1", "-shared", "-fPIC", "-I", B.CSRC, src,
                            os.path.join(B.CSRC, "gemm_plan.cpp"), "-o", so], check=True)
            _lib = ctypes.CDLL(so)
            _lib.stream_of.restype = ctypes.c_double
        finally:
            shutil.rmtree(d, ignore_errors=True)
    return _lib


def stream_us(m, k, ncb):
    return _load().stream_of(m, k, ctypes.c_long(ncb), int(m <= 16 and m * k <= 32768))


def gemm_plan(m, k, n, batch=1, room=2 ** 62):
    lib = _load()
    o = (ctypes.c_double * 7)()
    lib.plan_of(m, k, len(n), (ctypes.c_int * len(n))(*n), batch, ctypes.c_size_t(room), o)
    return Plan(*(int(x) for x in o[:6]), o[6])
