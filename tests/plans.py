"""The launch plans of csrc/plans.h (host arithmetic) as ctypes functions: compiled with the host
compiler behind a few C entry points, for the tests of launchers without a device."""
import ctypes
import os
import subprocess
import tempfile

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "wan2-ti2v-5b_amd", "csrc")
SHIM = """
#include "plans.h"
using namespace wan;
extern "C" {
void attention(int B, int H, int Lq, int keys, int cus, size_t scratch, int* out, size_t* bytes) {
  const SplitPlan p = split_plan(B, H, Lq, keys, cus, scratch);
  out[0] = p.from; out[1] = p.blocks; out[2] = p.splits;
  *bytes = p.bytes;
}
void rows(long long blocks, int threads, unsigned* out) {
  const RowGrid g = row_grid(blocks, threads);
  out[0] = g.x; out[1] = g.y;
}
int threads(int W) { return row_threads(W); }
void gemm(int M, int N, int K, long long ldx, int cus, size_t scratch, int* out, size_t* bytes) {
  const GemmPlan p = gemm_plan(M, N, K, ldx, cus, scratch);
  out[0] = p.rows; out[1] = p.from; out[2] = p.rest; out[3] = p.splits;
  *bytes = gemm_plan_bytes(p);
}
}
"""


def load() -> ctypes.CDLL:
    with tempfile.TemporaryDirectory() as d:
        src, lib = os.path.join(d, "plans.cpp"), os.path.join(d, "plans.so")
        with open(src, "w") as f:
            f.write(SHIM)
        subprocess.run([os.environ.get("CXX", "g++"), "-std=c++17", "-O1", "-Wall", "-Werror", "-shared", "-fPIC",
                        "-I", CSRC, src, "-o", lib], check=True)
        return ctypes.CDLL(lib)


def gemm(lib, M, N, K, ldx=None, cus=256, scratch=0):
    """(tile rows, whole tiles before the split, split tiles, parts of each, scratch bytes)"""
    out, n = (ctypes.c_int * 4)(), ctypes.c_size_t()
    lib.gemm(M, N, K, ctypes.c_longlong(K if ldx is None else ldx), cus, ctypes.c_size_t(scratch), out, ctypes.byref(n))
    return (*out, n.value)


def rows(lib, blocks, threads):
    """(workgroups along x, along y)"""
    out = (ctypes.c_uint * 2)()
    lib.rows(ctypes.c_longlong(blocks), threads, out)
    return tuple(out)


def attention(lib, B, H, Lq, keys, cus=256, scratch=1 << 40):
    """(whole blocks, split blocks, parts of each, scratch bytes)"""
    out, n = (ctypes.c_int * 3)(), ctypes.c_size_t()
    lib.attention(B, H, Lq, keys, cus, ctypes.c_size_t(scratch), out, ctypes.byref(n))
    return (*out, n.value)
