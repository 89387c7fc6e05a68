"""The host's choices in transformer_amd/csrc/plans.h, compiled for the tests: which grid, tile or split a size takes, so that
a test of a variant can assert that its sizes reach it."""
import ctypes
import functools
import os
import subprocess
import tempfile
from collections import namedtuple

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

_SOURCE = r"""
#include "plans.h"
using namespace mla;
extern "C" {
int one_per_cu(int64_t n_bh, int64_t n, int square) { return single_tiles_one_per_cu(TileGrid{n_bh, n, square != 0}); }
int two_per_cu(int64_t n_bh, int64_t n, int square) { return single_tiles_two_per_cu(TileGrid{n_bh, n, square != 0}); }
void nl(int64_t M, int64_t N, int64_t K, int64_t* o) {
  const NlPlan p = nl_plan(M, N, K);
  o[0] = p.kind, o[1] = p.n_nt, o[2] = p.n_wide, o[3] = p.n_rest;
}
void wg(int64_t M, int64_t N, int64_t K, int64_t* o) {
  const WgPlan p = wg_plan(M, N, K);
  o[0] = p.narrow, o[1] = p.S, o[2] = p.seg, o[3] = p.nt, o[4] = p.kt, o[5] = p.part_bytes;
}
}
"""

NlPlan = namedtuple("NlPlan", "kind n_nt n_wide n_rest")
WgPlan = namedtuple("WgPlan", "narrow S seg nt kt part_bytes")
NL_WIDE, NL_HALF, NL_SMALL = range(3)


@functools.lru_cache(None)
def _lib():
    with tempfile.TemporaryDirectory() as d:
        src, out = os.path.join(d, "plans.cpp"), os.path.join(d, "plans.so")
        with open(src, "w") as f:
            f.write(_SOURCE)
        subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-I",
                        os.path.join(ROOT, "transformer_amd", "csrc"), src, "-o", out], check=True)
        return ctypes.CDLL(out)


def _plan(name, n, *sizes):
    o = (ctypes.c_int64 * n)()
    getattr(_lib(), name)(*(ctypes.c_int64(s) for s in sizes), o)
    return list(o)


def norm_linear(M, N, K):
    return NlPlan(*_plan("nl", 4, M, N, K))


def weight_grad(M, N, K):
    return WgPlan(*_plan("wg", 6, M, N, K))


def single_tiles(n_bh, T, square=True):
    """(forward and dQ, dK/dV): whether causal attention of ``n_bh`` (b, h) of T rows runs a tile a workgroup."""
    n = ctypes.c_int64((T + 127) // 128)
    return (bool(_lib().two_per_cu(ctypes.c_int64(n_bh), n, int(square))),
            bool(_lib().one_per_cu(ctypes.c_int64(n_bh), n, int(square))))
