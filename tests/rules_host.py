"""The launch rules of csrc/fhog_grid.h, built with the host compiler.

load(dir) returns a ctypes library of C wrappers around the rules, which are plain
C++. Causal codes are the C ABI's; CUS is the number of compute units that the tests
give them.
"""

from __future__ import annotations

import ctypes
import pathlib
import shutil
import subprocess

import pytest

CSRC = pathlib.Path(__file__).resolve().parent.parent / "flash-hog_amd" / "csrc"
CUS = 256

WRAPPERS = r"""
#include "fhog_grid.h"
using fhog::Mask;
static Mask mask(int causal, int nq, int nk) { return Mask{causal != 0, nq, nk, causal == 2 ? nk - nq : 0}; }
extern "C" {
int fwd_pair(int c, int nq, int nk, int np, int d, int cus) { return fhog::fwd_pair_rule(mask(c, nq, nk), np, d, cus); }
int bwd_pair(int c, int nq, int nk, int np, int cus) { return fhog::bwd_pair_rule(mask(c, nq, nk), np, cus); }
int bwd_k64(int c, int nq, int nk, int np, int cus) { return fhog::bwd_k64_rule(mask(c, nq, nk), np, cus); }
int bwd_qpair(int c, int nq, int nk, int np, int d, int cus) { return fhog::bwd_qpair_rule(mask(c, nq, nk), np, d, cus); }
int bwd_q64(int c, int nq, int nk, int np, int cus) { return fhog::bwd_q64_rule(mask(c, nq, nk), np, cus); }
int bwd_waves(int c, int nq, int nk, int np, int d, int bytes, int cus) {
  return fhog::bwd_pair_waves(mask(c, nq, nk), np, d, bytes, cus);
}
int stage1_fused(int c, int nq, int nk) { return fhog::stage1_fused_rule(mask(c, nq, nk)); }
int stage1_pairs(int c, int nq, int nk, int np, int cus) { return fhog::stage1_pairs_rule(mask(c, nq, nk), np, cus); }
int stage1_qpair(int c, int nq, int nk, int np, int cus) { return fhog::stage1_qpair_rule(mask(c, nq, nk), np, cus); }
int stage2_pair(int c, int nq, int nk, int np, int cus) { return fhog::stage2_pair_rule(mask(c, nq, nk), np, cus); }
int q32_deal(int c, int nq, int nk, int np, int cus) { return fhog::q32_deal_rule(mask(c, nq, nk), np, cus); }
double q32_folded(int c, int nq, int nk, int np, int cus) { return fhog::q32_load(mask(c, nq, nk), np, cus).folded; }
double q32_dealt(int c, int nq, int nk, int np, int cus) { return fhog::q32_load(mask(c, nq, nk), np, cus).dealt; }
int pairing(int c, int nq, int nk, int nb, int np, int resident, int waves) {
  return fhog::block_pairing(mask(c, nq, nk), nb, np, resident, waves);
}
long sees(int c, int nq, int nk, int rows, int keys) { return fhog::blocks_see(mask(c, nq, nk), rows, keys != 0); }
int folded_percent(int c, int nq, int nk) { return fhog::folded_percent(mask(c, nq, nk)); }
int near_square(int c, int nq, int nk, int parts) { return fhog::near_square(mask(c, nq, nk), parts); }
int fold(int c, int nb, int np, int cus) { return fhog::fold_rank(c != 0, nb, np, cus); }
int chunk(int np, int nranks, int resident) { return fhog::grid_chunk(np, nranks, resident); }
}
"""


def load(directory):
    cxx = shutil.which("g++") or shutil.which("c++") or shutil.which("clang++")
    if cxx is None:
        pytest.skip("no host C++ compiler")
    (directory / "rules.cpp").write_text(WRAPPERS)
    cmd = [cxx, "-std=c++20", "-O1", "-Wall", "-Werror", "-shared", "-fPIC", f"-I{CSRC}", str(directory / "rules.cpp"),
           "-o", str(directory / "rules.so")]
    subprocess.run(cmd, check=True)
    lib = ctypes.CDLL(str(directory / "rules.so"))
    lib.sees.restype = ctypes.c_long
    lib.q32_folded.restype = lib.q32_dealt.restype = ctypes.c_double
    return lib


def stage2_order(r, causal, nq, nk, npairs):
    """`pairs` of bwdbwd_k_kernel: 128-key blocks, two workgroups per CU."""
    return r.pairing(causal, nq, nk, (nk + 127) // 128, npairs, 2 * CUS, 2)


def one_wave_order(r, causal, nq, nk, n, npairs):
    """`pairs` of the kernels with 256-row blocks of the n queries or keys, one workgroup per CU."""
    return r.pairing(causal, nq, nk, (n + 255) // 256, npairs, CUS, 1)
