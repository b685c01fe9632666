"""csrc/sparse_steps.h compiled for the host: a sparse plan's steps and where launches keep them.  Helper module, not
collected by pytest."""

from __future__ import annotations

import ctypes as C
import functools
import os
import subprocess
import tempfile

import numpy as np

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "instantmimic_amd", "csrc")

SOURCE = r"""
#include "sparse_steps.h"
using namespace im;
extern "C" {
// tables LP .. BJ, then FL .. RK by their places; out: the words (null: their number), counts[0 .. 1] the steps
int steps(const int32_t *const *tables, const int *sizes, int nlevels, uint32_t *out, int *counts) {
  im_sparse_plan pl;
  pl.nlevels = nlevels;
  for (int i = 0; i < NTABLES; ++i) pl.table[i].assign(tables[i], tables[i] + sizes[i]);
  const WaveSteps w = wave_steps(pl);
  counts[0] = w.nfactor, counts[1] = w.nbackward;
  if (out) std::copy(w.words.begin(), w.words.end(), out);
  return (int)w.words.size();
}
long init_bytes(const int *s, int njmax) { return (long)init_lds_bytes({s[0], s[1], s[2], s[3]}, njmax); }
void update(const int *s, int nworld, int ncu, long *out) {
  const SparseUpdate u = sparse_update_layout({s[0], s[1], s[2], s[3]}, nworld, ncu);
  out[0] = u.waves, out[1] = u.staged_rows, out[2] = (long)u.lds;
}
void resident(const int *s, int njmax, int tables, int kept, int nworld, int ncu, long *out) {
  const int waves[] = {16, 12, 8, 4};
  const SparseResident r = sparse_resident_layout({s[0], s[1], s[2], s[3]}, njmax, tables, kept, waves, 4, nworld, ncu);
  out[0] = r.waves, out[1] = r.staged_rows, out[2] = r.step_words, out[3] = (long)r.lds, out[4] = r.per_cu;
}
}
"""

TABLES = ["SH_LP", "SH_LT", "SH_ES", "SH_EC", "SH_RP", "SH_RAB", "SH_RKL", "SH_ORIG", "SH_BL", "SH_BS", "SH_BI", "SH_BJ",
          "SH_PM", "SH_SA", "SH_SB", "SH_SM", "SH_PAIR", "SH_FL", "SH_FR", "SH_RS", "SH_RKP", "SH_RK"]  # fmt: skip


@functools.lru_cache(maxsize=None)
def lib():
    with tempfile.TemporaryDirectory() as tmp:
        src, out = os.path.join(tmp, "layout.cpp"), os.path.join(tmp, "layout.so")
        with open(src, "w") as f:
            f.write(SOURCE)
        subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-fPIC", "-shared", "-I", CSRC, src, "-o", out], check=True)
        so = C.CDLL(out)
    so.init_bytes.restype = C.c_long
    return so


class Layout:
    """Of one plan (``SparseHessianPlan``)."""

    def __init__(self, plan, nv: int, terms: int):
        t = [np.ascontiguousarray(plan.tables[k], np.int32) for k in TABLES]
        ptr = (C.c_void_p * len(t))(*(a.ctypes.data for a in t))
        size = (C.c_int * len(t))(*(len(a) for a in t))
        counts = (C.c_int * 2)()
        n = lib().steps(ptr, size, plan.levels, None, counts)
        self.words = np.zeros(n, np.uint32)
        lib().steps(ptr, size, plan.levels, C.c_void_p(self.words.ctypes.data), counts)
        self.nfactor, self.nbackward = counts
        up = lambda x: (x + 3) & ~3  # noqa: E731
        self.nv, self.terms = nv, terms
        self.sizes = (C.c_int * 4)(nv, plan.nslots, n, sum(up(len(plan.tables[k])) for k in TABLES[-5:]) + up(nv))

    def init_bytes(self, njmax: int) -> int:
        return lib().init_bytes(self.sizes, njmax)

    def update(self, nworld: int, ncu: int = 256):
        """(worlds per workgroup, staged rows, bytes)"""
        out = (C.c_long * 3)()
        lib().update(self.sizes, nworld, ncu, out)
        return tuple(out)

    def resident(self, njmax: int, nworld: int, ncu: int = 256):
        """(worlds per workgroup, staged rows, words of steps in LDS, bytes, workgroups of a CU)"""
        out = (C.c_long * 5)()
        lib().resident(self.sizes, njmax, (self.terms + self.nv + 4) & ~3, 4 * self.nv + 4 * njmax, nworld, ncu, out)
        return tuple(out)
