"""The plan of the batched product (qtip_amd/csrc/qtip_gemm_plan.h) compiled for the host, and cases that reach every form."""
import ctypes
import functools
import os
import subprocess
import tempfile

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CUS = 256
FEW, SHARED, ROWS = range(3)

SHIM = r"""
#include "qtip_gemm_plan.h"
using namespace qtip;
static void put(const GemmPlan& g, int* out) {
  const int v[] = {g.form, g.NB, g.RG, g.S, g.wl_per};
  for (int i = 0; i < 5; ++i) out[i] = v[i];
}
extern "C" int plan_of(int m, int k, int bits, int nb, int cus, int split, int fine, int* out) {
  const GemmParts p = gemm_plan(m, k, bits, nb, cus, split, fine);
  put(p.first, out);
  put(p.rest, out + 5);
  return p.m0;
}
extern "C" int pass_of(int m, int k, int bits, int left, int cus, int split, int fine) {
  return next_pass(m, k, bits, left, cus, split, fine);
}
extern "C" int slot_of(int m, int k, int bits, int nb, int split, int fine) { return plan_slot(m, k, bits, nb, split, fine); }
extern "C" void few_place(int lane, int batch, int k, int wl, int units, int nst, int last_half, uint32_t* out) {
  const FewPlace p = few_activations(lane, batch, k, wl, units, nst, last_half);
  out[0] = p.so;
  out[1] = p.vo;
}
"""


@functools.lru_cache(None)
def library():
    with tempfile.TemporaryDirectory() as d:
        src, lib = os.path.join(d, "shim.cpp"), os.path.join(d, "shim.so")
        with open(src, "w") as f:
            f.write(SHIM)
        subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-I", os.path.join(ROOT, "qtip_amd", "csrc"), src, "-o",
                        lib], check=True)
        return ctypes.CDLL(lib)


def plan(m, k, bits, batch, split=True, fine=True):
    """Matrix rows of the first launch, (form, NB, RG, S, wl_per) of it and of the second."""
    out = (ctypes.c_int * 10)()
    m0 = library().plan_of(m, k, bits, batch, CUS, int(split), int(fine), out)
    return m0, tuple(out[:5]), tuple(out[5:])


def launches(m, k, bits, batch, fine):
    """(form, NB, RG, cut into ranges, k ends inside a stage) of every launch of a product with scratch."""
    seen, left = set(), batch
    while left:
        nb = library().pass_of(m, k, bits, left, CUS, 1, int(fine))
        m0, *parts = plan(m, k, bits, nb, True, fine)
        for rows, (form, NB, RG, S, _) in zip((m0, m - m0), parts):
            if rows:
                inside = k % (64 * 8 // RG) != 0 if form == ROWS else k // 32 % 2 == 1
                seen.add((form, NB, RG, S > 1, inside))
        left -= nb
    return seen


# (m, k, rows), long sums or not, and a form among the launches: every kernel that is compiled, cut into ranges and not where a
# plan has both, with a last tile that is not full
FORMS = [
    (32, 512, 2, False, (FEW, 1, 1, False, False)), (96, 32, 3, False, (FEW, 1, 1, False, True)),
    (32, 2048, 13, False, (FEW, 1, 1, True, False)), (32, 1120, 7, False, (FEW, 1, 1, True, True)),
    (16416, 512, 5, False, (FEW, 1, 2, False, False)), (16416, 32, 2, False, (FEW, 1, 2, False, True)),
    (32, 8192, 15, False, (FEW, 1, 2, True, False)), (4992, 2080, 2, False, (FEW, 1, 2, True, True)),
    (96, 512, 17, False, (SHARED, 2, 2, False, False)), (32, 32, 31, False, (SHARED, 2, 2, False, True)),
    (544, 2048, 19, False, (SHARED, 2, 2, True, False)), (32, 2080, 23, False, (SHARED, 2, 2, True, True)),
    (96, 512, 37, False, (ROWS, 2, 2, False, False)), (32, 160, 33, False, (ROWS, 2, 2, False, True)),
    (32, 512, 150, False, (ROWS, 2, 2, True, False)), (32, 1120, 35, False, (ROWS, 2, 2, True, True)),
    (4992, 512, 200, False, (ROWS, 2, 4, False, False)), (32, 32, 39, False, (ROWS, 2, 4, False, True)),
    (1248, 2048, 200, False, (ROWS, 2, 4, True, False)), (2080, 1120, 250, False, (ROWS, 2, 4, True, True)),
    (5632, 512, 190, False, (ROWS, 4, 2, False, False)), (5632, 160, 190, False, (ROWS, 4, 2, False, True)),
    (3328, 512, 150, False, (ROWS, 4, 2, True, False)), (3328, 832, 150, False, (ROWS, 4, 2, True, True)),
    (8224, 512, 250, False, (ROWS, 4, 4, False, False)), (16416, 96, 100, False, (ROWS, 4, 4, False, True)),
    (2080, 2048, 250, False, (ROWS, 4, 4, True, False)), (4992, 1120, 200, False, (ROWS, 4, 4, True, True)),
    (16416, 512, 250, False, (ROWS, 8, 4, False, False)), (16416, 160, 250, False, (ROWS, 8, 4, False, True)),
    (2080, 4096, 250, False, (ROWS, 8, 4, True, False)), (8192, 1120, 150, False, (ROWS, 8, 4, True, True)),
    (16416, 3328, 70, False, (ROWS, 6, 8, True, False)),
    (1248, 512, 806, True, (ROWS, 2, 4, False, False)), (1248, 2048, 806, True, (ROWS, 4, 2, False, False)),
    (544, 8192, 400, True, (ROWS, 4, 2, True, False)), (544, 11008, 400, True, (ROWS, 4, 4, True, False)),
    (4992, 512, 806, True, (ROWS, 4, 8, False, False)), (4992, 32, 400, True, (ROWS, 4, 8, False, True)),
    (8224, 512, 1000, True, (ROWS, 6, 8, False, False)), (12288, 32, 650, True, (ROWS, 6, 8, False, True)),
    (2048, 8192, 1030, True, (ROWS, 6, 8, True, False)), (1248, 8192, 806, True, (ROWS, 8, 4, True, False)),
    (4096, 928, 1030, True, (ROWS, 8, 4, False, True)), (6144, 512, 2030, True, (ROWS, 8, 8, False, False)),
    (22016, 32, 509, True, (ROWS, 8, 8, False, True)), (4096, 28672, 806, True, (ROWS, 8, 8, True, False)),
    (8224, 2080, 2040, True, (ROWS, 2, 2, True, True)), (14336, 8192, 1400, True, (ROWS, 8, 4, True, False)),
]
# of the largest matrices, at 3 and 4 bits
SHARED_FORMS = [(22016, 4096, 15, False, (SHARED, 1, 2, False, False)), (8192, 11008, 13, False, (SHARED, 1, 2, True, False)),
                (32768, 4128, 13, False, (SHARED, 1, 2, False, True))]
