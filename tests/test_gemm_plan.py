"""How the batched product is cut into launches and where its waves read (qtip_gemm_plan.h), compiled for the host."""
import ctypes
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CUS = 256

SHIM = r"""
#include "qtip_gemm_plan.h"
using namespace qtip;
extern "C" void plan_of(int m, int k, int bits, int nb, int cus, int split, int* out) {
  const GemmParts p = gemm_plan(m, k, bits, nb, cus, split);
  const int v[] = {p.m0, p.first.NB, p.first.RG, p.first.S, p.first.wl_per, p.rest.NB, p.rest.RG, p.rest.S, p.rest.wl_per};
  for (int i = 0; i < 9; ++i) out[i] = v[i];
}
extern "C" void few_place(int lane, int batch, int k, int wl, int units, int nst, int last_half, uint32_t* out) {
  const FewPlace p = few_activations(lane, batch, k, wl, units, nst, last_half);
  out[0] = p.so;
  out[1] = p.vo;
}
"""


@pytest.fixture(scope="module")
def native(tmp_path_factory):
    d = tmp_path_factory.mktemp("gemm_plan")
    (d / "shim.cpp").write_text(SHIM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-Wno-unused-function", "-shared", "-fPIC", "-I",
                    os.path.join(ROOT, "qtip_amd", "csrc"), str(d / "shim.cpp"), "-o", str(d / "shim.so")], check=True)
    return ctypes.CDLL(str(d / "shim.so"))


def plan(native, m, k, bits, batch, split=True):
    out = (ctypes.c_int * 9)()
    native.plan_of(m, k, bits, batch, CUS, int(split), out)
    return out[0], tuple(out[1:5]), tuple(out[5:])


@pytest.mark.parametrize("k", [32, 64, 96, 832, 928, 2080, 4096, 28672])
@pytest.mark.parametrize("m", [32, 1056, 4096, 22016])
def test_few_rows_read_their_activations_only(native, m, k):
    """Every load of activations that gemm_few_kernel issues (the first whether or not the wave has a wave-load, then one for
    each) lies inside the batch, or has a lane offset out of range by itself and a scalar offset inside."""
    place = (ctypes.c_uint32 * 2)()
    nwl, odd = (k // 32 + 1) // 2, k // 32 % 2
    for batch in (2, 5, 16):
        _, (NB, RG, S, wl_per), _ = plan(native, m, k, 2, batch)
        assert NB == 0
        KS, size = 16 // RG, batch * k * 2
        for s in sorted({0, S - 1}):
            wl1 = min((s + 1) * wl_per, nwl)
            for ks in range(KS):
                first = s * wl_per + ks
                nst = max(0, -(-(wl1 - first) // KS))
                half = bool(odd and nst and first + KS * (nst - 1) == nwl - 1)
                for units in (1, 0):
                    for lane in range(64):
                        native.few_place(lane, batch, k, first, units, nst, int(half), place)
                        so, vo = place
                        for t in range(nst if units and nst else 1):
                            last = half and t == nst - 1 and lane >= 32  # (the kernel takes these lanes out of range)
                            assert so <= size
                            if vo < 0x7FFFFF00 and not (last and t):
                                assert so + vo + 32 + 16 <= size, (batch, s, ks, lane, t)
                            so += KS * 128
