"""Which matrices a matvec cuts into half units (qtip_matvec_half.h), compiled for the host."""
import ctypes
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CUS = 256


@pytest.fixture(scope="module")
def half(tmp_path_factory):
    d = tmp_path_factory.mktemp("half")
    src, lib = d / "shim.cpp", d / "shim.so"
    src.write_text('#include "qtip_matvec_half.h"\nextern "C" int half(int bits, int left, int whole, int full, int S, int wl, int cus) '
                   '{ return qtip::half_units(bits, left, whole, full, S, wl, cus); }\n'
                   'extern "C" int apart(int bits, int left, int whole, int S, int wl, int cus) '
                   '{ return qtip::half_apart(bits, left, whole, S, wl, cus); }\n')
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-I", os.path.join(ROOT, "qtip_amd", "csrc"), str(src), "-o",
                    str(lib)], check=True)
    native = ctypes.CDLL(str(lib))

    def of(m, k, bits, S=1, cus=CUS, apart=False):
        full = cus // S
        blocks, wl = m // 32, ((k // 32 + 3) // 4 + S - 1) // S
        if apart:
            return native.apart(bits, blocks % full, blocks // full, S, wl, cus)
        return bool(native.half(bits, blocks % full, blocks // full, full, S, wl, cus))
    return of


# matrices that do not fill the chip and were slower in halves, by the wave-loads of a wave
SLOWER = ([(m, k, 4, 1) for m in (512, 1024, 2048, 4096) for k in (1024, 2048, 3072)] +
          [(m, k, 4, 1) for m in (2048, 4096) for k in (4096, 4608, 5120)] + [(4096, k, 4, 1) for k in (5504, 6144, 7168)] +
          [(2048, k, 4, 2) for k in (4096, 6144, 8192, 11008, 14336)] + [(1024, k, 4, 2) for k in (4096, 6144, 8192)] +
          [(1024, k, 4, 4) for k in (8192, 14336, 28672)] + [(4096, 4608, 3, 1), (4096, 14336, 3, 1), (2048, 28672, 3, 2)])
FASTER = ([(m, k, 4, 1) for m in (512, 1024, 2048) for k in (6144, 7168, 8192, 11008, 14336)] +
          [(4096, k, 4, 1) for k in (8192, 11008, 14336)] + [(2048, 28672, 4, 2), (1024, 14336, 4, 2), (1024, 49152, 4, 4)] +
          [(m, k, 3, 1) for m in (512, 1024, 2048) for k in (4608, 5120, 6144, 8192, 11008, 14336)] +
          [(4096, k, 3, 1) for k in (6144, 7168, 8192, 9216, 11008)] + [(1024, 28672, 3, 4)])


def test_matrices_are_cut_where_that_was_faster(half):
    assert not [c for c in SLOWER if half(*c)]
    assert not [c for c in FASTER if not half(*c)]


def test_two_bits_and_left_over_blocks(half):
    for m, k, S in ((4096, 1024, 1), (4096, 4096, 1), (32, 128, 1), (2048, 8192, 2), (1024, 49152, 4)):
        assert half(m, k, 2, S)
    # behind whole units: at 2 bits, which end on an even item, and at most half a round
    assert half(10240, 4096, 2) and half(12288, 4096, 2) and not half(12320, 4096, 2) and not half(10240, 6144, 2)
    assert not any(half(10240, 4096, bits) for bits in (3, 4))
    assert not any(half(m, 8192, bits) for m in (8192, 16384, 4128) for bits in (2, 3, 4))


def test_halves_lie_on_one_xcd_where_that_was_faster(half):
    apart = lambda m, k, bits, S=1: half(m, k, bits, S, apart=True)
    for m, k, S in ((512, 1024, 1), (2048, 4096, 1), (4096, 2048, 1), (1024, 8192, 1), (512, 28672, 2), (1024, 14336, 2), (256, 28672, 4)):
        assert apart(m, k, 2, S) == 0
    for m, k, S in ((2048, 11008, 1), (2048, 14336, 1), (4096, 5504, 1), (4096, 11008, 1), (1024, 28672, 2), (1024, 49152, 4)):
        assert apart(m, k, 2, S) == {1: 3, 2: 2, 4: 1}[S]
    for bits in (3, 4):
        assert [apart(512, 24576, bits, S) for S in (1, 2, 3, 4, 5, 8)] == [3, 2, 0, 1, 0, 0]
    assert apart(12288, 4096, 2) == apart(10240, 8192, 2) == 0  # behind whole units


def _units(left, lg):
    """(block, row half) of each workgroup of the half units, as matvec_kernel takes them."""
    r = 2 * left
    for w in range(r):
        paired = w < (r >> (lg + 1)) << (lg + 1)
        yield ((w >> (lg + 1)) << lg) + (w & ((1 << lg) - 1)) if paired else w >> 1, (w >> lg if paired else w) & 1


@pytest.mark.parametrize("lg", (0, 1, 2, 3))
def test_every_half_is_taken_once(lg):
    for left in range(1, 129):
        assert sorted(_units(left, lg)) == [(b, h) for b in range(left) for h in (0, 1)]
