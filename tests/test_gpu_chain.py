"""GPU: the layer boundary and the input transform in front of a matvec against float64, every size and bit width they are
compiled for, with as many partial results in front as are requested ahead (two) and more."""
import pytest
import torch

from qtip_amd import ops
from qtip_amd.utils.matmul_had import had_bits, sign_rows

pytestmark = pytest.mark.gpu


def _hadamard(n):
    h = torch.ones(1, 1, dtype=torch.float64, device="cuda")
    while h.shape[0] < n:
        h = torch.cat([torch.cat([h, h], 1), torch.cat([h, -h], 1)])
    return h


def _matrix(m, k, bits, g):
    packed = torch.randint(-32768, 32768, (m * k * bits // 16,), dtype=torch.int16, generator=g, device="cuda")
    tlut = torch.randn(512, 2, generator=g, device="cuda").half().reshape(-1)
    return packed, tlut, ops.decode(packed, tlut, m, k, bits).double()


def _close(parts, w, xt):
    """xt in fp16 (2**-11 of a value at most, and the neighbouring value where a sum in another order crosses over), sums in fp32."""
    want = w @ xt
    assert (parts.double().sum(0) - want).norm() <= 6e-4 * want.norm()


@pytest.mark.parametrize("bits", (2, 3, 4))
@pytest.mark.parametrize("k", ops.RHT_IN_MATVEC_SIZES)
@pytest.mark.parametrize("before", (1, 2, 3, 5))
def test_boundary_in_front_of_a_matvec(bits, k, before):
    g = torch.Generator(device="cuda").manual_seed(k + 10 * bits + before)
    packed, tlut, w = _matrix(96, k, bits, g)
    prev = torch.randn(before, k, generator=g, device="cuda")
    post = torch.randn(k, generator=g, device="cuda")
    res, norm, su = (torch.randn(k, generator=g, device="cuda").half() for _ in range(3))
    parts, x_new = ops.decompress_matvec_parts_chain(packed, tlut, 96, k, bits, prev, post, k**-0.5, res[None], norm, 1e-5, su,
                                                     k**-0.5)
    h = _hadamard(k)
    x = res.double() + (h @ prev.double().sum(0)) * k**-0.5 * post.double()
    # both terms of the sum and the sum itself are rounded to fp16
    assert (x_new.reshape(-1).double() - x).norm() <= 6e-4 * x.norm()
    xn = x_new.reshape(-1).double()
    n = (xn * (xn.square().mean() + 1e-5).rsqrt()).half().double()
    _close(parts, w, h @ ((n * norm.double()).half().double() * su.double()) * k**-0.5)


@pytest.mark.parametrize("bits", (2, 3, 4))
@pytest.mark.parametrize("k", ops.RHT_IN_MATVEC_SIZES)
def test_input_transform_in_front_of_a_matvec(bits, k):
    g = torch.Generator(device="cuda").manual_seed(k + bits)
    packed, tlut, w = _matrix(96, k, bits, g)
    x, su = (torch.randn(k, generator=g, device="cuda").half() for _ in range(2))
    parts = ops.decompress_matvec_parts_rht(packed, x, su, k**-0.5, tlut, 96, k, bits)
    _close(parts, w, _hadamard(k) @ (x.double() * su.double()) * k**-0.5)


# (k, table order, ranges): 64 and 32 columns, rows that do and do not fill a tile of 16 or a k tile of 32, A from 1 to 256,
# ranges that start inside a tile, buffers that do and do not reach into the table (from 224 rows of 64 on)
MIXES = ((5504, 172, 2), (11008, 172, 2), (11008, 172, 1), (13824, 108, 3), (14336, 28, 2), (14336, 28, 1), (7168, 28, 5),
         (5120, 20, 1), (4992, 156, 2), (3328, 52, 1), (1280, 20, 4), (1536, 12, 1), (1024, 1, 1), (16384, 1, 2), (128, 1, 1))


@pytest.mark.parametrize("bits,m", ((2, 96), (2, 3232), (3, 96), (4, 96)))
@pytest.mark.parametrize("k,order,ranges", MIXES)
@pytest.mark.parametrize("signs", (True, False))
def test_table_transform_in_front_of_a_matvec(k, order, ranges, m, bits, signs):
    """Against the transform's own launch in fp32.  A sign vector of other values than +-1 takes three planes."""
    g = torch.Generator(device="cuda").manual_seed(k + 10 * bits + ranges)
    packed, tlut, w = _matrix(m, k, bits, g)
    x, su = (torch.randn(k, generator=g, device="cuda").half() for _ in range(2))
    if signs:
        su = torch.where(su < 0, -1.0, 1.0).half()
    hb = had_bits(None, order, True, "cuda") if order > 1 else None
    rows = sign_rows(hb, order, k // ops.matvec_mix_columns(k, order, ranges) // order, "cuda")
    parts = ops.decompress_matvec_parts_mix(packed, x, su, k**-0.5, rows, order, tlut, m, k, bits, ranges)
    assert parts.shape == (ranges, m)
    xt = ops.rht((x.float() * su.float())[None], order=order, had_bits=hb, scale=k**-0.5, out_dtype=torch.float32)
    _close(parts, w, xt.reshape(-1).double())


def test_table_transform_refusals():
    """Fewer than 32 columns, more than 256 rows of 64, a range past the staging area, k inside a wave-load."""
    for k, order, ranges in ((832, 52, 1), (28672, 28, 4), (16384, 1, 1), (4800, 150, 1), (4096 + 32, 129, 1), (11008, 172, 0)):
        assert ops.matvec_mix_columns(k, order, ranges) == 0
    z = torch.zeros(11008, device="cuda").half()
    packed, tlut, _ = _matrix(32, 11008, 2, torch.Generator(device="cuda").manual_seed(0))
    with pytest.raises(ValueError):
        ops.decompress_matvec_parts_mix(packed, z, z, 1.0, torch.zeros(171, 8, dtype=torch.int32, device="cuda"), 172, tlut, 32, 11008, 2)


# row blocks that fill less than half of the chip: pairs of halves on one XCD and side by side, one to four ranges of k
@pytest.mark.parametrize("bits", (2, 3, 4))
@pytest.mark.parametrize("m,k,ranges", ((32, 4224, 1), (288, 8192, 1), (4096, 4608, 1), (256, 8192, 2), (160, 8320, 3), (1024, 16384, 4)))
def test_half_units_of_matrices_that_do_not_fill_the_chip(m, k, ranges, bits):
    """Every row once: sums of k exact products in fp32 against float64 (a chain of k / 64 on the matrix cores and 16 waves)."""
    g = torch.Generator(device="cuda").manual_seed(m + k + bits)
    packed, tlut, w = _matrix(m, k, bits, g)
    x = torch.randn(k, generator=g, device="cuda").half()
    got = ops.decompress_matvec_parts(packed, x, tlut, m, k, bits, ranges).double().sum(0)
    want, size = w @ x.double(), w.abs() @ x.double().abs()
    assert ((got - want).abs() <= size * (k / 64 + 24) * 2.0**-24).all()
    if ranges == 1:
        one = ops.decompress_matvec(packed, x, tlut, m, k, bits).reshape(-1).double()
        assert ((one - want).abs() <= size * (k / 64 + 24) * 2.0**-24).all()
