"""GPU: the layer boundary and the input transform in front of a matvec against float64, every size and bit width they are
compiled for, with as many partial results in front as are requested ahead (two) and more."""
import pytest
import torch

from qtip_amd import ops

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
