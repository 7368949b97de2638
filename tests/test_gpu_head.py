"""GPU: the end of a decoded token (last boundary, final norm, output matrix) in one launch against float64."""
import pytest
import torch

from qtip_amd import ops

pytestmark = pytest.mark.gpu


def _operands(vocab, n, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    head = torch.randn(vocab, n, generator=g, device="cuda").half()
    x = (torch.randn(1, n, generator=g, device="cuda") * 3).half()
    w = (torch.rand(n, generator=g, device="cuda") + 0.5).half()
    return g, head, x, w


def _check(got, head, xn):
    """fp32 sums of n products (a lane's chain of n / 64 + 8, six levels over lanes), rounded to fp16 once."""
    n = head.shape[1]
    want = head.double() @ xn.reshape(-1).double()
    size = head.double().abs() @ xn.reshape(-1).double().abs()
    bound = want.abs() * 2.0**-11 + size * (n / 64 + 14) * 2.0**-24 * 1.001 + 2.0**-25
    assert ((got.double() - want).abs() <= bound).all()


# vocabularies around the rows of a workgroup (16) and of the chip (4096), rows around a load (512 values)
@pytest.mark.parametrize("vocab", (1, 15, 17, 4095, 4097, 9001))
@pytest.mark.parametrize("n", (8, 256, 504, 512, 520, 1000, 4096, 5120, 8184, 8192))
def test_head_of_a_residual_stream(vocab, n):
    _, head, x, w = _operands(vocab, n, vocab + n)
    xn = ops.rmsnorm(x, w, 1e-5)
    y = ops.token_head(head, x, w, 1e-5)
    _check(y, head, xn)
    assert torch.equal(ops.token_head(head, x, w, 1e-5, out_dtype=torch.float32), y.float())


@pytest.mark.parametrize("n", ops.RHT_IN_MATVEC_SIZES)
@pytest.mark.parametrize("nparts", (1, 2, 3, 5))
@pytest.mark.parametrize("vocab", (33, 5000))
def test_head_behind_the_last_boundary(n, nparts, vocab):
    """The residual stream is that of the boundary's own launch; the sum of its squares runs in another order, so that a
    value of the norm may be the neighbouring fp16 one: in 2-norm far below the rounding of the result, 2.8e-4."""
    g, head, x, w = _operands(vocab, n, n + nparts)
    parts = torch.randn(nparts, n, generator=g, device="cuda")
    post = torch.randn(n, generator=g, device="cuda") / 64
    scale = 32.0 * n**-0.5
    x_new, _ = ops.rht_chain(parts[:, None], post, scale, x, w, 1e-5, torch.ones(n, device="cuda").half(), 1.0)
    y = ops.token_head(head, x, w, 1e-5, parts, post, scale, torch.float32)
    want = head.double() @ ops.rmsnorm(x_new, w, 1e-5).reshape(-1).double()
    assert (y.double() - want).norm() <= 3.5e-4 * want.norm()


def test_zeros_stay_zeros_with_ragged_rows():
    """The values that pad a ragged row take no part, whatever the reciprocal of a zero norm is."""
    head = torch.randn(40, 520, device="cuda").half()
    y = ops.token_head(head, torch.zeros(1, 520, device="cuda").half(), torch.ones(520, device="cuda").half(), 1e-5)
    assert torch.equal(y, torch.zeros_like(y))


def test_refusals():
    head, x, w = torch.zeros(8, 64, device="cuda").half(), torch.zeros(64, device="cuda").half(), torch.ones(64, device="cuda").half()
    with pytest.raises(ValueError):
        ops.token_head(head, x[:32], w, 1e-5)
    with pytest.raises(ValueError):
        ops.token_head(head, x, w, 1e-5, torch.zeros(1, 64, device="cuda"), torch.zeros(64, device="cuda"), 1.0)
    with pytest.raises(ops._lib.QtipLibraryError):
        ops.token_head(torch.zeros(8, 60, device="cuda").half(), x[:60], w[:60].clone(), 1e-5)
