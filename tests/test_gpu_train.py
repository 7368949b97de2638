"""Training-side parity: gradients of the differentiable forward against a float64 dense model."""
import numpy as np
import pytest
import torch

from oracle import qtip_oracle as O
from synth import make_layer

pytestmark = pytest.mark.gpu


def _matrix(n, transpose):
    return torch.from_numpy(O.hadamard_transform(np.eye(n), transpose=transpose).T.copy())  # y = M @ x


@pytest.mark.parametrize("m,k,bs", [(128, 256, 4), (192, 128, 1), (96, 160, 3)])
def test_gradients_of_input_and_sign_vectors(m, k, bs):
    from qtip_amd.codebook.bitshift import BitshiftLinear
    from qtip_amd.utils import matmul_had as mh
    dev = torch.device("cuda:0")
    K = 2
    L = make_layer(m, k, K, seed=m + k)
    tlut = torch.from_numpy(L["tlut"]).to(dev)
    mod = BitshiftLinear(16, 16, 16, K, 2, 9, "quantlut_sym", tlut=tlut, has_kernel=True)
    tr = torch.from_numpy(L["packed"]).to(dev)
    g = torch.Generator().manual_seed(1)
    x = torch.randn(bs, k, generator=g).half().to(dev).requires_grad_(True)
    SU = torch.from_numpy(L["SU"]).to(dev).requires_grad_(True)
    SV = torch.from_numpy(L["SV"]).to(dev).requires_grad_(True)
    hl, Kl = mh.get_hadK(k)
    hr, Kr = mh.get_hadK(m)
    y = mod(x, tr, SU, SV, hl, hr, Kl, Kr, 0, 8, mode="train-recons")
    w = torch.randn(bs, m, generator=g).to(dev)
    (y.float() * w).sum().backward()

    # float64 dense model of lib/codebook/bitshift.py:428-472
    W = torch.from_numpy(O.decode_kernel(L["packed"], L["tlut"], m, k, K).astype(np.float64))
    A, B = _matrix(k, True), _matrix(m, False)
    xd = x.detach().cpu().double().requires_grad_(True)
    SUd = SU.detach().cpu().double().requires_grad_(True)
    SVd = SV.detach().cpu().double().requires_grad_(True)
    yd = (((xd * SUd) @ A.T / 32) @ W.T @ B.T) * (SVd * 32)
    (yd * w.cpu().double()).sum().backward()

    def close(a, b, tol):
        a, b = a.detach().cpu().double(), b.detach().double()
        return float((a - b).abs().max() / b.abs().max()) <= tol

    assert close(y, yd, 1e-2)
    assert close(x.grad, xd.grad, 2e-2)
    assert close(SU.grad, SUd.grad, 2e-2)
    assert close(SV.grad, SVd.grad, 2e-2)
    assert x.grad.dtype == torch.float16 and SV.grad.dtype == torch.float32


def test_hadamard_function_gradient_is_the_transposed_transform():
    from qtip_amd.utils import matmul_had as mh
    dev = torch.device("cuda:0")
    for n in (256, 160, 96):  # 160 = 20 * 8 and 96 = 12 * 8: tables that are not symmetric
        had, K = mh.get_hadK(n)
        x = torch.randn(5, n, device=dev, requires_grad=True)
        y = mh.matmul_hadU_cuda(x, had, K)
        gy = torch.randn(5, n, device=dev)
        (y * gy).sum().backward()
        M = _matrix(n, False).float().to(dev)
        assert torch.allclose(y.detach(), x.detach() @ M.T, atol=1e-4)
        assert torch.allclose(x.grad, gy @ M, atol=1e-4)
        # and it inverts: hadUt(hadU(x)) = x
        z = mh.matmul_hadUt_cuda(y.detach(), had, K)
        assert torch.allclose(z, x.detach(), atol=1e-4)


def test_train_fixW_mode_matches_eval():
    from qtip_amd.linear.quantized_linear import QuantizedLinear
    dev = torch.device("cuda:0")
    m, k, K = 128, 256, 3
    L = make_layer(m, k, K, seed=9)
    outs = {}
    for mode in ("eval", "train-fixW"):
        lin = QuantizedLinear(k, m, 16, 16, 16, K, 2, 9, "quantlut_sym", mode=mode).to(dev)
        with torch.no_grad():
            lin.trellis.copy_(torch.from_numpy(L["packed"]))
            lin.tlut.copy_(torch.from_numpy(L["tlut"]))
            lin.SU.copy_(torch.from_numpy(L["SU"]))
            lin.SV.copy_(torch.from_numpy(L["SV"]))
        x = torch.randn(4, k, generator=torch.Generator().manual_seed(2)).half().to(dev)
        outs[mode] = lin(x).float()
    err = (outs["eval"] - outs["train-fixW"]).abs().max() / outs["eval"].abs().max()
    assert err < 2e-2


@pytest.mark.parametrize("rows,n", [(1, 32), (3, 96), (17, 256), (16, 260), (300, 1248), (2049, 4992)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
def test_scale_columns_gradients(rows, n, dtype):
    """Both gradients of x * s in one pass.  The column sum of r products errs by r 2^-24 times the sum of
    their magnitudes at most."""
    from qtip_amd.utils.matmul_had import scale_columns
    g = torch.Generator(device="cuda").manual_seed(rows + n)
    x = torch.randn(rows, n, generator=g, device="cuda").requires_grad_(True)
    s = torch.randn(n, generator=g, device="cuda").to(dtype).requires_grad_(True)
    gy = torch.randn(n, rows, generator=g, device="cuda").T  # a strided gradient
    y = scale_columns(x, s)
    gx, gs = torch.autograd.grad(y, (x, s), gy)
    assert torch.equal(y, x * s) and torch.equal(gx, gy * s) and gs.dtype == dtype
    prod = gy.double() * x.detach().double()
    tol = prod.abs().sum(0) * rows * 2.0**-24 + prod.sum(0).abs() * (2.0**-11 if dtype == torch.float16 else 0)
    assert bool(((gs.double() - prod.sum(0)).abs() <= tol).all())


def test_second_derivatives_pass_through_the_fused_steps():
    from qtip_amd.utils import matmul_had as mh
    n = 96
    had, K = mh.get_hadK(n)
    x = torch.randn(6, n, device="cuda", requires_grad=True)
    s = torch.randn(n, device="cuda", requires_grad=True)

    def grads(f):
        y = f(x, s)
        gx, gs = torch.autograd.grad((y**2).sum(), (x, s), create_graph=True)
        return torch.autograd.grad((gx**2).sum() + (gs**2).sum(), (x, s))

    fused = grads(lambda x, s: mh.hadU_cast(mh.scale_columns(x, s), had, K, True, 0.25, torch.float32))
    M = _matrix(n, True).float().cuda()
    plain = grads(lambda x, s: (x * s) @ M.T * 0.25)
    for a, b in zip(fused, plain):
        assert torch.allclose(a, b, rtol=1e-4, atol=1e-4 * float(b.abs().max()))


def _module(m, k, kernel):
    from qtip_amd.codebook.bitshift import BitshiftLinear
    from qtip_amd.utils import matmul_had as mh
    g = torch.Generator(device="cuda").manual_seed(m + k)
    rand = lambda *s: torch.randn(*s, generator=g, device="cuda")
    mod = BitshiftLinear(16, 16, 16, 2, 2, 9, "quantlut_sym", tlut=rand(512, 2).half(), has_kernel=kernel)
    tr = torch.randint(-32768, 32768, (m // 16 * k // 16, 32), dtype=torch.int16, generator=g, device="cuda")
    if not kernel:
        tr = mod.cb.unpack_trellis(tr, 256)
    (hl, kl), (hr, kr) = mh.get_hadK(k), mh.get_hadK(m)
    call = lambda *a: mod(a[0], tr, a[1], a[2], hl, hr, kl, kr, 0, 8, mode="train-recons")
    return call, [rand(20, k), rand(k).sign(), rand(m) / k**0.5], rand(3, 20, m)


def _gradients(call, leaves, gy, **kw):
    leaves = [t.detach().clone().requires_grad_() for t in leaves]
    return torch.autograd.grad(call(*leaves), leaves, gy, **kw)


def _close(a, b):  # (the same roundings to fp16 along either route, sums of a few hundred in another order)
    a, b = ([t.detach().double() for t in l] for l in (a, b))
    return all(float((p - q).norm() / q.norm()) <= 2.0**-10 for p, q in zip(a, b))


@pytest.mark.parametrize("kernel", [True, False])
def test_batched_gradients(kernel):
    """A batch of output gradients in one call is the calls one by one: nothing is launched on what has no memory."""
    call, leaves, gy = _module(256, 512, kernel)
    got = _gradients(call, leaves, gy, is_grads_batched=True)
    each = [_gradients(call, leaves, g) for g in gy]
    assert _close(got, [torch.stack(t) for t in zip(*each)])


def test_traced_and_fake_training_step():
    """The step of a module without a kernel can be traced, compiled and run on fake tensors, as it consists of torch's and
    registered operations then."""
    from torch._subclasses.fake_tensor import FakeTensorMode
    from torch.fx.experimental.proxy_tensor import make_fx
    call, leaves, gy = _module(256, 512, False)
    want = _gradients(call, leaves, gy[0])
    for backend in ("eager", "aot_eager"):
        torch._dynamo.reset()
        assert _close(_gradients(torch.compile(call, backend=backend), leaves, gy[0]), want)
    torch._dynamo.reset()
    graph = make_fx(call)(*[t.clone().requires_grad_() for t in leaves])
    assert sum("hadamard" in str(n.target) for n in graph.graph.nodes) == 2
    other = [t * 1.5 for t in leaves]
    assert _close([graph(*other)], [call(*other)])
    with FakeTensorMode(allow_non_fake_inputs=True) as mode:
        fake = [mode.from_tensor(t.detach().clone().requires_grad_()) for t in leaves]
        grads = torch.autograd.grad(call(*fake), fake, mode.from_tensor(gy[0]))
    assert [g.shape for g in grads] == [t.shape for t in leaves]


def test_step_over_a_batch_of_inputs():
    call, leaves, _ = _module(256, 512, False)
    x = torch.stack([leaves[0], 2 * leaves[0]])
    su = leaves[1].clone().requires_grad_()
    y = torch.func.vmap(lambda t: call(t, su, leaves[2]))(x)
    assert _close([y], [torch.stack([call(t, su, leaves[2]) for t in x])])


@pytest.mark.parametrize("rows", [250, 3000])
def test_kernel_product_of_rows_that_start_anywhere(rows):
    """BitshiftLinearKernelAG and rows_product of many rows take rows off 16 bytes and rows that are not contiguous, as a library
    product does: the values of an aligned copy."""
    from qtip_amd.codebook.bitshift import BitshiftLinear, BitshiftLinearKernelAG
    m, k = 256, 512
    g = torch.Generator(device="cuda").manual_seed(rows)
    tr = torch.randint(-32768, 32768, (m * k * 2 // 16,), dtype=torch.int16, generator=g, device="cuda")
    mod = BitshiftLinear(16, 16, 16, 2, 2, 9, "quantlut_sym", has_kernel=True,
                         tlut=torch.randn(512, 2, generator=g, device="cuda").half()).cuda()
    x = torch.randn(rows, k, generator=g, device="cuda").half()
    off = torch.empty(rows * k + 3, dtype=torch.float16, device="cuda")[3:].view(rows, k).copy_(x)
    wide = torch.stack([x, x], -1)[..., 0]
    tlut = mod._tlut16(x.device)
    with torch.no_grad():
        mod.cb.recons_lut()
        for form in (off, wide):
            a, b = (BitshiftLinearKernelAG.apply(t, tr, m, k, 16, 9, 2, 2, mod.cb.lut) for t in (x, form))
            assert torch.equal(a, b)
            assert torch.equal(mod.rows_product(x, tr, tlut, m, k), mod.rows_product(form, tr, tlut, m, k))
