"""Transforms of many rows on the matrix cores against float64 matrices, at the edges of their tiling."""
import numpy as np
import pytest
import scipy.linalg
import torch

pytestmark = pytest.mark.gpu


def _transform(x, n, transpose):
    """sqrt(n) * (H_K (x) H_p) x in float64 on the device (x: float64 rows)."""
    from qtip_amd.utils.matmul_had import get_hadK
    had, K = get_hadK(n)
    p = n // K
    z = x.view(-1, K, p) @ torch.from_numpy(scipy.linalg.hadamard(p).astype(np.float64)).cuda()
    if had is not None:
        h = had.double().cuda()
        z = (h.T if transpose else h) @ z
    return z.reshape(-1, n)


# power-of-two parts of 8 to 2048: one to sixteen rows per pass, table orders that fill their k tiles and
# ones that leave 4 to 28 padding rows, one and two slices (53248, 57344), a workgroup of one to eight tiles
@pytest.mark.parametrize("n", [256, 832, 928, 1120, 1248, 3328, 5120, 10240, 11008, 12288, 14336, 16384, 22016, 28672,
                               53248, 57344])
@pytest.mark.parametrize("rows", [24, 37])
def test_rows_against_float64(n, rows):
    _check_rows(n, rows)


# short rows, which take the matrix form from more rows on: either side of the line for fp16 and for fp32 values
@pytest.mark.parametrize("n,rows", [(64, 515), (64, 519), (64, 1107), (64, 1131), (256, 130), (256, 160), (256, 290),
                                    (512, 147), (768, 48), (768, 103), (832, 61), (1024, 81), (1248, 13), (1248, 41),
                                    (1280, 69), (2240, 17), (2240, 39), (3072, 35), (3456, 40), (4992, 19)])
def test_short_rows_against_float64(n, rows):
    _check_rows(n, rows)


# few rows, whose passes are shared by several workgroups: one pass and many, shares that do not divide a pass's waves
@pytest.mark.parametrize("n,rows", [(928, 9), (1248, 7), (4992, 5), (5504, 5), (10240, 7), (11008, 3), (11008, 130),
                                    (13824, 5), (14336, 67), (22016, 2), (28672, 6), (28672, 100), (57344, 11)])
def test_few_rows_against_float64(n, rows):
    _check_rows(n, rows)


def test_rows_in_place():
    """A transform over its own input, which workgroups that share a row cannot be given."""
    from qtip_amd import _lib
    from qtip_amd.utils.matmul_had import get_hadK, had_bits
    n, rows = 11008, 20
    had, K = get_hadK(n)
    x = torch.randn(rows, n, generator=torch.Generator(device="cuda").manual_seed(0), device="cuda").half()
    ref = _transform(x.double(), n, True) * n**-0.5
    bits = had_bits(had, K, True, "cuda")
    st = torch.cuda.current_stream().cuda_stream
    assert _lib.lib().qtip_rht(x.data_ptr(), _lib.QTIP_F16, x.data_ptr(), _lib.QTIP_F16, 1, rows, n, K, bits.data_ptr(), None, None,
                               n**-0.5, st) == 0
    assert float((x.double() - ref).abs().max()) <= 1e-3 * float(ref.abs().max())  # fp16 results


def _check_rows(n, rows):
    from qtip_amd import ops
    from qtip_amd.utils.matmul_had import get_hadK, had_bits
    had, K = get_hadK(n)
    g = torch.Generator(device="cuda").manual_seed(n + rows)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda")
    for dt_in, dt_out, transpose, pre_kind, scale_in in (
            (torch.float16, torch.float16, True, "sign", 1.0), (torch.float16, torch.float32, False, "real", 1.0),
            (torch.float32, torch.float16, True, "sign", 1.0), (torch.float32, torch.float32, False, "real", 1e-6),
            (torch.float16, torch.float32, False, None, 1.0), (torch.float32, torch.float32, True, None, 1e6)):
        x = (rnd(rows, n) * scale_in).to(dt_in)
        pre = post = None
        if pre_kind:
            pre = torch.sign(rnd(n) + 1e-5)
            pre = (pre if pre_kind == "sign" else pre * (0.5 + torch.rand(n, generator=g, device="cuda"))).half()
            post = rnd(n)
        got = ops.rht(x, order=K, had_bits=had_bits(had, K, transpose, "cuda") if K > 1 else None, pre=pre, post=post,
                      out_dtype=dt_out)
        ref = _transform(x.double() * (1 if pre is None else pre.double()), n, transpose) * n**-0.5
        ref = ref * (1 if post is None else post.double())
        # exact products, fp32 sums of n terms (n * 2^-24 in the worst case, sqrt(n) of it in these) and fp16 results
        tol = 1e-3 if dt_out == torch.float16 else 1e-5
        assert got.dtype == dt_out and float((got.double() - ref).abs().max()) <= tol * float(ref.abs().max())


@pytest.mark.parametrize("n", [928, 4096, 11008, 28672, 57344])
@pytest.mark.parametrize("sign", [True, False])
def test_rows_with_prologue_and_residual(n, sign):
    """The element-wise neighbours folded into the many-row form: same fp16 rounding points as the
    single-row forms, whose sums run in another order (an fp16 ulp)."""
    from qtip_amd import ops
    from qtip_amd.utils.matmul_had import get_hadK, had_bits
    had, K = get_hadK(n)
    rows = 29
    g = torch.Generator(device="cuda").manual_seed(n)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda")
    bits = had_bits(had, K, True, "cuda") if K > 1 else None
    pre = torch.sign(rnd(n) + 1e-5)
    pre = (pre if sign else pre * 1.25).half()
    w = (1 + 0.1 * rnd(n)).half()
    x, gu, res = rnd(rows, n).half(), rnd(rows, 2 * n).half(), rnd(rows, n).half()
    kw = dict(order=K, had_bits=bits, pre=pre, out_dtype=torch.float16)
    close = lambda a, b: float((a.float() - b.float()).abs().max()) <= 2e-3 * float(b.float().abs().max())
    if n <= 16384:  # the single-row form of the norm holds the vector in registers
        got = ops.rht(x, pre_mode=ops.PRE_RMSNORM, norm_weight=w, eps=1e-5, **kw)
        one = torch.cat([ops.rht(x[i:i + 1], pre_mode=ops.PRE_RMSNORM, norm_weight=w, eps=1e-5, **kw) for i in (0, 17, 28)])
        assert close(got[[0, 17, 28]], one)
    got = ops.rht(gu, pre_mode=ops.PRE_SILU_MUL, **kw)
    one = torch.cat([ops.rht(gu[i:i + 1], pre_mode=ops.PRE_SILU_MUL, **kw) for i in (0, 17, 28)])
    assert close(got[[0, 17, 28]], one)
    got = ops.rht(x, residual=res, **kw)
    one = torch.cat([ops.rht(x[i:i + 1], residual=res[i:i + 1], **kw) for i in (0, 17, 28)])
    assert close(got[[0, 17, 28]], one)


@pytest.mark.parametrize("n", [11008, 832, 14336])
def test_infinities_and_nan_stay_what_they_are(n):
    """One infinity in a row of fp32 values makes every element of its transform infinite (a sum of it and finite
    values), with the signs the single-row form gives; a NaN fills its own row only."""
    from qtip_amd import ops
    from qtip_amd.utils import matmul_had as mh
    had, order = mh.get_hadK(n)
    bits = mh.had_bits(had, order, False, "cuda")
    x = torch.randn(48, n, generator=torch.Generator().manual_seed(n)).cuda()
    x[3, 7] = float("inf")
    x[20, n - 1] = -float("inf")
    x[41, 100] = float("nan")
    y = ops.rht(x, order=order, had_bits=bits)
    for r in (3, 20):
        assert torch.equal(y[r:r + 1], ops.rht(x[r:r + 1].clone(), order=order, had_bits=bits))
        assert bool(torch.isinf(y[r]).all())
    bad = ~torch.isfinite(y).all(1)
    assert torch.isnan(y[41]).all() and bad.nonzero().flatten().tolist() == [3, 20, 41]


@pytest.mark.parametrize("n,K", [(688, 172), (624, 156), (344, 172), (108, 108), (1200, 300), (2048, 512)])
@pytest.mark.parametrize("rows", [96, 300])
def test_orders_the_matrix_form_does_not_take(n, K, rows, monkeypatch):
    """Large orders over parts of fewer than 8 points, and orders above 256, run as library products from the rows on
    from which those are faster; either route against float64: exact products, fp32 sums of n terms."""
    from qtip_amd.utils import matmul_had as mh
    g = torch.Generator(device="cuda").manual_seed(n + rows)
    had = mh.get_hadK(n)[0].cuda() if K < 256 else torch.randint(0, 2, (K, K), generator=g, device="cuda").float() * 2 - 1
    taken, many = [], mh.rht_many_rows
    monkeypatch.setattr(mh, "rht_many_rows", lambda *a, **k: taken.append(1) or many(*a, **k))
    h64 = torch.from_numpy(scipy.linalg.hadamard(n // K).astype(np.float64)).cuda()
    for dtype, tol in ((torch.float32, 1e-5), (torch.float16, 2.0**-10)):
        x = torch.randn(n, rows, generator=g, device="cuda").to(dtype).T  # (no contiguous rows)
        for transpose in (False, True):
            z = (had.T if transpose else had).double() @ (x.double().reshape(rows, K, n // K) @ h64)
            ref = z.reshape(rows, n) / n**0.5
            taken.clear()
            outs = [mh.matmul_hadU_cuda(x, had, K, transpose), mh.hadU_cast(x, had, K, transpose, 1.0, dtype)]
            assert len(taken) == (2 if rows * K >= 24000 else 0)
            for y in outs:
                assert y.dtype == dtype and float((y.double() - ref).abs().max()) <= tol * float(ref.abs().max())


def test_projection_whose_orders_the_matrix_form_does_not_take(monkeypatch):
    """A dense-route projection with 172 * 4 outputs and 156 * 4 inputs: 300 rows at once against 50 at a time, which
    take the kernel (fp16 activations and results: another order of sums moves some by a rounding)."""
    from qtip_amd.codebook import bitshift
    from qtip_amd.utils.matmul_had import get_hadK
    m, k, rows = 688, 624, 300
    g = torch.Generator(device="cuda").manual_seed(1)
    tr = torch.randint(-32768, 32768, (m // 16 * k // 16, 32), dtype=torch.int16, generator=g, device="cuda")
    mod = bitshift.BitshiftLinear(16, 16, 16, 2, 2, 9, "quantlut_sym", has_kernel=False,
                                  tlut=torch.randn(512, 2, generator=g, device="cuda").half())
    su = torch.randint(0, 2, (k,), generator=g, device="cuda").half() * 2 - 1
    sv = torch.randn(m, generator=g, device="cuda")
    x = torch.randn(rows, k, generator=g, device="cuda").half()
    (hl, kl), (hr, kr) = get_hadK(k), get_hadK(m)
    taken, many = [], bitshift.rht_many_rows
    monkeypatch.setattr(bitshift, "rht_many_rows", lambda *a, **kw: taken.append(1) or many(*a, **kw))
    call = lambda t: mod(t, tr, su, sv, hl, hr, kl, kr, 0, 8)
    with torch.no_grad():
        want = torch.cat([call(x[i:i + 50]) for i in range(0, rows, 50)])
        assert not taken
        got = call(x)
    assert len(taken) == 2 and float((got.float() - want.float()).norm() / want.float().norm()) <= 2.0**-10


@pytest.mark.parametrize("rows", [150, 300])
def test_kernel_projection_of_a_callers_large_order(rows, monkeypatch):
    """A table of order 300 from the caller on both sides of a kernel-packed projection: its transforms run as library products, as
    they do without a kernel; 50 rows at a time take the kernel's (another order of sums, fp16 activations and results)."""
    from qtip_amd.codebook import bitshift
    m = k = 4800
    g = torch.Generator(device="cuda").manual_seed(2)
    tr = torch.randint(-32768, 32768, (m * k * 2 // 16,), dtype=torch.int16, generator=g, device="cuda")
    mod = bitshift.BitshiftLinear(16, 16, 16, 2, 2, 9, "quantlut_sym", has_kernel=True,
                                  tlut=torch.randn(512, 2, generator=g, device="cuda").half())
    had = torch.randint(0, 2, (300, 300), generator=g, device="cuda").float() * 2 - 1
    su = torch.randint(0, 2, (k,), generator=g, device="cuda").half() * 2 - 1
    sv = torch.randn(m, generator=g, device="cuda")
    x = torch.randn(rows, k, generator=g, device="cuda").half()
    taken, many = [], bitshift.rht_many_rows
    monkeypatch.setattr(bitshift, "rht_many_rows", lambda *a, **kw: taken.append(1) or many(*a, **kw))
    call = lambda t: mod(t, tr, su, sv, had, had, 300, 300, 0, 8)
    with torch.no_grad():
        want = torch.cat([call(x[i:i + 50]) for i in range(0, rows, 50)])
        assert not taken
        got = call(x)
    assert len(taken) == 2 and float((got.float() - want.float()).norm() / want.float().norm()) <= 2.0**-10


@pytest.mark.parametrize("n", [11008, 4096, 12288])
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
def test_many_rows_that_start_off_16_bytes(n, dtype):
    """Rows and vectors at any element offset take the route of aligned ones, to the same bits."""
    from qtip_amd import ops
    from qtip_amd.utils.matmul_had import get_hadK, had_bits
    had, K = get_hadK(n)
    bits = had_bits(had, K, True, "cuda") if K > 1 else None
    rows = 96
    g = torch.Generator(device="cuda").manual_seed(n)

    def both(*shape, dt):
        off = torch.empty(int(np.prod(shape)) + 1, dtype=dt, device="cuda")[1:].view(*shape)
        off.copy_(torch.randn(*shape, generator=g, device="cuda"))
        assert off.data_ptr() % 16 and off.is_contiguous()
        return off, off.clone()

    x, pre, post = both(rows, n, dt=dtype), both(n, dt=torch.float16), both(n, dt=torch.float32)
    got, want = (ops.rht(x[i], order=K, had_bits=bits, pre=pre[i], post=post[i]) for i in (0, 1))
    assert torch.equal(got, want)
    if dtype == torch.float16:
        res, w = both(rows, n, dt=torch.float16), both(n, dt=torch.float16)
        got, want = (ops.rht(x[i], order=K, had_bits=bits, residual=res[i], pre_mode=ops.PRE_RMSNORM, norm_weight=w[i],
                             eps=1e-5) for i in (0, 1))
        assert torch.equal(got, want)
    m = 64
    packed = torch.randint(-32768, 32768, (m * n * 2 // 16,), dtype=torch.int16, generator=g, device="cuda")
    tlut = torch.randn(1024, generator=g, device="cuda").half()
    sv = both(m, dt=torch.float32)
    got, want = (ops.linear(x[i], packed, tlut, pre[i], sv[i], bits, K, None, 1, m, n, 2, n**-0.5 / 32, m**-0.5 * 32)
                 for i in (0, 1))
    assert torch.equal(got, want)


@pytest.mark.parametrize("K,p", [(256, 8), (256, 128), (250, 16), (173, 64), (6, 32), (1, 8), (1, 16), (1, 64), (12, 8)])
@pytest.mark.parametrize("rows", [24, 61])
def test_any_order_of_signs(K, p, rows):
    """A caller's own +-1 matrix of any order up to the largest the matrix form takes, and short rows, against float64."""
    from qtip_amd import ops
    from qtip_amd.utils.matmul_had import had_bits
    n = K * p
    g = torch.Generator(device="cuda").manual_seed(n + rows)
    had = torch.randint(0, 2, (K, K), generator=g, device="cuda").float() * 2 - 1 if K > 1 else torch.ones(1, 1, device="cuda")
    h64 = torch.from_numpy(scipy.linalg.hadamard(p).astype(np.float64)).cuda()
    for dtype in (torch.float16, torch.float32):
        x = torch.randn(rows, n, generator=g, device="cuda").to(dtype)
        for transpose in (False, True):
            bits = had_bits(had, K, transpose, "cuda") if K > 1 else None
            z = (had.T if transpose else had).double() @ (x.double().view(rows, K, p) @ h64)
            ref = z.reshape(rows, n) / n**0.5
            y = ops.rht(x, order=K, had_bits=bits, out_dtype=torch.float32)
            # exact products, fp32 sums of n terms
            assert float((y.double() - ref).abs().max()) <= 1e-5 * float(ref.abs().max())


@pytest.mark.parametrize("n,line16,line32", [(5120, 7, 12), (11008, 3, 8), (28672, 5, 12), (57344, 10, 10)])
def test_rows_with_a_residual_either_side_of_the_line(n, line16, line32):
    """A residual behind few rows: below the line between the forms every row has the bits of a launch of its own, on it the
    matrix form rounds some of them to the neighbouring fp16 value."""
    from qtip_amd import ops
    from qtip_amd.utils.matmul_had import get_hadK, had_bits
    had, K = get_hadK(n)
    g = torch.Generator(device="cuda").manual_seed(n)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda")
    kw = dict(order=K, had_bits=had_bits(had, K, False, "cuda"), post=rnd(n), out_dtype=torch.float16)
    for dtype, line in ((torch.float16, line16), (torch.float32, line32)):
        x, res = rnd(line, n).to(dtype), rnd(line, n).half()
        one = torch.cat([ops.rht(x[i:i + 1], residual=res[i:i + 1], **kw) for i in range(line)])
        assert torch.equal(ops.rht(x[:-1], residual=res[:-1], **kw), one[:-1])
        got = ops.rht(x, residual=res, **kw)
        # (exact values within half an fp16 step and the fp32 sums' error of each other; twice for a rounding of two sums)
        assert not torch.equal(got, one) and float((got.float() - one.float()).abs().max()) <= 2.0**-9 * float(one.abs().max())


@pytest.mark.parametrize("n,kind,line", [(10240, "post32", 20), (14336, "post32", 14), (14336, "pre32", 14), (16384, "post32", 13),
                                         (28672, "post32", 14), (11008, "post32", 8), (11008, "pre32", 6), (22016, "post32", 5),
                                         (22016, "pre32", 3), (57344, "post32", 10), (4992, "norm", 4), (9984, "silu", 4),
                                         (11008, "norm", 3), (14336, "silu", 5), (5120, "norm", 7)])
def test_rows_either_side_of_the_line(n, kind, line):
    """The row counts from which few rows take the matrix form: one below it every row has the bits of a launch of its own,
    on it the sums run in another order, with the same rounding points."""
    from qtip_amd import ops
    from qtip_amd.utils.matmul_had import get_hadK, had_bits
    had, K = get_hadK(n)
    g = torch.Generator(device="cuda").manual_seed(n)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda")
    kw = dict(order=K, had_bits=had_bits(had, K, True, "cuda") if K > 1 else None)
    x = rnd(line, 2 * n if kind == "silu" else n)
    if kind == "post32":
        kw.update(post=rnd(n))
    else:
        kw.update(pre=torch.sign(rnd(n) + 1e-5).half())
    if kind in ("norm", "silu"):
        x = x.half()
        kw.update(dict(pre_mode=ops.PRE_SILU_MUL) if kind == "silu" else
                  dict(pre_mode=ops.PRE_RMSNORM, norm_weight=(1 + 0.1 * rnd(n)).half(), eps=1e-5))
    one = torch.cat([ops.rht(x[i:i + 1], **kw) for i in range(line)])
    assert torch.equal(ops.rht(x[:-1], **kw), one[:-1])
    got = ops.rht(x, **kw)
    # fp32 sums of n terms; a prologue's fp16 values may round the other way (a norm's sum of squares in another order)
    tol = 2e-3 if kind in ("norm", "silu") else 1e-5
    assert float((got.float() - one.float()).abs().max()) <= tol * float(one.abs().max())
    assert kind in ("norm", "silu") or not torch.equal(got, one)  # (fp16 results may all round the same way)


@pytest.mark.parametrize("n,rows", [(928, 3), (4992, 4), (5120, 2), (5120, 7), (8960, 6), (11008, 3), (11008, 11), (14336, 5), (16384, 6),
                                    (16384, 48), (28672, 9), (57344, 5), (57344, 9), (57344, 11)])
@pytest.mark.parametrize("sign", [True, False])
def test_few_rows_with_prologue_and_residual_against_float64(n, rows, sign):
    """Either form of few rows with element-wise neighbours, sharing workgroups among them."""
    from qtip_amd import ops
    from qtip_amd.utils.matmul_had import get_hadK, had_bits
    had, K = get_hadK(n)
    g = torch.Generator(device="cuda").manual_seed(n + rows)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda")
    bits = {t: had_bits(had, K, t, "cuda") if K > 1 else None for t in (True, False)}
    pre = torch.sign(rnd(n) + 1e-5)
    pre = (pre if sign else pre * (0.5 + torch.rand(n, generator=g, device="cuda"))).half()
    w, post = (1 + 0.1 * rnd(n)).half(), rnd(n)
    x, gu, res = rnd(rows, n).half(), rnd(rows, 2 * n).half(), rnd(rows, n).half()
    d = x.double()
    normed = w.double() * (d * torch.rsqrt(d.pow(2).mean(-1, keepdim=True) + 1e-5)).half().double()
    gate, up = gu.double().split(n, -1)
    cases = [(x, dict(pre=pre, residual=res), d * pre.double(), res.double()), (x, dict(post=post, residual=res), d, res.double()),
             (gu, dict(pre=pre, pre_mode=ops.PRE_SILU_MUL),
              ((gate * torch.sigmoid(gate)).half().double() * up).half().double() * pre.double(), 0.0)]
    if n <= 16384 or rows >= 5:  # (the norm of longer rows has the matrix form alone)
        cases.append((x, dict(pre=pre, pre_mode=ops.PRE_RMSNORM, norm_weight=w, eps=1e-5), normed.half().double() * pre.double(), 0.0))
    for src, kw, ref, more in cases:
        t = "pre" in kw
        got = ops.rht(src, order=K, had_bits=bits[t], out_dtype=torch.float16, **kw)
        ref = _transform(ref, n, t) * n**-0.5 * (post.double() if "post" in kw else 1.0) + more
        # fp16 results; a prologue's fp16 values on the edge that round the other way move all elements of a row by 2^-11 / sqrt(n) each
        assert float((got.double() - ref).abs().max()) <= 1e-3 * float(ref.abs().max()), kw.keys()
