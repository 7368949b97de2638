"""A whole projection by one call of the library against the same launches made one by one (lib/codebook/bitshift.py:
415-472)."""
import pytest
import torch

from qtip_amd import ops
from qtip_amd.linear.quantized_linear import QuantizedLinear
from qtip_amd.utils.matmul_had import get_hadK, had_bits

pytestmark = pytest.mark.gpu
DEV = "cuda"


# one row: input transform inside the matvec (4096) and beside it, split and whole k; more: each batch form and the
# last row count of the fused product; table orders on either side
@pytest.mark.parametrize("m,k,rows", [(32, 4096, 1), (4096, 4096, 1), (832, 11008, 1), (11008, 928, 1), (4096, 4096, 2),
                                      (1120, 832, 17), (11008, 4096, 64), (4096, 11008, 129), (64, 2048, 192)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("bits", [2, 3, 4])
def test_linear_is_its_launches(m, k, rows, dtype, bits):
    g = torch.Generator(device=DEV).manual_seed(m + k + rows + bits)
    packed = torch.randint(-32768, 32768, (m * k * bits // 16,), dtype=torch.int16, generator=g, device=DEV)
    tlut = torch.randn(1024, generator=g, device=DEV).half()
    su = (torch.randint(0, 2, (k,), generator=g, device=DEV) * 2 - 1).half()
    sv = torch.randn(m, generator=g, device=DEV)
    x = torch.randn(rows, k, generator=g, device=DEV).to(dtype)
    (tin, oin), (tout, oout) = get_hadK(k), get_hadK(m)
    bin_ = had_bits(None, oin, True, DEV) if oin > 1 else None
    bout = had_bits(None, oout, False, DEV) if oout > 1 else None
    s_in, s_out = k**-0.5 / 32, m**-0.5 * 32
    got = ops.linear(x, packed, tlut, su, sv, bin_, oin, bout, oout, m, k, bits, s_in, s_out)
    if rows == 1 and oin == 1 and dtype == torch.float16 and k in ops.RHT_IN_MATVEC_SIZES:
        y = ops.decompress_matvec_parts_rht(packed, x.reshape(-1), su, s_in, tlut, m, k, bits)
    else:
        xt = ops.rht(x, order=oin, had_bits=bin_, pre=su, scale=s_in, out_dtype=torch.float16)
        y = (ops.decompress_matvec_parts(packed, xt.reshape(-1), tlut, m, k, bits) if rows == 1
             else ops.decompress_gemm(packed, xt, tlut, m, k, bits, out_dtype=torch.float16))
    parts = y.shape[0] if rows == 1 else 1
    want = ops.rht(y if parts > 1 else y.reshape(rows, m), order=oout, had_bits=bout, post=sv, scale=s_out,
                   out_dtype=dtype, in_parts=parts).reshape(rows, m)
    assert got.dtype == dtype and torch.equal(got, want)


# ranges of k added by the output transform: one workgroup per row (2, 4, 8 values a thread, 2 to 16 ranges), the matrix form at
# 128 columns (2, 4 ranges; a last pass that is not full) and 64 (two), and the sizes on the other side of each line
@pytest.mark.parametrize("m,k,rows", [(2048, 28672, 17), (2048, 4096, 8), (4096, 2048, 64), (4096, 4096, 4), (4096, 4096, 5), (2048, 4096, 2),
                                      (8192, 11008, 7), (8192, 4096, 33),
                                      (5120, 2048, 45), (3072, 8192, 65), (3072, 4096, 17), (12288, 4096, 19), (11008, 4096, 17),
                                      (11008, 8192, 40), (928, 8192, 400), (832, 4096, 40)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
def test_linear_cut_along_k_is_its_launches(m, k, rows, dtype):
    test_linear_is_its_launches(m, k, rows, dtype, 2)


@pytest.mark.parametrize("m,k,rows", [(928, 8192, 400), (4096, 4096, 250), (2048, 28672, 300), (11008, 2048, 1000), (64, 96, 7)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
def test_linear_with_long_sums_is_its_launches(m, k, rows, dtype):
    """ops.linear(long_sums=True) gives the bits of decompress_gemm(long_sums=True) between its transforms."""
    bits = 2
    g = torch.Generator(device=DEV).manual_seed(m + k + rows)
    packed = torch.randint(-32768, 32768, (m * k * bits // 16,), dtype=torch.int16, generator=g, device=DEV)
    tlut = torch.randn(1024, generator=g, device=DEV).half()
    su = (torch.randint(0, 2, (k,), generator=g, device=DEV) * 2 - 1).half()
    sv, x = torch.randn(m, generator=g, device=DEV), torch.randn(rows, k, generator=g, device=DEV).to(dtype)
    (_, oin), (_, oout) = get_hadK(k), get_hadK(m)
    bin_ = had_bits(None, oin, True, DEV) if oin > 1 else None
    bout = had_bits(None, oout, False, DEV) if oout > 1 else None
    s_in, s_out = k**-0.5 / 32, m**-0.5 * 32
    got = ops.linear(x, packed, tlut, su, sv, bin_, oin, bout, oout, m, k, bits, s_in, s_out, long_sums=True)
    xt = ops.rht(x, order=oin, had_bits=bin_, pre=su, scale=s_in, out_dtype=torch.float16)
    y = ops.decompress_gemm(packed, xt, tlut, m, k, bits, out_dtype=torch.float16, long_sums=True)
    assert torch.equal(got, ops.rht(y, order=oout, had_bits=bout, post=sv, scale=s_out, out_dtype=dtype))


def test_linear_refuses_what_does_not_fit():
    packed = torch.zeros(64 * 64 * 2 // 16, dtype=torch.int16, device=DEV)
    args = dict(tlut=torch.zeros(1024, dtype=torch.float16, device=DEV), su=torch.ones(64, dtype=torch.float16, device=DEV),
                sv=torch.ones(64, device=DEV), had_in=None, order_in=1, had_out=None, order_out=1, m=64, k=64, bits=2,
                scale_in=1.0, scale_out=1.0)
    x = torch.zeros(3, 64, dtype=torch.float16, device=DEV)
    assert ops.linear(x, packed, **args).shape == (3, 64)
    for bad in (dict(x=x[:, :32]), dict(x=x[:0]), dict(x=x.cpu()), dict(su=args["su"][:32]), dict(sv=args["sv"].half()),
                dict(bits=3), dict(order_in=3), dict(packed=packed[:-1])):
        with pytest.raises((ValueError, TypeError)):
            ops.linear(**{**args, "x": x, "packed": packed, **bad})


def test_dense_rows_rule():
    """The row count of the dense route: past 2048 rows, or 2^24 results of fewer than 4096 columns; an instance's own
    dense_rows_min (whatever its value) grows with the matrix."""
    lin = QuantizedLinear(1024, 512, 16, 16, 16, 2, 2, 9, "quantlut_sym", dtype=torch.float16).cuda()
    with torch.no_grad():
        lin(torch.zeros(1, 1024, device="cuda", dtype=torch.float16))
    book = lin.codebook_class
    shapes = ((4096, 4096), (57344, 4096), (8192, 8192), (8160, 8192), (28672, 8192), (8192, 28672), (16384, 8192))
    assert book.dense_rows_min is None and {book.dense_rows_from(m, n) for m, n in shapes} == {2049}
    assert [book.dense_rows_from(m, n) for m, n in ((8192, 2048), (8224, 2048), (28672, 1024), (512, 32))] == [2049, 2041, 586, 2049]
    for rows_min in (193, 194):
        book.dense_rows_min = rows_min
        assert [book.dense_rows_from(m, n) for m, n in shapes[:5]] == [rows_min, rows_min, rows_min * 4 // 3, rows_min, rows_min * 5 // 3]
        assert book.dense_rows_from(8192, 28672) == rows_min * 8 // 3 and book.takes_dense(rows_min, 512, 1024)
    book.dense_rows_min = 2
    assert book.dense_rows_from(4096, 4096) == 2 and book.dense_rows_from(28672, 8192) == 3


@pytest.mark.parametrize("m,k,bits", [(13824, 5120, 3), (16384, 8192, 2), (8192, 16384, 4), (28672, 1024, 2), (512, 1024, 3)])
def test_rows_around_the_dense_route(m, k, bits, monkeypatch):
    """Either side of the row count from which a matrix is decoded to dense fp16 (2049, 586 for the short rows of 28672x1024),
    against float64 from the decoded weights: fp32 sums of k products (error at most k 2^-24 of the sum of magnitudes, far
    less in fact) and a rounding to fp16."""
    from qtip_amd.codebook.bitshift import BitshiftLinearKernelAG
    g = torch.Generator(device="cuda").manual_seed(m)
    lin = QuantizedLinear(k, m, 16, 16, 16, bits, 2, 9, "quantlut_sym", dtype=torch.float16).cuda()
    lin.trellis.copy_(torch.randint(-32768, 32768, lin.trellis.shape, dtype=torch.int16, generator=g, device="cuda"))
    lin.tlut.copy_(torch.randn(512, 2, generator=g, device="cuda"))
    with torch.no_grad():
        lin(torch.zeros(1, k, device="cuda", dtype=torch.float16))
        book = lin.codebook_class
        book.cb.recons_lut()
        edge = book.dense_rows_from(m, k)
        assert edge == (586 if m == 28672 else 2049) and book.takes_dense(edge, m, k) and not book.takes_dense(edge - 1, m, k)
        tl = book._tlut16(torch.device("cuda", 0))
        pick = torch.arange(0, m, 37, device="cuda")
        w = ops.decode(lin.trellis.reshape(-1), tl.reshape(-1), m, k, bits)[pick].double()
        dense, decode = [], ops.decode
        monkeypatch.setattr(ops, "decode", lambda *a: dense.append(1) or decode(*a))
        for rows in (edge - 1, edge):
            x = torch.randn(rows, k, generator=g, device="cuda").half()
            want, size = x.double() @ w.T, x.double().abs() @ w.abs().T
            for product in (lambda: book.rows_product(x, lin.trellis, tl, m, k),
                            lambda: BitshiftLinearKernelAG.apply(x, lin.trellis, m, k, 16, 9, bits, 2, book.cb.lut)):
                dense.clear()
                y = product()
                assert len(dense) == (1 if rows == edge else 0)
                assert y.shape == (rows, m) and y.dtype == torch.float16
                assert bool(((y[:, pick].double() - want).abs() <= 2.0**-11 * want.abs() + 2.0**-20 * size).all())


def test_native_call_takes_what_fits_and_leaves_the_rest():
    """The native functions behind a projection and the torch op: the bits of the way through the checks where the
    operands fit, None for everything that they do not describe."""
    from qtip_amd import _lib, ops
    m, k, bits, rows = 96, 256, 3, 5
    g = torch.Generator(device="cuda").manual_seed(3)
    packed = torch.randint(-32768, 32768, (m * k * bits // 16,), dtype=torch.int16, generator=g, device="cuda")
    tlut = torch.randn(512, 2, generator=g, device="cuda").half()
    su, sv = torch.ones(k, device="cuda").half(), torch.ones(m, device="cuda")
    x = torch.randn(rows, k, generator=g, device="cuda").half()
    st = torch.cuda.current_stream().cuda_stream
    from qtip_amd.utils.matmul_had import get_hadK, had_bits
    order = get_hadK(m)[1]
    table = had_bits(get_hadK(m)[0], order, False, "cuda")

    def call(x=x, packed=packed, tlut=tlut, su=su, sv=sv, table=table, m=m, k=k, bits=bits, copy_rows=96):
        return _lib.host().linear(x, packed, tlut, su, sv, None, 1, table, order, m, k, bits, 0.5, 2.0, False, copy_rows, st)

    want = ops.rht(ops.decompress_gemm(packed, ops.rht(x, pre=su, scale=0.5, out_dtype=torch.float16), tlut, m, k, bits,
                                       out_dtype=torch.float16), order=order, had_bits=table, post=sv, scale=2.0)
    assert torch.equal(call(), want) and torch.equal(call(packed=packed.view(torch.uint8)), want)
    wide = torch.zeros(rows, 2 * k, device="cuda").half()
    off = torch.zeros(k + 1, device="cuda").half()[1:]
    for kw in (dict(x=wide[:, ::2]), dict(x=wide[:, :k]), dict(x=x.double()), dict(x=x[0]), dict(x=x[:0]), dict(x=x.cpu()),
               dict(packed=packed[:-1]), dict(packed=packed.float()), dict(packed=None), dict(tlut=tlut.float()),
               dict(su=su.float()), dict(su=su[:-1]), dict(su=off, copy_rows=1), dict(sv=sv.half()), dict(table=None),
               dict(table=table[:1] if table.numel() > 1 else table.float()), dict(m=m + 1), dict(k=k - 32), dict(bits=5),
               dict(x=x.to_sparse())):
        assert call(**kw) is None, kw
    seen = []
    torch.vmap(lambda v: seen.append(call(x=v)) or v)(x.expand(2, rows, k))
    assert seen == [None]
    row = x[:1]
    assert torch.equal(_lib.host().matvec(packed, row, tlut, m, k, bits, 0, 0, st)[0],
                       ops.decompress_matvec(packed, row, tlut, m, k, bits, split_k=False))
    for args in ((packed, row.float(), tlut), (packed, x, tlut), (packed.cpu(), row, tlut), (packed, row, tlut[:256])):
        assert _lib.host().matvec(*args, m, k, bits, 0, 0, st) is None
    with pytest.raises(TypeError):
        _lib.host().matvec(packed, row, tlut)


def test_without_the_native_module(monkeypatch):
    """Every caller of the native functions has its own way to the same launches: the same bits."""
    from qtip_amd import _lib, ops
    from qtip_amd.codebook import register_shape
    from qtip_amd.llama_decode import LlamaConfig, LlamaDecoder
    m, k, bits = 96, 256, 3
    g = torch.Generator(device="cuda").manual_seed(4)
    packed = torch.randint(-32768, 32768, (m // 16 * k // 16, 16 * bits), dtype=torch.int16, generator=g, device="cuda")
    tlut = torch.randn(512, 2, generator=g, device="cuda").half()
    su, sv = torch.ones(k, device="cuda").half(), torch.ones(m, device="cuda")
    xs = [torch.randn(rows, k, generator=g, device="cuda").half() for rows in (1, 5, 40)]
    from qtip_amd.utils.matmul_had import get_hadK, had_bits
    order = get_hadK(m)[1]
    table = had_bits(get_hadK(m)[0], order, False, "cuda")
    model = LlamaDecoder(LlamaConfig(hidden=256, heads=4, kv_heads=2, layers=1, ffn=512, vocab=64, K=2), 64, device="cuda")
    ids, pos = torch.arange(20, device="cuda")[None], torch.arange(20, device="cuda")

    def outputs():
        with torch.no_grad():
            return [ops.linear(x, packed.reshape(-1), tlut, su, sv, None, 1, table, order, m, k, bits, 0.5, 2.0) for x in xs] + [
                register_shape(m, k, bits)(packed, xs[0], tlut), model(ids, pos)]

    native = outputs()
    assert _lib.host()
    monkeypatch.setattr(_lib, "_host", False)
    assert all(torch.equal(a, b) for a, b in zip(native, outputs()))
