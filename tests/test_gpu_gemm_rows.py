"""The batched decompress-GEMM at the edges of its batch tiles, row-block pairs and column slices, against
the decoded weights (bit-exact elsewhere) multiplied in float64."""
import pytest
import torch

from gemm_plan import FORMS, SHARED_FORMS

pytestmark = pytest.mark.gpu


# odd numbers of row blocks and of column blocks, one block, ranges of k that end inside a stage
@pytest.mark.parametrize("m,k", [(32, 32), (96, 96), (160, 2080), (1056, 832), (1248, 3328), (4096, 11008)])
@pytest.mark.parametrize("bits", [2, 3, 4])
def test_batch_tiles(m, k, bits):
    from qtip_amd import ops
    g = torch.Generator(device="cuda").manual_seed(m + k + bits)
    packed = torch.randint(-32768, 32768, (m * k * bits // 16,), dtype=torch.int16, generator=g, device="cuda")
    tlut = torch.randn(1024, generator=g, device="cuda").half()
    w = ops.decode(packed, tlut, m, k, bits).double()
    for batch in (1, 2, 16, 17, 32, 33, 64, 65, 128, 129, 200):
        x = torch.randn(batch, k, generator=g, device="cuda").half()
        ref = x.double() @ w.T
        got = ops.decompress_gemm(packed, x, tlut, m, k, bits, round_f16=False)
        # exact products, fp32 sums of k terms
        assert float((got.double() - ref).abs().max()) <= 1e-5 * float(ref.abs().max())
        wide = ops.decompress_gemm(packed, x, tlut, m, k, bits)
        half = ops.decompress_gemm(packed, x, tlut, m, k, bits, out_dtype=torch.float16)
        assert torch.equal(wide, got.half().float()) and torch.equal(half.float(), wide)


def test_fp16_results_are_rounded_ones():
    from qtip_amd import ops
    x = torch.zeros(2, 64, dtype=torch.float16, device="cuda")
    packed = torch.zeros(64 * 64 * 2 // 16, dtype=torch.int16, device="cuda")
    with pytest.raises(ValueError):
        ops.decompress_gemm(packed, x, torch.zeros(1024, dtype=torch.float16, device="cuda"), 64, 64, 2, round_f16=False,
                            out_dtype=torch.float16)


@pytest.mark.parametrize("k", [1 << 23, (1 << 24) + 32])
def test_activations_beyond_two_gib(k):
    """As many rows as pass the reach of 32-bit offsets (128 of 2^23 columns, 64 of 2^24) against float64 in pieces."""
    from qtip_amd import ops
    m, bits, rows = 32, 2, 128
    g = torch.Generator(device="cuda").manual_seed(k)
    packed = torch.randint(-32768, 32768, (m * k * bits // 16,), dtype=torch.int16, generator=g, device="cuda")
    tlut = torch.randn(1024, generator=g, device="cuda").half()
    x = torch.randn(rows, k, generator=g, device="cuda", dtype=torch.float16)
    y = ops.decompress_gemm(packed, x, tlut, m, k, bits, round_f16=False).double()
    w = ops.decode(packed, tlut, m, k, bits)
    want, size = torch.zeros(2, rows, m, dtype=torch.float64, device="cuda")
    for c in range(0, k, 1 << 20):
        a, b = x[:, c:c + (1 << 20)].double(), w[:, c:c + (1 << 20)].double().T.contiguous()
        want += a @ b
        size += a.abs() @ b.abs()
    # fp32 sums in chains of a few thousand products whose errors add like their square roots: 2^-20 of the magnitudes
    assert bool(((y - want).abs() <= 2.0**-20 * size).all())


def _check_product(m, k, batch, bits, long_sums):
    from qtip_amd import ops
    g = torch.Generator(device="cuda").manual_seed(m + k + batch)
    packed = torch.randint(-32768, 32768, (m * k * bits // 16,), dtype=torch.int16, generator=g, device="cuda")
    tlut = torch.randn(1024, generator=g, device="cuda").half()
    w = ops.decode(packed, tlut, m, k, bits).double()
    x = torch.randn(batch, k, generator=g, device="cuda").half()
    ref, size = x.double() @ w.T, x.double().abs() @ w.abs().T
    half = ops.decompress_gemm(packed, x, tlut, m, k, bits, out_dtype=torch.float16, long_sums=long_sums)
    # exact products, fp32 sums of k terms: chains of at most k / 32 additions, whose errors add like their square roots;
    # rounding to fp16 (normal numbers: the smallest are 2^-14)
    assert bool(((half.double() - ref).abs() <= 2.0**-11 * ref.abs() + 2.0**-24 + 2.0**-20 * size).all())
    if not long_sums:
        got = ops.decompress_gemm(packed, x, tlut, m, k, bits, round_f16=False)
        assert bool(((got.double() - ref).abs() <= 2.0**-21 * size).all())
        assert torch.equal(half, got.half())


@pytest.mark.parametrize("m,k,batch,long_sums", [c[:4] for c in FORMS])
@pytest.mark.parametrize("bits", [2, 3, 4])
def test_every_form(m, k, batch, long_sums, bits):
    """Every kernel of the batched product, cut along k and not, k ending inside a stage and not (FORMS says which case is which,
    and a test without a GPU that it is)."""
    _check_product(m, k, batch, bits, long_sums)


@pytest.mark.parametrize("m,k,batch", [c[:3] for c in SHARED_FORMS])
@pytest.mark.parametrize("bits", [3, 4])
def test_every_form_of_the_largest_matrices(m, k, batch, bits):
    _check_product(m, k, batch, bits, False)


def test_long_sums_are_for_fp16_results():
    from qtip_amd import ops
    x = torch.zeros(2, 64, dtype=torch.float16, device="cuda")
    packed = torch.zeros(64 * 64 * 2 // 16, dtype=torch.int16, device="cuda")
    with pytest.raises(ValueError):
        ops.decompress_gemm(packed, x, torch.zeros(1024, dtype=torch.float16, device="cuda"), 64, 64, 2, long_sums=True)


# row counts between and at the edges of batch tiles, odd numbers of row-block pairs, ranges of k that end inside a stage and
# inside a 64-column piece
@pytest.mark.parametrize("m,k,batch,bits", [(1056, 928, 9, 2), (96, 32, 2, 3), (1248, 2080, 16, 4), (32768, 2144, 13, 2),
                                            (16384, 8192, 5, 3), (22016, 4096, 16, 4), (64, 32, 17, 2), (544, 96, 40, 3), (96, 160, 150, 4), (512, 2048, 31, 3), (4096, 4096, 45, 4),
                                            (1056, 2080, 130, 2), (8192, 4096, 61, 3), (12288, 2144, 90, 4), (8192, 1248, 250, 3),
                                            (5632, 992, 1000, 2), (10240, 1120, 512, 4), (22016, 4096, 700, 3), (16416, 2080, 1030, 2),
                                            (1728, 832, 2048, 4)])
def test_forms_of_many_rows(m, k, batch, bits):
    from qtip_amd import ops
    g = torch.Generator(device="cuda").manual_seed(m + k + batch)
    packed = torch.randint(-32768, 32768, (m * k * bits // 16,), dtype=torch.int16, generator=g, device="cuda")
    tlut = torch.randn(1024, generator=g, device="cuda").half()
    w = ops.decode(packed, tlut, m, k, bits).double()
    x = torch.randn(batch, k, generator=g, device="cuda").half()
    ref, size = x.double() @ w.T, x.double().abs() @ w.abs().T
    got = ops.decompress_gemm(packed, x, tlut, m, k, bits, round_f16=False)
    # exact products, fp32 sums of k terms: chains of k / 32 additions, whose errors add like their square roots
    assert bool(((got.double() - ref).abs() <= 2.0**-21 * size).all())
    half = ops.decompress_gemm(packed, x, tlut, m, k, bits, out_dtype=torch.float16)
    assert torch.equal(half, got.half())


@pytest.mark.parametrize("m,k,batch", [(64, 32, 5), (128, 96, 16), (1056, 928, 11), (64, 32, 40), (128, 96, 20),
                                       (2048, 832, 100), (1056, 928, 200)])
def test_infinite_table_entry_stays_in_its_rows(m, k, batch):
    """Where k ends inside a stage, what stands in for the missing weights is met by zeros: it must not be a table entry the
    row does not hold (state 0 selects entry 0)."""
    from qtip_amd import ops
    g = torch.Generator(device="cuda").manual_seed(k)
    packed = torch.randint(-32768, 32768, (m * k * 2 // 16,), dtype=torch.int16, generator=g, device="cuda")
    tlut = torch.randn(512, 2, generator=g, device="cuda").half()
    tlut[0] = float("inf")
    w = ops.decode(packed, tlut.reshape(-1), m, k, 2)
    finite = w.isfinite().all(1)
    assert bool(finite.any()) and not bool(finite.all())
    x = torch.randn(batch, k, generator=g, device="cuda").half()
    got = ops.decompress_gemm(packed, x, tlut.reshape(-1), m, k, 2, round_f16=False)
    ref, size = x.double() @ w[finite].double().T, x.double().abs() @ w[finite].double().abs().T
    assert bool(((got[:, finite].double() - ref).abs() <= 2.0**-21 * size).all())
    assert not bool(got[:, ~finite].isfinite().any())


# forms of up to 16 rows (the last two share their activations through LDS), from 17 rows on, cut along k or not; k that ends
# in the middle of a 64-column piece, and slices without a piece
@pytest.mark.parametrize("m,k,batch,bits", [(64, 32, 5, 2), (128, 96, 16, 3), (1056, 928, 11, 4), (64, 32, 40, 4), (128, 96, 20, 2),
                                            (2048, 832, 100, 3), (1056, 928, 200, 2), (4096, 11040, 45, 2), (5632, 992, 1000, 4), (22016, 96, 509, 2), (12288, 928, 650, 3),
                                            (32768, 4128, 6, 4), (32768, 4128, 16, 3)])
@pytest.mark.parametrize("entry", [0, 5])
def test_infinities_are_those_of_the_product(m, k, batch, bits, entry):
    """One infinite value in the table: rows that hold it give the infinity, or NaN where two meet with opposite signs, as
    the product of the decoded matrix does, and nothing outside the matrix adds to them."""
    from qtip_amd import ops
    g = torch.Generator(device="cuda").manual_seed(k + batch)
    packed = torch.randint(-32768, 32768, (m * k * bits // 16,), dtype=torch.int16, generator=g, device="cuda")
    tlut = torch.randn(512, 2, generator=g, device="cuda").half()
    tlut[entry, 0] = float("inf")
    w = ops.decode(packed, tlut.reshape(-1), m, k, bits)
    x = torch.randn(batch, k, generator=g, device="cuda").half()
    x[x == 0] = 1
    got = ops.decompress_gemm(packed, x, tlut.reshape(-1), m, k, bits, round_f16=False)
    pos, neg = (x > 0).float(), (x < 0).float()
    wp, wn = (w == float("inf")).float(), (w == -float("inf")).float()
    up = (pos @ wp.T + neg @ wn.T) > 0
    down = (pos @ wn.T + neg @ wp.T) > 0
    fine = ~(up | down)
    assert bool((up ^ down).any())
    wf = w.double().nan_to_num(0, 0, 0)
    ref, size = x.double() @ wf.T, x.double().abs() @ wf.abs().T
    for got, off in ((got, 0), (ops.decompress_gemm(packed, x, tlut.reshape(-1), m, k, bits, out_dtype=torch.float16,
                                                    long_sums=True), 2.0**-11)):
        assert bool(got[up & down].isnan().all())
        assert bool((got[up & ~down] == float("inf")).all()) and bool((got[down & ~up] == -float("inf")).all())
        assert bool(((got.double() - ref).abs() <= off * ref.abs() + 2.0**-20 * size + 2.0**-24)[fine].all())


@pytest.mark.parametrize("m,k,bits", [(8192, 28672, 2), (4096, 4096, 3), (11008, 2048, 4), (28672, 8192, 2)])
def test_error_of_unrounded_results(m, k, bits):
    """The 2-norm error of sums cut into S ranges of KS slices of chains of L additions, 1.6e-8 sqrt(5 + 5 L + 1.5 KS + S), at
    the cut that bounds it (up to 32, 64 and 128 rows 8, 4 and 2 slices; ranges of at least 1024 and 512 columns while they fit
    256 CUs), with a tenth more for the sample; rounded results are off by their rounding, long sums or not."""
    from qtip_amd import ops
    g = torch.Generator(device="cuda").manual_seed(k)
    packed = torch.randint(-32768, 32768, (m * k * bits // 16,), dtype=torch.int16, generator=g, device="cuda")
    tlut = torch.randn(1024, generator=g, device="cuda").half()
    w = ops.decode(packed, tlut, m, k, bits).double()
    for batch in (2, 16, 24, 40, 100, 300, 1000):
        x = torch.randn(batch, k, generator=g, device="cuda").half()
        ref = x.double() @ w.T
        KS, RG, least = (8, 2, 16) if batch <= 32 else (4, 2, 8) if batch <= 64 else (2, 4, 8)
        S = 1
        while S < 16 and -(-m // 64 // RG) * S * 2 <= 256 and k // 64 // (2 * S) >= least:
            S *= 2
        bound = 1.1 * 1.6e-8 * (5 + 5 * k / 32 / KS / S + 1.5 * KS + S) ** 0.5
        y = ops.decompress_gemm(packed, x, tlut, m, k, bits, round_f16=False)
        assert float((y.double() - ref).norm() / ref.norm()) <= bound, batch
        for long_sums in (False, True):
            y = ops.decompress_gemm(packed, x, tlut, m, k, bits, out_dtype=torch.float16, long_sums=long_sums)
            assert float((y.double() - ref).norm() / ref.norm()) <= 2.1e-4
