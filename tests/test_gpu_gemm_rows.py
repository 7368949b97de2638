"""The batched decompress-GEMM at the edges of its batch tiles, row-block pairs and column slices, against
the decoded weights (bit-exact elsewhere) multiplied in float64."""
import pytest
import torch

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
