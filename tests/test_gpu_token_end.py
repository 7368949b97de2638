"""GPU: the end of LlamaDecoder.decode_fused where the one launch of ops.token_head does not take what the layers leave."""
import pytest
import torch

from qtip_amd.llama_decode import LlamaConfig, LlamaDecoder

pytestmark = pytest.mark.gpu


def _step(fused):
    cfg = LlamaConfig(hidden=2048, heads=16, kv_heads=4, layers=2, ffn=172 * 32, vocab=512)
    model = LlamaDecoder(cfg, max_cache_len=64, fused=fused)
    return model, torch.tensor([[7]], device="cuda"), torch.tensor([0], device="cuda")


@pytest.mark.parametrize("fused", (True, False))
@pytest.mark.parametrize("answers", ((True, False), (False,)))
def test_a_head_that_does_not_launch_reads_the_whole_stream(fused, answers, monkeypatch):
    """Logits of norm and library product against those of the one launch.  Each is one rounding to fp16 (2.8e-4 in 2-norm) away
    from the sums of a norm whose values may be the neighbouring ones in fp16 (as much again)."""
    model, tok, pos = _step(fused)
    with torch.no_grad():
        want = model.decode_fused(tok, pos)
        asked = iter(answers)
        monkeypatch.setattr(model, "_head_launches", lambda x: next(asked))
        got = model.decode_fused(tok, pos)
    assert next(asked, None) is None
    assert (got - want).norm() <= 8e-4 * want.norm()


@pytest.mark.parametrize("dtype", (torch.float16, torch.bfloat16))
def test_autocast_casts_the_output_matrix(dtype):
    """A region of autocast computes the product of the output matrix in its own type, as it does for the module's prompt."""
    model, tok, pos = _step(True)
    with torch.no_grad():
        plain = model.decode_fused(tok, pos)
        with torch.autocast("cuda", dtype=dtype):
            got = model.decode_fused(tok, pos)
            assert model.decode_fused(tok, pos, float_logits=False).dtype == dtype
    assert got.dtype == torch.float32 and torch.equal(got, got.to(dtype).float())
    # two roundings of the norm and one of the result
    assert (got - plain).norm() <= (1e-3 if dtype == torch.float16 else 8e-3) * plain.norm()
