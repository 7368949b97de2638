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
