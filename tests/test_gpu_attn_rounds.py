"""Decode attention at the edges of its rounds of keys and values, one workgroup per head and key ranges, against the
float64 attention over the cache it leaves."""
import pytest
import torch

from qtip_amd import ops

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("heads,kv,D", [(4, 4, 128), (8, 2, 64), (2, 1, 256)])
@pytest.mark.parametrize("splits", [1, 3, 8])
def test_rounds(heads, kv, D, splits):
    slots = 2100
    g = torch.Generator(device=DEV).manual_seed(heads + D + splits)
    qkv = torch.randn((heads + 2 * kv) * D, generator=g, device=DEV).half()
    kc = torch.randn(1, kv, slots, D, generator=g, device=DEV).half()
    vc = torch.randn(1, kv, slots, D, generator=g, device=DEV).half()
    freq = 1.0 / (10000.0**(torch.arange(0, D, 2, device=DEV).float() / D))
    for pos in (0, 1, 126, 127, 128, 255, 256, 257, 383, 384, 511, 512, 700, 1023, 1024, 2099):
        k1, v1 = kc.clone(), vc.clone()
        got = ops.decode_attention(qkv, k1, v1, torch.tensor([pos], device=DEV), freq, heads, kv, D, key_splits=splits)
        ang = (pos * freq).repeat(2)
        c, s = ang.cos().half(), ang.sin().half()
        q = qkv[:heads * D].view(heads, D)
        q = q * c + torch.cat((-q[:, D // 2:], q[:, :D // 2]), 1) * s
        keys = k1[0, :, :pos + 1].double().repeat_interleave(heads // kv, 0)
        vals = v1[0, :, :pos + 1].double().repeat_interleave(heads // kv, 0)
        p = torch.softmax((keys @ q.double()[:, :, None])[..., 0] / D**0.5, -1)
        ref = (p[:, None] @ vals)[:, 0]
        # the rotation's cos / sin may differ by an fp16 step (2^-11 of a query) and the result is rounded once
        err = (got.view(heads, D).double() - ref).abs().max()
        assert float(err) <= 2**-8 * float(ref.abs().max()), (pos, float(err))
        assert torch.equal(v1[0, :, pos], qkv[(heads + kv) * D:].view(kv, D))
