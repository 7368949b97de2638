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


@pytest.mark.parametrize("splits", [1, 4])
@pytest.mark.parametrize("pos", [3, 130, 700])
def test_infinite_scores_and_stale_slots(pos, splits):
    """Keys whose score is -inf weigh nothing (the first ones a wave meets among them), an infinite value stays one, a score of
    +inf or NaN makes its head NaN, and what stands in slots from the position on is not looked at."""
    heads, D, slots = 4, 128, 1024
    g = torch.Generator(device=DEV).manual_seed(pos)
    qkv = torch.randn(3 * heads * D, generator=g, device=DEV).half()
    qkv[:heads * D] = qkv[:heads * D].abs() + 0.5  # with no rotation every element of a query is positive
    freq = torch.zeros(D // 2, device=DEV)
    kc = torch.randn(1, heads, slots, D, generator=g, device=DEV).half()
    vc = torch.randn(1, heads, slots, D, generator=g, device=DEV).half()
    kc[:, :, pos:], vc[:, :, pos:] = float("nan"), float("nan")
    low = torch.arange(0, pos, 2, device=DEV)  # head 0, 2: every other key at -inf, head 1: one of +inf, head 2: an infinite value
    kc[0, 0, low, 5] = kc[0, 2, low, 5] = -float("inf")
    kc[0, 1, pos - 1, 7] = float("inf")
    vc[0, 2, 1, 9] = float("inf")
    out = ops.decode_attention(qkv, kc, vc, torch.tensor([pos], device=DEV), freq, heads, heads, D, key_splits=splits).view(heads, D)
    q = qkv[:heads * D].view(heads, 1, D).double()
    p = torch.softmax((kc[0, :, :pos + 1].double() @ q.transpose(1, 2).contiguous())[..., 0] / D**0.5, -1)
    ref = (p[:, None] @ vc[0, :, :pos + 1].double())[:, 0]
    assert bool(out[1].isnan().all()) and bool(ref[1].isnan().all())
    for h in (0, 3):
        assert float((out[h].double() - ref[h]).abs().max()) <= 2**-9 * float(ref[h].abs().max())
    assert float(out[2, 9]) == float(ref[2, 9]) == float("inf") and bool(out[2, :9].isfinite().all())


@pytest.mark.parametrize("form,D", [("plain", 64), ("plain", 128), ("plain", 256), ("rht", 64), ("rht", 128), ("rht3", 64),
                                    ("rht3", 128)])
def test_rotation_rounds_every_product(form, D):
    """The cached key of a token is fp16(fp16(k * cos) + fp16(rotate_half(k) * sin)) bit for bit in every form of the launch."""
    from qtip_amd.utils.matmul_had import get_hadK, had_bits
    heads, kv, slots, pos = 8, 2, 64, 37
    g = torch.Generator(device=DEV).manual_seed(D)
    n = (heads + 2 * kv) * D
    freq = 1.0 / (10000.0**(torch.arange(0, D, 2, device=DEV).float() / D))
    where = torch.tensor([pos], device=DEV)
    caches = lambda: [torch.zeros(1, kv, slots, D, device=DEV).half() for _ in range(2)]
    probe = torch.zeros(n, device=DEV).half()
    probe[heads * D:heads * D + D // 2] = 1  # a key of ones in front of zeros: cosines in its first half, sines in the other
    kc, vc = caches()
    ops.decode_attention(probe, kc, vc, where, freq, heads, kv, D)
    c, s = (t.repeat(2) for t in kc[0, 0, pos].split(D // 2))
    kc, vc = caches()
    if form == "plain":
        qkv = torch.randn(n, generator=g, device=DEV).half()
        ops.decode_attention(qkv, kc, vc, where, freq, heads, kv, D)
    else:  # whole numbers, whose transforms are exact in fp32 and in fp16 after the division by 8
        parts = torch.randint(-8, 9, (2, n), generator=g, device=DEV).float()
        sizes = [n] if form == "rht" else [heads * D, kv * D, kv * D]
        views = parts.split(sizes, dim=1)
        tables = [get_hadK(m) for m in sizes]
        bits = [had_bits(h, o, False, DEV) if o > 1 else None for h, o in tables]
        qkv = torch.cat([ops.rht(v.sum(0, keepdim=True), order=o, had_bits=b, scale=0.125, out_dtype=torch.float32)[0]
                         for v, (_, o), b in zip(views, tables, bits)])
        assert torch.equal(qkv, qkv.half().float())
        qkv = qkv.half()
        if form == "rht":
            ops.decode_attention_rht(parts, None, 0.125, bits[0], tables[0][1], kc, vc, where, freq, heads, kv, D)
        else:
            ops.decode_attention_rht3(list(views), [None] * 3, [0.125] * 3, bits, [o for _, o in tables], kc, vc, where, freq,
                                      heads, kv, D)
    k = qkv[heads * D:(heads + kv) * D].view(kv, D)
    turned = torch.cat((-k[:, D // 2:], k[:, :D // 2]), 1)
    assert torch.equal(kc[0, :, pos], k * c + turned * s)
    assert torch.equal(vc[0, :, pos], qkv[(heads + kv) * D:].view(kv, D))
