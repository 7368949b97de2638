"""GPU: attention over ranges of the keys that the position gives, put together in front of o's matvec, against the launch of one
range and the plain matvec behind it."""
import pytest
import torch

from qtip_amd import ops
from qtip_amd.llama_decode import LlamaConfig, LlamaDecoder, generate
from qtip_amd.utils.matmul_had import get_hadK, had_bits

pytestmark = pytest.mark.gpu


def _used(pos, slots, ranges, heads):
    n = min(pos + 1, slots)
    return 1 if n < (640 if heads > 40 else 380) else min(ranges, n // 160)


# positions around the lines between the numbers of ranges, the first, and the last of a cache
@pytest.mark.parametrize("pos,slots", ((0, 64), (1, 64), (378, 512), (379, 512), (478, 512), (479, 512), (638, 1024), (639, 1024),
                                       (1000, 1024), (1023, 1024), (4095, 4096)))
@pytest.mark.parametrize("heads,kv,D,S", ((32, 32, 128, 1), (32, 8, 128, 2), (64, 8, 128, 1), (16, 4, 128, 3), (32, 4, 64, 1)))
@pytest.mark.parametrize("vectors", (1, 3))
def test_shares_and_the_matvec_that_reads_them(pos, slots, heads, kv, D, S, vectors):
    g = torch.Generator(device="cuda").manual_seed(pos + heads + vectors)
    n = [heads * D, kv * D, kv * D]
    n = n if vectors == 3 else [sum(n)]
    buf = torch.randn(S, sum(n), generator=g, device="cuda") * 0.3
    parts = list(buf.split(n, dim=1))
    post = [torch.randn(v, generator=g, device="cuda").sign() for v in n]
    tables = [get_hadK(v) for v in n]
    bits = [had_bits(h, o, False, "cuda") if o > 1 else None for h, o in tables]
    order, scale = [o for _, o in tables], [v**-0.5 * 4 for v in n]
    caches = [torch.randn(1, kv, slots, D, generator=g, device="cuda").half() for _ in range(2)]
    freq = 10000.0 ** (-torch.arange(0, D, 2, device="cuda").float() / D)
    p = torch.tensor([pos], device="cuda")
    c0, c1 = [c.clone() for c in caches], [c.clone() for c in caches]
    if vectors == 1:
        want = ops.decode_attention_rht(parts[0], post[0], scale[0], bits[0], order[0], *c0, p, freq, heads, kv, D)
    else:
        want = ops.decode_attention_rht3(parts, post, scale, bits, order, *c0, p, freq, heads, kv, D)
    shares = ops.decode_attention_shares(parts, post, scale, bits, order, *c1, p, freq, heads, kv, D)
    assert all(torch.equal(a, b) for a, b in zip(c0, c1))
    used = _used(pos, slots, shares.shape[1], heads)
    s = shares[:, :used].double()
    w = (s[..., D:D + 1] - s[..., D:D + 1].amax(1, keepdim=True)).exp()
    out = ((w * s[..., :D]).sum(1) / (w * s[..., D + 1:D + 2]).sum(1)).reshape(-1)
    # fp32 sums, one rounding to fp16 (2**-12 of a value in the mean)
    assert (want.double() - out).norm() <= 4e-4 * out.norm()

    k, m, K = heads * D, 64, 2
    packed = torch.randint(-32768, 32768, (m * k * K // 16,), dtype=torch.int16, generator=g, device="cuda")
    tlut = torch.randn(1024, generator=g, device="cuda").half()
    su = torch.randn(k, generator=g, device="cuda").sign().half()
    a = ops.decompress_matvec_parts_rht(packed, out.half(), su, k**-0.5, tlut, m, k, K)
    b = ops.decompress_matvec_parts_shares(packed, shares, p, slots, su, k**-0.5, tlut, m, k, K)
    # (a value of the attention may be the neighbouring one in fp16, and so may one of its transform)
    assert (a.double() - b.double()).norm() <= 6e-4 * a.double().norm()


@pytest.mark.parametrize("fused", (True, False))
def test_one_recording_serves_every_context(fused):
    """A run from 300 to 600 keys, one to three ranges: the recorded step gives the eager steps' tokens."""
    cfg = LlamaConfig(hidden=2048, heads=16, kv_heads=4, layers=2, ffn=172 * 32, vocab=512)
    ids = torch.randint(0, cfg.vocab, (1, 300), generator=torch.Generator().manual_seed(3)).cuda()
    model = LlamaDecoder(cfg, max_cache_len=640, fused=fused)
    assert all(layer.attends_into_o() for layer in model.layers)
    a, _, _ = generate(model, ids, 300, use_graph=True)
    assert model.cfg.attn_key_splits == 1
    b, _, _ = generate(LlamaDecoder(cfg, max_cache_len=640, fused=fused), ids, 300, use_graph=False)
    assert torch.equal(a, b)


def test_a_callers_own_ranges_keep_their_launch():
    cfg = LlamaConfig(hidden=2048, heads=16, kv_heads=4, layers=1, ffn=172 * 32, vocab=512)
    model = LlamaDecoder(cfg, max_cache_len=512)
    for c in model.k_cache + model.v_cache:
        c.normal_()
    tok, pos = torch.zeros(1, 1, dtype=torch.int64, device="cuda"), torch.tensor([400], device="cuda")
    with torch.no_grad():
        a = model.decode_fused(tok, pos)
        cfg.attn_key_splits = 3
        b = model.decode_fused(tok, pos)
    assert (a - b).norm() <= 4e-3 * a.norm()


def test_a_further_request_needs_no_eager_step(monkeypatch):
    """The step of a further request is recorded at once, and with an eager step again where a layer has been replaced."""
    cfg = LlamaConfig(hidden=2048, heads=16, kv_heads=4, layers=2, ffn=172 * 32, vocab=512)
    g = torch.Generator().manual_seed(3)
    a, b = (torch.randint(0, cfg.vocab, (1, n), generator=g).cuda() for n in (20, 33))
    model = LlamaDecoder(cfg, max_cache_len=64)
    steps = []
    inner = model.decode_fused
    monkeypatch.setattr(model, "decode_fused", lambda *args, **kw: steps.append(torch.cuda.is_current_stream_capturing()) or
                        inner(*args, **kw))
    for ids in (a, b, a):
        got, _, _ = generate(model, ids, 12)
        assert torch.equal(got, generate(LlamaDecoder(cfg, max_cache_len=64), ids, 12, use_graph=False)[0])
    assert steps == [False, True, True, True]
    del steps[:]
    model.layers[1] = LlamaDecoder(cfg, max_cache_len=64).layers[1]
    assert torch.equal(generate(model, a, 12)[0], got) and steps == [False, True]
    drawn = [generate(model, b, 12, temperature=0.7, top_k=4)[0] for _ in range(2) if torch.manual_seed(7)]
    assert torch.equal(*drawn)


@pytest.mark.parametrize("fused", (True, False))
def test_a_callers_own_ranges_run_in_the_attentions_own_launch(fused, monkeypatch):
    """Which launches a token takes: ranges by the position and o's matvec on their shares, or the caller's count of ranges."""
    cfg = LlamaConfig(hidden=2048, heads=16, kv_heads=4, layers=2, ffn=172 * 32, vocab=512)
    model = LlamaDecoder(cfg, max_cache_len=512, fused=fused)
    tok, pos = torch.zeros(1, 1, dtype=torch.int64, device="cuda"), torch.tensor([400], device="cuda")
    took = []

    def watch(name):
        inner = getattr(ops, name)
        monkeypatch.setattr(ops, name, lambda *args, **kw: took.append((name, kw.get("key_splits"))) or inner(*args, **kw))

    own = "decode_attention_rht" if fused else "decode_attention_rht3"
    for name in ("decode_attention_shares", "decompress_matvec_parts_shares", "decode_attention", "decode_attention_rht",
                 "decode_attention_rht3"):
        watch(name)
    with torch.no_grad():
        model.decode_fused(tok, pos)
        assert took == [("decode_attention_shares", None), ("decompress_matvec_parts_shares", None)] * 2
        for ranges in (3, 8):
            del took[:]
            cfg.attn_key_splits = ranges
            model.decode_fused(tok, pos)
            assert took == [(own, ranges)] * 2
