"""The prompt's attention kernel and the fused launches of a decoder layer over many tokens."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu


def _rotate(x, cos, sin):
    h = x.shape[-1] // 2
    return x * cos + torch.cat([-x[..., h:], x[..., :h]], -1) * sin


@pytest.mark.parametrize("n,past,slots,heads,kv,hd", [
    (1, 0, 1, 1, 1, 64), (12, 0, 32, 4, 4, 128), (63, 0, 64, 4, 1, 64), (64, 1, 65, 2, 2, 128), (65, 130, 200, 8, 2, 128),
    (200, 0, 333, 4, 2, 64), (129, 900, 1088, 2, 1, 128), (3, 2000, 4096, 4, 4, 128)])
def test_prefill_attention(n, past, slots, heads, kv, hd):
    """Keys bit for bit the fp16 rotary embedding, values copied, output against float64 from the rounded queries
    and keys: probabilities are rounded to fp16 (2^-11 of each), and so is the result."""
    from qtip_amd import ops
    g = torch.Generator(device="cuda").manual_seed(n + past)
    rand = lambda *s: torch.randn(*s, generator=g, device="cuda").half()
    wide = rand(n, (heads + 2 * kv) * hd + 8)
    q, k, v = wide[:, :-8].split([heads * hd, kv * hd, kv * hd], -1)
    kc, vc = rand(1, kv, slots, hd), rand(1, kv, slots, hd)
    kc[:, :, past + n:] = float("nan")  # slots behind the last query are not looked at
    vc[:, :, past + n:] = float("nan")
    pos = torch.arange(past, past + n, device="cuda")
    f = pos[:, None].float() * torch.rand(hd // 2, generator=g, device="cuda")
    emb = torch.cat([f, f], -1)
    cos, sin = emb.cos().half(), emb.sin().half()
    kc0, vc0 = kc.clone(), vc.clone()
    out = ops.prefill_attention(q, k, v, cos, sin, kc, vc, pos, heads, kv, hd)
    rows = lambda t, h: t.reshape(n, h, hd).transpose(0, 1)
    kc0[0, :, past:past + n] = _rotate(rows(k, kv), cos, sin)
    vc0[0, :, past:past + n] = rows(v, kv)
    same = lambda a, b: torch.equal(a.view(torch.int16), b.view(torch.int16))
    assert same(kc[:, :, :past + n], kc0[:, :, :past + n]) and same(vc[:, :, :past + n], vc0[:, :, :past + n])
    qr = _rotate(rows(q, heads), cos, sin).double()
    kk = kc0[0, :, :past + n].double().repeat_interleave(heads // kv, 0)
    vv = vc0[0, :, :past + n].double().repeat_interleave(heads // kv, 0)
    s = qr @ kk.transpose(1, 2) / math.sqrt(hd)
    s.masked_fill_(torch.arange(past + n, device="cuda")[None, :] > pos[:, None], -math.inf)
    p = s.softmax(-1)
    want = (p @ vv).transpose(0, 1).reshape(n, -1)
    bound = (p @ vv.abs()).transpose(0, 1).reshape(n, -1)
    # roundings of the probabilities and of the result, and the fp32 scores' error in the exponent
    assert bool(((out.double() - want).abs() <= 2.0**-10 * bound + 1e-6).all())


@pytest.mark.parametrize("n,heads,kv,hd", [(12, 4, 4, 128), (64, 4, 1, 64), (150, 8, 8, 128), (333, 8, 2, 128)])
def test_prefill_probabilities_are_not_rounded_to_fp16(n, heads, kv, hd):
    """Output against float64: one rounding to fp16 (2^-11 of the value, 2^-25 below the normal range) beside the
    error of fp32 scores and sums: a score of up to 8 errs by hd 2^-24 of its terms' magnitudes at most and by a few 2^-22 in
    fact, and so does the probability relative to itself, 2^-18 of the weighted magnitudes with room to spare.
    Probabilities of 11 bits err by 2^-12 of them."""
    from qtip_amd import ops
    g = torch.Generator(device="cuda").manual_seed(n + hd)
    rand = lambda *s: torch.randn(*s, generator=g, device="cuda").half()
    q, k, v = rand(n, heads * hd), rand(n, kv * hd), rand(n, kv * hd)
    kc, vc = rand(1, kv, n, hd), rand(1, kv, n, hd)
    pos = torch.arange(n, device="cuda")
    one = torch.ones(n, hd, device="cuda").half()
    out = ops.prefill_attention(q, k, v, one, torch.zeros_like(one), kc, vc, pos, heads, kv, hd)
    rows = lambda t, h: t.double().reshape(n, h, hd).transpose(0, 1)
    kk, vv = (rows(t, kv).repeat_interleave(heads // kv, 0) for t in (k, v))
    s = rows(q, heads) @ kk.transpose(1, 2).contiguous() / math.sqrt(hd)
    p = s.masked_fill_(pos[None, :] > pos[:, None], -math.inf).softmax(-1)
    back = lambda t: t.transpose(0, 1).reshape(n, -1)
    want, size = back(p @ vv), back(p @ vv.abs())
    assert bool(((out.double() - want).abs() <= 2.0**-11 * want.abs() + 2.0**-25 + 2.0**-18 * size).all())


def test_prefill_attention_skips_positions_outside_the_cache():
    from qtip_amd import ops
    kc = torch.ones(1, 1, 4, 64, device="cuda", dtype=torch.float16)
    vc = kc.clone()
    x = torch.randn(3, 64, device="cuda").half()
    one, zero = torch.ones_like(x), torch.zeros_like(x)
    out = ops.prefill_attention(x, x, x, one, zero, kc, vc, torch.tensor([-1, 4, 2**32 + 1], device="cuda"), 1, 1, 64)
    assert bool((kc == 1).all()) and bool((vc == 1).all()) and bool((out[1:] == 1).all())


@pytest.mark.parametrize("fused", [True, False])
@pytest.mark.parametrize("hidden,heads,kv,ffn,n", [(256, 4, 2, 832, 12), (512, 4, 4, 1376, 77), (640, 5, 5, 1728, 40),
                                                   (256, 2, 1, 832, 300)])
def test_layer_over_many_tokens(hidden, heads, kv, ffn, n, fused):
    """The fused launches against the module-by-module layer (which a forward hook makes it take), whole and in two
    pieces; fp16 rounding points are the same, sums are in another order."""
    from qtip_amd.llama_decode import LlamaConfig, LlamaDecoder
    cfg = LlamaConfig(hidden=hidden, heads=heads, kv_heads=kv, layers=2, ffn=ffn, vocab=96)
    model = LlamaDecoder(cfg, max_cache_len=n + 9, seed=n, fused=fused)
    ids = torch.randint(0, 96, (1, n), generator=torch.Generator().manual_seed(1)).cuda()
    at = torch.arange(n, device="cuda")

    def run(cut=None):
        for c in model.k_cache + model.v_cache:
            c.zero_()
        with torch.no_grad():
            if cut:
                lg = torch.cat([model(ids[:, :cut], at[:cut]), model(ids[:, cut:], at[cut:])], 1)
            else:
                lg = model(ids, at)
        return [lg] + [c.clone() for c in model.k_cache + model.v_cache]

    with torch.no_grad():
        assert model.layers[0].rows_ok(model.embed[ids][0], model.k_cache[0], model.v_cache[0], at)
    got = run()
    pieces = run(n // 2) if n >= 24 else got
    seen = []
    hooks = [l.o.register_forward_hook(lambda *a: seen.append(1)) for l in model.layers]
    want = run()
    for h in hooks:
        h.remove()
    assert len(seen) == 2
    for other in (got, pieces):
        for a, b in zip(other, want):
            assert float((a.double() - b.double()).norm() / b.double().norm()) <= 5e-3


def test_hooks_see_the_modules():
    """A hook on the inner module of a projection, or on all modules, is called for a prompt as for a token."""
    from torch.nn.modules.module import register_module_forward_hook
    from qtip_amd.llama_decode import LlamaConfig, LlamaDecoder
    model = LlamaDecoder(LlamaConfig(hidden=256, heads=4, kv_heads=2, layers=1, ffn=832, vocab=96), max_cache_len=32)
    ids, at = torch.zeros(1, 20, dtype=torch.int64, device="cuda"), torch.arange(20, device="cuda")
    seen = []
    with torch.no_grad():
        model(ids, at)
        inner = model.layers[0].o.codebook_class
        for hook in (inner.register_forward_hook(lambda *a: seen.append(a[0])),
                     register_module_forward_hook(lambda *a: seen.append(a[0]))):
            seen.clear()
            model(ids, at)
            hook.remove()
            assert any(m is inner for m in seen)


@pytest.mark.parametrize("which", ["k_cache", "v_cache", "both"])
def test_caches_that_start_off_16_bytes(which):
    """Such a cache goes module by module, as any other the attention kernel does not take."""
    from qtip_amd.llama_decode import LlamaConfig, LlamaDecoder
    model = LlamaDecoder(LlamaConfig(hidden=256, heads=4, kv_heads=2, layers=2, ffn=832, vocab=96), max_cache_len=32)
    ids, at = torch.arange(20, device="cuda")[None], torch.arange(20, device="cuda")

    def run():
        with torch.no_grad():
            return [model(ids, at)] + [c.clone() for c in model.k_cache + model.v_cache]

    want = run()
    for name in ("k_cache", "v_cache") if which == "both" else (which,):
        caches = getattr(model, name)
        caches[1] = torch.zeros(caches[1].numel() + 3, dtype=torch.float16, device="cuda")[3:].view_as(caches[1])
    assert not model.layers[1].rows_ok(model.embed[ids][0], model.k_cache[1], model.v_cache[1], at)
    for a, b in zip(run(), want):  # (sums in another order before the fp16 rounding points)
        assert float((a.double() - b.double()).norm() / b.double().norm()) <= 5e-3


def test_layer_input_that_starts_off_16_bytes():
    from qtip_amd.llama_decode import LlamaConfig, LlamaDecoder
    model = LlamaDecoder(LlamaConfig(hidden=256, heads=4, kv_heads=2, layers=1, ffn=832, vocab=96), max_cache_len=32)
    at = torch.arange(20, device="cuda")
    cos, sin = model.rope(at)
    x = torch.empty(20 * 256 + 1, dtype=torch.float16, device="cuda")[1:].view(1, 20, 256)
    x.copy_(torch.randn(x.shape, generator=torch.Generator().manual_seed(0)))
    assert not model.layers[0].rows_ok(x[0], model.k_cache[0], model.v_cache[0], at)
    with torch.no_grad():
        got, want = (model.layers[0](t, cos, sin, model.k_cache[0], model.v_cache[0], at, None, causal=True)
                     for t in (x, x.clone()))
    assert float((got.double() - want.double()).norm() / want.double().norm()) <= 5e-3


def test_one_mask_for_all_layers(monkeypatch):
    """Layers that go module by module share one mask, plain ones need none; a hook on a layer, and a layer of the
    caller's own, get the tensor."""
    from qtip_amd import llama_decode
    model = llama_decode.LlamaDecoder(llama_decode.LlamaConfig(hidden=256, heads=4, kv_heads=2, layers=3, ffn=832, vocab=96),
                                      max_cache_len=32)
    ids, at = torch.zeros(1, 20, dtype=torch.int64, device="cuda"), torch.arange(20, device="cuda")
    made, masks, make = [], [], llama_decode._causal_mask
    monkeypatch.setattr(llama_decode, "_causal_mask", lambda *a: made.append(1) or make(*a))

    def run():
        made.clear()
        with torch.no_grad():
            return model(ids, at)

    run()
    assert not made
    hooks = [l.o.register_forward_hook(lambda *a: None) for l in model.layers]
    want = run()
    assert len(made) == 1
    for h in hooks:
        h.remove()
    hook = model.layers[1].register_forward_hook(lambda mod, args, out: masks.append(args[6]))
    run()
    hook.remove()
    assert len(made) == 1

    class Own(torch.nn.Module):

        def __init__(self, layer):
            super().__init__()
            self.layer = layer

        def forward(self, x, cos, sin, k_cache, v_cache, cache_position, attn_mask):
            masks.append(attn_mask)
            return self.layer(x, cos, sin, k_cache, v_cache, cache_position, attn_mask)

    model.layers[2] = Own(model.layers[2])
    got = run()
    assert len(made) == 1 and float((got - want).norm() / want.norm()) <= 5e-3
    assert len(masks) == 2 and all(torch.equal(m, make(32, at)) for m in masks)


def test_a_layer_without_a_mask_attends_to_every_slot():
    from qtip_amd.llama_decode import LlamaConfig, LlamaDecoder
    model = LlamaDecoder(LlamaConfig(hidden=256, heads=4, kv_heads=2, layers=1, ffn=832, vocab=96), max_cache_len=32)
    g = torch.Generator(device="cuda").manual_seed(0)
    at, x = torch.arange(20, device="cuda"), torch.randn(1, 20, 256, generator=g, device="cuda").half()
    cos, sin = model.rope(at)
    k, v = (torch.randn(1, 2, 32, 64, generator=g, device="cuda").half() for _ in range(2))
    layer = model.layers[0]
    every = torch.ones(1, 1, 20, 32, dtype=torch.bool, device="cuda")
    with torch.no_grad():
        got, want, causal = (layer(x, cos, sin, k, v, at, mask, causal=c) for mask, c in ((None, False), (every, False), (None, True)))
    far = lambda a, b: float((a.double() - b.double()).norm() / b.double().norm())
    assert far(got, want) <= 5e-3 < far(causal, want)


def test_a_hook_in_front_of_a_layer_may_replace_the_mask():
    from qtip_amd.llama_decode import LlamaConfig, LlamaDecoder
    model = LlamaDecoder(LlamaConfig(hidden=256, heads=4, kv_heads=2, layers=2, ffn=832, vocab=96), max_cache_len=32)
    ids, at = torch.arange(20, device="cuda")[None], torch.arange(20, device="cuda")
    near = (at[:, None] - torch.arange(32, device="cuda")[None, :]).abs()[None, None] < 4

    def window(mod, args):
        return args[:6] + (args[6] & near,)

    with torch.no_grad():
        plain = model(ids, at)
        hook = model.layers[1].register_forward_pre_hook(window)
        got = model(ids, at)
        hook.remove()
        # the same mask by hand
        x, (cos, sin) = model.embed[ids], model.rope(at)
        causal = torch.arange(32, device="cuda")[None, :] <= at[:, None]
        for layer, mask, k, v in zip(model.layers, (causal, causal & near), model.k_cache, model.v_cache):
            x = layer(x, cos, sin, k, v, at, mask.view(1, 1, 20, 32))
        want = (model.norm(x) @ model.lm_head.T).float()
    far = lambda a, b: float((a - b).norm() / b.norm())
    assert far(got, want) <= 5e-3 < far(plain, want)


@pytest.mark.parametrize("form", ["strided", "off", "shared"])
def test_rotary_tables_of_the_callers_own(form):
    """Tables the attention kernel does not read as they stand go module by module."""
    from qtip_amd.llama_decode import LlamaConfig, LlamaDecoder
    model = LlamaDecoder(LlamaConfig(hidden=256, heads=4, kv_heads=2, layers=2, ffn=832, vocab=96), max_cache_len=32)
    ids, at = torch.arange(20, device="cuda")[None], torch.arange(20, device="cuda")
    rope = model.rope

    def own(positions):
        if form == "strided":
            return tuple(t.transpose(2, 3).contiguous().transpose(2, 3) for t in rope(positions))
        if form == "off":
            return tuple(torch.empty(t.numel() + 1, dtype=t.dtype, device="cuda")[1:].view_as(t).copy_(t) for t in rope(positions))
        return tuple(t[:, :, :1] for t in rope(positions))  # one angle for every token

    with torch.no_grad():
        want = model(ids, at)
        model.rope = own
        got = model(ids, at)
    far = float((got - want).norm() / want.norm())
    assert got.isfinite().all() and (far > 5e-3 if form == "shared" else far <= 5e-3)


@pytest.mark.parametrize("hd", [64, 128])
def test_infinite_values_and_scores(hd):
    """An infinite value makes the outputs infinite that weigh it, and only those; keys with a score of minus infinity, however
    many come first, do not count; a NaN key leaves the queries before its tile alone."""
    from qtip_amd import ops
    past, n, heads, inf = 70, 150, 3, float("inf")
    slots = past + n
    g = torch.Generator(device="cuda").manual_seed(hd)
    q, k, v = (torch.randn(heads, m, hd, generator=g, device="cuda").half() for m in (n, slots, slots))
    v[0, 140, 5], v[0, 200, 9] = inf, -inf  # of queries 70 and 130
    q[1, :, 3] = q[1, :, 3].abs() + 0.01
    k[1, :past, 3] = -inf
    k[2, 160, 7] = math.nan
    pos = torch.arange(past, slots, device="cuda")
    one = torch.ones(n, hd, device="cuda").half()
    kc, vc = k[None].clone(), v[None].clone()
    rows = lambda t: t.transpose(0, 1).reshape(n, heads * hd).contiguous()
    out = ops.prefill_attention(rows(q), rows(k[:, past:]), rows(v[:, past:]), one, torch.zeros_like(one), kc, vc, pos, heads, heads, hd)
    out = out.view(n, heads, hd).transpose(0, 1)
    s = (q.double() @ k.double().transpose(1, 2).contiguous() / math.sqrt(hd))
    p = s.masked_fill(torch.arange(slots, device="cuda")[None, :] > pos[:, None], -inf).softmax(-1)
    want = p @ v.double().nan_to_num(posinf=0.0, neginf=0.0)
    size = p @ v.double().abs().nan_to_num(posinf=0.0)
    want[0, 70:, 5], want[0, 130:, 9] = inf, -inf
    # probabilities (2^-11 each where an infinity is about) and the result rounded to fp16
    near = lambda h, at: bool(((out[h][at].double() - want[h][at]).abs() <= 2.0**-10 * size[h][at]).all())
    assert torch.equal(out[0, 70:, 5].float(), want[0, 70:, 5].float()) and torch.equal(out[0, 130:, 9].float(), want[0, 130:, 9].float())
    finite = torch.tensor([c not in (5, 9) for c in range(hd)], device="cuda")
    assert near(0, (slice(None), finite)) and near(0, slice(0, 64))
    assert near(1, slice(None))
    assert near(2, slice(0, 64)) and out[2, 90:].isnan().all()


@pytest.mark.parametrize("order", ["descending", "gaps", "shuffled", "late"])
def test_positions_in_any_order(order):
    """Keys go to the slots of their positions and a query sees the slots up to its own, whatever order they come in."""
    from qtip_amd import ops
    n, slots, heads, kv, hd = 90, 300, 4, 2, 64
    g = torch.Generator(device="cuda").manual_seed(5)
    q, k, v = (torch.randn(n, h * hd, generator=g, device="cuda").half() for h in (heads, kv, kv))
    kc, vc = (torch.randn(1, kv, slots, hd, generator=g, device="cuda").half() for _ in range(2))
    pos = {"descending": torch.arange(n).flip(0), "gaps": torch.arange(n) * 3 + 1, "late": torch.arange(slots - n, slots),
           "shuffled": torch.randperm(slots, generator=torch.Generator().manual_seed(1))[:n]}[order].cuda()
    one = torch.ones(n, hd, device="cuda").half()
    wk, wv = kc.clone(), vc.clone()
    wk[0, :, pos] = k.view(n, kv, hd).transpose(0, 1)
    wv[0, :, pos] = v.view(n, kv, hd).transpose(0, 1)
    out = ops.prefill_attention(q, k, v, one, torch.zeros_like(one), kc, vc, pos, heads, kv, hd)
    assert torch.equal(kc, wk) and torch.equal(vc, wv)
    kk, vv = (t[0].double().repeat_interleave(heads // kv, 0) for t in (wk, wv))
    s = q.double().view(n, heads, hd).transpose(0, 1) @ kk.transpose(1, 2).contiguous() / math.sqrt(hd)
    p = s.masked_fill(torch.arange(slots, device="cuda")[None, :] > pos[:, None], -math.inf).softmax(-1)
    want, size = ((p @ t).transpose(0, 1).reshape(n, -1) for t in (vv, vv.abs()))
    # the rounding of the result and fp32 scores (as test_prefill_probabilities_are_not_rounded_to_fp16 derives)
    assert bool(((out.double() - want).abs() <= 2.0**-11 * want.abs() + 2.0**-25 + 2.0**-18 * size).all())


@pytest.mark.parametrize("k,m,rows,mode,residual", [
    (4096, 4096, 40, 0, True), (11008, 4096, 100, 2, True), (4096, 22016, 17, 1, False), (928, 1248, 33, 1, True),
    (5120, 1728, 200, 2, False), (2048, 8192, 12, 1, True), (28672, 8192, 70, 2, True)])
def test_projection_of_a_prompt_in_one_call(k, m, rows, mode, residual):
    """linear_rows gives the bits of its launches one by one, the ranges of a cut product added on the way or not."""
    from qtip_amd import ops
    from qtip_amd.utils.matmul_had import get_hadK, had_bits
    g = torch.Generator(device="cuda").manual_seed(k + rows)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda")
    packed = torch.randint(-32768, 32768, (m * k * 2 // 16,), dtype=torch.int16, generator=g, device="cuda")
    tlut, su, sv = rnd(512, 2).half(), torch.sign(rnd(k)).half(), rnd(m)
    x, w = rnd(rows, 2 * k if mode == 2 else k).half(), (1 + 0.1 * rnd(k)).half()
    res = rnd(rows, m).half() if residual else None
    (hk, ki), (hm, ko) = get_hadK(k), get_hadK(m)
    bi, bo = (had_bits(h, o, t, "cuda") if o > 1 else None for h, o, t in ((hk, ki, True), (hm, ko, False)))
    for long_sums in (False, True):
        got = ops.linear_rows(x, packed, tlut, su, sv, bi, ki, bo, ko, m, k, 2, 0.01, 0.02, long_sums, mode,
                              w if mode == 1 else None, 1e-5, res)
        xt = ops.rht(x, order=ki, had_bits=bi, pre=su, scale=0.01, out_dtype=torch.float16, pre_mode=mode,
                     norm_weight=w if mode == 1 else None, eps=1e-5)
        y = ops.decompress_gemm(packed, xt, tlut, m, k, 2, out_dtype=torch.float16, long_sums=long_sums)
        want = ops.rht(y, order=ko, had_bits=bo, post=sv, scale=0.02, out_dtype=torch.float16, residual=res)
        assert torch.equal(got, want), long_sums
    assert ops.linear_rows(x[:, ::2], packed, tlut, su, sv, bi, ki, bo, ko, m, k, 2, 1.0, 1.0, False, 0, None, 0.0, None) is None
    assert ops.linear_rows(x, packed, tlut, su, sv, bi, ki, bo, ko, m, k, 2, 1.0, 1.0, False, mode, w[1:], 0.0, res) is None


@pytest.mark.parametrize("rows,n", [(1, 8), (3, 17), (5, 1024), (2, 4096), (7, 8200), (1000, 4096), (2, 16384), (3, 16383)])
def test_norm_of_rows(rows, n):
    """rmsnorm_rows (and the module, which calls it) against the formula in float64 with its fp16 rounding points."""
    from qtip_amd import ops
    from qtip_amd.llama_decode import RMSNorm
    g = torch.Generator(device="cuda").manual_seed(n)
    store = torch.randn(rows * n + 1, generator=g, device="cuda").half()
    mod = RMSNorm(n, 1e-5).cuda()
    mod.weight.data = (1 + 0.1 * torch.randn(n, generator=g, device="cuda")).half()
    for x in (store[:-1].view(rows, n), store[1:].view(rows, n)):  # on 16 bytes, and not
        h = x.double()
        ref = mod.weight.double() * (h * torch.rsqrt(h.pow(2).mean(-1, keepdim=True) + 1e-5)).half().double()
        got = ops.rmsnorm_rows(x, mod.weight, 1e-5)
        assert torch.equal(mod(x), got) and torch.equal(mod(x.view(1, rows, n))[0], got)
        # two roundings to fp16, either of which a value on the edge may take the other way
        assert bool(((got.double() - ref).abs() <= 2e-3 * ref.abs() + 1e-7).all())
    assert torch.equal(mod(x.float().half().requires_grad_(True)), mod.weight * (
        x.float() * torch.rsqrt(x.float().pow(2).mean(-1, keepdim=True) + 1e-5)).half())  # gradients: the formula
    assert mod(x.float()).dtype == torch.float32 and mod(x[:0]).shape == (0, n)


@pytest.mark.parametrize("n,half", [(1, 32), (33, 64), (1000, 64), (5, 3)])
def test_rotary_tables(n, half):
    """The tables of the library passes, the angles' fp32 products and their cosines rounded to fp16, bit for bit."""
    from qtip_amd import ops
    inv = 10000.0 ** (-torch.arange(half, device="cuda", dtype=torch.float32) / half)
    pos = torch.randint(0, 4096, (n,), generator=torch.Generator(device="cuda").manual_seed(n), device="cuda")
    emb = torch.cat([pos.float()[:, None] * inv[None]] * 2, dim=-1)
    cos, sin = ops.rotary_tables(pos, inv)
    assert torch.equal(cos, emb.cos().half()) and torch.equal(sin, emb.sin().half())


def test_norm_carries_tangents():
    """Forward-mode derivatives of the norm, of its input and of its weight, against reverse mode."""
    from torch.autograd import forward_ad
    from qtip_amd.llama_decode import RMSNorm
    g = torch.Generator(device="cuda").manual_seed(5)
    x, t = (torch.randn(4, 512, generator=g, device="cuda").half() for _ in range(2))
    mod = RMSNorm(512, 1e-5).cuda()
    w = (1 + 0.1 * torch.randn(512, generator=g, device="cuda")).half()
    for dual in ("input", "weight"):
        f = lambda v: torch.func.functional_call(mod, {"weight": w}, v) if dual == "input" else \
            torch.func.functional_call(mod, {"weight": v}, x)
        at, along = (x, t) if dual == "input" else (w, t[0])
        with forward_ad.dual_level():
            y, tangent = forward_ad.unpack_dual(f(forward_ad.make_dual(at, along)))
        want = torch.autograd.functional.jvp(f, at, along)  # by reverse mode, twice
        assert torch.equal(y, want[0]) and tangent is not None
        # fp16 products and roundings on the way, in another order
        assert float((tangent.float() - want[1].float()).norm()) <= 2.0**-8 * float(want[1].float().norm())


def test_traced_norm_and_rotary_tables_follow_their_input():
    from qtip_amd.llama_decode import LlamaConfig, LlamaDecoder, RMSNorm
    g = torch.Generator(device="cuda").manual_seed(6)
    x, other = (torch.randn(4, 512, generator=g, device="cuda").half() for _ in range(2))
    mod = RMSNorm(512, 1e-5).cuda()
    # (a product of two values and a sum of 512 of them in another order: a value on the edge rounds the other way)
    assert float((torch.jit.trace(mod, x)(other).float() - mod(other).float()).abs().max()) <= 2.0**-9 * float(mod(other).abs().max())
    model = LlamaDecoder(LlamaConfig(hidden=256, heads=4, kv_heads=2, layers=1, ffn=512, vocab=64, K=2), 64, device="cuda")
    pos = torch.arange(9, device="cuda")
    traced = torch.jit.trace(lambda p: model.rope(p), (pos,))
    assert all(torch.equal(a, b) for a, b in zip(traced(pos + 30), model.rope(pos + 30)))


def test_more_rows_and_positions_than_a_launch_has_threads():
    """2^26 + 3 rows of 8 values (a wave each), and 2^26 + 3 positions of 64 angles: past 2^32 threads, the first and the last ones."""
    from qtip_amd import ops
    rows = 2**26 + 3
    pick = torch.tensor([0, 1, 2**20 - 1, 2**20, 2**26 - 1, 2**26, rows - 1], device="cuda")
    w = (1 + 0.1 * torch.randn(8, device="cuda")).half()
    x = torch.randn(rows, 8, device="cuda", dtype=torch.float16)
    assert torch.equal(ops.rmsnorm_rows(x, w, 1e-5)[pick], ops.rmsnorm_rows(x[pick], w, 1e-5))
    del x
    inv = 10000.0 ** (-torch.arange(64, device="cuda", dtype=torch.float32) / 64)
    pos = torch.randint(0, 4096, (rows,), device="cuda")
    for big, few in zip(ops.rotary_tables(pos, inv), ops.rotary_tables(pos[pick], inv)):
        assert torch.equal(big[pick], few)


@pytest.mark.parametrize("k,m,rows,mode,residual", [(4096, 4096, 2, 0, True), (4096, 22016, 5, 1, False), (11008, 4096, 3, 2, True),
                                                    (5120, 28672, 9, 1, False), (28672, 8192, 11, 2, True), (928, 1248, 7, 2, True)])
def test_projection_of_few_rows_in_one_call(k, m, rows, mode, residual):
    """(The rows below those of a prompt, for callers of the native entry: the same check.)"""
    test_projection_of_a_prompt_in_one_call(k, m, rows, mode, residual)
