"""Performance cases of the framework: what a program that uses it has it do, through its public
entry points, at the sizes of the Llama-architecture models its tests and benchmark run.

A case is a dict of plain values; "kind" names the entry point:

  linear      QuantizedLinear.forward without gradients: one quantized projection on `rows` tokens,
              from a single decoded token over small serving batches to a prompt
  op          the registered torch op quip_lib::decompress_matvec_qtip_{m}_1_{k}_{bits}
  decode      one decoded token: LlamaDecoder.decode_fused recorded into a HIP graph, as a
              generation loop holds it, with `context` tokens in the key / value caches
  generate    one whole request: generate() with a prompt and greedily decoded tokens
  prefill     LlamaDecoder.forward over a prompt
  train       forward and backward of one projection with gradients for the input and both sign
              vectors, as fine-tuning runs it
  decompress  decode_compressed: packed trellis to the dense fp16 matrix

Weights are random: any bitstream is a valid trellis walk, the table is N(0, 1) with the second
column centred, and the sign vectors carry a 1 / sqrt(fan-in) scale, so that activations have the
spread they have in a trained model.
"""
import math

import torch

import qtip_amd.codebook as codebook
from qtip_amd.linear.quantized_linear import QuantizedLinear
from qtip_amd.llama_decode import LlamaConfig, LlamaDecoder, generate
from qtip_amd.utils.kernel_decompress import decode_compressed

DEVICE = "cuda"
VOCAB = 32000

# (hidden, heads, kv heads, ffn): the decoder shapes of the tests and the benchmark
ARCHS = ((2048, 16, 4, 5504), (4096, 32, 32, 11008), (4096, 32, 8, 14336), (5120, 40, 40, 13824),
         (8192, 64, 8, 28672))
# widths off the usual ones: odd multiples of 32, every one a table order times a power of two
ODD_WIDTHS = (832, 928, 1120, 1248, 1728, 3328, 4992)


def listed():
    return [
        # one token through a small square projection: the shortest call there is
        dict(name="linear_4096_2bit_1row", kind="linear", k=4096, m=4096, bits=2, rows=1),
        # one token through the largest fused projection of the flagship 2-bit set
        dict(name="linear_57344_2bit_1row", kind="linear", k=8192, m=57344, bits=2, rows=1),
        # a serving batch at the size the batched kernel is quoted on
        dict(name="linear_28672_4bit_16rows", kind="linear", k=8192, m=28672, bits=4, rows=16),
        # a larger, odd batch through a table-order width
        dict(name="linear_down_3bit_45rows", kind="linear", k=11008, m=4096, bits=3, rows=45),
        # a ragged prompt through a fused projection
        dict(name="linear_22016_2bit_1000rows", kind="linear", k=4096, m=22016, bits=2, rows=1000),
        # the torch op a caller of the reference's kernel binds to
        dict(name="op_4096_11008_3bit", kind="op", m=4096, k=11008, bits=3),
        # one decoded token, fused q/k/v and up/gate
        dict(name="decode_fused_2bit", kind="decode", hidden=4096, heads=32, kv_heads=32, ffn=11008, layers=8,
             bits=2, fused=True, context=500),
        # one decoded token of a wide grouped-query model in the layout of the published checkpoints
        dict(name="decode_separate_4bit", kind="decode", hidden=8192, heads=64, kv_heads=8, ffn=28672, layers=4,
             bits=4, fused=False, context=900),
        # one request from prompt to the last token
        dict(name="generate_2bit", kind="generate", hidden=4096, heads=32, kv_heads=32, ffn=11008, layers=8, bits=2,
             fused=False, prompt=150, tokens=64),
        # a prompt through decoder layers and head
        dict(name="prefill_2bit_1000", kind="prefill", hidden=4096, heads=32, kv_heads=32, ffn=11008, layers=4,
             bits=2, fused=True, prompt=1000),
        # a fine-tuning step of one projection, in single precision as the fine-tuning scripts run it
        dict(name="train_11008_2bit_2048rows", kind="train", k=4096, m=11008, bits=2, rows=2048, dtype="float32"),
        # dense weights of a large projection
        dict(name="decompress_8192x28672_4bit", kind="decompress", m=8192, k=28672, bits=4),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _projection(rng):
    """(k, m) of a projection of one of the decoder shapes, now and then off the usual widths."""
    if rng.random() < 0.25:
        return rng.choice(ODD_WIDTHS), rng.choice(ODD_WIDTHS)
    d, heads, kv, ffn = rng.choice(ARCHS)
    kvd = kv * (d // heads)
    return rng.choice(((d, d), (d, d + 2 * kvd), (d, kvd), (d, ffn), (d, 2 * ffn), (ffn, d)))


def draw(rng):
    kind = rng.choice(("linear", "linear", "linear", "op", "decode", "generate", "prefill", "train", "decompress"))
    bits = rng.choice((2, 3, 4))
    if kind == "linear":
        k, m = _projection(rng)
        return dict(kind=kind, k=k, m=m, bits=bits, rows=_log_int(rng, 1, 2000))
    if kind in ("op", "decompress"):
        k, m = _projection(rng)
        return dict(kind=kind, m=m, k=k, bits=bits)
    if kind == "train":
        k, m = _projection(rng)
        rows = min(_log_int(rng, 16, 4000), max(16, 2048 * 4096 * 11008 // (k * m)))
        return dict(kind=kind, k=k, m=m, bits=bits, rows=rows, dtype=rng.choice(("float16", "float32")))
    hidden, heads, kv_heads, ffn = rng.choice(ARCHS)
    arch = dict(kind=kind, hidden=hidden, heads=heads, kv_heads=kv_heads, ffn=ffn, bits=bits,
                fused=rng.random() < 0.5)
    most = max(1, 8 * 4096 // hidden // (2 if hidden > 4096 else 1))
    if kind == "decode":
        return dict(arch, layers=rng.randint(1, most), context=_log_int(rng, 8, 1000))
    if kind == "prefill":
        return dict(arch, layers=rng.randint(1, max(1, most // 2)),
                    prompt=_log_int(rng, 16, 1000 if hidden <= 4096 else 500))
    return dict(arch, layers=rng.randint(1, max(1, most // 2)), prompt=_log_int(rng, 4, 1500 if hidden <= 4096 else 500),
                tokens=rng.randint(8, 64))


# ---- inputs -----------------------------------------------------------------------------------

def _generator(seed):
    return torch.Generator(device=DEVICE).manual_seed(seed)


def _trellis(shape, g):
    return torch.randint(-32768, 32768, shape, dtype=torch.int16, generator=g, device=DEVICE)


def _table(g):
    t = torch.randn(512, 2, generator=g, device=DEVICE)
    t[:, 1] -= t[:, 1].mean()
    return t.half()


def _signs(n, g):
    return torch.randint(0, 2, (n,), generator=g, device=DEVICE).float() * 2 - 1


def _fill(lin, g, gain=1.0):
    with torch.no_grad():
        lin.trellis.copy_(_trellis(lin.trellis.shape, g))
        lin.tlut.copy_(_table(g))
        lin.SU.copy_(_signs(lin.in_features, g))
        lin.SV.copy_(_signs(lin.out_features, g) * (gain / math.sqrt(lin.in_features)))
    return lin


def _linear(case, g, mode="eval"):
    lin = QuantizedLinear(case["k"], case["m"], 16, 16, 16, case["bits"], 2, 9, "quantlut_sym", dtype=torch.float16,
                          mode=mode).to(DEVICE)
    return _fill(lin, g)


def _model(case, slots, g):
    cfg = LlamaConfig(hidden=case["hidden"], heads=case["heads"], kv_heads=case["kv_heads"], layers=case["layers"],
                      ffn=case["ffn"], vocab=VOCAB, K=case["bits"])
    model = LlamaDecoder(cfg, max_cache_len=slots, device=DEVICE, fused=case["fused"], random_init=False)
    for layer in model.layers:
        for name, lin in layer.named_modules():
            if isinstance(lin, QuantizedLinear):
                # what a block adds to the residual stream is small beside it, as in a trained model
                _fill(lin, g, 0.1 if name in ("o", "down") else 1.0)
    # a peaked next-token distribution: token t is followed by successor[t]
    successor = torch.randperm(VOCAB, generator=g, device=DEVICE)
    model.embed.copy_(torch.randn(VOCAB, cfg.hidden, generator=g, device=DEVICE))
    model.lm_head[successor] = model.embed * 0.02
    return model


def prepare(case, seed):
    g = _generator(seed)
    kind = case["kind"]
    if kind == "linear":
        x = torch.randn(case["rows"], case["k"], generator=g, device=DEVICE).half()
        return dict(kind=kind, lin=_linear(case, g), x=x)
    if kind == "op":
        m, k, bits = case["m"], case["k"], case["bits"]
        return dict(kind=kind, op=codebook.register_shape(m, k, bits), trellis=_trellis((m // 16 * k // 16, 16 * bits), g),
                    x=torch.randn(1, k, generator=g, device=DEVICE).half(), tlut=_table(g))
    if kind == "decompress":
        m, k, bits = case["m"], case["k"], case["bits"]
        from qtip_amd.codebook.bitshift import quantlut_sym
        return dict(kind=kind, m=m, k=k, bits=bits, trellis=_trellis((m * k * bits // 16,), g),
                    lut=quantlut_sym(_table(g), 16, 9))
    if kind == "train":
        dtype = getattr(torch, case["dtype"])
        lin = _linear(case, g, mode="train-recons")
        # fine-tuning turns the sign vectors into parameters
        su, sv = lin.SU.to(dtype), lin.SV.clone()
        del lin.SU, lin.SV
        lin.SU = torch.nn.Parameter(su)
        lin.SV = torch.nn.Parameter(sv)
        x = torch.randn(case["rows"], case["k"], generator=g, device=DEVICE).to(dtype).requires_grad_(True)
        gy = torch.randn(case["rows"], case["m"], generator=g, device=DEVICE).to(dtype)
        return dict(kind=kind, lin=lin, x=x, gy=gy)
    if kind == "prefill":
        n = case["prompt"]
        ids = torch.randint(0, VOCAB, (1, n), generator=g, device=DEVICE)
        model = _model(case, (n + 256) // 64 * 64, g)
        return dict(kind=kind, model=model, ids=ids, positions=torch.arange(n, device=DEVICE))
    if kind == "generate":
        n, new = case["prompt"], case["tokens"]
        ids = torch.randint(0, VOCAB, (1, n), generator=g, device=DEVICE)
        model = _model(case, (n + new + 255) // 256 * 256, g)
        return dict(kind=kind, model=model, ids=ids, tokens=new,
                    keys=[c[:, :, :n + new - 1] for c in model.k_cache],
                    values=[c[:, :, :n + new - 1] for c in model.v_cache])
    # decode: the step of a generation loop, recorded once
    ctx = case["context"]
    model = _model(case, 1024, g)
    for c in model.k_cache + model.v_cache:
        c[:, :, :ctx] = torch.randn(c[:, :, :ctx].shape, generator=g, device=DEVICE).half()
    tok = torch.randint(0, VOCAB, (1, 1), generator=g, device=DEVICE)
    pos = torch.tensor([ctx], device=DEVICE)
    with torch.no_grad():
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            model.decode_fused(tok, pos)
        torch.cuda.current_stream().wait_stream(side)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            logits = model.decode_fused(tok, pos)
    return dict(kind=kind, model=model, tok=tok, pos=pos, graph=graph,
                out=[logits] + [c[:, :, ctx] for c in model.k_cache + model.v_cache])


@torch.no_grad()
def _infer(state):
    kind = state["kind"]
    if kind == "linear":
        return state["lin"](state["x"])
    if kind == "op":
        return state["op"](state["trellis"], state["x"], state["tlut"])
    if kind == "decompress":
        return decode_compressed(16, 9, state["bits"], 1, state["m"], state["k"], state["trellis"], state["lut"])
    if kind == "prefill":
        model = state["model"]
        return [model(state["ids"], state["positions"])] + model.k_cache + model.v_cache
    if kind == "generate":
        ids, _, _ = generate(state["model"], state["ids"], state["tokens"])
        return [ids] + state["keys"] + state["values"]
    state["graph"].replay()
    return state["out"]


def run(state):
    if state["kind"] == "train":
        y = state["lin"](state["x"])
        gx, gsu, gsv = torch.autograd.grad(y, (state["x"], state["lin"].SU, state["lin"].SV), state["gy"])
        return [y.detach(), gx, gsu, gsv]
    return _infer(state)


# ---- what a pass cannot do without --------------------------------------------------------------

def _layer_weights(case):
    d, kvd = case["hidden"], case["kv_heads"] * (case["hidden"] // case["heads"])
    return d * (d + 2 * kvd) + d * d + 3 * d * case["ffn"]


def _tokens(case, new, past):
    """(bytes, flops) of one forward of `new` tokens behind `past` cached ones: packed weights, keys and
    values, vector operands, head and logits."""
    d, kvd, layers = case["hidden"], case["kv_heads"] * (case["hidden"] // case["heads"]), case["layers"]
    w = _layer_weights(case) * layers
    pairs = new * past + new * (new + 1) // 2
    nbytes = (w * case["bits"] / 8 + layers * (4 * kvd * (past + new) + 30 * d + 6 * case["ffn"]) + 2 * VOCAB * d +
              new * (2 * d + 4 * VOCAB))
    flops = 2.0 * new * (w + VOCAB * d) + 4.0 * layers * d * pairs
    return nbytes, flops


def work(case):
    kind = case["kind"]
    if kind in ("linear", "op", "decompress", "train"):
        m, k = case["m"], case["k"]
        packed = m * k * case["bits"] / 8
        if kind == "linear":
            rows = case["rows"]
            return dict(bytes=packed + 2048 + 2 * k + 4 * m + 2 * rows * (k + m), flops=2.0 * rows * m * k)
        if kind == "op":
            return dict(bytes=packed + 2048 + 2 * k + 4 * m, flops=2.0 * m * k)
        if kind == "decompress":
            return dict(bytes=packed + 4 * 65536 + 2 * m * k, flops=0)
        size = 2 if case["dtype"] == "float16" else 4
        # input and output gradient in, output and input gradient out; two products
        return dict(bytes=packed + 2048 + case["rows"] * (k + m) * 2 * size + 2 * (size * k + 4 * m),
                    flops=4.0 * case["rows"] * m * k)
    if kind == "decode":
        nbytes, flops = _tokens(case, 1, case["context"])
    else:
        nbytes, flops = _tokens(case, case["prompt"], 0)
        for i in range(case.get("tokens", 1) - 1):
            b, f = _tokens(case, 1, case["prompt"] + i)
            nbytes, flops = nbytes + b, flops + f
    return dict(bytes=nbytes, flops=flops)


def tolerance(case):
    """About four times the distance measured between a pass and the same pass in float64 between its
    fp16 rounding points (linear, train, op) or along another route through the code (a decoded token
    module by module, a prompt in pieces through the batched kernels)."""
    kind = case["kind"]
    if kind == "decompress":
        return "exact"  # table entries, copied
    if kind == "op":
        return {"rel": 6e-7, "max": 5e-6}  # fp32 sums of k exact products; measured 1.5e-7, 6e-7
    if kind in ("linear", "train"):
        # fp16 activations behind a transform, the product rounded to fp16, fp16 or fp32 results: a sum in
        # another order moves some of them to the neighbouring fp16 value; measured 1.4e-4, 9.8e-4
        return {"rel": 6e-4, "max": 4e-3}
    # whole layers: the roundings of every sub-layer accumulate; measured 6.2e-4, 4.3e-3, no token
    return {"rel": 2.5e-3, "max": 2e-2, "differ": 0.0}
