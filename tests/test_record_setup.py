"""A further request records its step at once: what the layers keep for it exists before the recording."""
import contextlib
import copy
import pickle
import types

import pytest
import torch

from qtip_amd import llama_decode, ops
from qtip_amd.linear.quantized_linear import QuantizedLinear
from qtip_amd.llama_decode import DecoderLayer, LlamaConfig, LlamaDecoder, generate

SETUP = ("_fused", "_grouped", "_grouped_plain")
TABLE_ORDER = dict(hidden=1280, heads=20, kv_heads=20, layers=2, ffn=832, vocab=96)  # 1280 = 20 * 64, stacked sign vectors
POWER_OF_2 = dict(hidden=2048, heads=16, kv_heads=4, layers=2, ffn=832, vocab=96)


def _drop(model, names):
    for layer in model.layers:
        for name in names:
            layer.__dict__.pop(name, None)


@pytest.fixture
def steps(monkeypatch):
    """generate() on the host: graphs and streams that only say whether a step runs or is recorded."""
    log = types.SimpleNamespace(recording=False, seen=[])

    class Graph:
        def replay(self):
            pass

    @contextlib.contextmanager
    def graph(_):
        log.recording = True
        try:
            yield
        finally:
            log.recording = False

    stream = types.SimpleNamespace(wait_stream=lambda other: None)
    for name, fake in (("CUDAGraph", Graph), ("graph", graph), ("Stream", lambda: stream), ("current_stream", lambda: stream),
                       ("stream", lambda s: contextlib.nullcontext()), ("synchronize", lambda: None)):
        monkeypatch.setattr(torch.cuda, name, fake)
    monkeypatch.setattr(ops, "greedy_pick", lambda *args: None)
    return log


def _host_model(log, cfg):
    model = LlamaDecoder(LlamaConfig(**cfg), max_cache_len=32, device="cpu", random_init=False)
    model.fused = False
    logits = torch.zeros(1, 1, cfg["vocab"])

    def decode_fused(tok, pos, float_logits=True):
        names = ("_fused", "_grouped") + (("_grouped_plain",) if cfg is TABLE_ORDER else ())
        log.seen.append((log.recording, all(name in layer.__dict__ for layer in model.layers for name in names)))
        for layer in model.layers:
            layer.grouped_ok() or layer.grouped_plain_ok()
        return logits

    model.forward = lambda ids, pos: logits
    model.decode_fused = decode_fused
    return model


@pytest.mark.parametrize("cfg", (TABLE_ORDER, POWER_OF_2))
@pytest.mark.parametrize("names", (SETUP, ("_grouped", "_grouped_plain"), ("_grouped_plain",), ("_fused",)))
def test_nothing_is_set_up_inside_a_recording(steps, cfg, names):
    model = _host_model(steps, cfg)
    ids = torch.zeros(1, 4, dtype=torch.int64)
    generate(model, ids, 1)
    assert [recording for recording, _ in steps.seen] == [False, True]
    del steps.seen[:]
    generate(model, ids, 1)
    assert steps.seen == [(True, True)]
    _drop(model, names)
    del steps.seen[:]
    generate(model, ids, 1)
    assert steps.seen[-1] == (True, True)
    if "_fused" in names:  # the forms recorded with dropped projections went with them
        assert [recording for recording, _ in steps.seen] == [False, True]


def test_a_step_of_someones_own_layers_runs_before_it_is_recorded(steps):
    model = _host_model(steps, POWER_OF_2)
    layer = model.layers[1]
    layer.decode_fused = lambda *args, **kw: None
    for _ in range(2):
        del steps.seen[:]
        generate(model, torch.zeros(1, 4, dtype=torch.int64), 1)
        assert [recording for recording, _ in steps.seen] == [False, True]


class _Foreign(torch.nn.Module):
    """A layer that brings what the fused step asks of one, and no more."""
    fused = False

    def _fused_linears(self):
        return {}

    def grouped_ok(self):
        return False

    grouped_plain_ok = grouped_ok


class _OwnStep(DecoderLayer):
    def decode_fused(self, *args, **kw):
        raise NotImplementedError


class _OwnForward(DecoderLayer):
    pass


@pytest.mark.parametrize("kind,ranges", ((None, 1), (_Foreign, 8), (_OwnStep, 8), (_OwnForward, 1)))
def test_key_ranges_of_someones_own_layers_go_by_the_context(steps, kind, ranges):
    """Only the step of this module's layers cuts the keys by the position."""
    model = _host_model(steps, POWER_OF_2)
    model.max_cache_len = 2048
    if kind is _Foreign:
        model.layers[1] = kind()
    elif kind is not None:
        model.layers[1].__class__ = kind
    generate(model, torch.zeros(1, ops.ATTN_SPLIT_FROM, dtype=torch.int64), 1, use_graph=False)
    assert model.cfg.attn_key_splits == ranges


@pytest.mark.parametrize("through", (copy.deepcopy, lambda layers: pickle.loads(pickle.dumps(layers))))
def test_a_copy_has_nothing_recorded(steps, through):
    """What a step sets up with the process is not part of a file."""
    model = _host_model(steps, POWER_OF_2)
    ids = torch.zeros(1, 4, dtype=torch.int64)
    generate(model, ids, 1)
    model.layers = through(model.layers)
    del steps.seen[:]
    generate(model, ids, 1)
    assert [recording for recording, _ in steps.seen] == [False, True]
    del steps.seen[:]
    generate(model, ids, 1)
    assert steps.seen == [(True, True)]


@pytest.mark.parametrize("through", (copy.copy, copy.deepcopy, lambda model: pickle.loads(pickle.dumps(model))))
def test_a_model_from_a_file_makes_its_set_up_anew(through):
    """Set-up written by an earlier version lacks what this one keeps with it."""
    cfg = LlamaConfig(**TABLE_ORDER)
    model = LlamaDecoder(cfg, max_cache_len=32, device="cpu", random_init=False, fused=False)
    for layer in model.layers:
        assert layer.grouped_plain_ok()
        for lin in layer._fused_linears().values():
            lin.__dict__.pop("_mix_rows")
    for layer in (through(layer) for layer in model.layers):
        assert not any(name in layer.__dict__ for name in SETUP)
        assert all("_mix_rows" in lin.__dict__ for lin in layer._fused_linears().values()) and layer.grouped_plain_ok()
        assert torch.equal(layer._su_qkv, torch.stack([layer.q_proj.SU, layer.k_proj.SU, layer.v_proj.SU]))
    assert all(name in layer.__dict__ for layer in model.layers for name in SETUP)  # (the copied ones keep theirs)


def test_a_recording_that_fails_ends_the_request(steps, monkeypatch):
    """One attempt: the library's stream is not the caller's any more after a recording that was cut off."""
    model = _host_model(steps, POWER_OF_2)
    ids = torch.zeros(1, 4, dtype=torch.int64)
    generate(model, ids, 1)
    tries = []

    def refuse(*args, **kw):
        tries.append(steps.recording)
        raise RuntimeError("cut off")

    monkeypatch.setattr(model, "decode_fused", refuse)
    with pytest.raises(RuntimeError, match="cut off"):
        generate(model, ids, 1)
    assert tries == [True]


@pytest.mark.gpu
@pytest.mark.parametrize("names", (SETUP, ("_grouped", "_grouped_plain")))
@pytest.mark.parametrize("cfg", (TABLE_ORDER, POWER_OF_2))
def test_requests_on_dropped_set_up(cfg, names):
    cfg = LlamaConfig(**cfg)
    ids = torch.randint(0, cfg.vocab, (1, 20), generator=torch.Generator().manual_seed(3)).cuda()
    model = LlamaDecoder(cfg, max_cache_len=64, fused=False)
    want, _, _ = generate(LlamaDecoder(cfg, max_cache_len=64, fused=False), ids, 12, use_graph=False)
    assert torch.equal(generate(model, ids, 12)[0], want)
    _drop(model, names)
    generate(model, ids, 1)  # recorded, never replayed
    assert torch.equal(generate(model, ids, 12, use_graph=False)[0], want)
    assert torch.equal(generate(model, ids, 12)[0], want)
    if cfg.hidden == 1280:
        for layer in model.layers:
            assert torch.equal(layer._su_qkv, torch.stack([layer.q_proj.SU, layer.k_proj.SU, layer.v_proj.SU]))


@pytest.mark.gpu
@pytest.mark.parametrize("fused", (True, False))
def test_sign_tables_are_made_where_a_matvec_reads_them(fused, monkeypatch):
    """Of a layer with a power-of-two hidden size and a table order behind it: down's alone."""
    cfg = LlamaConfig(hidden=2048, heads=16, kv_heads=4, layers=2, ffn=172 * 32, vocab=96)
    model = LlamaDecoder(cfg, max_cache_len=64, fused=fused)
    made, inner = [], llama_decode.sign_rows
    monkeypatch.setattr(llama_decode, "sign_rows", lambda bits, K, A, dev: made.append(K) or inner(bits, K, A, dev))
    generate(model, torch.zeros(1, 20, dtype=torch.int64, device="cuda"), 4)
    assert made == [172] * cfg.layers


@pytest.mark.gpu
def test_a_step_recorded_behind_a_prompt():
    """A prompt sets up the tables of the transforms, which is all that a recording of the step copies from host memory; it goes
    without the sign tables of the transforms inside matvecs and is replayed beside steps that have them."""
    cfg = LlamaConfig(hidden=2048, heads=16, kv_heads=4, layers=2, ffn=172 * 32, vocab=96)
    model = LlamaDecoder(cfg, max_cache_len=64)
    ids = torch.randint(0, cfg.vocab, (1, 20), generator=torch.Generator().manual_seed(3)).cuda()
    tok, pos = torch.zeros(1, 1, dtype=torch.int64, device="cuda"), torch.tensor([20], device="cuda")
    with torch.no_grad():
        model(ids, torch.arange(20, device="cuda"))
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            got = model.decode_fused(tok, pos)
        for t in (3, 50, 3):
            tok.fill_(t)
            graph.replay()
            want = model.decode_fused(tok, pos)
            torch.cuda.synchronize()
            # (down's input transform may give the neighbouring value in fp16)
            assert (got - want).norm() <= 2.5e-3 * want.norm()


@pytest.mark.gpu
@pytest.mark.parametrize("m,k,inside", ((8192, 11008, True), (8192, 13824, False), (8192, 14336, False), (5120, 14336, True), (4096, 14336, True)))
def test_a_transform_inside_a_matvec_makes_a_range_that_pays(m, k, inside):
    lin = QuantizedLinear(k, m, 16, 16, 16, 2, 2, 9, "quantlut_sym", dtype=torch.float16, mode="eval").cuda()
    assert (llama_decode._FusedLinear(lin).mix_rows() is not None) == inside
