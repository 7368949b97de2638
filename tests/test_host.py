"""CPU: host logic and the C-ABI surface (no kernel launches)."""
import ctypes
import os
import re

import numpy as np
import pytest
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _declared_symbols():
    text = open(os.path.join(ROOT, "include", "qtip_hip.h")).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(qtip_[a-z0-9_]+)\s*\(", text)))


def test_library_exports_every_declared_symbol():
    from qtip_amd import _lib
    assert os.path.exists(_lib.LIB_PATH), "build with python -m qtip_amd.build"
    handle = ctypes.CDLL(_lib.LIB_PATH)
    declared = _declared_symbols()
    assert len(declared) >= 7
    for name in declared:
        assert hasattr(handle, name), name
    assert sorted(_lib.EXPORTED_SYMBOLS) == declared
    assert _lib.lib().qtip_abi_version() == _lib.ABI_VERSION
    assert b"shape" in _lib.lib().qtip_error_string(-1)


def test_measurement_aids_live_in_a_library_of_their_own():
    """libqtip_hip.so exports no probe; bench_probe/libqtip_probe.so exports what its header declares."""
    from qtip_amd import _lib
    import bench_probe
    main = ctypes.CDLL(_lib.LIB_PATH)
    assert os.path.exists(bench_probe.LIB_PATH), "build with python -m bench_probe"
    probe = ctypes.CDLL(bench_probe.LIB_PATH)
    text = open(os.path.join(ROOT, "bench_probe", "qtip_probe.h")).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    names = sorted(set(re.findall(r"\b(qtip_probe_[a-z0-9_]+)\s*\(", text)))
    assert names == ["qtip_probe_issue", "qtip_probe_stream_read"]
    for name in names:
        assert hasattr(probe, name), name
        assert not hasattr(main, name), name


def test_python_host_never_routes_through_the_shared_scratch_entry_point():
    """qtip_decompress_matvec_noalloc keeps its partial sums in one array per GPU, so overlapping
    calls race: it is for callers of the C ABI that accept that.  The package's own wrappers (which
    serve any number of streams) bind it but never call it."""
    import glob
    hits = []
    for path in glob.glob(os.path.join(ROOT, "qtip_amd", "**", "*.py"), recursive=True):
        for n, line in enumerate(open(path), 1):
            if "qtip_decompress_matvec_noalloc" in line and not path.endswith("_lib.py"):
                hits.append((path, n))
    assert hits == []


def test_argument_rejection_without_gpu():
    # rejected arguments return a negative code before anything touches the device
    from qtip_amd import _lib
    L = _lib.lib()
    buf = ctypes.create_string_buffer(4096)
    p = ctypes.cast(buf, ctypes.c_void_p)
    null = ctypes.c_void_p(0)
    assert L.qtip_decompress_matvec(p, p, p, p, 33, 64, 2, null, 0, null) == -1
    assert L.qtip_decompress_matvec(p, p, p, p, 64, 64, 5, null, 0, null) == -1
    assert L.qtip_decompress_matvec(null, p, p, p, 64, 64, 2, null, 0, null) == -2
    assert L.qtip_decode(p, p, null, 64, 64, 2, null) == -2
    assert L.qtip_decompress_gemm(p, p, p, p, 64, 64, 2, 0, 0, null, 0, null) == -1
    assert L.qtip_gemm_workspace_bytes(33, 64, 2, 8) == 0
    assert L.qtip_rht(p, 0, p, 0, 1, 1, 100, 1, null, null, null, 1.0, null) == -1  # not a power of two
    assert L.qtip_rht(p, 0, p, 0, 1, 1, 12 * 64, 12, null, null, null, 1.0, null) == -2  # table missing
    assert L.qtip_rht(p, 7, p, 0, 1, 1, 64, 1, null, null, null, 1.0, null) == -5
    assert L.qtip_matvec_split(33, 64, 2) == 0 and L.qtip_matvec_split(64, 64, 7) == 0
    assert L.qtip_decompress_matvec_parts(p, p, p, p, 64, 64, 2, 0, null) in (-1, 100, 101)  # bad nparts (or no device)
    assert L.qtip_decompress_matvec_parts(null, p, p, p, 64, 64, 2, 1, null) == -2


def test_cpu_tensors_raise():
    from qtip_amd import ops
    with pytest.raises(ValueError):
        ops.decode(torch.zeros(64 * 64 * 2 // 16, dtype=torch.int16), torch.zeros(512, 2, dtype=torch.float16), 64, 64, 2)
    import qtip_amd.utils.matmul_had  # registers hadamard::hadamard (GPU implementation only)
    with pytest.raises(NotImplementedError):
        torch.ops.hadamard.hadamard(torch.zeros(2, 64), 1.0)


def test_has_kernel_gate():
    from qtip_amd.utils.kernel_check import has_kernel
    assert has_kernel('quantlut_sym', 16, 2, 2, 9, 16, 16)
    assert has_kernel('quantlut_sym', 16, 4, 2, 9, 16, 16)
    for bad in [('lut', 16, 2, 2, 9, 16, 16), ('quantlut_sym', 12, 2, 2, 9, 16, 16), ('quantlut_sym', 16, 5, 2, 9, 16, 16),
                ('quantlut_sym', 16, 1, 2, 9, 16, 16), ('quantlut_sym', 16, 2, 1, 9, 16, 16),
                ('quantlut_sym', 16, 2, 2, 10, 16, 16), ('quantlut_sym', 16, 2, 2, 9, 8, 16)]:
        assert not has_kernel(*bad)


def test_op_registry_names():
    import qtip_amd.codebook as cbk
    # every Llama-2 7B / 70B layer shape at every bit width, under the reference's naming scheme
    for m, k in [(4096, 4096), (12288, 4096), (22016, 4096), (4096, 11008), (10240, 8192), (8192, 8192),
                 (57344, 8192), (8192, 28672), (28672, 8192)]:
        for b in (2, 3, 4):
            assert (m, 1, k, b) in cbk.kdict
            assert hasattr(torch.ops.quip_lib, f"decompress_matvec_qtip_{m}_1_{k}_{b}")
    assert len([k for k in cbk.kernels if k[0] != 256]) == 61
    op = cbk.register_shape(64, 128, 3)
    assert op is cbk.kdict[(64, 1, 128, 3)]
    with pytest.raises(ValueError):
        cbk.register_shape(48, 128, 3)
    # fake (meta) implementation: shape/dtype only
    out = torch.ops.quip_lib.decompress_matvec_qtip_4096_1_4096_2(
        torch.empty(1, device="meta", dtype=torch.int16), torch.empty(1, 4096, device="meta"),
        torch.empty(512, 2, device="meta", dtype=torch.float16))
    assert out.shape == (1, 4096) and out.dtype == torch.float32


def test_quantlut_sym_matches_oracle():
    from oracle import qtip_oracle as O
    from qtip_amd.codebook.bitshift import quantlut_sym
    t = torch.randn(512, 2, generator=torch.Generator().manual_seed(0)).half()
    a = quantlut_sym(t, 16, 9).numpy().view(np.uint16)
    b = O.quantlut_sym(t.numpy()).view(np.uint16)
    assert np.array_equal(a, b)


def test_tlut_roundtrip_through_expanded_table():
    from qtip_amd.codebook.bitshift import quantlut_sym
    from qtip_amd.utils.kernel_decompress import _representatives, tlut_from_expanded
    t = torch.randn(512, 2, generator=torch.Generator().manual_seed(1)).half()
    back = tlut_from_expanded(quantlut_sym(t, 16, 9))
    seen = _representatives()[2]
    assert torch.equal(back[seen], t[seen])
    # every index some state hashes to is covered (all 512 are reachable)
    assert int(seen.sum()) == 512


def test_unpack_trellis_matches_oracle():
    from oracle import qtip_oracle as O
    from qtip_amd.codebook.bitshift import bitshift_codebook
    for K in (2, 3, 4):
        cb = bitshift_codebook(16, K, 2, 9, 'quantlut_sym', tlut=torch.zeros(512, 2, dtype=torch.float16))
        words = np.random.default_rng(K).integers(0, 65536, (6, 16 * K), dtype=np.uint16)
        got = cb.unpack_trellis(torch.from_numpy(words.view(np.int16)), 256).numpy()
        assert np.array_equal(got, O.unpack_trellis_natural(words, K))


def test_get_hadK_and_bits():
    from oracle import qtip_oracle as O
    from qtip_amd.utils import matmul_had as mh
    for n in (4096, 11008, 12288, 10240, 28672, 57344, 22016):
        had, K = mh.get_hadK(n)
        ohad, oK = O.get_hadK(n)
        assert K == oK
        if K > 1:
            assert np.array_equal(had.numpy(), ohad)
            assert np.array_equal(mh.get_hadK(n, transpose=True)[0].numpy(), ohad.T)
    with pytest.raises(AssertionError):
        mh.get_hadK(100)
    neg = np.random.default_rng(0).integers(0, 2, (20, 20)).astype(bool)
    w = mh._pack_bits(neg).view(np.uint32)
    for i in range(20):
        for j in range(20):
            b = j * 20 + i
            assert ((w[b >> 5] >> (b & 31)) & 1) == neg[i, j]


def test_had_bits_cache_follows_the_memory_not_the_object():
    """A caller's own table: a fresh view of the same memory hits the cache (no repacking, hence no
    device-to-host copy per forward), an in-place change or a new tensor misses, and an entry
    disappears with the storage it was packed from."""
    import gc
    from qtip_amd.utils import matmul_had as mh
    rng = np.random.default_rng(3)
    K = 8  # no built-in table of this order: the caller's own entry is used
    h = torch.from_numpy(np.where(rng.integers(0, 2, (K, K)) > 0, 1.0, -1.0).astype(np.float32))
    mh._bit_cache.clear()
    b0 = mh.had_bits(h, K, False, "cpu")
    n_entries = len(mh._bit_cache)
    assert mh.had_bits(h.data, K, False, "cpu") is b0          # another tensor object, same memory
    assert mh.had_bits(h.view(K, K), K, False, "cpu") is b0
    assert len(mh._bit_cache) == n_entries
    bt = mh.had_bits(h, K, True, "cpu")
    assert bt is not b0 and torch.equal(bt, torch.from_numpy(mh._pack_bits((h.numpy() < 0).T)))
    h[0, 0] = -h[0, 0]                                          # in-place edit: version bump, repacked
    b1 = mh.had_bits(h, K, False, "cpu")
    assert b1 is not b0 and torch.equal(b1, torch.from_numpy(mh._pack_bits(h.numpy() < 0)))
    h2 = h.clone()
    assert mh.had_bits(h2, K, False, "cpu") is not b1           # other memory: its own entry
    before = len(mh._bit_cache)
    del h2
    gc.collect()
    assert len(mh._bit_cache) == before - 1                     # freed storage: entry dropped
    with pytest.raises(ValueError):
        mh.had_bits(torch.zeros(K, K), K, False, "cpu")


def test_quantiser_entry_points_raise():
    from qtip_amd.codebook.bitshift import BitshiftLinear, bitshift_codebook
    cb = bitshift_codebook(16, 2, 2, 9, 'quantlut_sym')
    with pytest.raises(NotImplementedError):
        cb.quantize(None)
    with pytest.raises(NotImplementedError):
        bitshift_codebook(12, 2, 1, 16, '1mad')  # only 16-bit state windows are built
    with pytest.raises(ValueError):  # packing states needs device tensors
        cb.pack_trellis(torch.zeros(1, 128, dtype=torch.int32))
    with pytest.raises(ValueError):
        BitshiftLinear(16, 16, 16, 5, 2, 9, 'quantlut_sym', has_kernel=True)


def test_rope_scaling_follows_the_rotary_initialisers():
    """rope_inv_freq against the initialisers the reference's LlamaRotaryEmbedding uses
    (model/llama.py:39,185: transformers' ROPE_INIT_FUNCTIONS) for the static types."""
    import torch
    from qtip_amd.llama_decode import LlamaConfig, rope_inv_freq
    base = dict(hidden=4096, heads=32, rope_theta=500000.0)
    plain = rope_inv_freq(LlamaConfig(**base))
    want = 1.0 / (500000.0**(torch.arange(0, 128, 2, dtype=torch.float32) / 128))
    assert torch.equal(plain, want)
    lin = rope_inv_freq(LlamaConfig(**base, rope_scaling={"type": "linear", "factor": 4.0}))
    assert torch.allclose(lin, want / 4.0, rtol=0, atol=0)
    l3 = {"rope_type": "llama3", "factor": 8.0, "low_freq_factor": 1.0, "high_freq_factor": 4.0,
          "original_max_position_embeddings": 8192}
    got = rope_inv_freq(LlamaConfig(**base, rope_scaling=l3))
    # closed-form properties: short wavelengths untouched, long ones divided by the factor, monotone in between
    wavelen = 2 * torch.pi / want
    assert torch.equal(got[wavelen < 8192 / 4.0], want[wavelen < 8192 / 4.0])
    assert torch.allclose(got[wavelen > 8192 / 1.0], want[wavelen > 8192 / 1.0] / 8.0)
    mid = ~(wavelen < 8192 / 4.0) & ~(wavelen > 8192 / 1.0)
    assert mid.any() and bool(((got[mid] <= want[mid]) & (got[mid] >= want[mid] / 8.0)).all())
    try:
        from transformers import LlamaConfig as HFConfig
        from transformers.modeling_rope_utils import ROPE_INIT_FUNCTIONS
    except Exception:  # the library moved the table: the closed-form checks above stand alone
        return
    hf = HFConfig(hidden_size=4096, num_attention_heads=32, rope_theta=500000.0, rope_scaling=dict(l3),
                  max_position_embeddings=131072)
    ref, att = ROPE_INIT_FUNCTIONS["llama3"](hf, "cpu")
    assert att == 1.0 and torch.allclose(got, ref, rtol=1e-6, atol=0)
    with pytest.raises(NotImplementedError):
        rope_inv_freq(LlamaConfig(**base, rope_scaling={"rope_type": "dynamic", "factor": 2.0}))


def test_sampling_helpers_follow_the_generation_script():
    """top-k restriction and the exponential-race draw of eval/interactive_gen.py:15-40."""
    from qtip_amd.llama_decode import logits_to_probs, sample
    g = torch.Generator().manual_seed(0)
    logits = torch.randn(2, 50, generator=g)
    p = logits_to_probs(logits, temperature=0.6, top_k=5)
    assert torch.allclose(p.sum(-1), torch.ones(2))
    assert ((p > 0).sum(-1) == 5).all()
    top = logits.topk(5).indices
    assert all(set(torch.nonzero(p[i]).flatten().tolist()) == set(top[i].tolist()) for i in range(2))
    # ratios inside the kept set are those of softmax(logits / T)
    full = torch.softmax(logits / 0.6, -1)
    i0, i1 = top[0, 0], top[0, 1]
    assert abs(p[0, i0] / p[0, i1] - full[0, i0] / full[0, i1]) < 1e-4
    # top_k = 1 is greedy whatever the random draw
    torch.manual_seed(1)
    tok, _ = sample(logits[:, None, :], temperature=0.6, top_k=1)
    assert (tok.flatten() == logits.argmax(-1)).all()
    # the exponential race draws from the distribution: frequencies of a 3-way distribution
    torch.manual_seed(2)
    lg = torch.log(torch.tensor([0.7, 0.2, 0.1])).repeat(6000, 1)[:, None, :]
    tok, _ = sample(lg)
    freq = torch.bincount(tok.flatten(), minlength=3).float() / 6000
    assert (freq - torch.tensor([0.7, 0.2, 0.1])).abs().max() < 0.03


def test_bench_refuses_more_than_one_gpu():
    """bench.py measures one GPU: any other --gpus value ends with a message and a non-zero
    status before the library or a device is touched."""
    import os
    import subprocess
    import sys
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    r = subprocess.run([sys.executable, os.path.join(root, "bench.py"), "--gpus", "2"], capture_output=True,
                       text=True, timeout=120)
    assert r.returncode == 2
    assert "one GPU" in r.stderr and r.stdout.strip() == ""


def test_generate_refuses_requests_beyond_the_cache():
    """The fused decode step keeps its position in device memory and would silently drop keys past
    the cache; the request is checked on the host before anything runs."""
    from qtip_amd.llama_decode import FUSED_MAX_CACHE_LEN, LlamaConfig, LlamaDecoder, generate
    cfg = LlamaConfig(hidden=256, heads=4, kv_heads=2, layers=1, ffn=512, vocab=64)
    model = LlamaDecoder(cfg, max_cache_len=16, device="cpu")
    ids = torch.zeros((1, 10), dtype=torch.int64)
    with pytest.raises(ValueError, match="does not fit"):
        generate(model, ids, 8)  # positions up to 16 needed, slots 0..15 exist
    with pytest.raises(ValueError, match="does not fit"):
        generate(model, torch.zeros((1, 17), dtype=torch.int64), 1)
    assert model.supports_fused_decode()
    long = LlamaDecoder(cfg, max_cache_len=FUSED_MAX_CACHE_LEN + 1, device="cpu")
    assert not long.supports_fused_decode()  # generate() then decodes module by module
    with pytest.raises(ValueError, match="fused decode step covers"):
        long.decode_fused(torch.zeros((1, 1), dtype=torch.int64), torch.tensor([0]))


@pytest.mark.parametrize("n", [9, 30])
def test_forward_refuses_more_tokens_than_the_cache_has_slots(n):
    """From the shapes alone, before a layer runs: past the cache keys and values would be dropped."""
    from qtip_amd.llama_decode import LlamaConfig, LlamaDecoder
    model = LlamaDecoder(LlamaConfig(hidden=256, heads=4, kv_heads=2, layers=1, ffn=832, vocab=96), max_cache_len=8,
                         device="cpu", random_init=False)
    with torch.no_grad(), pytest.raises(ValueError, match="do not fit the key / value cache"):
        model(torch.zeros(1, n, dtype=torch.int64), torch.arange(n))


def test_had_bits_reads_a_table_once_for_both_directions(monkeypatch):
    """A training step needs a table and its transpose: the caller's copy is read back and checked once."""
    from qtip_amd.utils import matmul_had as mh
    h, K = mh.get_hadK(12 * 64)
    for own in (h.clone(), h.flip(0).contiguous()):  # equal to the built-in table, and another one
        mh.had_bits(own, K, False, "cpu")
        reads = []
        monkeypatch.setattr(mh.np, "abs", lambda *a: reads.append(1))
        bt = mh.had_bits(own, K, True, "cpu")
        monkeypatch.undo()
        assert not reads and torch.equal(bt, torch.from_numpy(mh._pack_bits((own.numpy() < 0).T)))
    assert not mh._table_signs(K).flags.writeable


def test_had_bits_packs_the_direction_asked_for(monkeypatch):
    """A forward pass asks for one direction of a table; the other is packed when something asks for it."""
    from qtip_amd.utils import matmul_had as mh
    h, K = mh.get_hadK(20 * 64)
    packed, pack = [], mh._pack_bits
    monkeypatch.setattr(mh, "_pack_bits", lambda neg: packed.append(1) or pack(neg))
    monkeypatch.setattr(mh, "_bit_cache", {})
    for own in (h.clone(), h.flip(0).contiguous()):
        mh._bit_cache.clear()
        for calls, transpose in ((1, True), (1, True), (2, False), (2, False)):
            bits = mh.had_bits(own, K, transpose, "cpu")
            assert len(packed) == calls
            neg = own.numpy() < 0
            assert torch.equal(bits, torch.from_numpy(pack(neg.T if transpose else neg)))
        packed.clear()
        own.neg_()
        assert torch.equal(mh.had_bits(own, K, False, "cpu"), torch.from_numpy(pack(~neg)))
        packed.clear()


@pytest.mark.parametrize("n,K", [(11008, 172), (1248, 156), (624, 156)])
def test_large_orders_in_host_memory(n, K):
    """From 96 rows on, orders from 100 on are products, which run on the CPU too; against float64."""
    from qtip_amd.utils import matmul_had as mh
    had, order = mh.get_hadK(n)
    assert order == K
    p = n // K
    h = torch.ones(1, 1, dtype=torch.float64)
    while h.shape[0] < p:
        h = torch.cat([torch.cat([h, h], 1), torch.cat([h, -h], 1)])
    x = torch.randn(96, n, generator=torch.Generator().manual_seed(n))
    for t in (False, True):
        ref = ((had.T if t else had).double() @ (x.double().view(96, K, p) @ h)).reshape(96, n) / n**0.5
        y = x.clone().requires_grad_()
        for out in (mh.matmul_hadU_cuda(x, had, K, t), mh.hadU_cast(x, had, K, t, 1.0, torch.float32), mh.matmul_hadU_cuda(y, had, K, t)):
            assert float((out.detach().double() - ref).abs().max()) <= 1e-5 * float(ref.abs().max())
        (g,) = torch.autograd.grad(out, y, x)
        back = ((had if t else had.T).double() @ (x.double().view(96, K, p) @ h)).reshape(96, n) / n**0.5
        assert float((g.double() - back).abs().max()) <= 1e-5 * float(back.abs().max())


@pytest.mark.parametrize("grad", [False, True])
def test_module_without_a_kernel_in_host_memory(grad):
    """Projection of large table orders on the CPU, 96 rows or more: input and output transforms are products."""
    from qtip_amd.codebook.bitshift import BitshiftLinear
    from qtip_amd.utils import matmul_had as mh
    m, k, K = 928, 1248, 2
    g = torch.Generator().manual_seed(2)
    mod = BitshiftLinear(16, 16, 16, K, 2, 9, "quantlut_sym", tlut=torch.randn(512, 2, generator=g).half(), has_kernel=False)
    states = torch.randint(0, 1 << 16, (m // 16 * k // 16, 128), generator=g)
    x = torch.randn(100, k, generator=g)
    SU, SV = torch.randn(k, generator=g).sign().half(), torch.randn(m, generator=g).requires_grad_(grad)
    (hl, kl), (hr, kr) = mh.get_hadK(k), mh.get_hadK(m)
    y = mod(x, states, SU, SV, hl, hr, kl, kr, 0, 8, mode="train-recons")
    w = mod.get_hatW(states, m, k).double()
    h8 = torch.tensor([[(-1.0)**bin(i & j).count("1") for j in range(8)] for i in range(8)], dtype=torch.float64)
    t = lambda v, had, n: (had.double() @ (v.reshape(-1, had.shape[0], 8) @ h8)).reshape(-1, n) / n**0.5
    want = t((t(x.double() * SU.double(), hl.T, k) / 32).half().double() @ w.T, hr, m) * SV.detach().double() * 32
    assert y.requires_grad == grad
    assert float((y.detach().double() - want).norm() / want.norm()) <= 2.0**-10  # the product's rounding to fp16, once


def test_native_host_module_leaves_host_tensors_to_the_checks():
    from qtip_amd import _lib
    x = torch.zeros(1, 256, dtype=torch.float16)
    packed, tlut = torch.zeros(256 * 256 // 8, dtype=torch.int16), torch.zeros(512, 2, dtype=torch.float16)
    assert _lib.host().matvec(packed, x, tlut, 256, 256, 2, 0, 0, 0) is None
    assert _lib.host().linear(x, packed, tlut, x[0], x[0].float(), None, 1, None, 1, 256, 256, 2, 1.0, 1.0, False, 96, 0) is None


def test_a_tensor_with_a_tangent_is_not_launchable():
    from torch.autograd import forward_ad
    from qtip_amd import ops
    x = torch.randn(3, 8)
    assert ops.launchable(x)
    with forward_ad.dual_level():
        d = forward_ad.make_dual(x, torch.ones_like(x))
        assert not d.requires_grad and not ops.launchable(d) and not ops.launchable(x, d) and ops.launchable(x)
    assert ops.launchable(x)
    seen = []
    torch.func.jvp(lambda v: seen.append(ops.launchable(v)) or v, (x,), (x,))
    assert seen == [False]


def test_nothing_is_launchable_while_a_trace_records():
    """(A recorded program would hold the output's allocation and not the launch that fills it.)"""
    from qtip_amd import ops
    x, seen = torch.randn(3, 8), []
    torch.jit.trace(lambda v: seen.append(ops.launchable(v)) or v + 1, (x,), check_trace=False)
    assert seen == [False] and ops.launchable(x)


def test_symbolic_traces_of_the_norm_and_the_rotary_tables():
    import torch.fx
    from qtip_amd.llama_decode import LlamaConfig, LlamaDecoder, RMSNorm

    class Rope(torch.nn.Module):

        def forward(self, p):
            return model.rope(p)

    x, mod = torch.randn(3, 8).half(), RMSNorm(8, 1e-5)
    assert torch.equal(torch.fx.symbolic_trace(mod)(x), mod(x))
    model = LlamaDecoder(LlamaConfig(hidden=256, heads=4, kv_heads=2, layers=0, ffn=512, vocab=64, K=2), 64, device="cpu")
    pos = torch.arange(9)
    assert all(torch.equal(a, b) for a, b in zip(torch.fx.symbolic_trace(Rope())(pos), model.rope(pos)))


def test_scripted_norm():
    from qtip_amd.llama_decode import RMSNorm
    x, mod = torch.randn(3, 8).half(), RMSNorm(8, 1e-5)
    assert torch.equal(torch.jit.script(mod)(x), mod(x))


@pytest.mark.parametrize("fused", [True, False])
def test_a_layer_holds_its_projections_and_norms(fused):
    """(A model saved whole by an earlier version has no more than these.)"""
    from qtip_amd.llama_decode import DecoderLayer, LlamaConfig
    layer = DecoderLayer(LlamaConfig(hidden=256, heads=4, kv_heads=2, layers=1, ffn=512, vocab=64, K=2), None, "cpu", fused=fused)
    assert not dict(layer.named_buffers(recurse=False)) and not dict(layer.named_parameters(recurse=False))


@pytest.mark.parametrize("there", [False, True])
def test_library_without_a_host_module_that_loads(there, tmp_path, monkeypatch):
    """The native host module shortens calls; a tree that holds the library alone has all of them."""
    from qtip_amd import _lib
    path = tmp_path / "_qtip_host.so"
    if there:
        path.write_bytes(b"for another interpreter")
    monkeypatch.setattr(_lib, "HOST_PATH", str(path))
    monkeypatch.setattr(_lib, "_host", None)
    with pytest.warns(RuntimeWarning, match="qtip_amd.build"):
        assert not _lib.host()
    assert not _lib.host()  # (asked once)


def test_host_module_of_another_version(tmp_path, monkeypatch):
    """A module for another version of the library is refused; one for another torch is left alone."""
    from qtip_amd import _lib
    for abi, version in ((None, None), (_lib.ABI_VERSION - 1, torch.__version__), (_lib.ABI_VERSION, "1.0")):
        path = tmp_path / f"host_{abi}_{version}.py"
        text = "def bind(*a): raise AssertionError('bound')\n"
        path.write_text(text if abi is None else text + f"abi_version = {abi}\ntorch_version = {str(version)!r}\n")
        monkeypatch.setattr(_lib, "HOST_PATH", str(path))
        monkeypatch.setattr(_lib, "_host", None)
        if abi == _lib.ABI_VERSION:
            with pytest.warns(RuntimeWarning, match="torch 1.0"):
                assert not _lib.host()
        else:
            with pytest.raises(_lib.QtipLibraryError, match="rebuild"):
                _lib.host()


def test_header_and_host_module_are_of_one_version():
    from qtip_amd import _lib
    text = open(os.path.join(ROOT, "include", "qtip_hip.h")).read()
    assert int(re.search(r"#define QTIP_ABI_VERSION (\d+)", text)[1]) == _lib.ABI_VERSION == _lib.host().abi_version
    assert _lib.host().torch_version == torch.__version__


def test_key_ranges_of_a_context():
    """One workgroup a head for short contexts; ranges fit the chip side by side, as many as the kernel takes."""
    from qtip_amd import ops
    line, many = ops.ATTN_SPLIT_FROM, ops.ATTN_SPLIT_FROM_MANY
    for heads in (None, 1, 8, 32, 40):
        assert [ops.attention_key_splits(c, heads) for c in (1, line - 1, line, 4096)] == [1, 1, 8, 8]
    assert ops.attention_key_splits(line) == 8
    for heads, ranges in ((41, 6), (64, 4), (128, 2), (256, 1), (300, 1)):
        assert [ops.attention_key_splits(c, heads) for c in (line, many - 1, many, 4096)] == [1, 1, ranges, ranges]
        assert ranges <= ops.ATTN_MAX_KEY_SPLITS


@pytest.mark.parametrize("K,A", ((172, 1), (28, 8), (20, 4), (108, 2), (1, 256), (1, 1)))
@pytest.mark.parametrize("transpose", (True, False))
def test_sign_rows_of_a_table(K, A, transpose):
    from scipy.linalg import hadamard
    from qtip_amd.utils import matmul_had as mh
    rows = mh.sign_rows(mh.had_bits(None, K, transpose, "cpu") if K > 1 else None, K, A, "cpu")
    neg = mh._table_signs(K).astype(bool) if K > 1 else np.zeros((1, 1), bool)
    full = np.kron(np.where(neg.T if transpose else neg, -1, 1), hadamard(A)) < 0
    bits = np.unpackbits(rows.numpy().view(np.uint8).reshape(K * A, 32), axis=1, bitorder="little").astype(bool)
    assert np.array_equal(bits[:, :K * A], full) and not bits[:, K * A:].any()


def test_sign_rows_are_made_once():
    """Also for transforms without a table."""
    from qtip_amd.utils import matmul_had as mh
    for K, A in ((1, 32), (12, 4)):
        bits = mh.had_bits(None, K, True, "cpu") if K > 1 else None
        assert mh.sign_rows(bits, K, A, "cpu") is mh.sign_rows(bits, K, A, "cpu")
    assert not torch.equal(mh.sign_rows(None, 1, 32, "cpu")[:256], mh.sign_rows(None, 1, 64, "cpu")[:256])


def test_bench_names_every_kernel_source_of_its_traffic_figure():
    """The digest that the counter figure is tied to covers the matvec's file and every header beside it that it includes."""
    import os
    import bench
    sources = bench.kernel_sources()
    assert len(set(sources)) == len(sources) and sources[0] == "qtip_hip.hip"
    for name in sources:
        with open(os.path.join(bench.KERNEL_DIR, name)) as f:
            lines = [l.split('"')[1] for l in f if l.startswith("#include \"") and "/" not in l.split('"')[1]]
        assert set(lines) <= set(sources), name
    assert {"qtip_chain.h", "qtip_device.h", "qtip_mix.h", "qtip_setup.h", "qtip_shares.h", "qtip_wht.h"} <= set(sources)
