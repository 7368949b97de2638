"""Randomised-Hadamard helpers on the HIP RHT kernel.

Counterpart of lib/utils/matmul_had.py: same names and argument meaning
(get_hadK, matmul_hadU_cuda, matmul_hadUt_cuda, op hadamard::hadamard).  The
reference runs a third-party CUDA Walsh-Hadamard kernel and then a dense
K x K matmul; here both steps (and optional sign / scale vectors) are one
kernel launch.  The order-K tables are the reference's
(lib/utils/matmul_had.py:129-95715), kept as packed sign bits in
hadamard_tables.npz.
"""
import functools
import os
import weakref

import numpy as np
import torch

from .. import ops

_ORDERS = (172, 156, 140, 124, 116, 108, 60, 52, 36, 28, 20, 12)
_npz = None
_float_tables = {}
_bit_cache = {}


@functools.lru_cache(maxsize=None)  # one per table order; reading the archive takes 0.1 ms
def _table_signs(order):
    global _npz
    if _npz is None:
        _npz = np.load(os.path.join(os.path.dirname(os.path.abspath(__file__)), "hadamard_tables.npz"),
                       allow_pickle=False)
    bits = np.unpackbits(_npz[f"had{order}"])[:order * order].reshape(order, order)
    bits.setflags(write=False)
    return bits  # 1 = -1


def is_pow2(n):
    return (n & (n - 1) == 0) and (n > 0)


def get_hadK(n, transpose=False):
    """(hadK float tensor or None, K): first table order dividing n in the
    reference's order of preference, cofactor must be a power of two
    (lib/utils/matmul_had.py:9-63)."""
    for order in _ORDERS:
        if n % order == 0:
            assert is_pow2(n // order)
            if order not in _float_tables:
                _float_tables[order] = torch.from_numpy(1.0 - 2.0 * _table_signs(order).astype(np.float32))
            had = _float_tables[order]
            return (had.T if transpose else had), order
    assert is_pow2(n)
    return None, 1


def _pack_bits(neg):
    """(K, K) boolean array neg[i][j] (True = -1) -> int32 words, column-major:
    bit j*K+i (little-endian) holds neg[i][j], the layout the kernel reads."""
    flat = np.ascontiguousarray(np.asarray(neg, dtype=np.uint8).T).reshape(-1)
    pad = (-flat.size) % 32
    flat = np.concatenate([flat, np.zeros(pad, dtype=np.uint8)])
    words = np.packbits(flat.reshape(-1, 8)[:, ::-1], axis=1).reshape(-1, 4)
    return np.ascontiguousarray(words).view("<u4").reshape(-1).view(np.int32)


def sign_rows(bits, K, A, device):
    """Signs of (table (x) H_A), K * A <= 256 rows of 8 words with bit j of row i set for -1, from the table's `bits` as had_bits
    returns them (None for K = 1); kept for the built-in tables and K = 1."""
    dev = torch.device(device)
    own = [None] if bits is None else [t for t in (False, True) if bits is _bit_cache.get((K, t, dev))]
    key = ("rows", K, A, own[0], dev) if own else None
    if key in _bit_cache:
        return _bit_cache[key]
    words = np.zeros(1, np.uint32) if bits is None else bits.cpu().numpy().view(np.uint32)
    table = np.unpackbits(words.view(np.uint8), bitorder="little")[:K * K].reshape(K, K).T
    i = np.arange(A)
    parity = i[:, None] & i[None, :]
    for s in (4, 2, 1):
        parity ^= parity >> s
    parity &= 1
    neg = (table[:, None, :, None] ^ parity[None, :, None, :]).reshape(K * A, K * A)
    rows = np.zeros((K * A, 256), np.uint8)
    rows[:, :K * A] = neg
    out = torch.from_numpy(np.packbits(rows, axis=1, bitorder="little").view(np.int32)).to(dev)
    if key:
        _bit_cache[key] = out
    return out


def had_bits(hadK, K, transpose, device):
    """Device int32 tensor of sign bits for the kernel, cached.

    hadK may be None (the built-in table of order K is used) or the caller's
    K x K tensor (as QuantizedLinear hands in); a caller-supplied tensor is
    read back once per storage, packed once per direction asked for, and must be a +-1 matrix.
    """
    dev = torch.device(device)
    if hadK is None or (K in _float_tables and hadK.data_ptr() == _float_tables[K].data_ptr()):
        key = (K, bool(transpose), dev)
        if key not in _bit_cache:
            neg = _table_signs(K).astype(bool)
            _bit_cache[key] = torch.from_numpy(_pack_bits(neg.T if transpose else neg)).to(dev)
        return _bit_cache[key]
    # a caller's own table: keyed by the memory it occupies, so a fresh view of the same table (what
    # a module hands in on every call) hits.  The entry holds a weak reference to the storage: while
    # that storage lives its address cannot belong to another tensor, and when it is freed the entry
    # goes with it (nothing of the caller's is kept alive).  An in-place change bumps `_version`.
    st = hadK.untyped_storage()
    key = (st.data_ptr(), hadK.storage_offset(), tuple(hadK.shape), tuple(hadK.stride()), hadK.dtype, dev)
    hit = _bit_cache.get(key)
    if hit is None or hit[0]() is not st or hit[1] != hadK._version:
        h = hadK.detach().to("cpu", torch.float32).numpy()
        if h.shape != (K, K) or not np.all(np.abs(h) == 1.0):
            raise ValueError("hadK must be a K x K matrix of +-1")
        neg = h < 0
        # a K x K table equal to the built-in one shares the built-in entries
        if K in _ORDERS and np.array_equal(neg, _table_signs(K)):
            neg = None
        if hit is None or hit[0]() is not st:
            weakref.finalize(st, _bit_cache.pop, key, None)
        hit = (weakref.ref(st), hadK._version, neg, {})
        _bit_cache[key] = hit
    # (a forward pass asks for one direction: packing and copying the other would be paid by every first call)
    neg, packed = hit[2:]
    bits = packed.get(bool(transpose))
    if bits is None:
        bits = had_bits(None, K, transpose, dev) if neg is None else \
            torch.from_numpy(_pack_bits(neg.T if transpose else neg)).to(dev)
        packed[bool(transpose)] = bits
    return bits


_dense_cache = {}


def _dense_sylvester(p, device):
    """H_p (Sylvester order, +-1 fp32) on the device, cached."""
    key = ("sylvester", p, torch.device(device))
    if key not in _dense_cache:
        h = torch.ones(1, 1)
        while h.shape[0] < p:
            h = torch.cat([torch.cat([h, h], 1), torch.cat([h, -h], 1)], 0)
        _dense_cache[key] = h.to(device)
    return _dense_cache[key]


_MANY_ROWS_DENSE_P = 256


def by_library(rows, n, K, on_gpu=True):
    """A transform of `rows` vectors of n = K * p runs as library products (rht_many_rows): orders and parts which
    the matrix form of the transform kernel does not take (p < 8, K > 256), from the rows on from which the
    products are faster than the kernel's one set of workgroups per row.  us, kernel / products, fp16: 688 = 172 * 4,
    96 / 300 / 1000 rows 43/61 123/60 382/61; 432 = 108 * 4 30/61 80/61 242/61; 172 * 1, 96 rows 67/63; 2048 = 512 * 4,
    96 rows 119/60; 4800 = 300 * 16, 96 rows 137/61.  In host memory, where the kernel does not run, from 96 rows on at
    every order from 100 on."""
    return rows >= 96 and K >= 100 and (not on_gpu or (rows * K >= 24000 and (n // K < 8 or K > 256)))


def rht_many_rows(x, hadK, K, transpose, pre=None, post=None, scale=None, out_dtype=None):
    """post * scale * (H_K (x) H_p)(pre * x) over the last axis of a (rows, n) fp16 / fp32 tensor,
    evaluated the way the reference does for every input (lib/utils/matmul_had.py:105-115: a
    dense K x K matmul with the table and a Walsh-Hadamard transform of the power-of-two part) -
    fp32 library GEMMs instead of the transform kernel (by_library says when)."""
    rows, n = x.shape
    p = n // K
    dev = x.device
    table = (hadK if hadK is not None else get_hadK(n)[0]).to(device=dev, dtype=torch.float32)
    M = table.T if transpose else table
    z = x.to(torch.float32)
    if pre is not None:
        z = z * pre.to(torch.float32)
    z = torch.matmul(M, z.view(rows, K, p))  # the table over the K axis, batched over the rows
    if p <= _MANY_ROWS_DENSE_P:
        z = torch.matmul(z.reshape(rows * K, p), _dense_sylvester(p, dev))
    else:  # long power-of-two parts: one workgroup of the transform kernel per p-point vector
        z = z.reshape(rows * K, p).contiguous()
        z = torch.cat([ops.rht(z[i:i + 65535], scale=1.0) for i in range(0, rows * K, 65535)], 0)
    z = z.view(rows, n) * (n**-0.5 if scale is None else scale)
    if post is not None:
        z = z * post.to(torch.float32)
    return z.to(out_dtype or x.dtype)


torch.library.define("hadamard::hadamard", "(Tensor x, float scale) -> Tensor")


@torch.library.register_fake("hadamard::hadamard")
def hadamard_abstract(x: torch.Tensor, scale: float) -> torch.Tensor:
    return torch.empty_like(x)


@torch.library.impl("hadamard::hadamard", "cuda")
def hadamard(x: torch.Tensor, scale: float) -> torch.Tensor:
    """Sylvester-ordered Walsh-Hadamard transform along the last axis times scale
    (what fast_hadamard_transform.hadamard_transform computes for the
    reference, lib/utils/matmul_had.py:99-102).  Last axis must be a power of two."""
    if x.dtype not in (torch.float16, torch.float32):
        return ops.rht(x.float().contiguous(), scale=scale).to(x.dtype)
    return ops.rht(x.contiguous(), scale=scale)


class _HadamardFn(torch.autograd.Function):
    """y = (H_K (x) H_{n/K}) x / sqrt(n) with the gradient the reference gets from the autograd
    support of its Walsh-Hadamard package plus the dense hadK matmul: the transform is linear and
    orthonormal, so grad_x = (H_K^T (x) H_{n/K}) grad_y / sqrt(n) - the same kernel with the
    order-K table transposed."""

    @staticmethod
    def forward(ctx, X, hadK, K, transpose):
        ctx.hadK, ctx.K, ctx.transpose = hadK, K, transpose
        return _hadU(X, hadK, K, transpose)

    @staticmethod
    def backward(ctx, grad):
        return _hadU(grad.contiguous(), ctx.hadK, ctx.K, not ctx.transpose), None, None, None


def _hadU(X, hadK, K, transpose):
    n = X.shape[-1]
    if K == 1:
        return torch.ops.hadamard.hadamard(X.contiguous(), n**(-0.5))
    x = X if X.dtype in (torch.float16, torch.float32) else X.float()
    if by_library(x.numel() // n, n, K, x.is_cuda):
        return rht_many_rows(x.reshape(-1, n).contiguous(), hadK, K, transpose).to(X.dtype).reshape(X.shape)
    out = ops.rht(x.contiguous(), order=K, had_bits=had_bits(hadK, K, transpose, X.device), out_dtype=x.dtype)
    return out.to(X.dtype).reshape(X.shape)


class _HadamardCastFn(torch.autograd.Function):
    """_HadamardFn of a (rows, n) fp16 / fp32 tensor with the scale and the cast that follow it in the same
    launch: out_dtype(scale * (H_K (x) H_{n/K}) x / sqrt(n)); the gradient takes the way back with its cast."""

    @staticmethod
    def forward(ctx, X, hadK, K, transpose, scale, out_dtype):
        ctx.args = (hadK, K, transpose, scale, X.dtype)
        return _hadU_cast(X, hadK, K, transpose, scale, out_dtype)

    @staticmethod
    def backward(ctx, grad):
        hadK, K, transpose, scale, in_dtype = ctx.args
        if not ops.launchable(grad):
            return (_hadU(grad.float().contiguous(), hadK, K, not transpose) * scale).to(in_dtype), None, None, None, None, None
        args = (grad, hadK, K, not transpose, scale, in_dtype)
        # (with create_graph the way back is itself recorded)
        gx = _HadamardCastFn.apply(*args) if torch.is_grad_enabled() else _hadU_cast(*args)
        return gx, None, None, None, None, None


def _hadU_cast(X, hadK, K, transpose, scale, out_dtype):
    n = X.shape[-1]
    if by_library(X.shape[0], n, K, X.is_cuda):
        return rht_many_rows(X.contiguous(), hadK, K, transpose, scale=n**-0.5 * scale, out_dtype=out_dtype)
    bits = had_bits(hadK, K, transpose, X.device) if K > 1 else None
    return ops.rht(X.contiguous(), order=K, had_bits=bits, scale=n**-0.5 * scale, out_dtype=out_dtype)


def hadU_cast(X, hadK, K, transpose, scale, out_dtype):
    """out_dtype(scale * matmul_hadU_cuda(X)), one launch; differentiable with respect to X."""
    if X.dtype not in (torch.float16, torch.float32) or not ops.launchable(X):
        return (matmul_hadU_cuda(X, hadK, K, transpose) * scale).to(out_dtype)
    return _HadamardCastFn.apply(X, hadK, K, transpose, scale, out_dtype)


class _ScaleColumnsFn(torch.autograd.Function):
    """x * s over the columns of a (rows, n) fp32 tensor; both gradients in one pass over grad and x."""

    @staticmethod
    def forward(ctx, x, s):
        ctx.save_for_backward(x, s)
        return x * s

    @staticmethod
    def backward(ctx, grad):
        x, s = ctx.saved_tensors
        if torch.is_grad_enabled() or grad.numel() == 0 or not ops.launchable(grad, x, s):
            return grad * s, (grad * x).sum(0).to(s.dtype)
        gx, gs = ops.scale_columns_grad(*(ops.aligned16(t.contiguous()) for t in (grad, x, s)))
        return gx, gs.to(s.dtype)


def scale_columns(x, s):
    """x * s for x (rows, n) and s (n,)."""
    if (x.requires_grad and s.requires_grad and x.is_cuda and s.device == x.device and x.dim() == 2
            and x.dtype == torch.float32 and s.dtype in (torch.float16, torch.float32) and s.shape == x.shape[1:]
            and x.shape[1] % 4 == 0 and ops.launchable(x, s)):
        return _ScaleColumnsFn.apply(x, s)
    return x * s


def matmul_hadU_cuda(X, hadK, K, transpose=False):
    """(H_K (x) H_{n/K}) X / sqrt(n) along the last axis (lib/utils/matmul_had.py:105-115);
    differentiable with respect to X."""
    if torch.is_grad_enabled() and X.requires_grad:
        return _HadamardFn.apply(X, hadK, K, transpose)
    return _hadU(X, hadK, K, transpose)


def matmul_hadUt_cuda(X, hadK, K):
    return matmul_hadU_cuda(X, hadK, K, transpose=True)
