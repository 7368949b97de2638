"""Tensor-level wrappers over the C ABI (include/qtip_hip.h).

Every function launches on the current stream of the tensors' device and
returns without synchronising.  Inputs are checked here (device, dtype,
contiguity, sizes) so that a bad argument raises instead of reaching a kernel.
"""
import contextlib
import ctypes
import math

import torch
from torch.autograd import forward_ad

from . import _lib
from ._lib import QTIP_F16, QTIP_F32, check, host, lib, require_cuda, stream_ptr

_DT = {torch.float16: QTIP_F16, torch.float32: QTIP_F32}
_Tensor, _F16, _F32, _BITS = torch.Tensor, torch.float16, torch.float32, (2, 3, 4)
_PACKED_TYPES = (torch.int16, torch.uint16, torch.int32, torch.uint8)

# scratch for split-k partial sums, one buffer per (device, stream): launches on one stream are
# ordered, launches on different streams must not share partial results
_WORKSPACE = {}
_WORKSPACE_BYTES = 8 << 20
_SPLIT = {}


def _workspace(device, need, stream=None):
    """Scratch of at least `need` bytes for the current stream (`stream`, if the caller has looked it up).  A request beyond the current
    buffer gets a larger one, and the smaller ones stay alive for the life of the process: a
    HIP graph recorded earlier still holds their addresses."""
    dev = device.index if device.index is not None else torch.cuda.current_device()
    key = (dev, stream_ptr(device) if stream is None else stream)
    held = _WORKSPACE.setdefault(key, [])
    if not held or held[-1].numel() < need:
        held.append(torch.empty(max(need, _WORKSPACE_BYTES), dtype=torch.uint8, device=device))
    return held[-1]


def matvec_split(m, k, bits, device):
    """Number of k splits the matvec kernel uses for this shape (cached per device)."""
    key = (m, k, bits, device.index)
    s = _SPLIT.get(key)
    if s is None:
        with _on(device):
            s = lib().qtip_matvec_split(m, k, bits)
        if s < 1:
            raise ValueError(f"unsupported matvec shape {m}x{k} at {bits} bits")
        _SPLIT[key] = s
    return s


def _ptr(t):
    return t.data_ptr() if t is not None else None


_HERE = contextlib.nullcontext()


def _on(device):
    """torch.cuda.device(device), which costs two device switches, only where that is not the current one."""
    return _HERE if torch.cuda.current_device() == device.index else torch.cuda.device(device)


# rows from which an input that does not start on 16 bytes is copied: the transforms of many rows read 16 bytes at a
# time, and without the copy every row goes back to workgroups of its own.  us, as it stands / copied: 11008 fp16, 96 rows
# 73/19, 1000 rows 669/29; 4096, 24 rows 14/18, 96 rows 23/18, 1000 rows 231/19; 28672, 1000 rows 1286/58
_ALIGN_ROWS = 96


def aligned16(t):
    """t (contiguous) or None, copied if it does not start on 16 bytes."""
    return t if t is None or t.data_ptr() % 16 == 0 else t.clone()


_is_compiling, _is_tracing, _modes = torch.compiler.is_compiling, torch.jit.is_tracing, torch._C._len_torch_dispatch_stack


def launchable(*tensors):
    """The tensors are memory that a launch can be given: nothing traces the program, and none of them is a wrapper
    (batched gradients, fake tensors) or carries a tangent.  What passes by torch's own or registered operations asks this
    first."""
    if _is_compiling() or _modes() or _is_tracing():
        return False
    try:
        for t in tensors:
            if not t.data_ptr() and t.numel():
                return False
        # (forward-mode derivatives: such a tensor has ordinary memory and no requires_grad)
        return forward_ad._current_level < 0 or all(forward_ad.unpack_dual(t).tangent is None for t in tensors)
    except RuntimeError:
        return False


def _check_packed(packed, m, k, bits):
    require_cuda(packed, "packed trellis", _PACKED_TYPES)
    if bits not in _BITS:
        raise ValueError(f"bits must be 2, 3 or 4 (got {bits})")
    if m % 32 or k % 32 or m <= 0 or k <= 0:
        raise ValueError(f"shape {m}x{k}: m and k must be positive multiples of 32")
    nbytes = packed.numel() * packed.element_size()
    if nbytes * 8 != bits * m * k:
        raise ValueError(f"packed trellis holds {nbytes} bytes, {m}x{k} at {bits} bits needs {bits * m * k // 8}")


def _check_tlut(tlut, device):
    require_cuda(tlut, "codebook (tlut)", torch.float16)
    if tlut.numel() != 1024:
        raise ValueError(f"codebook must hold 512 x 2 fp16 values (got {tuple(tlut.shape)})")
    if tlut.device != device:
        raise ValueError("codebook is on a different device")


def decode(packed, tlut, m, k, bits):
    """Kernel-packed trellis -> dense (m, k) fp16 weight matrix (bit-exact)."""
    _check_packed(packed, m, k, bits)
    _check_tlut(tlut, packed.device)
    out = torch.empty((m, k), dtype=torch.float16, device=packed.device)
    with _on(packed.device):
        check(lib().qtip_decode(_ptr(out), _ptr(packed), _ptr(tlut), m, k, bits, stream_ptr(packed.device)),
              "qtip_decode")
    return out


def decompress_matvec(packed, x, tlut, m, k, bits, out=None, split_k=True):
    """out[m] fp32 = decode(packed)[m,k] @ x[k]; x is fp16 with k elements."""
    dev = packed.device
    _check_packed(packed, m, k, bits)
    _check_tlut(tlut, dev)
    require_cuda(x, "x", _F16)
    if x.numel() != k or x.device != dev:
        raise ValueError(f"x must hold {k} fp16 values on {dev}")
    if out is None:
        out = torch.empty((m,), dtype=_F32, device=dev)
    else:
        require_cuda(out, "out", _F32)
        if out.numel() != m:
            raise ValueError(f"out must hold {m} fp32 values")
    stream = stream_ptr(dev)
    wsp, wsb = None, 0
    if split_k and matvec_split(m, k, bits, dev) > 1:
        ws = _workspace(dev, 16 * m * 4, stream)
        wsp, wsb = _ptr(ws), ws.numel()
    with _on(dev):
        check(lib().qtip_decompress_matvec(out.data_ptr(), packed.data_ptr(), x.data_ptr(), tlut.data_ptr(), m, k, bits,
                                           wsp, wsb, stream), "qtip_decompress_matvec")
    return out


def matvec_row(packed, x, tlut, m, k, bits):
    """decompress_matvec of operands that fit as they are, as a (1, m) tensor, in one native function; None for any other."""
    if not (isinstance(packed, _Tensor) and packed.is_cuda) or _is_compiling() or bits not in _BITS or (m | k) & 31:
        return None
    native = host()
    if not native:
        return None
    dev = packed.device
    stream = stream_ptr(dev)
    wsp, wsb = 0, 0
    if matvec_split(m, k, bits, dev) > 1:
        ws = _workspace(dev, 16 * m * 4, stream)
        wsp, wsb = ws.data_ptr(), ws.numel()
    y = native.matvec(packed, x, tlut, m, k, bits, wsp, wsb, stream)
    return y if y is None or isinstance(y, _Tensor) else check(y, "qtip_decompress_matvec")


def decompress_matvec_parts(packed, x, tlut, m, k, bits, nparts=None):
    """(S, m) fp32 partial sums of decode(packed) @ x over S ranges of k; their
    sum over axis 0 (in order) is the matvec.  S = nparts or matvec_split(...)."""
    _check_packed(packed, m, k, bits)
    _check_tlut(tlut, packed.device)
    require_cuda(x, "x", torch.float16)
    if x.numel() != k or x.device != packed.device:
        raise ValueError(f"x must hold {k} fp16 values on {packed.device}")
    S = int(nparts) if nparts is not None else matvec_split(m, k, bits, packed.device)
    parts = torch.empty((S, m), dtype=torch.float32, device=packed.device)
    with _on(packed.device):
        check(lib().qtip_decompress_matvec_parts(_ptr(parts), _ptr(packed), _ptr(x), _ptr(tlut), m, k, bits, S,
                                                 stream_ptr(packed.device)), "qtip_decompress_matvec_parts")
    return parts


RHT_IN_MATVEC_SIZES = (2048, 4096, 8192)


def decompress_matvec_parts_rht(packed, x_raw, su, scale, tlut, m, k, bits, nparts=None):
    """(S, m) fp32 partial sums of decode(packed) @ fp16(scale * H_k(su * x_raw)): the input
    transform of the layer runs inside the matvec launch (k in RHT_IN_MATVEC_SIZES)."""
    _check_packed(packed, m, k, bits)
    _check_tlut(tlut, packed.device)
    require_cuda(x_raw, "x", torch.float16)
    require_cuda(su, "su", torch.float16)
    if k not in RHT_IN_MATVEC_SIZES or x_raw.numel() != k or su.numel() != k:
        raise ValueError(f"x and su must hold k = {k} fp16 values, k in {RHT_IN_MATVEC_SIZES}")
    if x_raw.device != packed.device or su.device != packed.device:
        raise ValueError(f"x and su must be on {packed.device}")
    S = int(nparts) if nparts is not None else matvec_split(m, k, bits, packed.device)
    parts = torch.empty((S, m), dtype=torch.float32, device=packed.device)
    with _on(packed.device):
        check(lib().qtip_decompress_matvec_parts_rht(_ptr(parts), _ptr(packed), _ptr(x_raw), _ptr(su),
                                                     ctypes.c_float(scale), _ptr(tlut), m, k, bits, S,
                                                     stream_ptr(packed.device)), "qtip_decompress_matvec_parts_rht")
    return parts


def decompress_matvec_parts_mix(packed, x_raw, su, scale, sign_rows, order, tlut, m, k, bits, nparts=None):
    """decompress_matvec_parts_rht for k = order * 2^a where matvec_mix_columns(k, order, nparts) is not 0; sign_rows as
    utils.matmul_had.sign_rows makes them for that many columns."""
    _check_packed(packed, m, k, bits)
    _check_tlut(tlut, packed.device)
    require_cuda(x_raw, "x", torch.float16)
    require_cuda(su, "su", torch.float16)
    require_cuda(sign_rows, "sign_rows", torch.int32)
    S = int(nparts) if nparts is not None else matvec_split(m, k, bits, packed.device)
    cols = matvec_mix_columns(k, order, S)
    if x_raw.numel() != k or su.numel() != k:
        raise ValueError(f"x and su must hold k = {k} fp16 values")
    if not cols or sign_rows.numel() != k // cols * 8:
        raise ValueError(f"no transform of {k} = {order} * 2^a elements with such a table in front of {S} ranges")
    if any(t.device != packed.device for t in (x_raw, su, sign_rows)):
        raise ValueError(f"x, su and sign_rows must be on {packed.device}")
    parts = torch.empty((S, m), dtype=torch.float32, device=packed.device)
    with _on(packed.device):
        check(lib().qtip_decompress_matvec_parts_mix(_ptr(parts), _ptr(packed), _ptr(x_raw), _ptr(su), ctypes.c_float(scale),
                                                     _ptr(sign_rows), order, _ptr(tlut), m, k, bits, S,
                                                     stream_ptr(packed.device)), "qtip_decompress_matvec_parts_mix")
    return parts


def matvec_mix_columns(k, order, nparts):
    """Columns of the transform of k = order * 2^a elements that decompress_matvec_parts_mix runs in front of a matvec of nparts
    ranges; 0 where it does not."""
    return lib().qtip_matvec_mix_columns(k, order, nparts)


def decompress_matvec_parts_chain(packed, tlut, m, k, bits, prev_parts, post, scale_out, residual, norm_weight, eps,
                                  su, scale_in, nparts=None):
    """(parts, x_new): the boundary between two linear layers and the second layer's matvec in
    one launch - x_new = fp16(residual + fp16(post * scale_out * H(sum(prev_parts)))),
    parts = decode(packed) @ fp16(scale_in * H(su * rmsnorm(x_new))), the (S, m) fp32 partial sums.
    prev_parts: (S_prev, k) or (S_prev, 1, k) fp32; k in RHT_IN_MATVEC_SIZES."""
    _check_packed(packed, m, k, bits)
    _check_tlut(tlut, packed.device)
    require_cuda(prev_parts, "prev_parts", torch.float32)
    require_cuda(post, "post", torch.float32)
    require_cuda(residual, "residual", torch.float16)
    require_cuda(norm_weight, "norm_weight", torch.float16)
    require_cuda(su, "su", torch.float16)
    pp = prev_parts.reshape(prev_parts.shape[0], -1)
    if k not in RHT_IN_MATVEC_SIZES or pp.shape[1] != k:
        raise ValueError(f"prev_parts must hold vectors of k = {k} values, k in {RHT_IN_MATVEC_SIZES}")
    if any(t.numel() != k for t in (post, residual, norm_weight, su)):
        raise ValueError(f"post, residual, norm_weight and su must hold k = {k} values")
    if any(t.device != packed.device for t in (pp, post, residual, norm_weight, su)):
        raise ValueError(f"all operands must be on {packed.device}")
    S = int(nparts) if nparts is not None else matvec_split(m, k, bits, packed.device)
    parts = torch.empty((S, m), dtype=torch.float32, device=packed.device)
    x_new = torch.empty((1, k), dtype=torch.float16, device=packed.device)
    with _on(packed.device):
        check(lib().qtip_decompress_matvec_parts_chain(
            _ptr(parts), _ptr(packed), _ptr(tlut), m, k, bits, S, _ptr(pp), pp.shape[0], ctypes.c_size_t(pp.stride(0)),
            _ptr(post), ctypes.c_float(scale_out), _ptr(residual), _ptr(norm_weight), ctypes.c_float(eps), _ptr(su),
            ctypes.c_float(scale_in), _ptr(x_new), stream_ptr(packed.device)), "qtip_decompress_matvec_parts_chain")
    return parts, x_new


def decompress_matvec_group_chain(packed, tlut, m, k, bits, prev_parts, post, scale_out, residual, norm_weight, eps,
                                  su, scale_in, nparts=None):
    """decompress_matvec_parts_chain for up to three matrices that share the boundary and the
    input (separate q / k / v or gate / up projections) in one launch.  packed, tlut, m, su: lists,
    one entry per matrix.  Returns (parts (S, sum(m)) fp32 - matrix g's rows after those of
    matrix g - 1 -, x_new)."""
    n = len(packed)
    if not (1 <= n <= 3) or len(tlut) != n or len(m) != n or len(su) != n:
        raise ValueError("one to three matrices, with one table, row count and sign vector each")
    dev = packed[0].device
    for g in range(n):
        _check_packed(packed[g], m[g], k, bits)
        _check_tlut(tlut[g], dev)
        require_cuda(su[g], "su", torch.float16)
        if su[g].numel() != k or su[g].device != dev or packed[g].device != dev:
            raise ValueError(f"every su must hold k = {k} values on {dev}")
    require_cuda(prev_parts, "prev_parts", torch.float32)
    require_cuda(post, "post", torch.float32)
    require_cuda(residual, "residual", torch.float16)
    require_cuda(norm_weight, "norm_weight", torch.float16)
    pp = prev_parts.reshape(prev_parts.shape[0], -1)
    if k not in RHT_IN_MATVEC_SIZES or pp.shape[1] != k:
        raise ValueError(f"prev_parts must hold vectors of k = {k} values, k in {RHT_IN_MATVEC_SIZES}")
    if any(t.numel() != k for t in (post, residual, norm_weight)):
        raise ValueError(f"post, residual and norm_weight must hold k = {k} values")
    m_total = int(sum(m))
    S = int(nparts) if nparts is not None else matvec_split(m_total, k, bits, dev)
    parts = torch.empty((S, m_total), dtype=torch.float32, device=dev)
    x_new = torch.empty((1, k), dtype=torch.float16, device=dev)
    ptrs = lambda ts: (ctypes.c_void_p * n)(*[t.data_ptr() for t in ts])
    with _on(dev):
        check(lib().qtip_decompress_matvec_group_chain(
            _ptr(parts), n, ptrs(packed), ptrs(tlut), ptrs(su), (ctypes.c_int * n)(*[int(v) for v in m]), k, bits, S,
            _ptr(pp), pp.shape[0], ctypes.c_size_t(pp.stride(0)), _ptr(post), ctypes.c_float(scale_out),
            _ptr(residual), _ptr(norm_weight), ctypes.c_float(eps), ctypes.c_float(scale_in), _ptr(x_new),
            stream_ptr(dev)), "qtip_decompress_matvec_group_chain")
    return parts, x_new


def decompress_matvec_group(packed, x, tlut, m, k, bits, nparts=None):
    """Up to three matvecs of the same k and bit width in one launch, matrix g on its own fp16
    input x[g] (k values each; rows of one tensor will do).  Returns parts (S, sum(m)) fp32."""
    n = len(packed)
    if not (1 <= n <= 3) or len(tlut) != n or len(m) != n or len(x) != n:
        raise ValueError("one to three matrices, with one table, row count and input each")
    dev = packed[0].device
    for g in range(n):
        _check_packed(packed[g], m[g], k, bits)
        _check_tlut(tlut[g], dev)
        require_cuda(x[g], "x", torch.float16)
        if x[g].numel() != k or x[g].device != dev or packed[g].device != dev:
            raise ValueError(f"every x must hold k = {k} values on {dev}")
    m_total = int(sum(m))
    if nparts is not None:
        S = int(nparts)
    else:
        S = matvec_split(m_total, k, bits, dev)
        while k * 2 > S * 28 * 1024:  # every k range of x has to fit the kernel's staging area
            S *= 2
    parts = torch.empty((S, m_total), dtype=torch.float32, device=dev)
    ptrs = lambda ts: (ctypes.c_void_p * n)(*[t.data_ptr() for t in ts])
    with _on(dev):
        check(lib().qtip_decompress_matvec_group(_ptr(parts), n, ptrs(packed), ptrs(x), ptrs(tlut),
                                                 (ctypes.c_int * n)(*[int(v) for v in m]), k, bits, S,
                                                 stream_ptr(dev)), "qtip_decompress_matvec_group")
    return parts


def decompress_gemm(packed, x, tlut, m, k, bits, round_f16=True, out_dtype=torch.float32, long_sums=False):
    """(batch, m) = x[batch,k] (fp16) @ decode(packed)[m,k]^T on the matrix cores: fp32, rounded through
    fp16 on request, or with out_dtype=torch.float16 the rounded values themselves.  long_sums (fp16 results only): many
    rows faster, with fp32 sums in chains as long as those of a library product."""
    _check_packed(packed, m, k, bits)
    _check_tlut(tlut, packed.device)
    require_cuda(x, "x", torch.float16)
    if x.dim() != 2 or x.shape[1] != k or x.device != packed.device:
        raise ValueError(f"x must be (batch, {k}) fp16 on {packed.device}")
    if out_dtype not in _DT or (out_dtype == torch.float16 and not round_f16):
        raise ValueError("results are fp32, or fp16 when they are rounded")
    if long_sums and out_dtype != torch.float16:
        raise ValueError("long sums are for fp16 results")
    batch = x.shape[0]
    out = torch.empty((batch, m), dtype=out_dtype, device=packed.device)
    if batch == 0:
        return out
    L = lib()
    with _on(packed.device):
        need = (L.qtip_gemm_long_workspace_bytes if long_sums else L.qtip_gemm_workspace_bytes)(m, k, bits, batch)
        stream = stream_ptr(packed.device)
        wsp, wsb = None, 0
        if need:
            ws = _workspace(packed.device, need, stream)
            wsp, wsb = _ptr(ws), ws.numel()
        if out_dtype == torch.float16:
            product = L.qtip_decompress_gemm_long_f16 if long_sums else L.qtip_decompress_gemm_f16
            check(product(_ptr(out), _ptr(packed), _ptr(x), _ptr(tlut), m, k, bits, batch, wsp, wsb, stream),
                  "qtip_decompress_gemm_f16")
        else:
            check(L.qtip_decompress_gemm(_ptr(out), _ptr(packed), _ptr(x), _ptr(tlut), m, k, bits, batch,
                                         int(bool(round_f16)), wsp, wsb, stream), "qtip_decompress_gemm")
    return out


def _check_linear(x, packed, tlut, su, sv, had_in, order_in, had_out, order_out, m, k, bits):
    dev, rows = packed.device, x.shape[0]
    _check_packed(packed, m, k, bits)
    _check_tlut(tlut, dev)
    require_cuda(x, "x", (torch.float16, torch.float32))
    require_cuda(su, "su", torch.float16)
    require_cuda(sv, "sv", torch.float32)
    if x.shape != (rows, k) or not 1 <= rows <= 65535 or su.numel() != k or sv.numel() != m:
        raise ValueError(f"x must be (rows, {k}) with 1 to 65535 rows, su hold {k} and sv {m} values")
    if x.device != dev or su.device != dev or sv.device != dev:
        raise ValueError(f"x, su and sv must be on {dev}")
    for bits_t, order, n in ((had_in, order_in, k), (had_out, order_out, m)):
        p = n // order
        if n % order or p & (p - 1):
            raise ValueError(f"{n} is not {order} times a power of two")
        if order > 1:
            require_cuda(bits_t, "sign bits", torch.int32)
            if bits_t.numel() * 32 < order * order:
                raise ValueError("sign bits too short")
    return dev, rows


def _order_ok(t, order, n):
    p = n // order
    return not (n % order or p & (p - 1)) and (order == 1 or (
        isinstance(t, _Tensor) and t.is_cuda and t.dtype is torch.int32 and t.is_contiguous()
        and t.numel() * 32 >= order * order))


def linear(x, packed, tlut, su, sv, had_in, order_in, had_out, order_out, m, k, bits, scale_in, scale_out, long_sums=False):
    """A whole quantized projection in one call of the library: out (rows, m) in x's dtype = sv * scale_out * H_out(
    fp16(scale_in * H_in(su * x)) @ decode(packed)^T) for x (rows, k) fp16 / fp32; the launches, and the results bit
    for bit, of rht, decompress_matvec_parts[_rht] (one row) or decompress_gemm (more), rht.  had_in / had_out: sign
    bits of the table orders (None for order 1).  long_sums: the product is decompress_gemm's with long sums."""
    # a call whose operands fit is one native function's; any other goes through the checks one by one
    if isinstance(x, _Tensor) and x.is_cuda and not _is_compiling() and (native := host()):
        y = native.linear(x, packed, tlut, su, sv, had_in, order_in, had_out, order_out, m, k, bits, scale_in, scale_out,
                          long_sums, _ALIGN_ROWS, stream_ptr(x.device))
        if y is not None:
            return y if isinstance(y, _Tensor) else check(y, "qtip_linear")
    if not (isinstance(x, _Tensor) and isinstance(packed, _Tensor) and isinstance(tlut, _Tensor)
            and isinstance(su, _Tensor) and isinstance(sv, _Tensor) and packed.is_cuda
            and packed.dtype in _PACKED_TYPES and tlut.dtype is su.dtype is _F16 and sv.dtype is _F32
            and (x.dtype is _F16 or x.dtype is _F32)
            and x.device == (dev := packed.device) == tlut.device == su.device == sv.device
            and packed.is_contiguous() and x.is_contiguous() and tlut.is_contiguous() and su.is_contiguous()
            and sv.is_contiguous() and x.dim() == 2 and x.shape[1] == k and 1 <= (rows := x.shape[0]) <= 65535
            and su.numel() == k and sv.numel() == m and tlut.numel() == 1024
            and bits in _BITS and m > 0 and k > 0 and not (m | k) & 31
            and packed.numel() * packed.element_size() * 8 == bits * m * k
            and _order_ok(had_in, order_in, k) and _order_ok(had_out, order_out, m)):
        dev, rows = _check_linear(x, packed, tlut, su, sv, had_in, order_in, had_out, order_out, m, k, bits)
    dt = _DT[x.dtype]
    if rows >= _ALIGN_ROWS and (x.data_ptr() | su.data_ptr() | sv.data_ptr()) & 15:
        x, su, sv = map(aligned16, (x, su, sv))
    out = torch.empty((rows, m), dtype=x.dtype, device=dev)
    L = lib()
    with _on(dev):
        stream = stream_ptr(dev)
        size, run = ((L.qtip_linear_long_workspace_bytes, L.qtip_linear_long) if long_sums else
                     (L.qtip_linear_workspace_bytes, L.qtip_linear))
        need = size(m, k, bits, rows, order_in, dt)
        ws = torch.empty(need, dtype=torch.uint8, device=dev)
        check(run(out.data_ptr(), x.data_ptr(), dt, packed.data_ptr(), tlut.data_ptr(), su.data_ptr(),
                  sv.data_ptr(), _ptr(had_in), order_in, _ptr(had_out), order_out, m, k, bits, rows, scale_in,
                  scale_out, ws.data_ptr(), need, stream), "qtip_linear")
    return out


PRE_NONE, PRE_RMSNORM, PRE_SILU_MUL = 0, 1, 2


def linear_rows(x, packed, tlut, su, sv, had_in, order_in, had_out, order_out, m, k, bits, scale_in, scale_out, long_sums,
                pre_mode, norm_weight, eps, residual):
    """linear() for fp16 rows, two or more, with the element-wise work around the projection in the transforms (as rht takes
    it); None where an operand is not as the launches need it (contiguous, on 16 bytes), or without the native module."""
    if not (isinstance(x, _Tensor) and x.is_cuda) or _is_compiling() or not (native := host()):
        return None
    y = native.linear(x, packed, tlut, su, sv, had_in, order_in, had_out, order_out, m, k, bits, scale_in, scale_out, long_sums, 0,
                      stream_ptr(x.device), pre_mode, norm_weight, eps, residual)
    return y if y is None or isinstance(y, _Tensor) else check(y, "qtip_linear_rows")


def rht(x, order=1, had_bits=None, pre=None, post=None, scale=None, out_dtype=None, in_parts=1, pre_mode=PRE_NONE,
        norm_weight=None, eps=0.0, residual=None):
    """out[r] = post * scale * (H_order (x) H_p)(pre * f(x[r])) (+ residual) over the last axis.

    x: (..., n) fp16 or fp32 (with in_parts > 1: (in_parts, ..., n), summed on load).
    had_bits: int32 device tensor of packed sign bits for order > 1.  scale defaults to n ** -0.5.
    pre_mode / norm_weight / eps / residual: element-wise work of the surrounding layer folded
    into the same launch (see qtip_rht_fused in include/qtip_hip.h); with PRE_SILU_MUL the last
    axis of x holds [gate | up] and n is half of it.
    """
    require_cuda(x, "x", (torch.float16, torch.float32))
    n = x.shape[-1]
    if pre_mode == PRE_SILU_MUL:
        if n % 2:
            raise ValueError("gate|up input needs an even last dimension")
        n //= 2
    rows = x.numel() // x.shape[-1] // in_parts
    if n % order:
        raise ValueError(f"order {order} does not divide {n}")
    p = n // order
    if p & (p - 1):
        raise ValueError(f"{n} / {order} = {p} is not a power of two")
    if order > 1:
        require_cuda(had_bits, "had_bits", torch.int32)
        if had_bits.numel() * 32 < order * order:
            raise ValueError("had_bits too short")
    if pre is not None:
        require_cuda(pre, "pre", torch.float16)
        if pre.numel() != n:
            raise ValueError(f"pre must hold {n} values")
    if post is not None:
        require_cuda(post, "post", torch.float32)
        if post.numel() != n:
            raise ValueError(f"post must hold {n} values")
    out_dtype = out_dtype or x.dtype
    shape = list(x.shape[1:] if in_parts > 1 else x.shape)
    shape[-1] = n
    fused = pre_mode != PRE_NONE or residual is not None
    if pre_mode == PRE_RMSNORM:
        require_cuda(norm_weight, "norm_weight", torch.float16)
        if norm_weight.numel() != n or x.dtype != torch.float16:
            raise ValueError("RMSNorm prologue needs an fp16 input and an fp16 weight of the same length")
    if pre_mode not in (PRE_NONE, PRE_RMSNORM, PRE_SILU_MUL) or (pre_mode != PRE_NONE and in_parts != 1):
        raise ValueError("bad pre_mode")
    if residual is not None:
        require_cuda(residual, "residual", torch.float16)
        if out_dtype != torch.float16 or residual.numel() != rows * n:
            raise ValueError("residual needs fp16 output and one value per output element")
    out = torch.empty(shape, dtype=out_dtype, device=x.device)
    if rows == 0:
        return out
    if scale is None:
        scale = n ** -0.5
    p_pre, p_post = _ptr(pre), _ptr(post)
    if rows >= _ALIGN_ROWS and n % 8 == 0 and (x.data_ptr() | (p_pre or 0) | (p_post or 0) | (
            fused and ((_ptr(norm_weight) or 0) | (_ptr(residual) or 0)))) & 15:
        x, pre, post, norm_weight, residual = map(aligned16, (x, pre, post, norm_weight, residual))
        p_pre, p_post = _ptr(pre), _ptr(post)
    L = lib()
    with _on(x.device):
        width = x.shape[-1]
        xf = x.reshape(in_parts, rows, width) if in_parts > 1 else x.reshape(rows, width)
        of = out.reshape(rows, n)
        rf = residual.reshape(rows, n) if residual is not None else None
        step = 65535 if in_parts == 1 else rows
        if in_parts > 1 and rows > 65535:
            raise ValueError("too many rows for a split input")
        for r0 in range(0, rows, step):
            r1 = min(rows, r0 + step)
            src = xf if in_parts > 1 else xf[r0:r1]
            if fused:
                check(L.qtip_rht_fused(_ptr(of[r0:r1]), _DT[out_dtype], _ptr(src), _DT[x.dtype], in_parts, r1 - r0, n,
                                       order, _ptr(had_bits), p_pre, p_post, ctypes.c_float(scale), pre_mode,
                                       _ptr(norm_weight), ctypes.c_float(eps),
                                       _ptr(rf[r0:r1]) if rf is not None else _ptr(None),
                                       stream_ptr(x.device)), "qtip_rht_fused")
            else:
                check(L.qtip_rht(_ptr(of[r0:r1]), _DT[out_dtype], _ptr(src), _DT[x.dtype], in_parts, r1 - r0, n,
                                 order, _ptr(had_bits), p_pre, p_post, ctypes.c_float(scale),
                                 stream_ptr(x.device)), "qtip_rht")
    return out


def rht_fused_pre_rows(x, pre_rows, norm_weight, eps, order=1, had_bits=None, scale=None):
    """Input transforms of `rows` layers that read the same fp16 vector x (n values), one launch:
    row r = fp16(scale * H^T(pre_rows[r] * rmsnorm(x))).  pre_rows (rows, n) fp16.  -> (rows, n)."""
    require_cuda(x, "x", torch.float16)
    require_cuda(pre_rows, "pre_rows", torch.float16)
    require_cuda(norm_weight, "norm_weight", torch.float16)
    n = x.numel()
    if pre_rows.dim() != 2 or pre_rows.shape[1] != n or norm_weight.numel() != n or pre_rows.shape[0] > 65535:
        raise ValueError("pre_rows must be (rows, n) and norm_weight hold n values")
    p = n // order
    if n % order or p & (p - 1):
        raise ValueError(f"{n} is not {order} times a power of two")
    if order > 1:
        require_cuda(had_bits, "had_bits", torch.int32)
    out = torch.empty_like(pre_rows)
    with _on(x.device):
        check(lib().qtip_rht_fused_pre_rows(_ptr(out), _ptr(x), pre_rows.shape[0], n, order, _ptr(had_bits),
                                            _ptr(pre_rows), ctypes.c_float(scale if scale is not None else n ** -0.5),
                                            _ptr(norm_weight), ctypes.c_float(eps), stream_ptr(x.device)),
              "qtip_rht_fused_pre_rows")
    return out


def rht_post_rows(parts, post_rows, order=1, had_bits=None, scale=None, out_dtype=torch.float16):
    """Output transforms of `rows` layers of the same size in one launch: parts (S, rows, n) fp32
    (summed over S on load), post_rows (rows, n) fp32, one vector per row.  Returns (rows, n)."""
    require_cuda(parts, "parts", torch.float32)
    require_cuda(post_rows, "post_rows", torch.float32)
    if parts.dim() != 3 or post_rows.shape != parts.shape[1:]:
        raise ValueError("parts must be (S, rows, n) and post_rows (rows, n)")
    S, rows, n = parts.shape
    p = n // order
    if n % order or p & (p - 1) or rows > 65535:
        raise ValueError(f"{n} is not {order} times a power of two, or too many rows")
    if order > 1:
        require_cuda(had_bits, "had_bits", torch.int32)
    out = torch.empty((rows, n), dtype=out_dtype, device=parts.device)
    with _on(parts.device):
        check(lib().qtip_rht_post_rows(_ptr(out), _DT[out_dtype], _ptr(parts), _DT[torch.float32], S, rows, n, order,
                                       _ptr(had_bits), _ptr(post_rows),
                                       ctypes.c_float(scale if scale is not None else n ** -0.5),
                                       stream_ptr(parts.device)), "qtip_rht_post_rows")
    return out


def rht_silu_pair(parts, post, order=1, had_bits=None, scale=None):
    """fp16(fp16(silu(gate)) * up) of the transformed gate / up outputs in one launch.
    parts (S, n) fp32 with post (n,): gate and up are the halves of one transformed vector
    (returns (n / 2,)); parts (S, 2, n) with post (2, n): a transformed vector each (returns (n,))."""
    require_cuda(parts, "parts", torch.float32)
    require_cuda(post, "post", torch.float32)
    two = parts.dim() == 3
    if parts.dim() not in (2, 3) or post.shape != parts.shape[1:] or (two and parts.shape[1] != 2):
        raise ValueError("parts must be (S, n) with post (n,), or (S, 2, n) with post (2, n)")
    S, n = parts.shape[0], parts.shape[-1]
    if order > 1:
        require_cuda(had_bits, "had_bits", torch.int32)
    out = torch.empty(n if two else n // 2, dtype=torch.float16, device=parts.device)
    with _on(parts.device):
        check(lib().qtip_rht_silu_pair(_ptr(out), _ptr(parts), S, int(two), n, order, _ptr(had_bits), _ptr(post),
                                       ctypes.c_float(scale if scale is not None else n ** -0.5),
                                       stream_ptr(parts.device)), "qtip_rht_silu_pair")
    return out


def rht_silu_pair_ok(n, order, two_vectors):
    """Shapes qtip_rht_silu_pair takes (the vectorised form of the transform: rows of >= 8 values
    per workgroup, whole rows of the table mix for either half)."""
    p = n // order
    if n % order or p & (p - 1) or n <= 4096 or (not two_vectors and order % 2):
        return False
    pp, log_a = p, 0
    while pp > 1024:  # values per workgroup of the transform kernels
        pp >>= 1
        log_a += 1
    while pp > 64 and (order << (log_a + 1)) <= 64:
        pp >>= 1
        log_a += 1
    return pp >= 8


ATTN_MAX_KEY_SPLITS = 16


ATTN_SPLIT_FROM = 1024  # context length from which the key-range form is faster, of heads whose ranges fit the chip side by side
ATTN_SPLIT_FROM_MANY = 2560  # and of more heads than that


def attention_key_splits(context, heads=None):
    """Key ranges per head for decode attention over a context of `context` tokens: one workgroup per head below
    ATTN_SPLIT_FROM keys, 8 ranges from there on.  The ranges cost a second small launch, and every one of them repeats the
    transform of the new token: more than 40 heads (of `heads`, where given) keep one workgroup up to ATTN_SPLIT_FROM_MANY
    keys and then have as many ranges as 256 compute units hold.  us a launch with that transform, one range / eight: 32 heads
    of 128, 250 keys 9.0/11.7; 32 on 8, 900 keys 12.0/12.7, 1200 13.4/12.9, 2000 18.1/15.0, 4000 29.3/20.3; 32 on 32, 900
    12.0/12.6, 1200 16.5/13.9; 40, 900 13.8/15.5, 1200 17.8/15.8.  One / four / eight: 64 on 8, 1024 keys 12.5/16.2/21.2, 2000
    18.7/19.2/25.3, 2500 21.8/20.3/27.1, 4000 30.7/26.1/31.1; one / two / four: 128 on 8, 2500 23.1/24.0/29.3, 3000
    26.1/25.5/32.5."""
    if heads is not None and heads > 40:
        return 1 if context < ATTN_SPLIT_FROM_MANY else max(1, 256 // heads)
    return 1 if context < ATTN_SPLIT_FROM else 8


def _split_workspace(device, heads, head_dim, key_splits):
    if not 1 <= key_splits <= ATTN_MAX_KEY_SPLITS:
        raise ValueError(f"key_splits must be in 1..{ATTN_MAX_KEY_SPLITS} (got {key_splits})")
    if key_splits == 1:
        return None
    return torch.empty(heads * key_splits * (head_dim + 2), dtype=torch.float32, device=device)


def decode_attention(qkv, k_cache, v_cache, pos, inv_freq, heads, kv_heads, head_dim, key_splits=1):
    """Attention output (heads*head_dim,) fp16 of one new token: RoPE, cache write at `pos`
    (device int64 tensor with one element) and attention over cache slots 0..pos in one launch.
    k_cache / v_cache: (1, kv_heads, max_len, head_dim) fp16, updated in place."""
    require_cuda(qkv, "qkv", torch.float16)
    require_cuda(k_cache, "k_cache", torch.float16)
    require_cuda(v_cache, "v_cache", torch.float16)
    require_cuda(pos, "pos", torch.int64)
    require_cuda(inv_freq, "inv_freq", torch.float32)
    max_len = k_cache.shape[-2]
    if qkv.numel() != (heads + 2 * kv_heads) * head_dim or k_cache.numel() != kv_heads * max_len * head_dim \
            or v_cache.shape != k_cache.shape or inv_freq.numel() != head_dim // 2 or pos.numel() != 1:
        raise ValueError("decode_attention: inconsistent shapes")
    out = torch.empty(heads * head_dim, dtype=torch.float16, device=qkv.device)
    ws = _split_workspace(qkv.device, heads, head_dim, key_splits)
    with _on(qkv.device):
        check(lib().qtip_decode_attention(_ptr(out), _ptr(qkv), _ptr(k_cache), _ptr(v_cache), _ptr(pos),
                                          _ptr(inv_freq), heads, kv_heads, head_dim, max_len, key_splits, _ptr(ws),
                                          stream_ptr(qkv.device)), "qtip_decode_attention")
    return out


def decode_attention_rht(parts, post, scale, had_bits, order, k_cache, v_cache, pos, inv_freq, heads, kv_heads,
                         head_dim, key_splits=1):
    """decode_attention on the qkv projection's raw matvec result `parts` (S, n) fp32: the
    projection's output transform (order x power-of-two Hadamard, * post * scale, cast to fp16) runs
    in the attention kernel's prologue.  had_bits: the table's packed sign bits (None for order 1)."""
    require_cuda(parts, "parts", torch.float32)
    require_cuda(k_cache, "k_cache", torch.float16)
    require_cuda(v_cache, "v_cache", torch.float16)
    require_cuda(pos, "pos", torch.int64)
    require_cuda(inv_freq, "inv_freq", torch.float32)
    if post is not None:
        require_cuda(post, "post", torch.float32)
    if had_bits is not None:
        require_cuda(had_bits, "had_bits", torch.int32)
    n = (heads + 2 * kv_heads) * head_dim
    parts = parts.reshape(-1, n)
    max_len = k_cache.shape[-2]
    if k_cache.numel() != kv_heads * max_len * head_dim or v_cache.shape != k_cache.shape \
            or inv_freq.numel() != head_dim // 2 or pos.numel() != 1 or (post is not None and post.numel() != n) \
            or (order > 1 and had_bits is None):
        raise ValueError("decode_attention_rht: inconsistent shapes")
    out = torch.empty(heads * head_dim, dtype=torch.float16, device=parts.device)
    ws = _split_workspace(parts.device, heads, head_dim, key_splits)
    with _on(parts.device):
        check(lib().qtip_decode_attention_rht(_ptr(out), _ptr(parts), parts.shape[0], parts.stride(0),
                                              _ptr(post) if post is not None else None, float(scale),
                                              _ptr(had_bits) if had_bits is not None else None, int(order),
                                              _ptr(k_cache), _ptr(v_cache), _ptr(pos), _ptr(inv_freq), heads,
                                              kv_heads, head_dim, max_len, key_splits, _ptr(ws),
                                              stream_ptr(parts.device)),
              "qtip_decode_attention_rht")
    return out


def decode_attention_rht3(parts, post, scale, had_bits, order, k_cache, v_cache, pos, inv_freq, heads, kv_heads,
                          head_dim, key_splits=1):
    """decode_attention_rht for separate q / k / v projections: parts, post, scale, had_bits and
    order are 3-element lists (q, k, v); the three `parts` are (S, n_i) fp32 views into one
    partial-sum buffer (same number of parts and the same row stride)."""
    for i in range(3):
        require_cuda(parts[i], "parts", torch.float32, contiguous=False)
        if post[i] is not None:
            require_cuda(post[i], "post", torch.float32)
        if had_bits[i] is not None:
            require_cuda(had_bits[i], "had_bits", torch.int32)
        n = (heads if i == 0 else kv_heads) * head_dim
        if parts[i].dim() != 2 or parts[i].shape[1] != n or parts[i].stride(1) != 1 \
                or parts[i].shape[0] != parts[0].shape[0] or parts[i].stride(0) != parts[0].stride(0) \
                or (post[i] is not None and post[i].numel() != n) or (order[i] > 1 and had_bits[i] is None):
            raise ValueError("decode_attention_rht3: inconsistent shapes")
    require_cuda(k_cache, "k_cache", torch.float16)
    require_cuda(v_cache, "v_cache", torch.float16)
    require_cuda(pos, "pos", torch.int64)
    require_cuda(inv_freq, "inv_freq", torch.float32)
    max_len = k_cache.shape[-2]
    if k_cache.numel() != kv_heads * max_len * head_dim or v_cache.shape != k_cache.shape \
            or inv_freq.numel() != head_dim // 2 or pos.numel() != 1:
        raise ValueError("decode_attention_rht3: inconsistent shapes")
    dev = parts[0].device
    out = torch.empty(heads * head_dim, dtype=torch.float16, device=dev)
    ws = _split_workspace(dev, heads, head_dim, key_splits)
    vp = lambda ts: (ctypes.c_void_p * 3)(*[t.data_ptr() if t is not None else None for t in ts])
    with _on(dev):
        check(lib().qtip_decode_attention_rht3(_ptr(out), vp(parts), parts[0].shape[0], parts[0].stride(0), vp(post),
                                               (ctypes.c_float * 3)(*[float(v) for v in scale]), vp(had_bits),
                                               (ctypes.c_int * 3)(*[int(v) for v in order]), _ptr(k_cache),
                                               _ptr(v_cache), _ptr(pos), _ptr(inv_freq), heads, kv_heads, head_dim,
                                               max_len, key_splits, _ptr(ws), stream_ptr(dev)),
              "qtip_decode_attention_rht3")
    return out


def attention_share_ranges(heads):
    """Ranges of the keys that decode_attention_shares has room for: up to four, which is what o's matvec reads, and as many as leave
    each of 256 compute units a workgroup."""
    return max(1, min(4, 256 // heads))


def decode_attention_shares(parts, post, scale, had_bits, order, k_cache, v_cache, pos, inv_freq, heads, kv_heads, head_dim):
    """decode_attention_rht (one-element lists) or _rht3 (three) for decompress_matvec_parts_shares: the shares of the ranges
    of keys, (heads, ranges, head_dim + 4) fp32, as many of them in use as the position gives."""
    vectors = len(parts)
    dev = parts[0].device
    for i in range(vectors):
        require_cuda(parts[i], "parts", torch.float32, contiguous=False)
        require_cuda(post[i], "post", torch.float32)
        if had_bits[i] is not None:
            require_cuda(had_bits[i], "had_bits", torch.int32)
        n = (heads + 2 * kv_heads if vectors == 1 else heads if i == 0 else kv_heads) * head_dim
        if parts[i].dim() != 2 or parts[i].shape[1] != n or parts[i].stride(1) != 1 \
                or parts[i].shape[0] != parts[0].shape[0] or parts[i].stride(0) != parts[0].stride(0) \
                or post[i].numel() != n or (order[i] > 1 and had_bits[i] is None):
            raise ValueError("decode_attention_shares: inconsistent shapes")
    require_cuda(k_cache, "k_cache", torch.float16)
    require_cuda(v_cache, "v_cache", torch.float16)
    require_cuda(pos, "pos", torch.int64)
    require_cuda(inv_freq, "inv_freq", torch.float32)
    max_len = k_cache.shape[-2]
    if k_cache.numel() != kv_heads * max_len * head_dim or v_cache.shape != k_cache.shape \
            or inv_freq.numel() != head_dim // 2 or pos.numel() != 1:
        raise ValueError("decode_attention_shares: inconsistent shapes")
    ranges = attention_share_ranges(heads)
    shares = torch.empty((heads, ranges, head_dim + 4), dtype=torch.float32, device=dev)
    vp = lambda ts: (ctypes.c_void_p * vectors)(*[t.data_ptr() if t is not None else None for t in ts])
    with _on(dev):
        check(lib().qtip_decode_attention_shares(_ptr(shares), ranges, vectors, vp(parts), parts[0].shape[0], parts[0].stride(0),
                                                 vp(post), (ctypes.c_float * vectors)(*[float(v) for v in scale]), vp(had_bits),
                                                 (ctypes.c_int * vectors)(*[int(v) for v in order]), _ptr(k_cache), _ptr(v_cache),
                                                 _ptr(pos), _ptr(inv_freq), heads, kv_heads, head_dim, max_len, stream_ptr(dev)),
              "qtip_decode_attention_shares")
    return shares


def decompress_matvec_parts_shares(packed, shares, pos, max_len, su, scale, tlut, m, k, bits, nparts=None):
    """decompress_matvec_parts_rht on the attention output that the shares of decode_attention_shares give, with the position and
    the cache slots of that call."""
    _check_packed(packed, m, k, bits)
    _check_tlut(tlut, packed.device)
    require_cuda(shares, "shares", torch.float32)
    require_cuda(su, "su", torch.float16)
    require_cuda(pos, "pos", torch.int64)
    heads, ranges, dim = shares.shape[0], shares.shape[1], shares.shape[2] - 4
    if k not in RHT_IN_MATVEC_SIZES or heads * dim != k or su.numel() != k or pos.numel() != 1:
        raise ValueError(f"shares and su must be of k = {k} values, k in {RHT_IN_MATVEC_SIZES}")
    if any(t.device != packed.device for t in (shares, su, pos)):
        raise ValueError(f"shares, su and pos must be on {packed.device}")
    S = int(nparts) if nparts is not None else matvec_split(m, k, bits, packed.device)
    parts = torch.empty((S, m), dtype=torch.float32, device=packed.device)
    with _on(packed.device):
        check(lib().qtip_decompress_matvec_parts_shares(_ptr(parts), _ptr(packed), _ptr(shares), ranges, dim, _ptr(pos), max_len,
                                                        _ptr(su), ctypes.c_float(scale), _ptr(tlut), m, k, bits, S,
                                                        stream_ptr(packed.device)), "qtip_decompress_matvec_parts_shares")
    return parts


def prefill_attention(q, k, v, cos, sin, k_cache, v_cache, pos, heads, kv_heads, head_dim):
    """Causal attention of n new tokens against the cache, which gets their keys and values first: q (n, heads *
    head_dim), k / v (n, kv_heads * head_dim) fp16 with contiguous rows, cos / sin (n, head_dim) fp16, pos (n,) int64
    cache slots, caches (1, kv_heads, slots, head_dim) fp16.  Returns (n, heads * head_dim)."""
    n, slots = q.shape[0], k_cache.shape[2]
    for t, name, width in ((q, "q", heads * head_dim), (k, "k", kv_heads * head_dim), (v, "v", kv_heads * head_dim)):
        require_cuda(t, name, torch.float16, contiguous=False)
        if t.shape != (n, width) or t.stride(1) != 1:
            raise ValueError(f"{name} must be ({n}, {width}) with contiguous rows")
    for t, name in ((cos, "cos"), (sin, "sin")):
        require_cuda(t, name, torch.float16)
        if t.numel() != n * head_dim:
            raise ValueError(f"{name} must be ({n}, {head_dim})")
    for t, name in ((k_cache, "k_cache"), (v_cache, "v_cache")):
        require_cuda(t, name, torch.float16)
        if t.shape != (1, kv_heads, slots, head_dim):
            raise ValueError(f"{name} must be (1, {kv_heads}, slots, {head_dim})")
    require_cuda(pos, "pos", torch.int64)
    if pos.shape != (n,):
        raise ValueError(f"pos must hold {n} cache slots")
    out = torch.empty((n, heads * head_dim), dtype=torch.float16, device=q.device)
    with _on(q.device):
        check(lib().qtip_prefill_attention(_ptr(out), _ptr(q), _ptr(k), _ptr(v), q.stride(0), k.stride(0), v.stride(0),
                                           _ptr(cos), _ptr(sin), _ptr(k_cache), _ptr(v_cache), _ptr(pos), n, heads,
                                           kv_heads, head_dim, slots, stream_ptr(q.device)), "qtip_prefill_attention")
    return out


def rmsnorm(x, weight, eps):
    """weight * fp16(x * rsqrt(mean(x^2) + eps)) for one fp16 vector (model/llama.py:129-135)."""
    require_cuda(x, "x", torch.float16)
    require_cuda(weight, "weight", torch.float16)
    if x.numel() != weight.numel():
        raise ValueError("rmsnorm: x and weight differ in length")
    out = torch.empty_like(x)
    with _on(x.device):
        check(lib().qtip_rmsnorm(_ptr(out), _ptr(x), _ptr(weight), float(eps), x.numel(), stream_ptr(x.device)),
              "qtip_rmsnorm")
    return out


def rmsnorm_rows(x, weight, eps):
    """rmsnorm of every row of x (..., n)."""
    require_cuda(x, "x", torch.float16)
    require_cuda(weight, "weight", torch.float16)
    n = weight.numel()
    if x.dim() < 1 or x.shape[-1] != n or x.device != weight.device:
        raise ValueError(f"rmsnorm: rows must hold {n} values and be where the weight is")
    out = torch.empty_like(x)
    if x.numel():
        with _on(x.device):
            check(lib().qtip_rmsnorm_rows(_ptr(out), _ptr(x), _ptr(weight), float(eps), x.numel() // n, n, stream_ptr(x.device)),
                  "qtip_rmsnorm_rows")
    return out


def rotary_tables(positions, inv_freq):
    """(cos, sin), each (n, 2 * len(inv_freq)) fp16, of float(positions) * inv_freq, every angle twice."""
    require_cuda(positions, "positions", torch.int64)
    require_cuda(inv_freq, "inv_freq", torch.float32)
    n, half = positions.numel(), inv_freq.numel()
    cos, sin = (torch.empty((n, 2 * half), dtype=torch.float16, device=positions.device) for _ in range(2))
    if positions.device != inv_freq.device:
        raise ValueError("positions and inv_freq are on different devices")
    if n:
        with _on(positions.device):
            check(lib().qtip_rotary_tables(_ptr(cos), _ptr(sin), _ptr(positions), _ptr(inv_freq), n, half,
                                           stream_ptr(positions.device)), "qtip_rotary_tables")
    return cos, sin


TOKEN_HEAD_MAX = 8192  # values of a row that the waves of token_head hold in flight


def token_head(head, x, norm_weight, eps, parts=None, post=None, scale_out=0.0, out_dtype=torch.float16):
    """fp16(head @ rmsnorm(y)) as out_dtype (fp16 or fp32), (vocab,), for one token: y = x, or behind the last layer's
    projection y = fp16(x + fp16(post * scale_out * H(sum(parts)))).  head (vocab, n) fp16; parts (S, n) fp32, n in
    RHT_IN_MATVEC_SIZES."""
    require_cuda(head, "head", torch.float16)
    require_cuda(x, "x", torch.float16)
    require_cuda(norm_weight, "norm_weight", torch.float16)
    if head.dim() != 2 or out_dtype not in _DT:
        raise ValueError("head must be a matrix, out_dtype fp16 or fp32")
    vocab, n = head.shape
    if x.numel() != n or norm_weight.numel() != n or x.device != head.device or norm_weight.device != head.device:
        raise ValueError(f"x and norm_weight must hold {n} values on {head.device}")
    nparts, stride = 0, 0
    if parts is not None:
        require_cuda(parts, "parts", torch.float32)
        require_cuda(post, "post", torch.float32)
        parts = parts.reshape(parts.shape[0], -1)
        nparts, stride = parts.shape[0], parts.stride(0)
        if n not in RHT_IN_MATVEC_SIZES or parts.shape[1] != n or post.numel() != n or parts.device != head.device \
                or post.device != head.device:
            raise ValueError(f"parts and post must hold vectors of {n} values on {head.device}, n in {RHT_IN_MATVEC_SIZES}")
    out = torch.empty((vocab,), dtype=out_dtype, device=head.device)
    with _on(head.device):
        check(lib().qtip_token_head(_ptr(out), _DT[out_dtype], _ptr(head), vocab, n, _ptr(x), _ptr(parts), nparts,
                                    ctypes.c_size_t(stride), _ptr(post), float(scale_out), _ptr(norm_weight), float(eps),
                                    stream_ptr(head.device)), "qtip_token_head")
    return out


def greedy_pick(logits, tok, pos, history=None, history_base=0):
    """tok[0] = argmax(logits) (fp16 logits of one position, first index among equal maxima),
    history[pos - history_base] = tok when that slot exists, pos += 1 - the per-token bookkeeping
    of a greedy generation loop (eval/interactive_gen.py:43-69) in one launch, in place."""
    require_cuda(logits, "logits", torch.float16)
    require_cuda(tok, "tok", torch.int64)
    require_cuda(pos, "pos", torch.int64)
    if history is not None:
        require_cuda(history, "history", torch.int64)
    if tok.numel() != 1 or pos.numel() != 1:
        raise ValueError("greedy_pick: tok and pos hold one element each")
    with _on(logits.device):
        check(lib().qtip_greedy_pick(_ptr(logits), logits.numel(), _ptr(tok), _ptr(pos),
                                     _ptr(history) if history is not None else None,
                                     history.numel() if history is not None else 0, int(history_base),
                                     stream_ptr(logits.device)), "qtip_greedy_pick")


SAMPLE_PICK_MAX_TOP_K = 64


def sample_pick(logits, temperature, top_k, seed, counter, tok, pos, history=None, history_base=0):
    """Draw tok[0] from softmax(logits / temperature) restricted to the top_k largest logits
    (None: all), as eval/interactive_gen.py:15-40 does, with the bookkeeping of greedy_pick, in
    one launch.  counter: device int64 draw counter (advanced in place); seed: host integer."""
    require_cuda(logits, "logits", torch.float16)
    require_cuda(tok, "tok", torch.int64)
    require_cuda(pos, "pos", torch.int64)
    require_cuda(counter, "counter", torch.int64)
    if history is not None:
        require_cuda(history, "history", torch.int64)
    k = 0 if top_k is None else int(top_k)
    if tok.numel() != 1 or pos.numel() != 1 or counter.numel() != 1 or not (0 <= k <= SAMPLE_PICK_MAX_TOP_K):
        raise ValueError("sample_pick: tok, pos and counter hold one element each, top_k at most 64")
    with _on(logits.device):
        check(lib().qtip_sample_pick(_ptr(logits), logits.numel(), ctypes.c_float(temperature), k,
                                     ctypes.c_uint(int(seed) & 0xffffffff), _ptr(counter), _ptr(tok), _ptr(pos),
                                     _ptr(history) if history is not None else None,
                                     history.numel() if history is not None else 0, int(history_base),
                                     stream_ptr(logits.device)), "qtip_sample_pick")


# ---- packing tools ---------------------------------------------------------------------------

def repack(packed, m, k, bits, to_kernel=True):
    """Natural packing <-> kernel packing of a 16x16-tile, V=2 trellis (same shape and dtype out).
    to_kernel=True is the re-pack of lib/algo/finetune.py:196-201, False its inverse
    (lib/utils/kernel_decompress.py:19-24)."""
    _check_packed(packed, m, k, bits)
    out = torch.empty_like(packed)
    with _on(packed.device):
        check(lib().qtip_repack(_ptr(out), _ptr(packed), m, k, bits, 1 if to_kernel else 0,
                                stream_ptr(packed.device)), "qtip_repack")
    return out


def _check_natural(packed, T, K, V):
    require_cuda(packed, "packed", (torch.int16, torch.uint16))
    if V not in (1, 2) or K * V > 16 or T % V or (T * K) % 16:
        raise ValueError(f"unsupported natural packing T={T} K={K} V={V}")
    nw = T * K // 16
    if packed.numel() % nw:
        raise ValueError(f"packed holds {packed.numel()} words, not a multiple of {nw} per tile")
    return packed.numel() // nw


def unpack_trellis(packed, T, K, V):
    """Natural packing (ntiles, T*K/16) int16/uint16 -> (ntiles, T/V) int32 states
    (lib/codebook/bitshift.py:329-353)."""
    ntiles = _check_natural(packed, T, K, V)
    states = torch.empty((ntiles, T // V), dtype=torch.int32, device=packed.device)
    with _on(packed.device):
        check(lib().qtip_unpack_trellis(_ptr(states), _ptr(packed), ntiles, T, K, V, stream_ptr(packed.device)),
              "qtip_unpack_trellis")
    return states


def pack_trellis(states, K, V):
    """(ntiles, T/V) states -> natural packing (ntiles, T*K/16) uint16
    (lib/codebook/bitshift.py:294-327).  Raises, like the reference's assert, when consecutive
    states do not overlap by 16 - K*V bits (this check synchronises with the device)."""
    require_cuda(states, "states", torch.int32)
    if states.dim() != 2:
        raise ValueError("states must be (ntiles, T/V)")
    ntiles, ns = states.shape
    T = ns * V
    if V not in (1, 2) or K * V > 16 or (T * K) % 16:
        raise ValueError(f"unsupported natural packing T={T} K={K} V={V}")
    packed = torch.empty((ntiles, T * K // 16), dtype=torch.uint16, device=states.device)
    bad = torch.zeros(1, dtype=torch.int32, device=states.device)
    with _on(states.device):
        check(lib().qtip_pack_trellis(_ptr(packed), _ptr(states), ntiles, T, K, V, _ptr(bad),
                                      stream_ptr(states.device)), "qtip_pack_trellis")
    nbad = int(bad.item())
    if nbad:
        raise ValueError(f"pack_trellis: {nbad} consecutive state pairs are not a bitshift trellis walk")
    return packed


def decode_natural(packed, lut, m, n, td_x, td_y, K, V):
    """Natural packing -> dense (m, n) in the dtype of `lut`, the expanded (V, 65536) table of the
    codebook (fp16 or fp32): get_hatW(unpack_trellis(.)) of lib/codebook/bitshift.py:329-381."""
    T = td_x * td_y
    ntiles = _check_natural(packed, T, K, V)
    if m % td_x or n % td_y or ntiles != (m // td_x) * (n // td_y) or td_y % V:
        raise ValueError(f"packed does not describe a {m}x{n} matrix of {td_x}x{td_y} tiles")
    require_cuda(lut, "lut", (torch.float16, torch.float32))
    if lut.shape != (V, 65536) or lut.device != packed.device:
        raise ValueError(f"lut must be ({V}, 65536) on {packed.device}")
    out = torch.empty((m, n), dtype=lut.dtype, device=packed.device)
    with _on(packed.device):
        check(lib().qtip_decode_natural(_ptr(out), _ptr(packed), _ptr(lut), _DT[lut.dtype], m, n, td_x, td_y, K, V,
                                        stream_ptr(packed.device)), "qtip_decode_natural")
    return out


def expand_table(tlut, nbits):
    """(2, 65536) value pairs of all states from a (2**nbits, 2) fp16 / fp32 table (quantlut_sym, transposed)."""
    require_cuda(tlut, "tlut", (torch.float16, torch.float32))
    if not 1 <= nbits <= 15 or tlut.shape != (1 << nbits, 2):
        raise ValueError(f"table must be (2**nbits, 2) with nbits up to 15 (got {tuple(tlut.shape)})")
    lut = torch.empty((2, 1 << 16), dtype=tlut.dtype, device=tlut.device)
    with _on(tlut.device):
        check(lib().qtip_expand_table(_ptr(lut), _ptr(tlut), _DT[tlut.dtype], nbits, 1, 1 << 16,
                                      stream_ptr(tlut.device)), "qtip_expand_table")
    return lut


def fold_table(lut):
    """(512, 2) fp16 table from the (65536, 2) fp16 / fp32 value pairs of all states, in any strides."""
    require_cuda(lut, "lut", (torch.float16, torch.float32), contiguous=False)
    if lut.shape != (1 << 16, 2):
        raise ValueError(f"lut must be (65536, 2) (got {tuple(lut.shape)})")
    tlut = torch.empty((512, 2), dtype=torch.float16, device=lut.device)
    with _on(lut.device):
        check(lib().qtip_fold_table(_ptr(tlut), _ptr(lut), _DT[lut.dtype], lut.stride(0), lut.stride(1),
                                    stream_ptr(lut.device)), "qtip_fold_table")
    return tlut


def scale_columns_grad(g, x, s):
    """(gx, gs) of y = x * s: g * s (rows, n) and the column sums of g * x (n,), fp32; g and x fp32, s fp16 / fp32."""
    require_cuda(g, "g", torch.float32)
    require_cuda(x, "x", torch.float32)
    require_cuda(s, "s", (torch.float16, torch.float32))
    if g.dim() != 2 or x.shape != g.shape or s.numel() != g.shape[1] or x.device != g.device or s.device != g.device:
        raise ValueError("g and x must be (rows, n) and s hold n values, on one device")
    rows, n = g.shape
    gx = torch.empty_like(g)
    gs = torch.empty(n, dtype=torch.float32, device=g.device)
    L = lib()
    ws = torch.empty(L.qtip_scale_columns_grad_workspace_bytes(rows, n), dtype=torch.uint8, device=g.device)
    with _on(g.device):
        check(L.qtip_scale_columns_grad(_ptr(gx), _ptr(gs), _ptr(g), _ptr(x), _ptr(s), _DT[s.dtype], rows, n, _ptr(ws),
                                        ws.numel(), stream_ptr(g.device)), "qtip_scale_columns_grad")
    return gx, gs


def rht_chain(parts, post, scale_out, residual, norm_weight, eps, pre, scale_in):
    """(x_new, xt) for one hidden-size vector per row, one launch:
    x_new = fp16(residual + fp16(post * scale_out * H(sum(parts)))),
    xt = fp16(scale_in * H(pre * rmsnorm(x_new))).  parts: (S, rows, n) fp32, n in {2048, 4096, 8192}."""
    require_cuda(parts, "parts", torch.float32)
    require_cuda(residual, "residual", torch.float16)
    require_cuda(norm_weight, "norm_weight", torch.float16)
    if parts.dim() != 3:
        raise ValueError("parts must be (S, rows, n)")
    S, rows, n = parts.shape
    if n not in (2048, 4096, 8192) or residual.numel() != rows * n or norm_weight.numel() != n:
        raise ValueError("rht_chain: unsupported or inconsistent shapes")
    if post is not None:
        require_cuda(post, "post", torch.float32)
    if pre is not None:
        require_cuda(pre, "pre", torch.float16)
    x_new = torch.empty((rows, n), dtype=torch.float16, device=parts.device)
    xt = torch.empty((rows, n), dtype=torch.float16, device=parts.device)
    with _on(parts.device):
        check(lib().qtip_rht_chain(_ptr(xt), _ptr(x_new), _ptr(parts), S, rows, n, _ptr(post), ctypes.c_float(scale_out),
                                   _ptr(residual), _ptr(norm_weight), ctypes.c_float(eps), _ptr(pre),
                                   ctypes.c_float(scale_in), stream_ptr(parts.device)), "qtip_rht_chain")
    return x_new, xt
