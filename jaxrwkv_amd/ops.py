"""Host-side operators over device tensors: thin, allocation + pointer plumbing around the C ABI.

Tensors are ``torch`` CUDA tensors (torch is used for device memory and streams only).  Every operator takes a
leading batch axis ``B`` -- what the reference gets from ``jax.vmap`` (rwkv7.py:419-431) -- and enqueues on the
current stream.  ``compat=True`` (default) reproduces ``AssociativeScanRWKV``; ``compat=False`` the sequential
``BaseRWKV``/``ScanRWKV`` conventions (they differ only in y[t] when new_starts[t+1], and in the returned state
when new_starts[length]).
"""
import ctypes

import torch
from torch.autograd import forward_ad

from . import _lib

_DT = {torch.float32: _lib.F32, torch.bfloat16: _lib.BF16}
_SA_DT = {torch.float32: torch.float32, torch.bfloat16: torch.float16}   # type of the WKV7 forward residual sa


def _stream():
    return torch._C._cuda_getCurrentRawStream(torch._C._cuda_getDevice())


def _p(t):
    return None if t is None else t.data_ptr()


def _dev(x, dtype=None):
    if not x.is_cuda:
        raise _lib.HipRwkvError("hiprwkv operators need CUDA (ROCm) tensors; there is no CPU path")
    if dtype is not None and x.dtype != dtype:
        x = x.to(dtype)
    return x.contiguous()


def _aligned(x):
    """x, or a copy of it where it does not lie on a 16-byte boundary (a slice of a flat array of parameters)."""
    return x if x.data_ptr() % 16 == 0 else x.clone()


# Placement of the (B,T,H,N) arrays one call touches.  Rows of different arrays at the same (token, head) are accessed
# together; when the arrays' base addresses are congruent modulo 1 KiB (any two large allocations of a caching
# allocator are: they start on 2 MiB boundaries) those rows compete for the same part of the memory system, and the
# write streams suffer most.  Measured on MI355X at B8 T4096 H32: the WKV7 forward with its residual 303 us with every
# array on a 2 MiB boundary, 284 us with the two outputs 128 and 256 bytes past one, 265 us with the inputs staggered
# as well; forward + backward 1619 / 1535 / 1469 us.  Offsets that are multiples of 1 KiB change nothing.  The operators
# therefore put every large array they allocate themselves at its own 128-byte step past the phase of the first input.
_PHASE_BYTES, _PHASES, _PHASED_MIN_BYTES = 128, 8, 1 << 20


def _phase(t):
    return (t.data_ptr() // _PHASE_BYTES) % _PHASES


def _empty_phased(shape, dtype, device, phase):
    """An uninitialised contiguous tensor whose address is ``phase`` 128-byte steps past a 1 KiB boundary (a view
    into a buffer 1 KiB larger); small tensors are allocated plainly."""
    n = dtype.itemsize
    for d in shape:
        n *= d
    if n < _PHASED_MIN_BYTES:
        return torch.empty(shape, dtype=dtype, device=device)
    buf = torch.empty(n + _PHASE_BYTES * _PHASES, dtype=torch.uint8, device=device)
    off = ((phase % _PHASES) * _PHASE_BYTES - buf.data_ptr()) % (_PHASE_BYTES * _PHASES)
    return buf[off:off + n].view(dtype).view(*shape)


def _empty_like_phased(ref, steps):
    """Like ``torch.empty_like(ref)``, ``steps`` 128-byte phases past ``ref``'s own."""
    if ref.nbytes < _PHASED_MIN_BYTES:
        return torch.empty_like(ref)
    return _empty_phased(tuple(ref.shape), ref.dtype, ref.device, _phase(ref) + steps)


def _length_ns(length, new_starts, B, T, device, keep=False):
    """``length`` as a contiguous (B,) int32 tensor (the kernels count a negative length as 0) and ``new_starts`` as a
    contiguous (B,T) bool one.  ``keep``: for a backward pass to come, so that ``length`` is never the caller's own memory."""
    if length is not None:
        if not torch.is_tensor(length) or length.device != device:
            length = torch.as_tensor(length, device=device)
        given = length
        if length.dtype != torch.int32:
            length = length.to(torch.int32)
        length = length.reshape(-1)
        if length.numel() == 1 and B > 1:
            length = length.expand(B)
        length = length.contiguous()
        assert length.numel() == B
        if keep and length.data_ptr() == given.data_ptr():
            length = length.clone()
    if new_starts is not None:
        if not torch.is_tensor(new_starts) or new_starts.device != device or new_starts.dtype != torch.bool:
            new_starts = torch.as_tensor(new_starts, device=device).to(torch.bool)
        if new_starts.dim() == 1:
            new_starts = new_starts[None].expand(B, T)
        new_starts = new_starts.contiguous()
        assert new_starts.shape == (B, T)
    return length, new_starts


def has_tangent(tensors):
    """Whether one of the tensors carries a forward-mode tangent (with or without autograd enabled)."""
    return forward_ad._current_level >= 0 and any(forward_ad.unpack_dual(t).tangent is not None for t in tensors)


def _needs_grad(*tensors):
    """Whether the call goes through its autograd function, which also is what refuses forward mode."""
    tensors = [t for t in tensors if t is not None]
    return (torch.is_grad_enabled() and any(t.requires_grad for t in tensors)) or has_tangent(tensors)


def autocast_elsewhere(x):
    """Whether ``torch.autocast`` makes products of x's dtype come out in another one."""
    dev = x.device.type
    return torch.is_autocast_enabled(dev) and torch.get_autocast_dtype(dev) != x.dtype


def _one_dtype(io, *tensors):
    """Kernels take one I/O dtype for all their operands: an operand of another would be read past its end."""
    for t in tensors:
        if t is not None and t.dtype != io:
            raise _lib.HipRwkvError(f"operand of {t.dtype} beside {io}")


def _flags(compat, force_seq=False, small_t=True, debug=0):
    return (_lib.LENGTH_I32 | (_lib.COMPAT_ASSOC if compat else 0) | (_lib.FORCE_SEQ if force_seq else 0)
            | (0 if small_t else _lib.NO_SMALL_T) | int(debug))


def handshake_failures():
    """Workgroups of the chunked kernels whose bounded hand-shake wait ran out since the library was loaded (their
    outputs are NaN).  Synchronises the current stream."""
    lib = _lib.load()
    n = ctypes.c_uint(0)
    _lib.check(lib.hiprwkv_handshake_failures(_stream(), ctypes.byref(n)), "hiprwkv_handshake_failures")
    return int(n.value)


def numeric_events():
    """Numeric events of the chunked kernels since the library was loaded: waves that capped a channel's decay over a
    chunk at e^-80 (its result is then inexact) and waves that found inf or NaN in a carried state of the bf16
    forward kernels (an IEEE-half operand overflowed: |state|, |sa|, |v| beyond 65504).  Synchronises the current
    stream."""
    lib = _lib.load()
    n = ctypes.c_uint(0)
    _lib.check(lib.hiprwkv_numeric_events(_stream(), ctypes.byref(n)), "hiprwkv_numeric_events")
    return int(n.value)


# ----------------------------------------------------------------------------- WKV7
def wkv7_fwd(r, w, k, v, a, b, s, length=None, new_starts=None, compat=True, want_sa=False, force_seq=False,
             small_t=True, debug_flags=0):
    """r,w,k,v,a,b (B,T,H,N) fp32|bf16; s (B,H,N,N) fp32|bf16.  Returns (new_s, y, sa|None); ``sa`` is fp32 for fp32
    inputs and fp16 for bf16 inputs.

    T <= 8 runs on the small-T (decode) kernel unless ``small_t=False``; otherwise on a chunked matrix-core kernel
    (fp16 operands for bf16 I/O, fp32 operands for fp32 I/O); ``force_seq`` selects the sequential fp32 kernel."""
    return _wkv7_fwd(r, w, k, v, a, b, s, length, new_starts, compat, want_sa, force_seq, small_t, debug_flags)[:3]


def _new_state(s, io, state_io):
    """Memory for a forward's new state beside the state ``s``, and the flag that goes with it.  ``state_io``: a caller rounds the state to
    the I/O type; from fp32 to bf16 the kernel does that (a launch of 3 us and 7 us of the host less)."""
    if state_io and s.dtype == torch.float32 and io == torch.bfloat16:
        return torch.empty(s.shape, dtype=io, device=s.device), _lib.NEW_STATE_IO
    return torch.empty_like(s), 0


def _wkv7_ends(io, B, T, H, N, device):
    """Memory that goes along to a backward in parts, None where the sequence runs whole."""
    nbytes = _lib.load().hiprwkv_wkv7_ends_bytes(_DT[io], B, T, H, N)
    return _workspace(nbytes, device) if nbytes else None


def _wkv7_fwd(r, w, k, v, a, b, s, length=None, new_starts=None, compat=True, want_sa=False, force_seq=False,
              small_t=True, debug_flags=0, want_ends=False, state_io=False):
    """``wkv7_fwd`` with a fourth result: with ``want_ends`` what lets the backward run the sequence in parts, where that is of use
    (fp32: filled here; bf16: memory that the backward fills).  ``state_io``: see ``_new_state``."""
    lib = _lib.load()
    io = r.dtype
    r, w, k, v, a, b = (_dev(x, io) for x in (r, w, k, v, a, b))
    s = _dev(s)
    B, T, H, N = r.shape
    assert s.shape == (B, H, N, N), (s.shape, r.shape)
    length, new_starts = _length_ns(length, new_starts, B, T, r.device)
    y = _empty_like_phased(r, 1)
    new_s, state_flag = _new_state(s, io, state_io)
    # the residual for the backward pass: fp32 beside fp32 I/O, fp16 beside bf16 I/O
    sa = _empty_phased((B, T, H, N), _SA_DT[io], r.device, _phase(r) + 2) if want_sa else None
    nbytes = 0 if force_seq else lib.hiprwkv_wkv7_fwd_workspace_bytes(_DT[io], B, T, H, N)
    ws = _workspace(nbytes, r.device) if nbytes else None
    ends = _wkv7_ends(io, B, T, H, N, r.device) if want_sa and want_ends and not force_seq else None
    fn, more = (lib.hiprwkv_wkv7_fwd_parts, ()) if ends is None else (lib.hiprwkv_wkv7_fwd_ends, (_p(ends),))
    rc = fn(_stream(), _DT[io], _DT[s.dtype], B, T, H, N, _p(w), _p(r), _p(k), _p(v), _p(a), _p(b),
            _p(s), _p(length), _p(new_starts), _p(y), _p(sa), _p(new_s), *more, _p(ws), nbytes,
            _flags(compat, force_seq, small_t, debug_flags) | state_flag)
    _lib.check(rc, "hiprwkv_wkv7_fwd")
    return new_s, y, sa, ends


def _packed_state(t, B, H, N):
    """(pointer tensor, batch stride in elements) of a state view whose sequences are H*N*N contiguous elements each."""
    assert t.is_cuda and t.shape[0] == B and t[0].numel() == H * N * N, (t.shape, (B, H, N))
    assert t[0].is_contiguous(), "a sequence's state must be contiguous"
    return t, (t.stride(0) if B > 1 else H * N * N)


def wkv7_step(r, w, k, v, a, b, s, new_s, length=None, new_starts=None, compat=True):
    """A decode step (T <= 8) on states inside a packed model state: ``s`` and ``new_s`` are views with a batch axis in
    front and H*N*N contiguous elements per sequence, e.g. ``state[:, layer, 2:]`` of a ``(B, L, 2+N, C)`` model state
    (rwkv7.py:176-180, 254-260); ``new_s`` is written in place (it may be ``s``).  Returns y.  No autograd."""
    lib = _lib.load()
    io = r.dtype
    r, w, k, v, a, b = (_dev(x, io) for x in (r, w, k, v, a, b))
    B, T, H, N = r.shape
    s, s_stride = _packed_state(s, B, H, N)
    new_s, ns_stride = _packed_state(new_s, B, H, N)
    assert s.dtype == new_s.dtype
    length, new_starts = _length_ns(length, new_starts, B, T, r.device)
    y = torch.empty_like(r)
    rc = lib.hiprwkv_wkv7_step(_stream(), _DT[io], _DT[s.dtype], B, T, H, N, _p(w), _p(r), _p(k), _p(v), _p(a), _p(b),
                               _p(s), s_stride, _p(length), _p(new_starts), _p(y), _p(new_s), ns_stride,
                               _flags(compat, False, True, 0))
    _lib.check(rc, "hiprwkv_wkv7_step")
    return y


def wkv7_bwd(r, w, k, v, a, b, s, length, new_starts, gy, sa, gs_out=None, compat=True, force_seq=False,
             debug_flags=0, ends=None, parts=False):
    """Cotangents (gr, gw, gk, gv, ga, gb, gs) of ``wkv7_fwd`` for cotangents gy of y and gs_out of new_s.

    bf16 inputs use the chunked MFMA kernels where they exist unless ``force_seq`` asks for the sequential ones.  ``ends``: the
    forward's (``_wkv7_fwd``), for the sequences in parts; with ``parts`` bf16 inputs need none."""
    lib = _lib.load()
    io = r.dtype
    r, w, k, v, a, b, gy = (_dev(x, io) for x in (r, w, k, v, a, b, gy))
    s = _dev(s)
    sa = _dev(sa, _SA_DT[io])
    gs_out = None if gs_out is None else _aligned(_dev(gs_out, s.dtype))
    B, T, H, N = r.shape
    length, new_starts = _length_ns(length, new_starts, B, T, r.device)
    gw, gr, gk, gv, ga, gb = (_empty_like_phased(r, i) for i in range(1, 7))
    gs = torch.empty_like(s)
    if parts and ends is None and io == torch.bfloat16 and not force_seq:
        ends = _wkv7_ends(io, B, T, H, N, r.device)
    if ends is None:
        fn, more, nbytes = lib.hiprwkv_wkv7_bwd, (), lib.hiprwkv_wkv7_bwd_workspace_bytes(B, T, H, N)
    else:
        ends = _aligned(_dev(ends))
        fn, more, nbytes = lib.hiprwkv_wkv7_bwd_ends, (_p(ends),), lib.hiprwkv_wkv7_bwd_ends_workspace_bytes(_DT[io], B, T, H, N)
    ws = torch.empty(nbytes, dtype=torch.uint8, device=r.device)
    rc = fn(_stream(), _DT[io], _DT[s.dtype], B, T, H, N, _p(w), _p(r), _p(k), _p(v), _p(a), _p(b),
            _p(s), _p(length), _p(new_starts), _p(gy), _p(sa), _p(gs_out), *more,
            _p(gw), _p(gr), _p(gk), _p(gv), _p(ga), _p(gb), _p(gs), _p(ws), nbytes,
            _flags(compat, force_seq, debug=debug_flags))
    _lib.check(rc, "hiprwkv_wkv7_bwd")
    return gr, gw, gk, gv, ga, gb, gs


class _Wkv7(torch.autograd.Function):
    """custom VJP, the counterpart of ``wkv7_cuda`` (rwkv7.py:442-446)."""

    @staticmethod
    def forward(ctx, r, w, k, v, a, b, s, length, new_starts, compat, force_seq):
        need = any(x.requires_grad for x in (r, w, k, v, a, b, s))
        new_s, y, sa, ends = _wkv7_fwd(r, w, k, v, a, b, s, length, new_starts, compat, want_sa=need, force_seq=force_seq,
                                       want_ends=need and r.dtype == torch.float32)
        ctx.compat = compat
        ctx.force_seq = force_seq
        ctx.save_for_backward(r, w, k, v, a, b, s, length, new_starts, sa, ends)
        return new_s, y

    @staticmethod
    def backward(ctx, gs_out, gy):
        r, w, k, v, a, b, s, length, new_starts, sa, ends = ctx.saved_tensors
        if gy is None:
            gy = torch.zeros_like(r)
        gr, gw, gk, gv, ga, gb, gs = wkv7_bwd(r, w, k, v, a, b, s, length, new_starts, gy, sa, gs_out, ctx.compat,
                                              ctx.force_seq, ends=ends, parts=True)
        return gr, gw, gk, gv, ga, gb, gs, None, None, None, None


def wkv7(r, w, k, v, a, b, s, length=None, new_starts=None, compat=True, force_seq=False, state_io=False):
    """Differentiable WKV7: returns (new_s, y).  ``force_seq`` runs the sequential fp32 kernels whatever the dtype.  ``state_io``: the
    caller will round new_s to r's type, so it may come in that already."""
    B, T = r.shape[:2]
    if not _needs_grad(r, w, k, v, a, b, s):
        return _wkv7_fwd(r, w, k, v, a, b, s, length, new_starts, compat, force_seq=force_seq, state_io=state_io)[:2]
    length, new_starts = _length_ns(length, new_starts, B, T, r.device, keep=True)
    return _Wkv7.apply(r, w, k, v, a, b, s, length, new_starts, compat, force_seq)


# ----------------------------------------------------------------------------- WKV6
def wkv6_fwd(r, k, v, w, u, s, length=None, new_starts=None, compat=True, force_seq=False, small_t=True,
             debug_flags=0, state_io=False):
    """r,k,v (B,T,H,N); w (B,T,H,N), or (H,N) for a log decay shared by all tokens (RWKV-5); u (H,N);
    s (B,H,N,N) [key, value].  Returns (new_s, y).

    T <= 8 runs on the small-T (decode) kernel unless ``small_t=False``; otherwise bf16 inputs run on the chunked
    MFMA kernel unless ``force_seq`` asks for the sequential fp32 one.  ``state_io``: see ``_new_state``."""
    lib = _lib.load()
    io = r.dtype
    B, T, H, N = r.shape
    r, k, v = (_dev(x, io) for x in (r, k, v))
    per_head = w.numel() == H * N and (B * T != 1 or w.dim() == 2)
    w = _dev(w.reshape(H, N) if per_head else w.reshape(B, T, H, N), io)
    u = _dev(u.reshape(H, N), io)
    s = _dev(s)
    length, new_starts = _length_ns(length, new_starts, B, T, r.device)
    y = _empty_like_phased(r, 1)
    new_s, state_flag = _new_state(s, io, state_io)
    nbytes = 0 if force_seq else lib.hiprwkv_wkv6_fwd_workspace_bytes(_DT[io], B, T, H, N)
    ws = _workspace(nbytes, r.device) if nbytes else None
    rc = lib.hiprwkv_wkv6_fwd_parts(_stream(), _DT[io], _DT[s.dtype], B, T, H, N, _p(r), _p(k), _p(v), _p(w), _p(u), _p(s),
                                    _p(length), _p(new_starts), _p(y), _p(new_s), _p(ws), nbytes,
                                    _flags(compat, force_seq, small_t, debug_flags) | state_flag | (_lib.W_PER_HEAD if per_head else 0))
    _lib.check(rc, "hiprwkv_wkv6_fwd")
    return new_s, y


def wkv6_step(r, k, v, w, u, s, new_s, length=None, new_starts=None, compat=True):
    """A decode step (T <= 8) on states inside a packed model state: ``s`` and ``new_s`` are views with a batch axis in
    front and H*N*N contiguous elements per sequence (rwkv6.py:221-224); ``new_s`` is written in place (it may be
    ``s``).  ``w`` (B,T,H,N) or the shared (H,N) decay.  Returns y.  No autograd."""
    lib = _lib.load()
    io = r.dtype
    B, T, H, N = r.shape
    r, k, v = (_dev(x, io) for x in (r, k, v))
    per_head = w.numel() == H * N and (B * T != 1 or w.dim() == 2)
    w = _dev(w.reshape(H, N) if per_head else w.reshape(B, T, H, N), io)
    u = _dev(u.reshape(H, N), io)
    s, s_stride = _packed_state(s, B, H, N)
    new_s, ns_stride = _packed_state(new_s, B, H, N)
    assert s.dtype == new_s.dtype
    length, new_starts = _length_ns(length, new_starts, B, T, r.device)
    y = torch.empty_like(r)
    flags = _flags(compat, False, True, 0) | (_lib.W_PER_HEAD if per_head else 0)
    rc = lib.hiprwkv_wkv6_step(_stream(), _DT[io], _DT[s.dtype], B, T, H, N, _p(r), _p(k), _p(v), _p(w), _p(u), _p(s),
                               s_stride, _p(length), _p(new_starts), _p(y), _p(new_s), ns_stride, flags)
    _lib.check(rc, "hiprwkv_wkv6_step")
    return y


def wkv6_bwd(r, k, v, w, u, s, length, new_starts, gy, gs_out=None, compat=True, force_seq=False, debug_flags=0):
    """Cotangents (gr, gk, gv, gw, gu, gs) of ``wkv6_fwd``; gu is summed over the batch here, and so is gw over batch
    and tokens when ``w`` is the shared (H,N) decay.

    bf16 inputs run on the chunked MFMA kernels unless ``force_seq`` asks for the sequential fp32 ones."""
    lib = _lib.load()
    io = r.dtype
    B, T, H, N = r.shape
    r, k, v, gy = (_dev(x, io) for x in (r, k, v, gy))
    per_head = w.numel() == H * N and (B * T != 1 or w.dim() == 2)
    w = _dev(w.reshape(H, N) if per_head else w.reshape(B, T, H, N), io)
    u = _dev(u.reshape(H, N), io)
    s = _dev(s)
    gs_out = None if gs_out is None else _dev(gs_out, s.dtype)
    length, new_starts = _length_ns(length, new_starts, B, T, r.device)
    gr, gk, gv, gw = (_empty_like_phased(r, i) for i in range(1, 5))
    gu = torch.empty((B, H, N), dtype=torch.float32, device=r.device)
    gs = torch.empty_like(s)
    nbytes = lib.hiprwkv_wkv6_bwd_workspace_bytes(B, T, H, N)
    ws = torch.empty(nbytes, dtype=torch.uint8, device=r.device)
    rc = lib.hiprwkv_wkv6_bwd(_stream(), _DT[io], _DT[s.dtype], B, T, H, N, _p(r), _p(k), _p(v), _p(w), _p(u), _p(s),
                              _p(length), _p(new_starts), _p(gy), _p(gs_out), _p(gr), _p(gk), _p(gv), _p(gw), _p(gu),
                              _p(gs), _p(ws), nbytes,
                              _flags(compat, force_seq, debug=debug_flags) | (_lib.W_PER_HEAD if per_head else 0))
    _lib.check(rc, "hiprwkv_wkv6_bwd")
    if per_head:
        gw = gw.float().sum((0, 1)).to(io)
    return gr, gk, gv, gw, gu.sum(0).to(io), gs


class _Wkv6(torch.autograd.Function):
    @staticmethod
    def forward(ctx, r, k, v, w, u, s, length, new_starts, compat, force_seq):
        new_s, y = wkv6_fwd(r, k, v, w, u, s, length, new_starts, compat, force_seq=force_seq)
        ctx.compat = compat
        ctx.force_seq = force_seq
        ctx.shapes = (w.shape, u.shape)
        ctx.save_for_backward(r, k, v, w, u, s, length, new_starts)
        return new_s, y

    @staticmethod
    def backward(ctx, gs_out, gy):
        r, k, v, w, u, s, length, new_starts = ctx.saved_tensors
        if gy is None:
            gy = torch.zeros_like(r)
        gr, gk, gv, gw, gu, gs = wkv6_bwd(r, k, v, w, u, s, length, new_starts, gy, gs_out, ctx.compat, ctx.force_seq)
        return gr, gk, gv, gw.reshape(ctx.shapes[0]), gu.reshape(ctx.shapes[1]), gs, None, None, None, None


def wkv6(r, k, v, w, u, s, length=None, new_starts=None, compat=True, force_seq=False, state_io=False):
    """Differentiable WKV6: returns (new_s, y).  ``force_seq`` and ``state_io`` as in ``wkv7``."""
    B, T = r.shape[:2]
    if not _needs_grad(r, k, v, w, u, s):
        return wkv6_fwd(r, k, v, w, u, s, length, new_starts, compat, force_seq=force_seq, state_io=state_io)
    length, new_starts = _length_ns(length, new_starts, B, T, r.device, keep=True)
    return _Wkv6.apply(r, k, v, w, u, s, length, new_starts, compat, force_seq)


# ----------------------------------------------------------------------------- WKV4
def wkv4_fwd(w_neg, u, k, v, s, length=None, new_starts=None, compat=True, want_ckpt=False):
    """w_neg = -exp(time_decay), u (C,); k,v (B,T,C); s (B,3,C).  Returns (new_s, wkv) -- receptance not applied.
    ``want_ckpt``: also return the checkpoint workspace that ``wkv4_bwd(..., ckpt=)`` takes (the state entering every
    16th step), so that the backward pass need not recompute it."""
    lib = _lib.load()
    io = k.dtype
    k, v, s, w_neg, u = (_dev(x, io) for x in (k, v, s, w_neg, u))
    B, T, C = k.shape
    assert s.shape == (B, 3, C) and w_neg.shape == (C,) and u.shape == (C,)
    length, new_starts = _length_ns(length, new_starts, B, T, k.device)
    y = torch.empty_like(k)
    new_s = torch.empty_like(s)
    if want_ckpt:
        nbytes = lib.hiprwkv_wkv4_bwd_workspace_bytes(B, T, C)
        ws = torch.empty(nbytes, dtype=torch.uint8, device=k.device)
        rc = lib.hiprwkv_wkv4_fwd_ckpt(_stream(), _DT[io], B, T, C, _p(w_neg), _p(u), _p(k), _p(v), _p(s), _p(length),
                                       _p(new_starts), _p(new_s), _p(y), _p(ws), nbytes, _flags(compat))
        _lib.check(rc, "hiprwkv_wkv4_fwd_ckpt")
        return new_s, y, ws
    rc = lib.hiprwkv_wkv4_fwd(_stream(), _DT[io], B, T, C, _p(w_neg), _p(u), _p(k), _p(v), _p(s), _p(length),
                              _p(new_starts), _p(new_s), _p(y), _flags(compat))
    _lib.check(rc, "hiprwkv_wkv4_fwd")
    return new_s, y


def wkv4_bwd(w_neg, u, k, v, s, length, new_starts, gy, gs_new=None, compat=True, ckpt=None):
    """Cotangents (gw, gu, gk, gv, gs) of ``wkv4_fwd``; gw, gu are summed over the batch here (rwkv4.py:351).
    ``ckpt``: the workspace ``wkv4_fwd(..., want_ckpt=True)`` returned for the same inputs."""
    lib = _lib.load()
    io = k.dtype
    k, v, s, w_neg, u, gy = (_dev(x, io) for x in (k, v, s, w_neg, u, gy))
    gs_new = None if gs_new is None else _dev(gs_new, io)
    B, T, C = k.shape
    length, new_starts = _length_ns(length, new_starts, B, T, k.device)
    gk, gv = torch.empty_like(k), torch.empty_like(v)
    gs = torch.empty_like(s)
    gw = torch.empty((B, C), dtype=torch.float32, device=k.device)
    gu = torch.empty((B, C), dtype=torch.float32, device=k.device)
    nbytes = lib.hiprwkv_wkv4_bwd_workspace_bytes(B, T, C)
    if ckpt is None:
        ws = torch.empty(nbytes, dtype=torch.uint8, device=k.device)
    else:
        ws = ckpt
        assert ws.dtype == torch.uint8 and ws.numel() >= nbytes and ws.is_cuda
    rc = lib.hiprwkv_wkv4_bwd(_stream(), _DT[io], B, T, C, _p(w_neg), _p(u), _p(k), _p(v), _p(gy), _p(s), _p(length),
                              _p(new_starts), _p(gs_new), _p(gw), _p(gu), _p(gk), _p(gv), _p(gs), _p(ws), nbytes,
                              _flags(compat) | (0 if ckpt is None else _lib.CKPT_READY))
    _lib.check(rc, "hiprwkv_wkv4_bwd")
    return gw.sum(0).to(io), gu.sum(0).to(io), gk, gv, gs


def _workspace(nbytes, device):
    return torch.empty(nbytes, dtype=torch.uint8, device=device)


def _wkv4_mix_fwd(w, u, k, v, r, s, length, new_starts, flags, want_ckpt):
    lib = _lib.load()
    io = k.dtype
    B, T, C = k.shape
    assert s.shape == (B, 3, C) and w.shape == (C,) and u.shape == (C,)
    y, new_s = torch.empty_like(k), torch.empty_like(s)
    ckpt = _workspace(lib.hiprwkv_wkv4_bwd_workspace_bytes(B, T, C), k.device) if want_ckpt else None
    nbytes = lib.hiprwkv_wkv4_mix_workspace_bytes(B, T, C)
    ws = _workspace(nbytes, k.device) if nbytes else None
    rc = lib.hiprwkv_wkv4_mix(_stream(), _DT[io], B, T, C, _p(w), _p(u), _p(k), _p(v), _p(r), _p(s), _p(length),
                              _p(new_starts), _p(new_s), _p(y), _p(ckpt), ckpt.numel() if want_ckpt else 0, _p(ws), nbytes,
                              flags)
    _lib.check(rc, "hiprwkv_wkv4_mix")
    return new_s, y, ckpt


class _Wkv4(torch.autograd.Function):
    """custom VJP, the counterpart of ``wkv4_cuda`` (rwkv4.py:379-383), with the receptance where ``r`` is given."""

    @staticmethod
    def forward(ctx, w, u, k, v, r, s, length, new_starts, flags):
        io = k.dtype
        k, v, s, u = (_dev(x, io) for x in (k, v, s, u))
        w, r = _aligned(_dev(w, io)), (None if r is None else _aligned(_dev(r, io)))
        new_s, y, ckpt = _wkv4_mix_fwd(w, u, k, v, r, s, length, new_starts, flags, True)
        ctx.flags = flags
        ctx.save_for_backward(w, u, k, v, r, s, length, new_starts, ckpt)
        ctx.set_materialize_grads(False)
        if not any(ctx.needs_input_grad[i] for i in (0, 1, 2, 3, 5)):
            ctx.mark_non_differentiable(new_s)            # the state does not depend on the receptance
        return new_s, y

    @staticmethod
    def backward(ctx, gs_new, gy):
        w, u, k, v, r, s, length, new_starts, ckpt = ctx.saved_tensors
        lib = _lib.load()
        io = k.dtype
        B, T, C = k.shape
        given = gy is not None
        gy = _aligned(_dev(gy, io)) if given else torch.zeros_like(k)
        gs_new = None if gs_new is None else _dev(gs_new, io)
        gk, gv, gs = torch.empty_like(k), torch.empty_like(v), torch.empty_like(s)
        gr = None if r is None else torch.empty_like(r)
        gw, gu = torch.empty_like(w), torch.empty_like(u)
        nbytes = lib.hiprwkv_wkv4_mix_bwd_workspace_bytes(B, T, C)
        ws = _workspace(nbytes, k.device)
        rc = lib.hiprwkv_wkv4_mix_bwd(_stream(), _DT[io], B, T, C, _p(w), _p(u), _p(k), _p(v), _p(r), _p(gy), _p(s),
                                      _p(length), _p(new_starts), _p(gs_new), _p(ckpt), ckpt.numel(), _p(gw), _p(gu), _p(gk),
                                      _p(gv), _p(gr), _p(gs), _p(ws), nbytes, ctx.flags | _lib.CKPT_READY)
        _lib.check(rc, "hiprwkv_wkv4_mix_bwd")
        return gw, gu, gk, gv, (gr if given else None), gs, None, None, None


def wkv4(w_neg, u, k, v, s, length=None, new_starts=None, compat=True):
    """Differentiable WKV4 in the op's convention (w_neg = -exp(time_decay), no receptance): returns (new_s, wkv)."""
    return _wkv4_apply(w_neg, u, k, v, None, s, length, new_starts, _flags(compat))


def _wkv4_apply(w, u, k, v, r, s, length, new_starts, flags):
    B, T = k.shape[:2]
    grad = _needs_grad(w, u, k, v, r, s)
    length, new_starts = _length_ns(length, new_starts, B, T, k.device, keep=grad)
    if grad:
        return _Wkv4.apply(w, u, k, v, r, s, length, new_starts, flags)
    u, k, v, s = (_dev(x, k.dtype) for x in (u, k, v, s))
    w, r = _aligned(_dev(w, k.dtype)), (None if r is None else _aligned(_dev(r, k.dtype)))
    return _wkv4_mix_fwd(w, u, k, v, r, s, length, new_starts, flags, False)[:2]


def wkv4_mix(r, k, v, w, u, s, length=None, new_starts=None, compat=True):
    """RWKV-4's ``inner_loop`` with a batch axis: the op with decay ``-exp(w)`` and its output times the receptance ``r``,
    all tensors in one dtype.  Returns (new_s, r wkv); differentiable in r, k, v, w, u and s."""
    return _wkv4_apply(w, u, k, v, r, s, length, new_starts, _flags(compat) | _lib.W_RAW)


# ----------------------------------------------------------------------------- RWKV-7 time-mixing stages
def _premix_fwd(k, a, k_k, k_a):
    lib = _lib.load()
    io = k.dtype
    H, N = k.shape[-2:]
    rows = k.numel() // (H * N)
    k_out, a_out, b_out = (torch.empty_like(k) for _ in range(3))
    rc = lib.hiprwkv_rwkv7_premix(_stream(), _DT[io], rows, H, N, _p(k), _p(a), _p(k_k), _p(k_a), _p(k_out), _p(a_out),
                                  _p(b_out))
    _lib.check(rc, "hiprwkv_rwkv7_premix")
    return k_out, a_out, b_out


def _postmix_fwd(y, r, k, v, g, ln_w, ln_b, r_k, eps):
    lib = _lib.load()
    io = y.dtype
    H, N = y.shape[-2:]
    rows = y.numel() // (H * N)
    out = torch.empty_like(y)
    rc = lib.hiprwkv_rwkv7_postmix(_stream(), _DT[io], rows, H, N, _p(y), _p(r), _p(k), _p(v), _p(g), _p(ln_w), _p(ln_b),
                                   _p(r_k), float(eps), _p(out))
    _lib.check(rc, "hiprwkv_rwkv7_postmix")
    return out


class _Premix(torch.autograd.Function):
    @staticmethod
    def forward(ctx, k, a, k_k, k_a):
        ctx.save_for_backward(k, a, k_k, k_a)
        return _premix_fwd(k, a, k_k, k_a)

    @staticmethod
    def backward(ctx, gk_out, ga_out, gb_out):
        k, a, k_k, k_a = ctx.saved_tensors
        lib = _lib.load()
        io = k.dtype
        H, N = k.shape[-2:]
        rows = k.numel() // (H * N)
        gk_out, ga_out, gb_out = (_dev(x, io) for x in (gk_out, ga_out, gb_out))
        gk, ga = torch.empty_like(k), torch.empty_like(a)
        gk_k, gk_a = (torch.empty(H, N, dtype=torch.float32, device=k.device) for _ in range(2))
        rc = lib.hiprwkv_rwkv7_premix_bwd(_stream(), _DT[io], rows, H, N, _p(k), _p(a), _p(k_k), _p(k_a), _p(gk_out),
                                          _p(ga_out), _p(gb_out), _p(gk), _p(ga), _p(gk_k), _p(gk_a))
        _lib.check(rc, "hiprwkv_rwkv7_premix_bwd")
        return gk, ga, gk_k.to(io), gk_a.to(io)


class _Postmix(torch.autograd.Function):
    @staticmethod
    def forward(ctx, y, r, k, v, g, ln_w, ln_b, r_k, eps):
        ctx.save_for_backward(y, r, k, v, g, ln_w, ln_b, r_k)
        ctx.eps = eps
        return _postmix_fwd(y, r, k, v, g, ln_w, ln_b, r_k, eps)

    @staticmethod
    def backward(ctx, gout):
        y, r, k, v, g, ln_w, ln_b, r_k = ctx.saved_tensors
        lib = _lib.load()
        io = y.dtype
        H, N = y.shape[-2:]
        rows = y.numel() // (H * N)
        gout = _dev(gout, io)
        gy, gr, gk, gv, gg = (torch.empty_like(y) for _ in range(5))
        gw, gb, grk = (torch.empty(H, N, dtype=torch.float32, device=y.device) for _ in range(3))
        rc = lib.hiprwkv_rwkv7_postmix_bwd(_stream(), _DT[io], rows, H, N, _p(y), _p(r), _p(k), _p(v), _p(g), _p(ln_w),
                                           _p(ln_b), _p(r_k), float(ctx.eps), _p(gout), _p(gy), _p(gr), _p(gk), _p(gv),
                                           _p(gg), _p(gw), _p(gb), _p(grk))
        _lib.check(rc, "hiprwkv_rwkv7_postmix_bwd")
        return gy, gr, gk, gv, gg, gw.to(io), gb.to(io), grk.to(io), None


def _ptr_array(tensors):
    return (ctypes.c_void_p * len(tensors))(*[t.data_ptr() for t in tensors])


def _shift_row(prev, B, C, io):
    """The token before t = 0 of every sequence as (tensor, batch stride in elements): rows of C contiguous elements,
    read where they lie when the stride allows it (a row of the packed model state), else from a dense copy."""
    assert prev.shape == (B, C), (prev.shape, (B, C))
    if not prev.is_cuda:
        raise _lib.HipRwkvError("hiprwkv operators need CUDA (ROCm) tensors; there is no CPU path")
    elem = 4 if io == torch.float32 else 2
    ok = (prev.dtype == io and (C == 1 or prev.stride(1) == 1) and prev.data_ptr() % 16 == 0
          and (B == 1 or (prev.stride(0) >= C and (prev.stride(0) * elem) % 16 == 0)))
    if not ok:
        prev = prev.to(io).contiguous()
    return prev, (prev.stride(0) if B > 1 else C)


def _shiftmix_fwd(x, prev, prev_stride, ns, mix):
    lib = _lib.load()
    io = x.dtype
    B, T, C = x.shape
    outs = [torch.empty_like(x) for _ in mix]
    rc = lib.hiprwkv_rwkv7_shiftmix(_stream(), _DT[io], B, T, C, len(mix), _p(x), _p(prev), prev_stride, _p(ns),
                                    _ptr_array(mix), _ptr_array(outs))
    _lib.check(rc, "hiprwkv_rwkv7_shiftmix")
    return tuple(outs)


class _ShiftMix(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x, prev, ns, *mix):
        prev_t, stride = _shift_row(prev, x.shape[0], x.shape[2], x.dtype)
        ctx.save_for_backward(x, prev_t, *mix)
        ctx.ns = ns
        return _shiftmix_fwd(x, prev_t, stride, ns, mix)

    @staticmethod
    def backward(ctx, *gs):
        x, prev, *mix = ctx.saved_tensors
        lib = _lib.load()
        io = x.dtype
        B, T, C = x.shape
        prev, stride = _shift_row(prev, B, C, io)         # a saved-tensor hook may have moved it
        gs = [_dev(g, io) for g in gs]
        dx = torch.empty_like(x)
        dprev = torch.empty((B, C), dtype=io, device=x.device)
        dmix = torch.empty((len(mix), C), dtype=torch.float32, device=x.device)
        rc = lib.hiprwkv_rwkv7_shiftmix_bwd(_stream(), _DT[io], B, T, C, len(mix), _p(x), _p(prev), stride,
                                            _p(ctx.ns), _ptr_array(mix), _ptr_array(gs), _p(dx), _p(dprev), C, _p(dmix))
        _lib.check(rc, "hiprwkv_rwkv7_shiftmix_bwd")
        return (dx, dprev, None) + tuple(dmix[i].to(io) for i in range(len(mix)))


def rwkv7_shiftmix(x, prev, new_starts, mix):
    """Token shift and interpolation of rwkv7.py:226-235 (six ``mix`` vectors, time mixing) and :192-195 (one, channel
    mixing): x (B,T,C); prev (B,C), the token before t = 0 (a row of the model state; read in place);
    new_starts (B,T) bool or None; mix a list of (C,) parameters.  Returns the tuple of x + sx*mix_i with
    sx = (new_starts ? 0 : previous token) - x.  Differentiable in x, prev and the mix vectors."""
    io = x.dtype
    B, T, C = x.shape
    assert len(mix) in (1, 6) and C % 8 == 0, (len(mix), C)
    x = _dev(x, io)
    mix2 = [_dev(m.reshape(C), io) for m in mix]
    _, ns = _length_ns(None, new_starts, B, T, x.device)
    if torch.is_grad_enabled() and any(t.requires_grad for t in (x, prev, *mix)):
        return _ShiftMix.apply(x, prev, ns, *mix2)
    prev_t, stride = _shift_row(prev, B, C, io)
    return _shiftmix_fwd(x, prev_t, stride, ns, mix2)


def _gate_fwd(x, p, kind):
    lib = _lib.load()
    io = x.dtype
    C = x.shape[-1]
    out = torch.empty_like(x)
    fn = (lib.hiprwkv_rwkv7_decay, lib.hiprwkv_rwkv7_agate)[kind]
    _lib.check(fn(_stream(), _DT[io], x.numel() // C, C, _p(x), _p(p), _p(out)), "hiprwkv_rwkv7_" + ("decay", "agate")[kind])
    return out


class _Gate(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x, p, kind):
        ctx.save_for_backward(x, p)
        ctx.kind = kind
        return _gate_fwd(x, p, kind)

    @staticmethod
    def backward(ctx, g):
        x, p = ctx.saved_tensors
        lib = _lib.load()
        io = x.dtype
        C = x.shape[-1]
        g = _dev(g, io)
        dx = torch.empty_like(x)
        dp = torch.empty(C, dtype=torch.float32, device=x.device)
        fn = (lib.hiprwkv_rwkv7_decay_bwd, lib.hiprwkv_rwkv7_agate_bwd)[ctx.kind]
        _lib.check(fn(_stream(), _DT[io], x.numel() // C, C, _p(x), _p(p), _p(g), _p(dx), _p(dp)),
                   "hiprwkv_rwkv7_" + ("decay", "agate")[ctx.kind] + "_bwd")
        return dx, dp.to(io), None


def _gate(x, p, kind):
    io = x.dtype
    C = x.shape[-1]
    assert C % 8 == 0, C
    x, p2 = _dev(x, io), _dev(p.reshape(C), io)
    if torch.is_grad_enabled() and (x.requires_grad or p.requires_grad):
        return _Gate.apply(x, p2, kind)
    return _gate_fwd(x, p2, kind)


def rwkv7_decay(x, w0):
    """The decay argument of the WKV op, rwkv7.py:237: ``-softplus(-(w0 + x)) - 0.5`` for x (..., C) (the low-rank
    term ``tanh(xw w1) w2``) and the parameter w0 (C,).  Differentiable in both."""
    return _gate(x, w0, 0)


def rwkv7_agate(x, a0):
    """The in-context learning rate, rwkv7.py:244: ``sigmoid(a0 + x)`` for x (..., C) and a0 (C,).  Differentiable."""
    return _gate(x, a0, 1)


def _relusq_fwd(x):
    out = torch.empty_like(x)
    rc = _lib.load().hiprwkv_rwkv7_relusq(_stream(), _DT[x.dtype], x.numel(), _p(x), _p(out))
    _lib.check(rc, "hiprwkv_rwkv7_relusq")
    return out


class _ReluSq(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x):
        ctx.save_for_backward(x)
        return _relusq_fwd(x)

    @staticmethod
    def backward(ctx, g):
        x, = ctx.saved_tensors
        g = _dev(g, x.dtype)
        dx = torch.empty_like(x)
        rc = _lib.load().hiprwkv_rwkv7_relusq_bwd(_stream(), _DT[x.dtype], x.numel(), _p(x), _p(g), _p(dx))
        _lib.check(rc, "hiprwkv_rwkv7_relusq_bwd")
        return dx


def rwkv7_relusq(x):
    """Channel mixing's activation, rwkv7.py:196: ``relu(x)**2`` in one pass; differentiable.  numel a multiple of 8."""
    assert x.numel() % 8 == 0, x.shape
    x = _dev(x, x.dtype)
    if torch.is_grad_enabled() and x.requires_grad:
        return _ReluSq.apply(x)
    return _relusq_fwd(x)


def _vmix_fwd(v, vf, x, v0):
    lib = _lib.load()
    io = v.dtype
    C = v.shape[-1]
    out = torch.empty_like(v)
    rc = lib.hiprwkv_rwkv7_vmix(_stream(), _DT[io], v.numel() // C, C, _p(v), _p(vf), _p(x), _p(v0), _p(out))
    _lib.check(rc, "hiprwkv_rwkv7_vmix")
    return out


class _VMix(torch.autograd.Function):
    @staticmethod
    def forward(ctx, v, vf, x, v0):
        ctx.save_for_backward(v, vf, x, v0)
        return _vmix_fwd(v, vf, x, v0)

    @staticmethod
    def backward(ctx, g):
        v, vf, x, v0 = ctx.saved_tensors
        lib = _lib.load()
        io = v.dtype
        C = v.shape[-1]
        g = _dev(g, io)
        dv, dvf, dx = (torch.empty_like(v) for _ in range(3))
        dv0 = torch.empty(C, dtype=torch.float32, device=v.device)
        rc = lib.hiprwkv_rwkv7_vmix_bwd(_stream(), _DT[io], v.numel() // C, C, _p(v), _p(vf), _p(x), _p(v0), _p(g),
                                        _p(dv), _p(dvf), _p(dx), _p(dv0))
        _lib.check(rc, "hiprwkv_rwkv7_vmix_bwd")
        return dv, dvf, dx, dv0.to(io)


def rwkv7_vmix(v, v_first, x, v0):
    """The value residual of the layers after the first, rwkv7.py:241-242: ``v + (v_first - v) sigmoid(v0 + x)`` for
    v, v_first, x (..., C) (x the low-rank term ``(xv v1) v2``) and the parameter v0 (C,).  Differentiable in all four."""
    io = v.dtype
    C = v.shape[-1]
    assert C % 8 == 0, C
    v, vf, x = (_dev(t, io) for t in (v, v_first, x))
    v02 = _dev(v0.reshape(C), io)
    if torch.is_grad_enabled() and any(t.requires_grad for t in (v, v_first, x, v0)):
        return _VMix.apply(v, vf, x, v02)
    return _vmix_fwd(v, vf, x, v02)


def rwkv7_premix(k, a, k_k, k_a):
    """k, a (..., H, N); k_k, k_a (H, N) or (H*N,).  Returns (k', a_i, b_i) of rwkv7.py:248-252, 257:
    kk = normalize_head(k k_k), k' = k (1 + (a - 1) k_a), a_i = -kk, b_i = kk a.  Differentiable in all four inputs
    (the backward kernel recomputes kk; parameter cotangents are summed over the tokens in fp32)."""
    io = k.dtype
    H, N = k.shape[-2:]
    k, a = _dev(k, io), _dev(a, io)
    k_k2, k_a2 = _dev(k_k.reshape(H, N), io), _dev(k_a.reshape(H, N), io)
    if torch.is_grad_enabled() and any(t.requires_grad for t in (k, a, k_k, k_a)):
        return _Premix.apply(k, a, k_k2, k_a2)
    return _premix_fwd(k, a, k_k2, k_a2)


def rwkv7_postmix(y, r, k, v, g, ln_w, ln_b, r_k, eps=64e-5):
    """y, r, k, v, g (..., H, N); ln_w, ln_b, r_k (H, N) or (H*N,).  Returns
    (group_norm_head(y) ln_w + ln_b + (r.k.r_k) v) g of rwkv7.py:263-265.  Differentiable in all eight tensors."""
    io = y.dtype
    H, N = y.shape[-2:]
    y, r, k, v, g = (_dev(x, io) for x in (y, r, k, v, g))
    ln_w2, ln_b2, r_k2 = (_dev(x.reshape(H, N), io) for x in (ln_w, ln_b, r_k))
    if torch.is_grad_enabled() and any(t.requires_grad for t in (y, r, k, v, g, ln_w, ln_b, r_k)):
        return _Postmix.apply(y, r, k, v, g, ln_w2, ln_b2, r_k2, eps)
    return _postmix_fwd(y, r, k, v, g, ln_w2, ln_b2, r_k2, eps)


# ----------------------------------------------------------------------------- RWKV-7 sub-block head and op inputs
LN_SHIFTMIX_MAX_C = 4096      # channels that one workgroup of the fused kernels spans


def _ln_shiftmix_fwd(x, dx, ln_w, ln_b, eps, prev, prev_stride, ns, length, mix, shift_out, stats):
    """``shift_out``: a (B,C) view with contiguous rows that receives the new shift row, or None."""
    lib = _lib.load()
    B, T, C = x.shape
    n_out = len(mix)
    outs = [torch.empty_like(x) for _ in range(max(n_out, 1))]
    xs = x if dx is None else torch.empty_like(x)
    rc = lib.hiprwkv_rwkv7_ln_shiftmix(_stream(), _DT[x.dtype], B, T, C, n_out, _p(x), _p(dx), _p(ln_w), _p(ln_b), eps,
                                       _p(prev), prev_stride, _p(ns), _p(length), _ptr_array(mix), _ptr_array(outs),
                                       _p(xs), _p(shift_out), C if shift_out is None else shift_out.stride(0), _p(stats))
    _lib.check(rc, "hiprwkv_rwkv7_ln_shiftmix")
    return xs, outs


class _LnShiftMix(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x, dx, ln_w, ln_b, prev, ns, length, eps, *mix):
        B, T, C = x.shape
        prev_t, stride = (None, C) if prev is None else _shift_row(prev, B, C, x.dtype)
        stats = torch.empty((B * T, 2), dtype=torch.float32, device=x.device)
        shift = None if prev is None else torch.empty((B, C), dtype=x.dtype, device=x.device)
        xs, outs = _ln_shiftmix_fwd(x, dx, ln_w, ln_b, eps, prev_t, stride, ns, length, mix, shift, stats)
        ctx.save_for_backward(xs, stats, ln_w, ln_b, prev_t, ns, length, *mix)
        ctx.has_dx, ctx.need_prev = dx is not None, prev is not None and ctx.needs_input_grad[4]
        ctx.set_materialize_grads(False)
        return (xs.view_as(xs) if dx is None else xs, shift) + tuple(outs)

    @staticmethod
    def backward(ctx, gx, gshift, *gs):
        xs, stats, ln_w, ln_b, prev, ns, length, *mix = ctx.saved_tensors
        lib = _lib.load()
        io = xs.dtype
        B, T, C = xs.shape
        n_out = len(mix)
        prev, stride = (None, C) if prev is None else _shift_row(prev, B, C, io)      # a saved-tensor hook may have moved it
        gs = [torch.zeros_like(xs) if g is None else _aligned(_dev(g, io)) for g in gs]
        gx, gshift = (None if g is None else _aligned(_dev(g, io)) for g in (gx, gshift))
        dxs = torch.empty_like(xs)
        dprev = torch.empty((B, C), dtype=io, device=xs.device) if ctx.need_prev else None
        dparam = torch.empty((n_out + 2, C), dtype=io, device=xs.device).unbind(0)
        nbytes = lib.hiprwkv_rwkv7_ln_shiftmix_bwd_workspace_bytes(B, T, C, n_out)
        ws = torch.empty(nbytes, dtype=torch.uint8, device=xs.device)
        rc = lib.hiprwkv_rwkv7_ln_shiftmix_bwd(_stream(), _DT[io], B, T, C, n_out, _p(xs), _p(stats), _p(ln_w), _p(ln_b),
                                               _p(prev), stride, _p(ns), _p(length), _ptr_array(mix), _ptr_array(gs),
                                               _p(gx), _p(gshift), _p(dxs), _p(dprev), _ptr_array(dparam), _p(ws), nbytes)
        _lib.check(rc, "hiprwkv_rwkv7_ln_shiftmix_bwd")
        return (dxs, dxs if ctx.has_dx else None, dparam[-2], dparam[-1], dprev, None, None, None) + tuple(dparam[:-2])


def rwkv7_ln_shiftmix(x, dx, ln, prev, new_starts, length, mix, eps=1e-5, shift_out=None):
    """The head of a sub-block in one pass: ``xs = x + dx`` (``dx`` may be None), ``xn = layer_norm(xs)`` with
    ``ln = {"weight", "bias"}``, then token shift and interpolation of ``xn`` as in ``rwkv7_shiftmix``.  Returns
    (xs, new shift row (B,C), the tuple of interpolations); the new shift row is ``xn`` of token ``(length - 1) mod T``.
    With an empty ``mix`` (``prev`` None) the one output is ``xn`` itself and there is no shift row.  ``shift_out``: write
    the shift row there (a (B,C) view with contiguous rows, no autograd).  ``length`` (B,) int32 or None; C at most
    ``LN_SHIFTMIX_MAX_C``.  Differentiable in x, dx, prev, the norm's and the mix parameters."""
    io = x.dtype
    B, T, C = x.shape
    assert len(mix) in (0, 1, 6) and C % 8 == 0 and C <= LN_SHIFTMIX_MAX_C, (len(mix), C)
    assert dx is None or dx.shape == x.shape, (dx.shape, x.shape)
    x = _dev(x, io)
    dx = None if dx is None else _dev(dx, io)
    ln_w, ln_b = (_aligned(_dev(ln[n].reshape(C), io)) for n in ("weight", "bias"))
    mix2 = [_dev(m.reshape(C), io) for m in mix]
    grad = _needs_grad(x, dx, ln_w, ln_b, prev, *mix2)
    length, new_starts = _length_ns(length, new_starts, B, T, x.device, keep=grad)
    if grad:
        if shift_out is not None:
            raise ValueError("rwkv7_ln_shiftmix: shift_out is for calls without autograd")
        xs, shift, *outs = _LnShiftMix.apply(x, dx, ln_w, ln_b, prev, new_starts, length, eps, *mix2)
        return xs, shift, outs
    _one_dtype(io, shift_out)
    prev_t, stride = (None, C) if prev is None else _shift_row(prev, B, C, io)
    if shift_out is None and prev is not None:
        shift_out = torch.empty((B, C), dtype=io, device=x.device)
    xs, outs = _ln_shiftmix_fwd(x, dx, ln_w, ln_b, eps, prev_t, stride, new_starts, length, mix2, shift_out, None)
    return xs, shift_out, outs


def _pre_fwd(xw, k, xa, v, vf, xv, w0, a0, v0, k_k, k_a):
    lib = _lib.load()
    H, N = k.shape[-2:]
    w, k_out, a_out, b_out = (torch.empty_like(k) for _ in range(4))
    v_out = None if vf is None else torch.empty_like(k)
    rc = lib.hiprwkv_rwkv7_pre(_stream(), _DT[k.dtype], k.numel() // (H * N), H, N, _p(xw), _p(k), _p(xa), _p(v), _p(vf),
                               _p(xv), _p(w0), _p(a0), _p(v0), _p(k_k), _p(k_a), _p(w), _p(k_out), _p(v_out), _p(a_out),
                               _p(b_out))
    _lib.check(rc, "hiprwkv_rwkv7_pre")
    return w, k_out, v_out, a_out, b_out


class _Pre(torch.autograd.Function):
    @staticmethod
    def forward(ctx, xw, k, xa, v, vf, xv, w0, a0, v0, k_k, k_a):
        ctx.save_for_backward(xw, k, xa, v, vf, xv, w0, a0, v0, k_k, k_a)
        return _pre_fwd(xw, k, xa, v, vf, xv, w0, a0, v0, k_k, k_a)

    @staticmethod
    def backward(ctx, gw, gk, gv, ga, gb):
        xw, k, xa, v, vf, xv, w0, a0, v0, k_k, k_a = ctx.saved_tensors
        lib = _lib.load()
        io = k.dtype
        H, N = k.shape[-2:]
        rows = k.numel() // (H * N)
        gw, gk, ga, gb = (_dev(g, io) for g in (gw, gk, ga, gb))
        dxw, dk, dxa = (torch.empty_like(k) for _ in range(3))
        dv = dvf = dxv = None
        if vf is not None:
            gv = _dev(gv, io)
            dv, dvf, dxv = (torch.empty_like(k) for _ in range(3))
        dparam = torch.empty((5, H * N), dtype=io, device=k.device).unbind(0)
        nbytes = lib.hiprwkv_rwkv7_pre_bwd_workspace_bytes(rows, H, N)
        ws = torch.empty(nbytes, dtype=torch.uint8, device=k.device)
        rc = lib.hiprwkv_rwkv7_pre_bwd(_stream(), _DT[io], rows, H, N, _p(xw), _p(k), _p(xa), _p(v), _p(vf), _p(xv), _p(w0),
                                       _p(a0), _p(v0), _p(k_k), _p(k_a), _p(gw), _p(gk), None if vf is None else _p(gv),
                                       _p(ga), _p(gb), None, None, None, None, None, _p(dxw), _p(dk), _p(dv), _p(dvf), _p(dxv), _p(dxa),
                                       _ptr_array(dparam), _p(ws), nbytes)
        _lib.check(rc, "hiprwkv_rwkv7_pre_bwd")
        dw0, da0, dk_k, dk_a, dv0 = dparam
        return dxw, dk, dxa, dv, dvf, dxv, dw0, da0, (None if vf is None else dv0), dk_k, dk_a


def rwkv7_pre(xw, k, xa, v, v_first, xv, w0, a0, v0, k_k, k_a):
    """``rwkv7_decay``, ``rwkv7_vmix``, ``rwkv7_agate`` and ``rwkv7_premix`` in one pass: xw, xa, xv the low-rank terms of
    decay, gate and value residual, k and v the projections, all (..., H, N); parameters (C,).  Returns (w, k', v', a_i,
    b_i), the WKV op's inputs.  The first layer has no value residual: ``v_first``, ``xv``, ``v0`` None, and v' is ``v``."""
    io = k.dtype
    C = k.shape[-2] * k.shape[-1]
    assert all(t is None or t.shape == k.shape for t in (xw, xa, v, v_first, xv)), [t if t is None else t.shape for t in (xw, k, xa, v, v_first, xv)]
    xw, k, xa, v = (_dev(t, io) for t in (xw, k, xa, v))
    w0, a0, k_k, k_a = (_dev(t.reshape(C), io) for t in (w0, a0, k_k, k_a))
    if v_first is None:
        args = (xw, k, xa, None, None, None, w0, a0, None, k_k, k_a)
    else:
        args = (xw, k, xa, v, _dev(v_first, io), _dev(xv, io), w0, a0, _dev(v0.reshape(C), io), k_k, k_a)
    w, k_out, v_out, a_out, b_out = _Pre.apply(*args) if _needs_grad(*args) else _pre_fwd(*args)
    return w, k_out, (v if v_first is None else v_out), a_out, b_out


# ----------------------------------------------------------------------------- RWKV-7 decode step
DECODE_MAX_ROWS = 256         # HIPRWKV_DECODE_MAX_ROWS
DECODE_HEAD_ROWS = 64         # up to here the head's product is a stream of its weights; beyond, the library's is faster


def _decode_tensors(params, C, F, vocab):
    """(argument name, tensor, shape after the layer axis) of every parameter of a decode step."""
    att, ffn = params["blocks"]["att"], params["blocks"]["ffn"]
    ln1, ln2 = params["blocks"]["ln1"], params["blocks"]["ln2"]
    vec = [(n, att[n]) for n in ("x_r", "x_w", "x_k", "x_v", "x_a", "x_g", "w0", "a0", "v0", "k_k", "k_a")]
    vec += [("ln1_w", ln1["weight"]), ("ln1_b", ln1["bias"]), ("ln2_w", ln2["weight"]), ("ln2_b", ln2["bias"]),
            ("lnx_w", att["ln_x"]["weight"]), ("lnx_b", att["ln_x"]["bias"]), ("ffn_x_k", ffn["x_k"])]
    out = [(n, t, (C,)) for n, t in vec]
    out += [(n, att[n]["weight"], (C, C)) for n in ("receptance", "key", "value", "output")]
    for n, d in (("w", "d_decay"), ("a", "d_aaa"), ("v", "d_mv"), ("g", "d_gate")):
        t1, t2 = att[n + "1"], att[n + "2"]
        out += [(n + "1", t1, (C, t1.shape[-1])), (n + "2", t2, (t1.shape[-1], C))]
    out += [("r_k", att["r_k"], (C // 64, 64)), ("ffn_key", ffn["key"]["weight"], (F, C)),
            ("ffn_value", ffn["value"]["weight"], (C, F))]
    return out


def rwkv7_decode(params, x, state, length, new_starts, compat=True):
    """A decode step of the whole RWKV-7 model from native code: x (B,T,C) the embedded tokens, state (B,L,2+64,C), length
    (B,) int32 or None, new_starts (B,T) bool or None.  Returns (logits, new state), or None where the step's kernels do
    not cover the call: they take bf16, contiguous stacked parameters, at most ``DECODE_MAX_ROWS`` tokens of which at most
    8 per sequence, and inner sizes that are multiples of 32.  No autograd."""
    B, T, C = x.shape
    bf = torch.bfloat16
    L, H, N = params["blocks"]["att"]["r_k"].shape
    head = params["head"]["weight"]
    F, vocab = params["blocks"]["ffn"]["key"]["weight"].shape[-2], head.shape[0]
    att = params["blocks"]["att"]
    dims = [att[n].shape[-1] for n in ("w1", "a1", "v1", "g1")]
    if (T > 8 or B * T > DECODE_MAX_ROWS or N != 64 or C != H * N or C > LN_SHIFTMIX_MAX_C or vocab % 16
            or any(d % 32 for d in (F, *dims)) or not x.is_cuda or x.dtype != bf
            or state.shape != (B, L, 2 + N, C) or state.dtype != bf or state.device != x.device or not state.is_contiguous()
            or state.data_ptr() % 16):
        return None
    A = _lib.Rwkv7DecodeArgs(B=B, T=T, L=L, C=C, H=H, F=F, vocab=vocab, d_decay=dims[0], d_aaa=dims[1], d_mv=dims[2],
                             d_gate=dims[3])
    tensors = [(n, t, (L,) + s) for n, t, s in _decode_tensors(params, C, F, vocab)]
    tensors += [(n + k, params[n]["weight" if k == "_w" else "bias"], (C,)) for n in ("ln0", "ln_out") for k in ("_w", "_b")]
    for name, t, shape in tensors + [("head", head, (vocab, C))]:
        ptr = t.data_ptr()
        if t.dtype != bf or t.shape != shape or not t.is_contiguous() or ptr % 16 or t.device != x.device:
            return None
        setattr(A, name, ptr)
    lib = _lib.load()
    x = x.contiguous()
    new_state, xn = torch.empty_like(state), torch.empty_like(x)
    logits = torch.empty((B, T, vocab), dtype=bf, device=x.device) if B * T <= DECODE_HEAD_ROWS else None
    nbytes = lib.hiprwkv_rwkv7_decode_workspace_bytes(ctypes.byref(A))
    ws = torch.empty(nbytes, dtype=torch.uint8, device=x.device)
    A.x, A.state, A.new_state, A.length, A.new_starts = _p(x), _p(state), _p(new_state), _p(length), _p(new_starts)
    A.xn, A.logits, A.workspace, A.workspace_bytes = _p(xn), _p(logits), _p(ws), nbytes
    A.flags = _lib.COMPAT_ASSOC if compat else 0
    _lib.check(lib.hiprwkv_rwkv7_decode(_stream(), ctypes.byref(A)), "hiprwkv_rwkv7_decode")
    return (xn @ head.T if logits is None else logits), new_state
