"""The stack of RWKV-7 blocks as one operator over whole sequences, with and without autograd (rwkv7.py:190-198, 223-291).

Autograd over the single steps spends longer on the host than the GPU needs for a training step of a small model (0.1B shape,
B=4 T=512: about 1000 launches, 23 ms against 13 ms of GPU time).  Here the whole stack is one node: the backward is
written out over the library's kernels and ``torch.mm``, writes every layer's parameter cotangents into their place in the
stacked arrays, and adds up nothing that a kernel can add on its way (the second cotangents of r, k and v, the value
residual's).  The low-rank factors of decay, gates and value residual run several to a launch (``hiprwkv_gemm``) in bf16.
"""
import ctypes

import torch
from torch.autograd.function import once_differentiable

from . import _lib, ops
from .rwkv7 import HipRWKV

#: parameter name -> path inside params["blocks"]; the order of the operator's arguments
PATHS = {n: ("att", n) for n in ("x_r", "x_w", "x_k", "x_v", "x_a", "x_g", "w0", "w1", "w2", "a0", "a1", "a2", "v0", "v1", "v2",
                                 "g1", "g2", "k_k", "k_a", "r_k")}
PATHS.update({n: ("att", n, "weight") for n in ("receptance", "key", "value", "output")})
PATHS.update(lnx_w=("att", "ln_x", "weight"), lnx_b=("att", "ln_x", "bias"), ffn_x_k=("ffn", "x_k"),
             ffn_key=("ffn", "key", "weight"), ffn_value=("ffn", "value", "weight"), ln1_w=("ln1", "weight"),
             ln1_b=("ln1", "bias"), ln2_w=("ln2", "weight"), ln2_b=("ln2", "bias"))
NAMES = tuple(PATHS)
MIX = ("x_r", "x_w", "x_k", "x_v", "x_a", "x_g")
EPS_X = 64e-5
_NONE, _TANH, _SIGMOID = 0, 1, 2             # hiprwkv_gemm_job.act without aux; with aux: add, tanh', sigmoid'
_LORA = (("w", _TANH), ("a", _NONE), ("g", _SIGMOID), ("v", _NONE))


def gather(blocks):
    out = []
    for path in PATHS.values():
        t = blocks
        for p in path:
            t = t[p]
        out.append(t)
    return out


def _gemm(jobs):
    """Several products in one launch: (out, x, w, km, kn, act, aux) with out (M, N), x (M, K) or, km, (K, M), w (N, K) or,
    kn, (K, N)."""
    arr = (_lib.GemmJob * len(jobs))()
    for j, (out, x, w, km, kn, act, aux) in zip(arr, jobs):
        j.out, j.x, j.w, j.aux = out.data_ptr(), x.data_ptr(), w.data_ptr(), None if aux is None else aux.data_ptr()
        j.M, j.N = out.shape
        j.K = x.shape[0] if km else x.shape[1]
        j.km, j.kn, j.act = km, kn, act
    _lib.check(_lib.load().hiprwkv_gemm(ops._stream(), len(jobs), arr), "hiprwkv_gemm")


def _grouped(p, like):
    """Whether the grouped products take the low-rank factors beside a (M, C) array: bf16, inner sizes multiples of 8, no
    operand of 2 GiB."""
    return (like.dtype == torch.bfloat16 and like.numel() < 2 ** 30
            and all(p[n].shape[-1] % 8 == 0 and p[n].shape[-1] * max(like.shape) < 2 ** 30 for n in ("w1", "a1", "v1", "g1")))


def _lora_pre_fwd(p, mix, names, k, v, v_first, keep):
    """``_lora_fwd`` and ``ops._pre_fwd`` for the products that ``_grouped`` takes: the second factors are made where the gates are.
    k, v, v_first (None: the first layer) (M, C); without ``keep`` the gate's result alone is there of the low-rank terms."""
    lib = _lib.load()
    M, C = k.shape
    H, N = p["r_k"].shape
    e = lambda: torch.empty_like(k)
    hid = {n: torch.empty((M, p[n + "1"].shape[-1]), dtype=k.dtype, device=k.device) for n, _ in names}
    _gemm([(hid[n], mix[n], p[n + "1"], 0, 1, act, None) for n, act in names])
    lora = {n: e() if keep or n == "g" else None for n, _ in names}
    w, k2, v2, a, b = e(), e(), None if v_first is None else e(), e(), e()
    sizes = (ctypes.c_int64 * len(names))(*(h.shape[1] for h in hid.values()))
    P = ops._p
    _lib.check(lib.hiprwkv_rwkv7_lora_pre(
        ops._stream(), ops._DT[k.dtype], M, H, N, ops._ptr_array(list(hid.values())), ops._ptr_array([p[n + "2"] for n, _ in names]),
        sizes, P(k), P(v), P(v_first), P(p["w0"]), P(p["a0"]), None if v_first is None else P(p["v0"]), P(p["k_k"]), P(p["k_a"]),
        ops._ptr_array(list(lora.values())) if keep else None, P(lora["g"]), P(w), P(k2), P(v2), P(a), P(b)), "hiprwkv_rwkv7_lora_pre")
    return hid, lora, (w, k2, v2, a, b)


def _lora_fwd(p, mix, names):
    """Hidden values (activation applied) and results of the low-rank terms ``names``; mix: name -> (M, C) input."""
    hid, out = {}, {}
    for n, act in names:
        h = mix[n] @ p[n + "1"]
        hid[n] = torch.tanh_(h) if act == _TANH else torch.sigmoid_(h) if act == _SIGMOID else h
        out[n] = hid[n] @ p[n + "2"]
    return hid, out


def _weight_grad(grad, name, a, b):
    if name in grad:
        torch.mm(a.T, b, out=grad[name])


def _lora_bwd(p, grad, mix, hid, gout, dmix, names):
    """From the cotangents ``gout`` of the low-rank terms: the parameters' cotangents into ``grad`` (those it has) and the
    inputs' into ``dmix`` (the value residual's is added to what is there)."""
    if _grouped(p, gout["w"]):
        dh = {n: gout[n].new_empty((len(gout[n]), p[n + "1"].shape[-1])) if hid[n] is None else torch.empty_like(hid[n]) for n, _ in names}
        _gemm([(dh[n], gout[n], p[n + "2"], 0, 0, act, hid[n] if act else None) for n, act in names])
        _gemm([(dmix[n], dh[n], p[n + "1"], 0, 0, 0, dmix[n] if n == "v" else None) for n, _ in names])
        jobs = ([(grad[n + "1"], mix[n], dh[n], 1, 1, _NONE, None) for n, _ in names if n + "1" in grad]
                + [(grad[n + "2"], hid[n], gout[n], 1, 1, _NONE, None) for n, _ in names if n + "2" in grad])
        if jobs:
            _gemm(jobs)
        return
    for n, act in names:
        _weight_grad(grad, n + "2", hid[n], gout[n])
        dh = gout[n] @ p[n + "2"].T
        if act == _TANH:
            dh = torch.ops.aten.tanh_backward(dh, hid[n])
        elif act == _SIGMOID:
            dh = torch.ops.aten.sigmoid_backward(dh, hid[n])
        _weight_grad(grad, n + "1", mix[n], dh)
        if n == "v":
            dmix[n].addmm_(dh, p[n + "1"].T)
        else:
            torch.mm(dh, p[n + "1"].T, out=dmix[n])


def _ln_mix(p, x, dx, ln, state_row, ns, length, mix, shift_out, keep):
    """``rwkv7_ln_shiftmix`` on (B,T,C) without autograd; ``keep``: also the statistics for the backward."""
    B, T, C = x.shape
    stats = torch.empty((B * T, 2), dtype=torch.float32, device=x.device) if keep else None
    prev, stride = ops._shift_row(state_row, B, C, x.dtype)
    xs, outs = ops._ln_shiftmix_fwd(x, dx, p[ln + "_w"], p[ln + "_b"], 1e-5, prev, stride, ns, length,
                                    [p[n] for n in mix], shift_out, stats)
    return xs, outs, (stats, prev, stride)


def _layer_fwd(i, p, x, dx, st, nst, v_first, ns, length, need):
    """One block on x (B,T,C) (+ dx): returns (x, dx, v_first, saved tensors).  st, nst: the layer's rows of the model
    states.  need: None without a backward to come, else the names of the parameters whose cotangents it will make."""
    keep = need is not None
    B, T, C = x.shape
    H, N = p["r_k"].shape
    M = B * T
    flat = lambda t: t.view(M, -1)
    heads = lambda t: t.view(B, T, H, N)
    x, outs, head1 = _ln_mix(p, x, dx, "ln1", st[:, 1], ns, length, MIX, nst[:, 1], keep)
    xr, xw, xk, xv, xa, xg = map(flat, outs)
    r, k, v = (torch.mm(a, p[n].T) for a, n in ((xr, "receptance"), (xk, "key"), (xv, "value")))
    # `covers` has seen the call's own tensors; under an autocast that the caller overlooked products come out in another type
    ops._one_dtype(x.dtype, r)
    mix = {"w": xw, "a": xa, "g": xg, "v": xv}
    names = _LORA if i else _LORA[:3]
    par = lambda n: p[n].reshape(C)
    if _grouped(p, r):
        hid, lora, pre = _lora_pre_fwd(p, mix, names, k, v, v_first if i else None, keep)
    else:
        hid, lora = _lora_fwd(p, mix, names)
        pre = ops._pre_fwd(heads(lora["w"]), heads(k), heads(lora["a"]), heads(v), heads(v_first) if i else None,
                           heads(lora["v"]) if i else None, par("w0"), par("a0"), par("v0") if i else None, par("k_k"), par("k_a"))
    if i == 0:
        v_first = v
    w, k2, v2, a, b = (None if t is None else heads(t) for t in pre)
    if i == 0:
        v2 = heads(v)
    s = st[:, 2:].reshape(B, H, N, N)
    new_s, yw, sa, ends = ops._wkv7_fwd(heads(r), w, k2, v2, a, b, s, length, ns, HipRWKV.assoc_compat, want_sa=keep,
                                        want_ends=keep and x.dtype == torch.float32)
    nst[:, 2:] = new_s.view(B, N, C)
    y = flat(ops._postmix_fwd(yw, heads(r), k2, v2, heads(lora["g"]), par("lnx_w"), par("lnx_b"), par("r_k"), EPS_X))
    dx1 = torch.mm(y, p["output"].T).view(B, T, C)
    x2, (xk2,), head2 = _ln_mix(p, x, dx1, "ln2", st[:, 0], ns, length, ("ffn_x_k",), nst[:, 0], keep)
    ff = torch.mm(flat(xk2), p["ffn_key"].T)
    fr = ops._relusq_fwd(ff)
    dx2 = torch.mm(fr, p["ffn_value"].T).view(B, T, C)
    saved = None
    if keep:
        # an operand of a weight's cotangent alone is kept for that weight only
        only = (lambda t, *names: t) if len(need) == len(NAMES) else (lambda t, *names: t if need.intersection(names) else None)
        saved = dict(x=x, head1=head1, xr=only(xr, "receptance"), xk=only(xk, "key"),
                     mix={n: only(t, n + "1", *(("value",) if n == "v" else ())) for n, t in mix.items()},
                     r=r, k=k, v=v, hid={n: hid[n] if act else only(hid[n], n + "2") for n, act in _LORA if n in hid}, lora=lora,
                     w=w, k2=k2, v2=v2, a=a, b=b, s=s, sa=sa, ends=ends, yw=yw, y=only(y, "output"), x2=x2, head2=head2,
                     xk2=only(flat(xk2), "ffn_key"), ff=ff, fr=only(fr, "ffn_value"))
    return x2, dx2, v_first, saved


def _vectors(grad, names, scratch):
    """The places for the cotangents of parameters that a kernel makes together: ``scratch`` for those nobody asked for."""
    return ops._ptr_array([grad.get(n, scratch) for n in names])


def _ln_mix_bwd(p, grad, scratch, xs, head, ln, ns, length, mix, gs, gx, gshift, need_prev):
    lib = _lib.load()
    stats, prev, stride = head
    io = xs.dtype
    B, T, C = xs.shape
    if prev.stride(1) != 1 or (B > 1 and prev.stride(0) != stride):
        prev, stride = ops._shift_row(prev, B, C, io)         # a saved-tensor hook has moved it
    dxs = torch.empty_like(xs)
    dprev = torch.empty((B, C), dtype=io, device=xs.device) if need_prev else None
    params = [p[n] for n in mix]
    nbytes = lib.hiprwkv_rwkv7_ln_shiftmix_bwd_workspace_bytes(B, T, C, len(mix))
    ws = ops._workspace(nbytes, xs.device)
    rc = lib.hiprwkv_rwkv7_ln_shiftmix_bwd(
        ops._stream(), ops._DT[io], B, T, C, len(mix), ops._p(xs), ops._p(stats), ops._p(p[ln + "_w"]), ops._p(p[ln + "_b"]),
        ops._p(prev), stride, ops._p(ns), ops._p(length), ops._ptr_array(params), ops._ptr_array(gs), ops._p(gx), ops._p(gshift),
        ops._p(dxs), ops._p(dprev), _vectors(grad, (*mix, ln + "_w", ln + "_b"), scratch), ops._p(ws), nbytes)
    _lib.check(rc, "hiprwkv_rwkv7_ln_shiftmix_bwd")
    return dxs, dprev


def _layer_bwd(i, p, grad, scratch, S, ns, length, g_x, g_dx, g_state, g_in, g_vfirst, v_first):
    """The cotangents of one block: g_x, g_dx of what it returns, g_state (or None) of its rows of the new model state (B,66,C).
    Fills ``grad`` (the layer's slices of the stacked cotangents, of those asked for; scratch: C elements) and ``g_in`` (or None), the cotangent of its rows of the input
    state; accumulates ``g_vfirst``.  Returns the cotangent of its input x (and of the dx added to it) and g_vfirst."""
    lib = _lib.load()
    x, x2 = S["x"], S["x2"]
    B, T, C = x.shape
    H, N = p["r_k"].shape
    M = B * T
    io = x.dtype
    flat = lambda t: t.view(M, -1)
    heads = lambda t: t.view(B, T, H, N)
    row = lambda j: None if g_state is None else g_state[:, j].contiguous()
    # channel mixing
    g2 = flat(g_dx)
    _weight_grad(grad, "ffn_value", g2, S["fr"])
    gf = torch.mm(g2, p["ffn_value"])
    gff = torch.empty_like(gf)
    _lib.check(lib.hiprwkv_rwkv7_relusq_bwd(ops._stream(), ops._DT[io], gf.numel(), ops._p(S["ff"]), ops._p(gf), ops._p(gff)),
               "hiprwkv_rwkv7_relusq_bwd")
    _weight_grad(grad, "ffn_key", gff, S["xk2"])
    gxk2 = torch.mm(gff, p["ffn_key"]).view(B, T, C)
    dx2, dprev = _ln_mix_bwd(p, grad, scratch, x2, S["head2"], "ln2", ns, length, ("ffn_x_k",), [gxk2], g_x, row(0), g_in is not None)
    if g_in is not None:
        g_in[:, 0] = dprev
    # time mixing: output projection, group norm and gate
    g1 = flat(dx2)
    _weight_grad(grad, "output", g1, S["y"])
    gy = torch.mm(g1, p["output"])
    e = lambda: torch.empty((B, T, H, N), dtype=io, device=x.device)
    gyw, gr1, gk1, gv1, gg = (e() for _ in range(5))
    nbytes = lib.hiprwkv_rwkv7_postmix_bwd2_workspace_bytes(M, H, N)
    ws = ops._workspace(nbytes, x.device)
    rc = lib.hiprwkv_rwkv7_postmix_bwd2(
        ops._stream(), ops._DT[io], M, H, N, ops._p(S["yw"]), ops._p(S["r"]), ops._p(S["k2"]), ops._p(S["v2"]),
        ops._p(S["lora"]["g"]), ops._p(p["lnx_w"]), ops._p(p["lnx_b"]), ops._p(p["r_k"]), EPS_X, ops._p(gy), ops._p(gyw),
        ops._p(gr1), ops._p(gk1), ops._p(gv1), ops._p(gg),
        _vectors(grad, ("lnx_w", "lnx_b", "r_k"), scratch), ops._p(ws), nbytes)
    _lib.check(rc, "hiprwkv_rwkv7_postmix_bwd2")
    # the recurrence
    gs_out = None if g_state is None else g_state[:, 2:].reshape(B, H, N, N)
    gr2, gw, gk2, gv2, ga, gb, gs = ops.wkv7_bwd(heads(S["r"]), S["w"], S["k2"], S["v2"], S["a"], S["b"], S["s"], length, ns,
                                                 gyw, S["sa"], gs_out, HipRWKV.assoc_compat, ends=S["ends"], parts=True)
    if g_in is not None:
        g_in[:, 2:] = gs.reshape(B, N, C)
    # gates
    par = lambda n: p[n].reshape(C)
    lora, dxw, dk, dxa, gr = S["lora"], e(), e(), e(), e()
    names = _LORA if i else _LORA[:3]
    if i:
        dv, dvf, dxv = e(), e(), e()
    else:
        dv, dvf, dxv = gv1.add_(gv2), None, None
        if g_vfirst is not None:
            dv.add_(g_vfirst)
    nbytes = lib.hiprwkv_rwkv7_pre_bwd_workspace_bytes(M, H, N)
    ws = ops._workspace(nbytes, x.device)
    P = ops._p
    rc = lib.hiprwkv_rwkv7_pre_bwd(
        ops._stream(), ops._DT[io], M, H, N, P(lora["w"]), P(S["k"]), P(lora["a"]), P(S["v"]), P(v_first) if i else None,
        P(lora["v"]) if i else None, P(par("w0")), P(par("a0")), P(par("v0")) if i else None, P(par("k_k")), P(par("k_a")),
        P(gw), P(gk1), P(gv1) if i else None, P(ga), P(gb), P(gk2), P(gv2) if i else None, P(gr1), P(gr2), P(gr),
        P(dxw), P(dk), P(dv) if i else None, P(dvf), P(dxv), P(dxa),
        _vectors(grad, ("w0", "a0", "k_k", "k_a", "v0"), scratch), P(ws), nbytes)
    _lib.check(rc, "hiprwkv_rwkv7_pre_bwd")
    if i:
        g_vfirst = dvf if g_vfirst is None else g_vfirst.add_(dvf)
    # projections
    gr, dk, dv = flat(gr), flat(dk), flat(dv)
    mix = S["mix"]
    for g, a, n in ((gr, S["xr"], "receptance"), (dk, S["xk"], "key"), (dv, mix["v"], "value")):
        _weight_grad(grad, n, g, a)
    dxr, dxk, dxv_ = torch.mm(gr, p["receptance"]), torch.mm(dk, p["key"]), torch.mm(dv, p["value"])
    dmix = {n: torch.empty_like(dxr) for n in ("w", "a", "g")}
    dmix["v"] = dxv_
    gout = {"w": flat(dxw), "a": flat(dxa), "g": flat(gg)}
    if i:
        gout["v"] = flat(dxv)
    _lora_bwd(p, grad, mix, S["hid"], gout, dmix, names)
    gmix = [t.view(B, T, C) for t in (dxr, dmix["w"], dxk, dxv_, dmix["a"], dmix["g"])]
    dx, dprev = _ln_mix_bwd(p, grad, scratch, x, S["head1"], "ln1", ns, length, MIX, gmix, dx2, row(1), g_in is not None)
    if g_in is not None:
        g_in[:, 1] = dprev
    return dx, g_vfirst


def _pack(tree, tensors):
    """``tree`` with its tensors moved to the list ``tensors`` and their places left in it."""
    if torch.is_tensor(tree):
        tensors.append(tree)
        return len(tensors) - 1, None
    if isinstance(tree, dict):
        return {k: _pack(v, tensors) for k, v in tree.items()}
    if isinstance(tree, (list, tuple)):
        return [_pack(v, tensors) for v in tree]
    return None, tree


def _unpack(tree, tensors):
    if isinstance(tree, dict):
        return {k: _unpack(v, tensors) for k, v in tree.items()}
    if isinstance(tree, list):
        return [_unpack(v, tensors) for v in tree]
    return tree[1] if tree[0] is None else tensors[tree[0]]


class _Blocks(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x, state, ns, length, *params):
        ctx.set_materialize_grads(False)
        need = {n for n, asked in zip(NAMES, ctx.needs_input_grad[4:]) if asked}
        x, dx, new_state, saved, v_first = _run(x, state, ns, length, params, need)
        tensors = []
        ctx.places = _pack([saved, v_first, ns, length], tensors)
        ctx.n = len(tensors)
        ctx.save_for_backward(*tensors, state, *params)
        return x, dx, new_state

    @staticmethod
    @once_differentiable              # create_graph=True: first cotangents as ever, an error for those of the cotangents
    def backward(ctx, g_x, g_dx, g_state):
        tensors = ctx.saved_tensors
        saved, v_first, ns, length = _unpack(ctx.places, tensors)
        state, *params = tensors[ctx.n:]
        L = params[0].shape[0]
        like = saved[-1]["x2"]
        io = like.dtype
        g_x = torch.zeros_like(like) if g_x is None else ops._dev(g_x, io)
        g_dx = torch.zeros_like(like) if g_dx is None else ops._dev(g_dx, io)
        g_state = None if g_state is None else ops._aligned(g_state.to(io))
        residual = ("v0", "v1", "v2")           # the first layer has no value residual
        grads = {n: torch.empty_like(t) for n, t, asked in zip(NAMES, params, ctx.needs_input_grad[4:])
                 if asked and (L > 1 or n not in residual)}
        for n in residual:
            if n in grads:
                grads[n][0].zero_()
        scratch = torch.empty(like.shape[-1], dtype=io, device=like.device)
        g_in = torch.empty_like(state) if ctx.needs_input_grad[1] else None
        g_vfirst = None
        layers = list(zip(*(t.unbind(0) for t in params)))
        glayers = list(zip(*(t.unbind(0) for t in grads.values()))) or [()] * L
        # products in the operands' own dtype even where the caller's backward runs under autocast
        with torch.autocast(like.device.type, enabled=False):
            for i in reversed(range(L)):
                dx, g_vfirst = _layer_bwd(i, dict(zip(NAMES, layers[i])), dict(zip(grads, glayers[i])), scratch, saved[i],
                                          ns, length, g_x, g_dx, None if g_state is None else g_state[:, i],
                                          None if g_in is None else g_in[:, i], g_vfirst, v_first)
                g_x = g_dx = dx
        return (g_x, g_in, None, None) + tuple(grads.get(n) for n in NAMES)


def _run(x, state, ns, length, params, need):
    L = params[0].shape[0]
    layers = list(zip(*(t.unbind(0) for t in params)))
    new_state = torch.empty_like(state, memory_format=torch.contiguous_format)      # the kernels write rows of neighbours
    dx = v_first = None
    saved = []
    for i in range(L):
        x, dx, v_first, S = _layer_fwd(i, dict(zip(NAMES, layers[i])), x, dx, state[:, i], new_state[:, i], v_first, ns,
                                       length, need)
        saved.append(S)
    if not state.is_contiguous():
        new_state = torch.empty_like(state).copy_(new_state)                          # in the order of the caller's
    return x, dx, new_state, saved, v_first


_FACTORS = ("w1", "w2", "a1", "a2", "v1", "v2", "g1", "g2")
_PRODUCTS = ("receptance", "key", "value", "output", "ffn_key", "ffn_value")       # torch looks at these itself


def covers(params, x, state):
    """Whether the operator takes the call: one dtype and device throughout, stacked parameters of the sizes that the kernels
    read, contiguous and on 16-byte boundaries."""
    io, dev, C = x.dtype, x.device, x.shape[-1]
    L = params[0].shape[0]
    n = L * C
    if not (io in ops._DT and x.is_cuda and state.dtype == io and state.device == dev and C <= ops.LN_SHIFTMIX_MAX_C):
        return False
    for name, t in zip(NAMES, params):
        if t.dtype != io or t.device != dev or t.shape[0] != L or not t.is_contiguous() or t.data_ptr() % 16:
            return False
        if name not in _PRODUCTS and name not in _FACTORS and t.numel() != n:
            return False
    p = dict(zip(NAMES, params))
    return all(p[f + "1"].shape[-2] == C and p[f + "2"].shape[-2:] == (p[f + "1"].shape[-1], C)
               and p[f + "1"].numel() == p[f + "2"].numel() == n * p[f + "1"].shape[-1] for f in "wavg")


#: rows x channels^2 up to which the stack is launched from native code: up to 1536 channels, and beyond.  A layer costs the host 0.3 ms
#: forward (and 0.8 backward) from Python; from some size on the library's large products, which the separate steps use, are worth it.
#: Of wide models they are better by more than the host's time, but for sizes that fill the native products' rounds.  Native / steps in ms:
#: forward of 24 layers of 2048 channels 1000 rows 5.8 / 7.7, 1100 7.3 / 8.0, 1200 8.2 / 8.2, 1400 8.6 / 8.2, 1600 9.1 / 9.3, 2000 9.7 / 10.1,
#: 2200 12.0 / 11.6, 2500 12.6 / 11.8, 4000 17.0 / 15.9; 6 of 4096, 300 rows 2.24 / 2.41, 600 3.5 / 3.2; 8 of 1536, 2500 rows 3.36 / 3.38, 4000
#: 4.5 / 4.6; 24 of 1024, 5000 rows 9.4 / 9.5, 8000 12.5 / 13.1; training steps of 4 of 2048, 1200 rows 5.2 / 5.7, 1600 6.18 / 6.19, 2400
#: 8.7 / 8.4; 4 of 1536, 3000 rows 7.5 / 8.0, 4000 9.56 / 9.56; 8 of 1024, 8000 rows 16.9 / 17.4.  NATIVE_ROWS bounds the workspace.
NATIVE_ROWS_C2, NATIVE_ROWS_C2_WIDE, NATIVE_ROWS = 9 * 10 ** 9, 5 * 10 ** 9, 8192


def _native(params, x, state, grad):
    """Whether native code launches the stack (``hiprwkv_rwkv7_stack_args``): bf16, all parameters or none trained and not the state,
    the shapes that the model has (the separate steps take any that multiply), channels in whole 128-column tiles."""
    B, T, C = x.shape
    M = B * T
    p = dict(zip(NAMES, params))
    L, H, N = p["r_k"].shape
    F = p["ffn_key"].shape[1]
    sizes = (F, *(p[f + "1"].shape[-1] for f in "wavg"))
    shapes = {"ffn_key": (L, F, C), "ffn_value": (L, C, F)}
    most = NATIVE_ROWS_C2 if C <= 1536 else NATIVE_ROWS_C2_WIDE
    return (x.dtype == torch.bfloat16 and M * C * C <= most and M <= NATIVE_ROWS and T > 8 and N == 64 and C == H * N
            and C % 128 == 0 and F <= 8 * C and all(d % 8 == 0 and max(d, C) * max(M, C, 256) < 2 ** 30 for d in sizes)
            and state.shape == (B, L, 2 + N, C) and state.is_contiguous() and state.data_ptr() % 16 == 0 and not ops.autocast_elsewhere(x)
            and all(p[n].shape == shapes.get(n, (L, C, C)) for n in _PRODUCTS)
            and not (grad and (state.requires_grad or not all(t.requires_grad for t in params))))


def _stack_args(x, state, s, ns, length, params, xs):
    """The arguments that both directions share."""
    p = dict(zip(NAMES, params))
    (L, H, _), (B, T, C) = p["r_k"].shape, x.shape
    A = _lib.Rwkv7StackArgs(B=B, T=T, L=L, C=C, H=H, F=p["ffn_key"].shape[1], d_decay=p["w1"].shape[-1], d_aaa=p["a1"].shape[-1],
                            d_mv=p["v1"].shape[-1], d_gate=p["g1"].shape[-1])
    A.x, A.state, A.s, A.length, A.new_starts, A.xs = map(ops._p, (x, state, s, length, ns, xs))
    A.param[:] = [t.data_ptr() for t in params]
    return A


def _stack_fwd(x, state, ns, length, params, compat, keep):
    """Returns (xs, dx, new_state) and, with ``keep``, what the backward reads besides them and the arguments."""
    lib = _lib.load()
    x = ops._aligned(x.contiguous())
    s = state[:, :, 2:].transpose(0, 1).contiguous()
    xs, dx, new_s, new_state = torch.empty_like(x), torch.empty_like(x), torch.empty_like(s), torch.empty_like(state)
    A = _stack_args(x, state, s, ns, length, params, xs)
    A.dx, A.new_s, A.new_state, A.flags = dx.data_ptr(), new_s.data_ptr(), new_state.data_ptr(), _lib.COMPAT_ASSOC if compat else 0
    sizes = [lib.hiprwkv_rwkv7_stack_saved_layer_bytes(ctypes.byref(A), i) for i in (0, A.L // 2, A.L - 1)] if keep else ()
    saved = [ops._workspace(sizes[0 if i == 0 else 2 if i == A.L - 1 else 1], x.device) for i in range(A.L if keep else 0)]
    arr = ops._ptr_array(saved)
    A.saved = ctypes.addressof(arr) if keep else None
    A.workspace_bytes = lib.hiprwkv_rwkv7_stack_workspace_bytes(ctypes.byref(A), 0)
    ws = ops._workspace(A.workspace_bytes, x.device)
    A.workspace = ws.data_ptr()
    _lib.check(lib.hiprwkv_rwkv7_stack_fwd(ops._stream(), ctypes.byref(A)), "hiprwkv_rwkv7_stack_fwd")
    new_state[:, :, 2:].copy_(new_s.transpose(0, 1))
    return xs, dx, new_state, (x, xs, s, *saved)


class _Stack(torch.autograd.Function):
    """``_Blocks`` launched from native code."""

    @staticmethod
    def forward(ctx, x, state, ns, length, compat, *params):
        ctx.set_materialize_grads(False)
        xs, dx, new_state, saved = _stack_fwd(x, state, ns, length, params, compat, True)
        ctx.compat, ctx.n = compat, len(saved)
        ctx.save_for_backward(*saved, state, ns, length, *params)
        return xs, dx, new_state

    @staticmethod
    @once_differentiable
    def backward(ctx, g_x, g_dx, g_state):
        lib = _lib.load()
        tensors = ctx.saved_tensors
        x, xs, s, *saved = map(ops._aligned, tensors[:ctx.n])
        state, ns, length, *params = tensors[ctx.n:]
        state = ops._aligned(state.contiguous())                      # a saved-tensor hook may have moved it
        params = [ops._aligned(t.contiguous()) for t in params]
        A = _stack_args(x, state, s, ns, length, params, xs)
        g_x, g_dx = (torch.zeros_like(x) if g is None else ops._aligned(ops._dev(g, x.dtype)) for g in (g_x, g_dx))
        if g_state is not None:
            g_state = g_state.to(x.dtype).transpose(0, 1)
            g_shift, g_s = g_state[:, :, :2].permute(2, 0, 1, 3).contiguous(), g_state[:, :, 2:].contiguous()
            A.g_shift, A.g_s = g_shift.data_ptr(), g_s.data_ptr()
        residual = ("v0", "v1", "v2")                                 # the first layer has no value residual
        grads = [None if A.L == 1 and n in residual else torch.empty_like(t) for n, t in zip(NAMES, params)]
        for n, g in zip(NAMES, grads):
            if g is not None and n in residual:
                g[0].zero_()
        A.grad[:] = [ops._p(g) for g in grads]
        out = torch.empty_like(x)
        A.g_xs, A.g_dx, A.g_x, A.flags = g_x.data_ptr(), g_dx.data_ptr(), out.data_ptr(), _lib.COMPAT_ASSOC if ctx.compat else 0
        arr = ops._ptr_array(saved)
        A.saved = ctypes.addressof(arr)
        A.workspace_bytes = lib.hiprwkv_rwkv7_stack_workspace_bytes(ctypes.byref(A), 1)
        ws = ops._workspace(A.workspace_bytes, x.device)
        A.workspace = ws.data_ptr()
        _lib.check(lib.hiprwkv_rwkv7_stack_bwd(ops._stream(), ctypes.byref(A)), "hiprwkv_rwkv7_stack_bwd")
        return (out if ctx.needs_input_grad[0] else None, None, None, None, None, *grads)


def run(params, x, state, ns, length, grad):
    """The stack on x (B,T,C) and state (B,L,2+N,C): returns (x, dx, new_state) whose sum x + dx is the residual stream."""
    if grad:
        length = None if length is None else length.clone()          # the caller may change its own before the backward
    if _native(params, x, state, grad):
        if grad:
            return _Stack.apply(x, state, ns, length, HipRWKV.assoc_compat, *params)
        return _stack_fwd(x, state, ns, length, params, HipRWKV.assoc_compat, False)[:3]
    if grad:
        return _Blocks.apply(x, state, ns, length, *params)
    return _run(x, state, ns, length, params, None)[:3]
