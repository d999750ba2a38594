"""RWKV-7 full-model harness around ``HipRWKV.inner_loop``: the caller of the WKV op, restated over torch tensors.

It mirrors the reference's ``RWKV.forward(params, tokens, state, length=, new_starts=)`` and ``default_state``
(/root/reference/src/jaxrwkv/llm.py:71-84, rwkv7.py:176-198, 223-291) with an explicit leading batch axis (the
reference batches with ``jax.vmap``).  Projections are torch's; the element-wise work between them (residual addition and
LayerNorm, token shift, gates, group norm) runs on fused kernels of this library, and the recurrence goes through
``HipRWKV.inner_loop``.  The parameter tree has the reference's names and stacked-per-layer shapes
(rwkv7.py:81-173) so that a converted checkpoint would drop in; ``randomize_weights`` follows the same schedules and
distributions with torch's generator (the reference's threefry streams cannot be reproduced without jax).

Model state per sequence, as in the reference (rwkv7.py:176-180, 254-260, 283-287): ``(L, 2 + N, C)`` in the
parameter dtype; row 0 = channel-mix token-shift state, row 1 = time-mix token-shift state, rows 2.. = the WKV state
of the layer, a flat reinterpretation of ``(H, N, N)`` [value row, key column].
"""
import itertools
import math

import torch
import torch.nn.functional as F

from . import blocks7, ops
from .rwkv7 import HipRWKV

HEAD_SIZE = 64


def layer_norm(x, w, eps=1e-5):
    """rwkv7.py:8-12"""
    return F.layer_norm(x.float(), (x.shape[-1],), w["weight"].float(), w["bias"].float(), eps).to(x.dtype)


def _orthogonal(gen, rows, cols, gain, device):
    """rwkv7.py:26-38: QR of a normal matrix with the sign fix, scaled by gain."""
    flat = torch.randn((max(rows, cols), min(rows, cols)), generator=gen, device=device, dtype=torch.float32)
    q, r = torch.linalg.qr(flat)
    q = q * torch.sign(torch.diagonal(r))[None] * gain
    return q if rows >= cols else q.T


def randomize_weights(seed, n_layer, n_embd, vocab_size, dtype=torch.bfloat16, device="cuda", zero_init=True):
    """Schedules and distributions of rwkv7.py:81-173.  ``zero_init=False`` replaces the zero-initialised matrices
    (output, ffn.value, the first LoRA factors) by small random ones, so that the recurrence reaches the logits --
    used by the parity tests; the reference's init makes every block's contribution vanish."""
    gen = torch.Generator(device=device)
    gen.manual_seed(seed)
    L, C, N = n_layer, n_embd, HEAD_SIZE
    H = C // N
    f32 = dict(device=device, dtype=torch.float32)
    lay = torch.arange(L, **f32)
    ratio_0_to_1 = lay / max(L - 1, 1)
    ratio_1_to_almost_0 = 1.0 - lay / L
    ddd = torch.arange(C, **f32) / C

    def small(*shape):
        if zero_init:
            return torch.zeros(shape, **f32)
        return 0.02 * torch.randn(shape, generator=gen, **f32)

    def orth_stack(rows, cols, gain):
        return torch.stack([_orthogonal(gen, rows, cols, gain, device) for _ in range(L)])

    att = {}
    for name, p in (("x_r", 0.2), ("x_w", 0.9), ("x_k", 0.7), ("x_v", 0.7), ("x_a", 0.9), ("x_g", 0.2)):
        att[name] = 1 - torch.pow(ddd[None], p * ratio_1_to_almost_0[:, None])
    linear = (torch.arange(C, **f32) / (C - 1) - 0.5)[None].repeat(L, 1)
    zz = ((torch.arange(C, **f32) % N) - (N - 1) / 2) / ((N - 1) / 2)
    zigzag = (zz * zz.abs())[None].repeat(L, 1)
    www = -6 + 6 * torch.pow(torch.arange(C, **f32)[None] / (C - 1), 1 + ratio_0_to_1[:, None] ** 0.3)
    d_decay = max(32, int(round((1.8 * (C ** 0.5)) / 32) * 32))
    d_mv = max(32, int(round((1.3 * (C ** 0.5)) / 32) * 32))
    d_gate = max(32, int(round((0.6 * (C ** 0.8)) / 32) * 32))
    att["w0"] = www + 0.5 + zigzag * 2.5
    att["w1"] = small(L, C, d_decay)
    att["w2"] = orth_stack(d_decay, C, 0.1)
    att["a0"] = -0.19 + zigzag * 0.3 + linear * 0.4
    att["a1"] = small(L, C, d_decay)
    att["a2"] = orth_stack(d_decay, C, 0.1)
    att["v0"] = 0.73 - linear * 0.4
    att["v1"] = small(L, C, d_mv)
    att["v2"] = orth_stack(d_mv, C, 0.1)
    att["g1"] = small(L, C, d_gate)
    att["g2"] = orth_stack(d_gate, C, 0.1)
    att["k_k"] = 0.71 - linear * 0.1
    att["k_a"] = 1.02 + torch.zeros_like(linear)
    att["r_k"] = torch.zeros((L, H, N), **f32) - 0.04
    att["receptance"] = {"weight": orth_stack(C, C, 1.0)}
    att["key"] = {"weight": orth_stack(C, C, 0.1)}
    att["value"] = {"weight": orth_stack(C, C, 1.0)}
    att["output"] = {"weight": small(L, C, C)}
    att["ln_x"] = {"bias": torch.zeros((L, C), **f32),
                   "weight": (((1 + lay) / L)[:, None] ** 0.7).repeat(1, C)}
    ffn = {"x_k": 1 - torch.pow(ddd[None], ratio_1_to_almost_0[:, None] ** 4),
           "key": {"weight": orth_stack(4 * C, C, 1.0)},
           "value": {"weight": small(L, C, 4 * C)}}
    head_scale = 0.5 if vocab_size <= C else 0.5 * math.sqrt(vocab_size / C)
    params = {
        "blocks": {"att": att, "ffn": ffn,
                   "ln1": {"bias": torch.zeros((L, C), **f32), "weight": torch.ones((L, C), **f32)},
                   "ln2": {"bias": torch.zeros((L, C), **f32), "weight": torch.ones((L, C), **f32)}},
        "emb": {"weight": (torch.rand((vocab_size, C), generator=gen, **f32) * 2 - 1) * 1e-4},
        "head": {"weight": _orthogonal(gen, vocab_size, C, head_scale, device)},
        "ln0": {"bias": torch.zeros(C, **f32), "weight": torch.ones(C, **f32)},
        "ln_out": {"bias": torch.zeros(C, **f32), "weight": torch.ones(C, **f32)},
    }
    return tree_map(lambda t: t.to(dtype).contiguous(), params)


def tree_map(fn, tree):
    return {k: tree_map(fn, v) if isinstance(v, dict) else fn(v) for k, v in tree.items()}


def layer_of(tree, i):
    return tree_map(lambda t: t[i], tree)


def unstack(tree, n_layer):
    """The per-layer trees of a tree of stacked parameters.  One ``unbind`` per parameter: its backward is one ``stack``,
    where a slice per layer would add a zero-filled copy of the whole stack per layer and parameter (0.1B shape, one
    training step: 860 launches and 5 ms of the GPU's time)."""
    split = tree_map(lambda t: t.unbind(0), tree)
    return [tree_map(lambda ts: ts[i], split) for i in range(n_layer)]


def _leaves(tree):
    for v in tree.values():
        if isinstance(v, dict):
            yield from _leaves(v)
        else:
            yield v


def _needs_grad(x, state, tree):
    """Whether a derivative is asked for with respect to anything that what follows depends on."""
    tensors = lambda: itertools.chain((x, state), _leaves(tree))
    return (torch.is_grad_enabled() and any(t.requires_grad for t in tensors())) or ops.has_tangent(tensors())


class RWKV7:
    """``forward`` / ``default_state`` with the reference's argument names; batched over the leading axis."""

    inner = HipRWKV
    #: use the fused kernels beside the recurrence, with or without autograd: ops.rwkv7_ln_shiftmix (up to
    #: ops.LN_SHIFTMIX_MAX_C channels; wider models: torch's norm and ops.rwkv7_shiftmix), rwkv7_pre, rwkv7_postmix, rwkv7_relusq
    fuse_mix = True

    @classmethod
    def default_state(cls, params, batch):
        """rwkv7.py:176-180 with a batch axis: zeros ``(B, L, 2 + N, C)`` in the parameter dtype."""
        emb = params["emb"]["weight"]
        L, H, N = params["blocks"]["att"]["r_k"].shape
        return torch.zeros((batch, L, 2 + N, emb.shape[1]), dtype=emb.dtype, device=emb.device)

    @classmethod
    def _shift(cls, x, prev, new_starts):
        """Token shift of rwkv7.py:227-229 / 192-194: previous token (state row for t = 0), zero at new_starts."""
        sx = torch.cat([prev[:, None], x[:, :-1]], dim=1)
        if new_starts is not None:
            sx = torch.where(new_starts[:, :, None], torch.zeros_like(sx), sx)
        return sx - x

    @classmethod
    def _interpolate(cls, x, prev, new_starts, mix):
        if cls.fuse_mix and not ops.has_tangent((x, prev, *mix)):
            return ops.rwkv7_shiftmix(x, prev, new_starts, mix)
        sx = cls._shift(x, prev, new_starts)
        return [x + sx * m for m in mix]

    @classmethod
    def _channel_mix(cls, xk, ffn):
        k = xk @ ffn["key"]["weight"].T
        k = ops.rwkv7_relusq(k) if cls.fuse_mix and not ops.has_tangent((k,)) else torch.square(torch.relu(k))
        return k @ ffn["value"]["weight"].T

    @classmethod
    def channel_mixing_seq(cls, x, state_row, ffn, last_idx, new_starts):
        """rwkv7.py:190-198; x is the norm's result.  Returns (output, new shift row)."""
        xk, = cls._interpolate(x, state_row, new_starts, [ffn["x_k"]])
        return cls._channel_mix(xk, ffn), x[torch.arange(x.shape[0], device=x.device), last_idx]

    @classmethod
    def time_mixing_seq(cls, x, shift_row, wkv_state, v_first, att, length, last_idx, new_starts, layer_id,
                        wkv_out=None):
        """rwkv7.py:223-267; x is the norm's result, wkv_state (B, N, C) the layer's rows 2.. of the model state.  With
        ``wkv_out`` (the same rows of the new model state; decode steps without autograd) the recurrence reads and writes the
        two views in place and the third result is None.  Returns (output, new shift row, new wkv state, v_first)."""
        mixed = cls._interpolate(x, shift_row, new_starts, [att[n] for n in blocks7.MIX])
        y, s_new, v_first = cls._time_mix(mixed, wkv_state, v_first, att, length, new_starts, layer_id, wkv_out)
        return y, x[torch.arange(x.shape[0], device=x.device), last_idx], s_new, v_first

    @classmethod
    def _time_mix(cls, mixed, wkv_state, v_first, att, length, new_starts, layer_id, wkv_out):
        """``time_mixing_seq`` from the six interpolations on."""
        xr, xw, xk, xv, xa, xg = mixed
        B, T, C = xr.shape
        H, N = att["r_k"].shape
        fused = cls.fuse_mix and not ops.has_tangent(itertools.chain(mixed, (wkv_state, v_first), _leaves(att)))
        heads = lambda t: t.reshape(B, T, H, N)
        r = heads(xr @ att["receptance"]["weight"].T)
        k = heads(xk @ att["key"]["weight"].T)
        v = heads(xv @ att["value"]["weight"].T)
        w_lora = heads(torch.tanh(xw @ att["w1"]) @ att["w2"])
        a_lora = heads((xa @ att["a1"]) @ att["a2"])
        v_lora = heads((xv @ att["v1"]) @ att["v2"]) if layer_id != 0 else None
        g = heads(torch.sigmoid(xg @ att["g1"]) @ att["g2"])
        if layer_id == 0:
            v_first = v.reshape(B, T, C)
        if fused:
            w, k, v, a, b = ops.rwkv7_pre(w_lora, k, a_lora, v, None if layer_id == 0 else heads(v_first), v_lora, att["w0"],
                                          att["a0"], att["v0"], att["k_k"], att["k_a"])
        else:
            par = lambda n: att[n].reshape(H, N)
            w = -F.softplus(-(par("w0") + w_lora).float()).to(xr.dtype) - 0.5
            if layer_id != 0:
                v = v + (heads(v_first) - v) * torch.sigmoid(par("v0") + v_lora)
            a = torch.sigmoid(par("a0") + a_lora)
            kk = k * par("k_k")
            kk = kk / torch.clamp(torch.linalg.vector_norm(kk.float(), dim=-1, keepdim=True), min=1e-12).to(kk.dtype)
            k = k * (1 + (a - 1) * par("k_a"))
            a, b = -kk, kk * a
        if wkv_out is not None:
            s_new, out = None, cls.inner.step_packed(r, w, k, v, a, b, wkv_state, wkv_out, length, new_starts)
        else:
            s_new, out = cls.inner.inner_loop(r, w, k, v, a, b, wkv_state.reshape(B, H, N, N), length, new_starts)
            s_new = s_new.reshape(B, N, C)
        if fused:
            y = ops.rwkv7_postmix(out, r, k, v, g, att["ln_x"]["weight"], att["ln_x"]["bias"], att["r_k"], 64e-5)
            y = y.reshape(B, T, C)
        else:
            # not F.group_norm: in torch 2.10 for ROCm its weight's and bias's cotangents are wrong beyond some 100 rows
            y = F.layer_norm(out.reshape(B, T, H, N).float(), (N,), eps=64e-5).reshape(B, T, C)
            y = (y * att["ln_x"]["weight"].float() + att["ln_x"]["bias"].float()).to(xr.dtype)
            bonus = ((r * k * att["r_k"]).sum(-1, keepdim=True) * v).reshape(B, T, C)
            y = (y + bonus) * g.reshape(B, T, C)
        return y @ att["output"]["weight"].T, s_new, v_first

    @classmethod
    def forward(cls, params, tokens, state, length=None, new_starts=None):
        """tokens (B,T) int; state (B,L,2+N,C); length (B,) or None (= T); new_starts (B,T) bool or None.
        Returns (logits (B,T,vocab), new state).  llm.py:71-84 + rwkv7.py:269-291."""
        B, T = tokens.shape
        L, H, N = params["blocks"]["att"]["r_k"].shape
        C = H * N
        x = params["emb"]["weight"][tokens]
        dev = x.device                              # the tokens themselves may lie in host memory
        if length is not None:
            length = torch.as_tensor(length, device=dev).to(torch.int32).reshape(-1).expand(B).contiguous()
        if new_starts is not None:
            new_starts = torch.as_tensor(new_starts, device=dev).to(torch.bool).expand(B, T).contiguous()
        # the separate steps carry forward-mode tangents where torch does; the recurrence refuses those that reach it
        fused = (cls.fuse_mix and C <= ops.LN_SHIFTMIX_MAX_C
                 and not ops.has_tangent(itertools.chain((x, state), _leaves(params))))
        # a subclass's own mixing methods get what they always got: the norm's result, and every argument as a tensor
        steps = any(getattr(cls, n).__func__ is not getattr(RWKV7, n).__func__ for n in ("time_mixing_seq", "channel_mixing_seq"))
        # where everything is this package's: decode steps from native code, whole sequences as one operator
        own = (fused and not steps and cls.inner.inner_loop == HipRWKV.inner_loop and not HipRWKV.force_seq
               and not ops.autocast_elsewhere(x))
        if own and T <= 8 and not _needs_grad(x, state, params):
            step = ops.rwkv7_decode(params, x, state, length, new_starts, HipRWKV.assoc_compat)
            if step is not None:
                return step
        # the fused norm takes one dtype: a norm held in another (fp32 beside bf16) is not rounded to it
        fits = lambda *lns: fused and all(t.dtype == x.dtype for ln in lns for t in ln.values())
        norm = lambda x, dx, ln: (ops.rwkv7_ln_shiftmix(x, dx, ln, None, None, None, [])[2][0] if fits(ln) else
                                  layer_norm(x if dx is None else x + dx, ln))
        x = norm(x, None, params["ln0"])
        # x is ln0's result here: a trainable norm counts as well as a trainable embedding.  What trains after the blocks does not.
        grad = _needs_grad(x, state, params["blocks"])
        stacked = blocks7.gather(params["blocks"]) if own and T > 8 else ()
        if stacked and blocks7.covers(stacked, x, state):
            x, dx, new_state = blocks7.run(stacked, x, state, new_starts, length, grad)
            return norm(x, dx, params["ln_out"]) @ params["head"]["weight"].T, new_state
        blocks = unstack(params["blocks"], L)
        head = not steps and fits(params["blocks"]["ln1"], params["blocks"]["ln2"])
        if steps:
            length = torch.full((B,), T, dtype=torch.int32, device=dev) if length is None else length
            new_starts = torch.zeros((B, T), dtype=torch.bool, device=dev) if new_starts is None else new_starts
        if not head:                                # xn[length - 1] with the wrap-around of negative indices
            last = torch.full((B,), T - 1, device=dev) if length is None else (length.long() - 1) % T
        # without autograd the layers write their rows of the new state where they belong; decode steps read and write the
        # recurrence's rows in place as well
        in_place = head and not grad and state.dtype == x.dtype and (C * x.element_size()) % 16 == 0
        packed = T <= 8 and hasattr(cls.inner, "step_packed") and not grad
        new_state = torch.empty_like(state) if (in_place or packed) else None
        in_place = in_place and new_state.is_contiguous()
        rows = []                                   # otherwise: the new state's parts in memory order, joined at the end
        v_first, dx = x, None
        for i, blk in enumerate(blocks):
            st, nst = state[:, i], (None if new_state is None else new_state[:, i])
            att, ffn, wkv_out = blk["att"], blk["ffn"], (nst[:, 2:] if packed else None)
            if head:
                x, shift1, mixed = ops.rwkv7_ln_shiftmix(x, dx, blk["ln1"], st[:, 1], new_starts, length,
                                                         [att[n] for n in blocks7.MIX], shift_out=nst[:, 1] if in_place else None)
                dx, wkv, v_first = cls._time_mix(mixed, st[:, 2:], v_first, att, length, new_starts, i, wkv_out)
                x, shift0, (xk,) = ops.rwkv7_ln_shiftmix(x, dx, blk["ln2"], st[:, 0], new_starts, length, [ffn["x_k"]],
                                                         shift_out=nst[:, 0] if in_place else None)
                dx = cls._channel_mix(xk, ffn)
            else:
                x = x if dx is None else x + dx
                dx, shift1, wkv, v_first = cls.time_mixing_seq(layer_norm(x, blk["ln1"]), st[:, 1], st[:, 2:], v_first, att, length,
                                                               last, new_starts, i, wkv_out)
                x = x + dx
                dx, shift0 = cls.channel_mixing_seq(layer_norm(x, blk["ln2"]), st[:, 0], ffn, last, new_starts)
            if new_state is None:
                rows += [shift0[:, None], shift1[:, None], wkv]
                continue
            if not in_place:
                nst[:, 0], nst[:, 1] = shift0, shift1
            if not packed:
                nst[:, 2:] = wkv
        if new_state is None:
            new_state = torch.cat([r.to(state.dtype) for r in rows], dim=1).reshape(state.shape)
        return norm(x, dx, params["ln_out"]) @ params["head"]["weight"].T, new_state
