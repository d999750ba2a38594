"""The fused sub-block head (residual addition, LayerNorm, token shift, interpolation) and the fused step between the
projections and the WKV op, forward and backward, against plain torch in fp32 on the same values.

fp32: results within 2e-5 of the array's rms plus 2e-5 relative (sums over up to 2056 channels; cotangents of parameters sum
over up to 135 tokens).  bf16: one rounding of the result (2^-8 relative) plus the roundings inside (xs, xn and a: 2^-9 of
their size each, entering a difference or a product: 1e-2 of the array's rms).
"""
import pytest
import torch

pytestmark = pytest.mark.gpu

TOL = {torch.float32: (2e-5, 2e-5), torch.bfloat16: (2.0 ** -8, 2e-2)}


def close(name, got, want, dtype):
    rtol, frac = TOL[dtype]
    want = want.double()
    bound = rtol * want.abs() + frac * want.pow(2).mean().sqrt().clamp(min=1.0)
    worst = ((got.double() - want).abs() / bound).max().item()
    assert worst <= 1.0, (name, worst)


def both(fn, ref, tensors, dtype):
    """Outputs and cotangents of fn on ``tensors`` and of ref on their fp32 copies, for the same random cotangents."""
    a = [t.clone().requires_grad_() for t in tensors]
    b = [t.float().requires_grad_() for t in tensors]
    ya, yb = fn(*a), ref(*b)
    g = torch.Generator("cuda").manual_seed(1)
    cot = [torch.randn(y.shape, device="cuda", generator=g).to(dtype) for y in ya]
    ga = torch.autograd.grad(ya, a, cot)
    gb = torch.autograd.grad(yb, b, [c.float() for c in cot])
    for i, (x, y) in enumerate(zip(ya, yb)):
        close(f"output {i}", x, y, dtype)
    for i, (x, y) in enumerate(zip(ga, gb)):
        close(f"cotangent {i}", x, y, dtype)
    with torch.no_grad():
        for x, y in zip(fn(*tensors), ya):
            assert torch.equal(x, y)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("n_mix", [0, 1, 6])
@pytest.mark.parametrize("B,T,C,with_dx", [(1, 1, 8, False), (3, 1, 128, True), (3, 45, 72, True), (2, 9, 2048, True), (2, 9, 2056, True),
                                           (1, 4100, 64, False)])
def test_ln_shiftmix(B, T, C, with_dx, n_mix, dtype):
    from jaxrwkv_amd import ops
    g = torch.Generator("cuda").manual_seed(B * T + C)
    n = lambda *s: torch.randn(s, device="cuda", generator=g).to(dtype)
    x, dx, w, b, prev, mix = n(B, T, C), n(B, T, C), 1 + 0.1 * n(C), 0.1 * n(C), n(B, C), [n(C).sigmoid() for _ in range(n_mix)]
    ns = torch.rand((B, T), device="cuda", generator=g) < 0.1
    length = torch.randint(0, T + 1, (B,), device="cuda", generator=g, dtype=torch.int32)
    extra = [dx] if with_dx else []

    def split(t):
        t = list(t)
        d = t.pop(1) if with_dx else None
        return t[0], d, t[1], t[2], t[3], t[4:]

    def fn(*t):
        x_, d_, w_, b_, p_, m_ = split(t)
        xs, shift, outs = ops.rwkv7_ln_shiftmix(x_, d_, {"weight": w_, "bias": b_}, p_ if n_mix else None,
                                                ns if n_mix else None, length if n_mix else None, m_)
        return [xs * 1, *outs] + ([shift] if n_mix else [p_ * 1])

    def ref(*t):
        x_, d_, w_, b_, p_, m_ = split(t)
        xs = x_ if d_ is None else x_ + d_
        if dtype == torch.bfloat16:                       # the stored residual stream is rounded; straight-through here
            xs = xs + (xs.bfloat16().float() - xs).detach()
        xn = torch.nn.functional.layer_norm(xs, (C,), w_, b_, 1e-5)
        if not n_mix:
            return [xs * 1, xn, p_ * 1]
        pv = torch.cat([p_[:, None], xn[:, :-1]], 1)
        sx = torch.where(ns[:, :, None], torch.zeros_like(pv), pv) - xn
        return [xs * 1] + [xn + sx * m for m in m_] + [xn[torch.arange(B, device="cuda"), (length.long() - 1) % T]]

    both(fn, ref, [x, *extra, w, b, prev, *mix], dtype)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("vmix", [False, True])
@pytest.mark.parametrize("rows,H", [(1, 1), (33, 3), (1100, 2)])
def test_pre(rows, H, vmix, dtype):
    from jaxrwkv_amd import ops
    g = torch.Generator("cuda").manual_seed(rows)
    n = lambda *s: torch.randn(s, device="cuda", generator=g).to(dtype)
    tok = [n(1, rows, H, 64) for _ in range(6 if vmix else 3)]           # xw, k, xa (, v, v_first, xv)
    par = [n(H * 64) for _ in range(5 if vmix else 4)]                   # w0, a0, k_k, k_a (, v0)

    def fn(*t):
        tk, p = list(t[:len(tok)]), list(t[len(tok):])
        if vmix:
            return ops.rwkv7_pre(*tk, p[0], p[1], p[4], p[2], p[3])
        w, k, v, a, b = ops.rwkv7_pre(*tk, tk[1], None, None, p[0], p[1], None, p[2], p[3])
        return [w, k, a, b]

    def ref(*t):
        tk = t[:len(tok)]
        p = [x.reshape(H, 64) for x in t[len(tok):]]
        w = -torch.nn.functional.softplus(-(p[0] + tk[0])) - 0.5
        a = torch.sigmoid(p[1] + tk[2])
        kk = torch.nn.functional.normalize(tk[1] * p[2], dim=-1)
        k = tk[1] * (1 + (a - 1) * p[3])
        if not vmix:
            return [w, k, -kk, kk * a]
        return [w, k, tk[3] + (tk[4] - tk[3]) * torch.sigmoid(p[4] + tk[5]), -kk, kk * a]

    both(fn, ref, tok + par, dtype)
