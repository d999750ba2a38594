"""RWKV-4's inner_loop with the decay and the receptance inside the kernels and the sequences cut into parts, against the op
on whole sequences (wkv4_fwd and wkv4_bwd with their own first pass) with the same steps in torch around it.

fp32: the parts carry the state and its cotangent over many steps at once, rounded in another order: 1e-5 of the array's rms plus
1e-5 relative (2e-5 and 1e-4 for cotangents, whose sums run over all tokens).  bf16: both sides round to bf16 at the same places,
so a result differs by at most one rounding (2^-7 relative) plus 2e-3 of the rms."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def close(name, got, want, rtol, frac):
    got, want = got.double(), want.double()
    bound = rtol * want.abs() + frac * want.pow(2).mean().sqrt() + 1e-30
    worst = ((got - want).abs() / bound).max().item()
    assert worst <= 1.0, (name, worst)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("compat", [True, False])
@pytest.mark.parametrize("B,T,C,p_reset", [(1, 1, 64, 0.0), (1, 15, 8, 0.2), (2, 16, 64, 0.1), (1, 17, 72, 0.0), (3, 700, 200, 0.01),
                                           (1, 2000, 64, 0.0), (9, 40, 4096, 0.02), (33, 33, 1024, 0.02)])
def test_inner_loop(B, T, C, p_reset, compat, dtype, monkeypatch):
    from jaxrwkv_amd import ops
    from jaxrwkv_amd.rwkv4 import HipRWKV
    monkeypatch.setattr(HipRWKV, "assoc_compat", compat)
    g = torch.Generator("cuda").manual_seed(T + C)
    n = lambda *s: torch.randn(s, device="cuda", generator=g)
    r, k, v = n(B, T, C).sigmoid(), n(B, T, C), n(B, T, C)
    w, u = n(C), 0.5 * n(C)
    s = torch.stack([n(B, C), n(B, C).abs() + 0.5, n(B, C)], 1)
    r, k, v, w, u, s = (t.to(dtype).requires_grad_() for t in (r, k, v, w, u, s))
    ns = torch.rand((B, T), device="cuda", generator=g) < p_reset
    length = torch.randint(0, T + 1, (B,), device="cuda", generator=g)
    go, gs = n(B, T, C).to(dtype), n(B, 3, C).to(dtype)

    new_s, out = HipRWKV.inner_loop(r, k, v, w, u, s, length, ns)
    gs = torch.where(new_s < -1e29, torch.zeros_like(gs), gs)             # the constant of a reset state
    grads = torch.autograd.grad((new_s, out), (r, k, v, w, u, s), (gs, go))
    with torch.no_grad():
        again = HipRWKV.inner_loop(r, k, v, w, u, s, length, ns)
    assert torch.equal(again[0], new_s) and torch.equal(again[1], out)

    with torch.no_grad():
        w_neg = -torch.exp(w.float()).to(dtype)
        ref_s, wkv = ops.wkv4_fwd(w_neg, u, k, v, s, length, ns, compat)
        gw, gu, gk, gv, gsi = ops.wkv4_bwd(w_neg, u, k, v, s, length, ns, go * r, gs, compat)
        want = (go * wkv, gk, gv, (gw.float() * w_neg.float()).to(dtype), gu, gsi)
    fine = ref_s > -1e29
    assert torch.equal(fine, new_s > -1e29)
    f32 = dtype == torch.float32
    tol = (1e-5, 1e-5) if f32 else (2.0 ** -7, 2e-3)
    close("out", out, r.detach() * wkv, *tol)
    close("state", new_s[fine], ref_s[fine], *tol)
    for name, a, b in zip(("r", "k", "v", "w", "u", "s"), grads, want):
        close("g" + name, a, b, *((1e-4, 2e-5) if f32 else tol))


@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
def test_a_reset_keeps_a_cotangent_that_is_not_finite_behind_it(bad):
    """Tokens before a reset do not depend on what comes after it, whatever its cotangent (one sequence of 64 channels: in parts
    of 16 tokens): bit for bit the cotangents that a finite one gives."""
    from jaxrwkv_amd.rwkv4 import HipRWKV
    g = torch.Generator("cuda").manual_seed(4)
    B, T, C, t0 = 1, 1000, 64, 605
    n = lambda *s: torch.randn(s, device="cuda", generator=g)
    s = torch.stack([n(B, C), n(B, C).abs() + 0.5, n(B, C)], 1)
    args = [t.requires_grad_() for t in (n(B, T, C).sigmoid(), n(B, T, C), n(B, T, C), n(C), 0.5 * n(C), s)]
    ns = torch.zeros((B, T), dtype=torch.bool, device="cuda")
    ns[:, t0] = True
    go = n(B, T, C)
    _, out = HipRWKV.inner_loop(*args, None, ns)
    want = torch.autograd.grad(out, args, go, retain_graph=True)
    go[:, 900] = bad
    got = torch.autograd.grad(out, args, go)
    for i in (0, 1, 2):
        assert torch.equal(got[i][:, :t0], want[i][:, :t0]) and torch.isfinite(got[i][:, :t0]).all()
    assert torch.equal(got[5], want[5])
    assert not torch.isfinite(got[2][:, t0:]).all()
