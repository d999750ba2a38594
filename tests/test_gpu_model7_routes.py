"""Results and gradients of the RWKV-7 model on the routes that a call can take, against another route of the same model."""
import pytest
import torch

pytestmark = pytest.mark.gpu

L, C, V = 2, 128, 208


def model(dtype, **kw):
    from jaxrwkv_amd.model7 import randomize_weights
    return randomize_weights(7, kw.get("L", L), kw.get("C", C), V, dtype=dtype, device="cuda", zero_init=False)


def leaves(tree, path=()):
    for k, v in tree.items():
        yield from leaves(v, path + (k,)) if isinstance(v, dict) else ((".".join(path + (k,)), v),)


def inputs(B, T, dtype, L=L, C=C):
    g = torch.Generator("cuda").manual_seed(T)
    return (torch.randint(0, V, (B, T), device="cuda", generator=g),
            (0.1 * torch.randn((B, L, 66, C), device="cuda", generator=g)).to(dtype))


def rel(a, b):
    a, b = a.double(), b.double()
    return ((a - b).norm() / b.norm().clamp(min=1e-30)).item()


@pytest.mark.parametrize("T", [3, 20])
def test_autocast(T, monkeypatch):
    """fp32 parameters under bf16 autocast: the fused steps are no further from the fp32 model than the separate ones are, which
    round at more places (half as much again for the chance in a rounding error's 2-norm, and 1e-2)."""
    from jaxrwkv_amd.model7 import RWKV7
    tok, state = inputs(3, T, torch.float32)
    g = torch.Generator("cuda").manual_seed(1)
    cot = [torch.randn(s, device="cuda", generator=g) for s in ((3, T, V), state.shape)]

    def run(autocast):
        params = model(torch.float32)
        ps = [p.requires_grad_() for _, p in leaves(params)]
        with torch.autocast("cuda", torch.bfloat16, enabled=autocast):
            outs = RWKV7.forward(params, tok, state)
        grads = torch.autograd.grad(outs, ps, [c.to(o.dtype) for c, o in zip(cot, outs)], allow_unused=True)
        return [*outs, *grads]

    exact, fused = run(False), run(True)
    monkeypatch.setattr(RWKV7, "fuse_mix", False)
    for i, (e, f, s) in enumerate(zip(exact, fused, run(True))):
        if s is not None and s.abs().max() > 0:
            assert rel(f, e) < 1.5 * rel(s, e) + 1e-2, (i, tuple(e.shape), rel(f, e), rel(s, e))


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("T", [1, 3, 20])
def test_frozen_embedding(T, dtype):
    """Gradients and results do not depend on what else is trainable: the same route, the same kernels, sums in the same order but
    for the atomics of the general path's group norm (fp32, 1e-5 of the 2-norm; rounded to bf16 2^-9 where a sum sits on an edge)."""
    from jaxrwkv_amd.model7 import RWKV7
    tok, state = inputs(3, T, dtype)

    def run(skip):
        ps = {n: p.requires_grad_(n not in skip) for n, p in leaves(model(dtype)) }
        params = tree(ps)
        logits, new_state = RWKV7.forward(params, tok, state)
        keep = [n for n in ps if n not in skip]
        grads = torch.autograd.grad(logits.float().square().mean() + new_state.float().square().mean(), [ps[n] for n in keep],
                                    allow_unused=True)
        return logits, new_state, dict(zip(keep, grads))

    def tree(flat):
        out = {}
        for name, t in flat.items():
            *path, last = name.split(".")
            at = out
            for p in path:
                at = at.setdefault(p, {})
            at[last] = t
        return out

    full, part = run(()), run(("emb.weight",))
    assert torch.equal(full[0], part[0]) and torch.equal(full[1], part[1])
    with torch.no_grad():
        plain = RWKV7.forward(model(dtype), tok, state)
    assert rel(part[0], plain[0]) < (1e-4 if dtype == torch.float32 else 3e-2)
    assert rel(part[1], plain[1]) < (1e-4 if dtype == torch.float32 else 3e-2)
    for n, g in part[2].items():
        assert g is not None, n
        if full[2][n].abs().max() > 0:
            assert rel(g, full[2][n]) < (1e-5 if dtype == torch.float32 else 2e-3), (n, rel(g, full[2][n]))


@pytest.mark.parametrize("grad", [False, True])
def test_state_in_another_memory_order(grad):
    from jaxrwkv_amd.model7 import RWKV7
    tok, state = inputs(3, 20, torch.bfloat16)
    params = model(torch.bfloat16)
    for _, p in leaves(params):
        p.requires_grad_(grad)
    other = state.transpose(2, 3).contiguous().transpose(2, 3)
    a, b = RWKV7.forward(params, tok, state), RWKV7.forward(params, tok, other)
    assert torch.equal(a[0], b[0]) and torch.equal(a[1], b[1]) and b[1].stride() == other.stride()


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("T", [5, 20])
def test_lengths_outside_the_sequence(T, dtype, monkeypatch):
    """The shift row is that of token (length - 1) mod T whatever the length; the recurrence counts a negative one as none."""
    from jaxrwkv_amd.model7 import RWKV7
    length = torch.tensor([-1, -2 * T - 2, 0, 1, T, T + 3, -(2 ** 31)], device="cuda", dtype=torch.int32)
    tok, state = inputs(len(length), T, dtype)
    params = model(dtype)
    with torch.no_grad():
        got = RWKV7.forward(params, tok, state, length)
        monkeypatch.setattr(RWKV7, "fuse_mix", False)
        want = RWKV7.forward(params, tok, state, length)
    for i in range(len(length)):
        for rows in (slice(0, 1), slice(1, 2), slice(2, 66)):           # a wrong token's row would be about 1 away
            assert rel(got[1][i, :, rows], want[1][i, :, rows]) < (1e-4 if dtype == torch.float32 else 3e-2), (i, rows)


@pytest.mark.parametrize("grad", [False, True])
@pytest.mark.parametrize("T", [3, 20])
def test_wide_models(T, grad, monkeypatch):
    """The route of models too wide for the fused head against the other one: sums of the norm in another order (fp32)."""
    from jaxrwkv_amd import ops
    from jaxrwkv_amd.model7 import RWKV7
    tok, state = inputs(3, T, torch.float32)
    ns = torch.rand((3, T), device="cuda", generator=torch.Generator("cuda").manual_seed(3)) < 0.1
    length = torch.tensor([1, T, 0], device="cuda", dtype=torch.int32)

    def run():
        params = model(torch.float32)
        ps = [p.requires_grad_(grad) for _, p in leaves(params)]
        outs = RWKV7.forward(params, tok, state, length, ns)
        return list(outs) + (list(torch.autograd.grad(outs, ps, [torch.ones_like(o) for o in outs])) if grad else [])

    want = run()
    monkeypatch.setattr(ops, "LN_SHIFTMIX_MAX_C", 64)
    for i, (a, b) in enumerate(zip(run(), want)):
        assert rel(a, b) < 2e-4, (i, tuple(a.shape), rel(a, b))


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("keep", [(), ("att.x_a", "att.v0"), ("ffn.key.weight",), ("att.w1", "att.g2", "att.ln_x.bias", "ln1.weight")])
def test_frozen_parameters_of_the_stack(keep, dtype):
    """Whatever of the blocks is frozen, the other cotangents and the state's are those of a full training step, bit for bit."""
    from jaxrwkv_amd.model7 import RWKV7
    tok, state = inputs(3, 45, dtype)
    g = torch.Generator("cuda").manual_seed(2)
    cot = [torch.randn(s, device="cuda", generator=g).to(dtype) for s in ((3, 45, V), state.shape)]

    def run(trains):
        params = model(dtype)
        ps = {n: p.requires_grad_() for n, p in leaves(params) if trains(n)}
        st = state.clone().requires_grad_()
        outs = RWKV7.forward(params, tok, st)
        return dict(zip(["state", *ps], torch.autograd.grad(outs, [st, *ps.values()], cot)))

    full = run(lambda n: True)
    part = run(lambda n: n.removeprefix("blocks.") in keep)
    assert len(part) == 1 + len(keep)
    for n, t in part.items():
        assert torch.equal(t, full[n]), n


def test_saved_tensors_kept_in_host_memory():
    """Saved tensors that come back as dense copies give the same bits."""
    from jaxrwkv_amd.model7 import RWKV7
    tok, state = inputs(3, 45, torch.bfloat16)
    params = model(torch.bfloat16)
    ps = [p.requires_grad_() for _, p in leaves(params)]

    def run():
        outs = RWKV7.forward(params, tok, state)
        return outs, (outs[0].float().square().sum() + outs[1].float().square().sum())

    _, loss = run()
    want = torch.autograd.grad(loss, ps)
    with torch.autograd.graph.save_on_cpu():
        _, loss = run()
    for a, b in zip(torch.autograd.grad(loss, ps), want):
        assert torch.equal(a, b)


def test_separate_steps_give_the_fused_ones_gradients(monkeypatch):
    """fp32 at more rows than one workgroup of a reduction takes (torch's group norm drops the cotangents of the others): the two
    formulations differ by the rounding of sums over 600 rows, 2e-4 as for the wide models."""
    from jaxrwkv_amd.model7 import RWKV7
    tok, state = inputs(4, 150, torch.float32)
    params = model(torch.float32)
    ps = [p.requires_grad_() for _, p in leaves(params)]
    g = torch.Generator("cuda").manual_seed(3)
    cot = [torch.randn(s, device="cuda", generator=g) for s in ((4, 150, V), state.shape)]

    def run():
        return torch.autograd.grad(RWKV7.forward(params, tok, state), ps, cot)

    want = run()
    monkeypatch.setattr(RWKV7, "fuse_mix", False)
    for (name, _), a, b in zip(leaves(params), run(), want):
        assert rel(a, b) < 2e-4, (name, rel(a, b))
