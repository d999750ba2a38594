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
    """fp32 parameters under bf16 autocast, fused and separate steps: both round products to bf16 and differ in where else they
    round, 3e-2 in the 2-norm as any two bf16 formulations of the model."""
    from jaxrwkv_amd.model7 import RWKV7
    tok, state = inputs(3, T, torch.float32)

    def run():
        params = model(torch.float32)
        ps = [p.requires_grad_() for _, p in leaves(params)]
        with torch.autocast("cuda", torch.bfloat16):
            logits, new_state = RWKV7.forward(params, tok, state)
        grads = torch.autograd.grad(logits.float().square().mean() + new_state.square().mean(), ps, allow_unused=True)
        return [logits, new_state, *grads]

    got = run()
    monkeypatch.setattr(RWKV7, "fuse_mix", False)
    for i, (a, b) in enumerate(zip(got, run())):
        if b is not None and b.abs().max() > 0:
            assert rel(a, b) < 3e-2, (i, tuple(a.shape), rel(a, b))
