"""What the operators hand to the library, on the CPU with the library stubbed out."""
import pytest
import torch

from tests import stub_library


def off(t):
    """The same values one element past a 16-byte boundary."""
    return torch.cat([torch.zeros(1, dtype=t.dtype), t.flatten()])[1:].view(t.shape)


@pytest.mark.parametrize("grad", [False, True])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_wkv4_receptance_and_decay_anywhere_in_memory(monkeypatch, dtype, grad):
    from jaxrwkv_amd.rwkv4 import HipRWKV
    stub_library.install(monkeypatch)
    B, T, C = 2, 5, 64
    n = lambda *s: torch.randn(s).to(dtype)
    r, w = off(n(B, T, C)), off(n(C))
    if grad:
        w.requires_grad_()
    assert r.data_ptr() % 16 and w.data_ptr() % 16
    new_s, out = HipRWKV.inner_loop(r, n(B, T, C), n(B, T, C), w, n(C), n(B, 3, C), None, None)
    assert not out.isnan().any()
    if grad:
        out.float().sum().backward()
        assert w.grad is not None


def test_wkv4_cotangent_anywhere_in_memory(monkeypatch):
    """The output's cotangent is the caller's own: with the receptance inside the op no product of torch's comes before it."""
    from jaxrwkv_amd.rwkv4 import HipRWKV
    stub_library.install(monkeypatch)
    n = lambda *s: torch.randn(s)
    w = n(64).requires_grad_()
    _, out = HipRWKV.inner_loop(n(2, 5, 64), n(2, 5, 64), n(2, 5, 64), w, n(64), n(2, 3, 64), None, None)
    torch.autograd.grad(out, w, off(n(2, 5, 64)))


@pytest.mark.parametrize("T", [3, 20])
def test_model_state_cotangent_anywhere_in_memory(monkeypatch, T):
    from tests.test_model7_routes import L, C, call, leaves, model
    stub_library.install(monkeypatch)
    params = model(torch.float32)
    ps = [p.requires_grad_() for _, p in leaves(params["blocks"])]
    _, new_state = call(params, T, B=1)
    torch.autograd.grad(new_state, ps, off(torch.randn(1, L, 66, C)), allow_unused=True)


def test_wkv4_state_and_receptance_are_apart(monkeypatch):
    """The new state has no derivative in the receptance: no graph, and no cotangent of zeros for it."""
    from jaxrwkv_amd.rwkv4 import HipRWKV
    stub_library.install(monkeypatch)
    n = lambda *s: torch.randn(s)
    r, k = n(2, 5, 64).requires_grad_(), n(2, 5, 64)
    new_s, out = HipRWKV.inner_loop(r, k, n(2, 5, 64), n(64), n(64), n(2, 3, 64), None, None)
    assert not new_s.requires_grad and torch.autograd.grad(out.sum(), r)[0] is not None
    k.requires_grad_()
    new_s, out = HipRWKV.inner_loop(r, k, n(2, 5, 64), n(64), n(64), n(2, 3, 64), None, None)
    gr, gk = torch.autograd.grad(new_s.sum(), (r, k), allow_unused=True)
    assert gr is None and gk is not None
