"""Which route a call of the RWKV-7 model takes and what it hands to the library, on the CPU with the library stubbed out."""
import pytest
import torch

from tests import stub_library

L, C, V = 2, 64, 32


def model(dtype):
    from jaxrwkv_amd.model7 import randomize_weights
    return randomize_weights(1, L, C, V, dtype=dtype, device="cpu", zero_init=False)


def leaves(tree, path=()):
    for k, v in tree.items():
        yield from leaves(v, path + (k,)) if isinstance(v, dict) else ((".".join(path + (k,)), v),)


def call(params, T, B=2, state=None, **kw):
    from jaxrwkv_amd.model7 import RWKV7
    tok = torch.arange(B * T).reshape(B, T) % V
    return RWKV7.forward(params, tok, RWKV7.default_state(params, B) if state is None else state, **kw)


@pytest.mark.parametrize("grad", [False, True])
@pytest.mark.parametrize("T", [3, 20])
def test_autocast_hands_over_one_type(monkeypatch, T, grad):
    """Products come out in autocast's type beside parameters of another: no kernel may be told one type and given the other."""
    stub = stub_library.install(monkeypatch)
    params = model(torch.float32)
    for _, p in leaves(params):
        p.requires_grad_(grad)
    with torch.autocast("cpu", torch.bfloat16):
        logits, new_state = call(params, T)
    assert logits.dtype == torch.bfloat16 and stub.calls
    if grad:
        (logits.float().sum() + new_state.float().sum()).backward()


def test_backward_inside_autocast(monkeypatch):
    stub_library.install(monkeypatch)
    params = model(torch.float32)
    for _, p in leaves(params):
        p.requires_grad_()
    logits, new_state = call(params, 20)
    with torch.autocast("cpu", torch.bfloat16):
        (logits.float().sum() + new_state.float().sum()).backward()
    assert all(p.grad.dtype == torch.float32 for _, p in leaves(params))
