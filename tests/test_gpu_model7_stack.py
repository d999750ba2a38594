"""The RWKV-7 stack launched from native code against the same stack in separate steps, both measured by the fp32 model.

Both round to bf16 in the same places but for sums, which the native code rounds once: its distance from the fp32 results (relative,
over an array) may exceed the separate steps' by what their own differs from draw to draw (a fifth) and by half a bf16 step of the
array's size, 2^-9, where an array has few elements."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _case(L, C, B, T, lengths, resets, seed=0):
    from jaxrwkv_amd import model7
    params = model7.randomize_weights(seed, L, C, 256, zero_init=False)
    g = torch.Generator("cuda").manual_seed(seed + T)
    blocks = model7.tree_map(lambda t: t, params["blocks"])
    state = 0.3 * torch.randn((B, L, 66, C), device="cuda", generator=g)
    x = torch.randn((B, T, C), device="cuda", generator=g)
    ns = torch.rand((B, T), device="cuda", generator=g) < 0.1 if resets else None
    length = torch.randint(1, T + 1, (B,), device="cuda", generator=g, dtype=torch.int32) if lengths else None
    cot = [torch.randn(s, device="cuda", generator=g) for s in ((B, T, C), (B, T, C), (B, L, 66, C))]
    return blocks, x.bfloat16(), state.bfloat16(), ns, length, [c.bfloat16() for c in cot]


def _run(case, dtype, grad, with_state):
    from jaxrwkv_amd import blocks7
    blocks, x, state, ns, length, cot = case
    params = [t.to(dtype).clone().requires_grad_(grad) for t in blocks7.gather(blocks)]
    x = x.to(dtype).requires_grad_(grad)
    out = blocks7.run(params, x, state.to(dtype), ns, length, grad)
    if not grad:
        return [o.float() for o in out]
    n = 3 if with_state else 2
    got = torch.autograd.grad(out[:n], [x, *params], [c.to(dtype) for c in cot[:n]], allow_unused=True)
    return [o.detach().float() for o in out] + [torch.zeros(1, device="cuda") if t is None else t.float() for t in got]


@pytest.mark.parametrize("L,C,B,T,lengths,resets,grad,with_state", [
    (1, 128, 1, 9, False, False, True, False),
    (2, 128, 3, 17, True, True, True, True),
    (3, 256, 2, 100, True, True, True, False),
    (2, 768, 1, 33, False, True, True, True),
    (2, 512, 4, 257, False, True, True, False),
    (3, 256, 1, 31, False, False, False, False),
    (2, 1024, 2, 65, True, True, False, False),
    (2, 768, 1, 700, False, True, False, False)])
def test_native_stack(L, C, B, T, lengths, resets, grad, with_state, monkeypatch):
    from jaxrwkv_amd import blocks7
    case = _case(L, C, B, T, lengths, resets)
    calls = []
    native = blocks7._native
    monkeypatch.setattr(blocks7, "_native", lambda *a: calls.append(native(*a)) or calls[-1])
    got = _run(case, torch.bfloat16, grad, with_state)
    assert calls == [True]
    monkeypatch.setattr(blocks7, "_native", lambda *a: False)
    steps = _run(case, torch.bfloat16, grad, with_state)
    want = _run(case, torch.float32, grad, with_state)
    for i, (a, b, w) in enumerate(zip(got, steps, want)):
        size = w.norm()
        assert torch.isfinite(a).all() and a.shape == w.shape
        assert (a - w).norm() <= 1.2 * (b - w).norm() + 2.0 ** -9 * size, (i, float((a - w).norm() / size), float((b - w).norm() / size))
