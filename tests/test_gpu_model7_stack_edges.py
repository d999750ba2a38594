"""The native stack where its dispatch goes and the plain cases do not: lengths at and below zero, the sequential rules for resets, one of
the two output cotangents alone, inner sizes and channel mixes of other widths with rows for either kind of product, training steps
at the sizes of large tiles, a second pass over one graph, captured graphs.  Measured as in test_gpu_model7_stack: its distance from
the fp32 model's results against that of the separate steps."""
import pytest
import torch

from tests.test_gpu_model7_stack import _case

pytestmark = pytest.mark.gpu


def _run(case, dtype, grad, which):
    from jaxrwkv_amd import blocks7
    blocks, x, state, ns, length, cot = case
    params = [t.to(dtype).clone().requires_grad_(grad) for t in blocks7.gather(blocks)]
    x = x.to(dtype).requires_grad_(grad)
    out = blocks7.run(params, x, state.to(dtype), ns, length, grad)
    if not grad:
        return [o.float() for o in out]
    got = torch.autograd.grad([out[i] for i in which], [x, *params], [cot[i].to(dtype) for i in which], allow_unused=True)
    return [o.detach().float() for o in out] + [torch.zeros(1, device="cuda") if t is None else t.float() for t in got]


def _compare(case, grad, which, monkeypatch):
    from jaxrwkv_amd import blocks7
    calls, native = [], blocks7._native
    monkeypatch.setattr(blocks7, "_native", lambda *a: calls.append(native(*a)) or calls[-1])
    got = _run(case, torch.bfloat16, grad, which)
    assert calls == [True]
    monkeypatch.setattr(blocks7, "_native", lambda *a: False)
    steps, want = _run(case, torch.bfloat16, grad, which), _run(case, torch.float32, grad, which)
    for i, (a, b, w) in enumerate(zip(got, steps, want)):
        size = w.norm()
        assert torch.isfinite(a).all() and a.shape == w.shape
        assert (a - w).norm() <= 1.2 * (b - w).norm() + 2.0 ** -9 * size, (i, float((a - w).norm() / size), float((b - w).norm() / size))


@pytest.mark.parametrize("compat", [True, False])
@pytest.mark.parametrize("which", [(0, 1, 2), (0,), (1,), (2,)])
def test_lengths_rules_and_single_cotangents(which, compat, monkeypatch):
    from jaxrwkv_amd.rwkv7 import HipRWKV
    monkeypatch.setattr(HipRWKV, "assoc_compat", compat)
    blocks, x, state, ns, _, cot = _case(2, 128, 4, 37, False, True)
    length = torch.tensor([0, -1, 37, 20], device="cuda", dtype=torch.int32)
    _compare((blocks, x, state, ns, length, cot), True, which, monkeypatch)


def _widths(case, F, sizes):
    """The first columns of the channel mix and of the low-rank factors, repeated where wider ones are asked for."""
    blocks = case[0]
    take = lambda t, dim, n: torch.cat([t] * -(-n // t.shape[dim]), dim).narrow(dim, 0, n).contiguous()
    att, ffn = dict(blocks["att"]), {k: dict(v) if isinstance(v, dict) else v for k, v in blocks["ffn"].items()}
    for f, d in zip("wavg", sizes):
        att[f + "1"], att[f + "2"] = take(att[f + "1"], 2, d), take(att[f + "2"], 1, d)
    ffn["key"]["weight"], ffn["value"]["weight"] = take(ffn["key"]["weight"], 1, F), take(ffn["value"]["weight"], 2, F)
    return (dict(blocks, att=att, ffn=ffn), *case[1:])


@pytest.mark.parametrize("F,sizes", [(200, (8, 24, 40, 72)), (1024, (136, 8, 16, 264)), (72, (64, 64, 64, 64))])
@pytest.mark.parametrize("B,T", [(1, 11), (2, 16), (3, 11), (1, 200)])
@pytest.mark.parametrize("grad", [False, True])
def test_widths(B, T, F, sizes, grad, monkeypatch):
    _compare(_widths(_case(2, 128, B, T, False, True), F, sizes), grad, (0, 1), monkeypatch)


@pytest.mark.parametrize("L,C,B,T", [(1, 768, 4, 512), (1, 1024, 3, 700), (1, 1536, 1, 1100), (1, 2048, 1, 600), (1, 2048, 3, 350)])
def test_training_steps_of_large_tiles(L, C, B, T, monkeypatch):
    _compare(_case(L, C, B, T, False, True), True, (0, 1), monkeypatch)


def _graph_inputs(seed):
    from jaxrwkv_amd import blocks7
    blocks, x, state, ns, length, cot = _case(2, 256, 2, 300, True, True, seed)
    return [t.clone() for t in blocks7.gather(blocks)], [x, state, ns, length, *cot]


def test_second_pass_over_one_graph():
    from jaxrwkv_amd import blocks7
    params, (x, state, ns, length, *cot) = _graph_inputs(3)
    for t in (x, *params):
        t.requires_grad_()
    out = blocks7.run(params, x, state, ns, length, True)
    first = torch.autograd.grad(out, [x, *params], cot, retain_graph=True)
    length.zero_()                                        # the caller's own, after the forward
    for a, b in zip(first, torch.autograd.grad(out, [x, *params], cot)):
        assert torch.equal(a, b)


@pytest.mark.parametrize("grad", [False, True])
def test_captured(grad):
    """Replays on other inputs, with eager work between them, equal eager passes bit for bit."""
    from jaxrwkv_amd import blocks7
    params, held = _graph_inputs(4)
    for t in params:
        t.requires_grad_(grad)

    def once():
        x, state, ns, length, *cot = held
        x = x.detach().requires_grad_(grad)
        out = blocks7.run(params, x, state, ns, length, grad)
        assert grad == out[0].requires_grad
        return [o.detach() for o in out] + (list(torch.autograd.grad(out, [x, *params], cot)) if grad else [])

    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        once()
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = once()
    for seed in (5, 6, 7):
        for h, new in zip(held, _graph_inputs(seed)[1]):
            h.copy_(new)
        want = [t.clone() for t in once()]
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(a, b) for a, b in zip(out, want))
