"""The stack of blocks as one operator (jaxrwkv_amd.blocks7) against the same model step by step under torch's autograd, and its
grouped products against torch.

The step-by-step path is the model with a recurrence class of its own (HipRWKV's op behind another class), so that both run the
same kernels but for the low-rank products.  fp32: sums in another order, 2e-4 of a result's rms in the 2-norm (gradients
of a two-layer model pass through about thirty of them).  bf16: both round at the same places but for the second cotangents of r,
k and v, which are added in fp32 here: a relative difference of 3e-2 in the 2-norm, what bf16 rounding does to these gradients
between any two formulations of the model."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def rel(a, b):
    a, b = a.double(), b.double()
    return ((a - b).norm() / b.norm().clamp(min=1e-30)).item()


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("L,B,T,C", [(1, 1, 9, 64), (2, 3, 45, 128), (3, 2, 130, 192)])
def test_blocks_equal_the_steps(L, B, T, C, dtype, monkeypatch):
    from jaxrwkv_amd.model7 import RWKV7, randomize_weights, tree_map
    from jaxrwkv_amd.rwkv7 import HipRWKV
    params = randomize_weights(T, L, C, 208, dtype=dtype, device="cuda", zero_init=False)
    g = torch.Generator("cuda").manual_seed(L)
    tok = torch.randint(0, 208, (B, T), device="cuda", generator=g)
    state = (0.1 * torch.randn((B, L, 66, C), device="cuda", generator=g)).to(dtype)
    length = torch.randint(0, T + 1, (B,), device="cuda", generator=g)
    ns = torch.rand((B, T), device="cuda", generator=g) < 0.1
    cot = [torch.randn((B, T, 208), device="cuda", generator=g).to(dtype),
           torch.randn((B, L, 66, C), device="cuda", generator=g).to(dtype)]

    class Same(HipRWKV):
        @classmethod
        def inner_loop(cls, *a):
            return HipRWKV.inner_loop(*a)

    def leaves(tree):
        for v in tree.values():
            yield from leaves(v) if isinstance(v, dict) else (v,)

    def run(twice):
        p = tree_map(lambda t: t.clone().requires_grad_(), params)
        st = state.clone().requires_grad_()
        outs = RWKV7.forward(p, tok, st, length, ns)
        ins = [st, *leaves(p)]
        grads = torch.autograd.grad(outs, ins, cot, allow_unused=True, retain_graph=twice)
        if twice:
            again = torch.autograd.grad(outs, ins, cot, allow_unused=True)
            assert all(torch.equal(a, b) for a, b in zip(grads[2:], again[2:]) if a is not None and a.dim() < 4)
        return list(outs) + list(grads)

    got = run(True)
    with torch.no_grad():
        plain = RWKV7.forward(params, tok, state, length, ns)
    assert torch.equal(plain[0], got[0]) and torch.equal(plain[1], got[1])
    monkeypatch.setattr(RWKV7, "inner", Same)
    want = run(False)
    limit = 2e-4 if dtype == torch.float32 else 3e-2
    for i, (a, b) in enumerate(zip(got, want)):
        if b is None or not b.abs().max() > 0:
            assert a is None or not a.abs().max() > 0, i
            continue
        assert rel(a, b) < limit, (i, a.shape, rel(a, b))


@pytest.mark.parametrize("M,N,K", [(8, 8, 8), (64, 64, 64), (72, 200, 40), (333, 64, 96), (1000, 136, 2048)])
@pytest.mark.parametrize("km,kn", [(0, 0), (0, 1), (1, 0), (1, 1)])
def test_grouped_products(M, N, K, km, kn):
    """The sum is rounded to bf16 before f and the result after it, each by at most 2^-8 of its size.  relu(x)^2 doubles the
    first: 3 * 2^-8 relative; where aux is added the first is relative to the product (below 5 here) and not to the sum: 5 * 2^-8,
    2e-2 of the rms of about 1."""
    from jaxrwkv_amd import blocks7
    if km:
        M = (M + 7) // 8 * 8
    g = torch.Generator("cuda").manual_seed(M + N)
    n = lambda *s: torch.randn(s, device="cuda", generator=g).bfloat16()
    x, w = n(K, M) if km else n(M, K), n(K, N) if kn else n(N, K)
    w = (w.float() / K ** 0.5).bfloat16()
    aux = n(M, N).sigmoid()
    prod = (x.float().T if km else x.float()) @ (w.float() if kn else w.float().T)
    h = aux.float()
    want = [prod, torch.tanh(prod), torch.sigmoid(prod), torch.relu(prod) ** 2, prod + h, prod * (1 - h * h), prod * h * (1 - h)]
    outs = [torch.full((M, N), 7.0, device="cuda", dtype=torch.bfloat16) for _ in want]
    blocks7._gemm([(o, x, w, km, kn, i if i < 4 else i - 4, None if i < 4 else aux) for i, o in enumerate(outs)])
    for i, (o, ref) in enumerate(zip(outs, want)):
        bound = 3 * 2.0 ** -8 * ref.abs() + 2e-2 * ref.pow(2).mean().sqrt()
        assert ((o.float() - ref).abs() <= bound).all(), (i, ((o.float() - ref).abs() / bound).max().item())


def test_create_graph_keeps_the_first_cotangents():
    """A caller that asks for a graph of the cotangents gets the cotangents as without; only differentiating those again is an
    error."""
    from jaxrwkv_amd.model7 import RWKV7, randomize_weights
    params = randomize_weights(3, 2, 128, 96, dtype=torch.bfloat16, device="cuda", zero_init=False)
    w = params["blocks"]["ffn"]["key"]["weight"].requires_grad_()
    tok = torch.randint(0, 96, (2, 20), device="cuda", generator=torch.Generator("cuda").manual_seed(1))
    logits, _ = RWKV7.forward(params, tok, RWKV7.default_state(params, 2))
    plain, = torch.autograd.grad(logits.float().square().mean(), w, retain_graph=True)
    graph, = torch.autograd.grad(logits.float().square().mean(), w, create_graph=True)
    assert torch.equal(plain, graph)
    with pytest.raises(RuntimeError):
        torch.autograd.grad(graph.float().sum(), w)
