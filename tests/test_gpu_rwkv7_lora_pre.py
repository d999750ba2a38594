"""The second low-rank products made where the gates are, against the two launches that they replace: the products add the same steps in
the same order and are rounded in the same place, so the results are equal bit for bit."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("keep", [True, False])
@pytest.mark.parametrize("first", [True, False])
@pytest.mark.parametrize("M,H,d", [(1, 1, (8, 8, 8, 8)), (63, 3, (64, 32, 128, 40)), (65, 2, (72, 136, 264, 64)), (260, 5, (128, 8, 96, 200))])
def test_products_and_gates(M, H, d, first, keep):
    from jaxrwkv_amd import blocks7, ops
    C = 64 * H
    g = torch.Generator("cuda").manual_seed(M)
    rnd = lambda *s, scale=1.0: (scale * torch.randn(s, device="cuda", generator=g)).bfloat16()
    names = blocks7._LORA[:3] if first else blocks7._LORA
    sizes = dict(zip("wagv", d))
    p = {n + "1": rnd(C, s, scale=C ** -0.5) for n, s in sizes.items()}
    p.update({n + "2": rnd(s, C, scale=s ** -0.5) for n, s in sizes.items()})
    p.update({n: rnd(C) for n in ("w0", "a0", "v0", "k_k", "k_a")}, r_k=rnd(H, 64))
    mix = {n: rnd(M, C) for n in sizes}
    k, v, vf = rnd(M, C), rnd(M, C), None if first else rnd(M, C)
    hid, lora, got = blocks7._lora_pre_fwd(p, mix, names, k, v, vf, keep)
    want = {n: torch.empty_like(k) for n, _ in names}
    blocks7._gemm([(want[n], hid[n], p[n + "2"], 0, 1, 0, None) for n, _ in names])
    heads = lambda t: None if t is None else t.view(M, H, 64)
    gates = ops._pre_fwd(heads(want["w"]), heads(k), heads(want["a"]), heads(v), heads(vf), heads(want.get("v")), p["w0"], p["a0"],
                         None if first else p["v0"], p["k_k"], p["k_a"])
    for n, _ in names:
        assert lora[n] is None and not keep and n != "g" or torch.equal(lora[n], want[n])
    for a, b in zip(got, gates):
        assert a is None and b is None or torch.equal(a, b.view(M, C))
