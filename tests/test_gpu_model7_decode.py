"""The native decode step (ops.rwkv7_decode) against the general path of the same model on the same weights.

Both round to bf16 at the same places but for the products' inner order and the low-rank activations (fp32 here, rounded
between there); a bf16 model of two layers is then within its own noise of the general path: logits and state within 3e-2 of
their rms in the 2-norm, and no element further than a tenth of the rms plus 5 percent."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def close(a, b):
    a, b = a.double(), b.double()
    rms = b.pow(2).mean().sqrt()
    assert ((a - b).pow(2).mean().sqrt() / rms).item() < 3e-2
    assert ((a - b).abs() <= 0.1 * rms + 0.05 * b.abs()).float().mean().item() > 0.999
    assert ((a - b).abs() / (rms + b.abs())).max().item() < 0.5


@pytest.mark.parametrize("compat", [True, False])
@pytest.mark.parametrize("B,T,C", [(1, 1, 64), (2, 8, 128), (15, 1, 192), (17, 1, 128), (5, 7, 128), (64, 1, 64), (65, 1, 128),
                                   (32, 8, 128), (256, 1, 192)])
def test_native_decode_step(B, T, C, compat, monkeypatch):
    from jaxrwkv_amd import ops
    from jaxrwkv_amd.model7 import RWKV7, randomize_weights
    from jaxrwkv_amd.rwkv7 import HipRWKV
    params = randomize_weights(B + T, 2, C, 208, dtype=torch.bfloat16, device="cuda", zero_init=False)
    g = torch.Generator("cuda").manual_seed(B)
    tok = torch.randint(0, 208, (B, T), device="cuda", generator=g)
    state = (0.1 * torch.randn((B, 2, 66, C), device="cuda", generator=g)).bfloat16()
    length = torch.randint(0, T + 1, (B,), device="cuda", generator=g)
    ns = torch.rand((B, T), device="cuda", generator=g) < 0.2
    calls = []
    native = ops.rwkv7_decode
    monkeypatch.setattr(HipRWKV, "assoc_compat", compat)
    monkeypatch.setattr(ops, "rwkv7_decode", lambda *a: calls.append(native(*a)) or calls[-1])
    with torch.no_grad():
        got = RWKV7.forward(params, tok, state, length, ns)
        assert calls and calls[0] is not None                       # the native step took the call
        monkeypatch.setattr(ops, "rwkv7_decode", lambda *a: None)
        want = RWKV7.forward(params, tok, state, length, ns)
    close(got[0], want[0])
    close(got[1], want[1])
    close(got[1][:, :, :2], want[1][:, :, :2])


def test_general_path_with_and_without_state_copies(monkeypatch):
    """Where the native step does not take the call, the recurrence on the packed state in place equals the one on dense
    copies of its rows bit for bit."""
    from jaxrwkv_amd import ops
    from jaxrwkv_amd.model7 import RWKV7, randomize_weights
    from jaxrwkv_amd.rwkv7 import HipRWKV
    monkeypatch.setattr(ops, "rwkv7_decode", lambda *a: None)
    params = randomize_weights(4, 2, 128, 208, dtype=torch.bfloat16, device="cuda", zero_init=False)
    g = torch.Generator("cuda").manual_seed(4)
    tok = torch.randint(0, 208, (33, 3), device="cuda", generator=g)
    state = (0.1 * torch.randn((33, 2, 66, 128), device="cuda", generator=g)).bfloat16()

    class Dense:
        inner_loop = HipRWKV.inner_loop

    with torch.no_grad():
        a = RWKV7.forward(params, tok, state)
        monkeypatch.setattr(RWKV7, "inner", Dense)
        b = RWKV7.forward(params, tok, state)
    assert torch.equal(a[0], b[0]) and torch.equal(a[1], b[1])


def test_calls_that_the_native_step_does_not_cover():
    from jaxrwkv_amd import ops
    from jaxrwkv_amd.model7 import randomize_weights
    params = randomize_weights(1, 1, 128, 208, dtype=torch.bfloat16, device="cuda", zero_init=False)
    x = torch.zeros((257, 1, 128), device="cuda", dtype=torch.bfloat16)
    st = torch.zeros((257, 1, 66, 128), device="cuda", dtype=torch.bfloat16)
    assert ops.rwkv7_decode(params, x, st, None, None) is None                          # too many tokens
    assert ops.rwkv7_decode(params, x[:1].float(), st[:1], None, None) is None          # not bf16
    assert ops.rwkv7_decode(params, x[:2], st[:4:2], None, None) is None                # a state that is not contiguous
    params["blocks"]["att"]["w0"] = params["blocks"]["att"]["w0"].float()
    assert ops.rwkv7_decode(params, x[:1], st[:1], None, None) is None


@pytest.mark.parametrize("B,T,C", [(1, 1, 768), (2, 1, 1088), (1, 2, 2048), (1, 1, 4096), (1, 2, 64), (3, 1, 1024)])
def test_native_decode_step_of_few_rows(B, T, C, monkeypatch):
    """Norms inside the products and second low-rank products inside the recurrence: two tokens of a sequence and
    of two, widths from one step of a wave to several, inner sizes beyond one round of requests, one row too many."""
    test_native_decode_step(B, T, C, True, monkeypatch)


@pytest.mark.parametrize("name", ["w2", "a2", "g2", "v2"])
@pytest.mark.parametrize("value", [float("inf"), float("-inf")])
def test_few_rows_with_a_factor_that_is_not_finite(name, value, monkeypatch):
    """The last row of a second low-rank factor is what requests beyond it re-read: it is not part of other rows' sums."""
    from jaxrwkv_amd import ops
    from jaxrwkv_amd.model7 import RWKV7, randomize_weights
    params = randomize_weights(3, 2, 128, 208, dtype=torch.bfloat16, device="cuda", zero_init=False)
    params["blocks"]["att"][name][1, -1, 5] = value
    g = torch.Generator("cuda").manual_seed(3)
    state = (0.1 * torch.randn((1, 2, 66, 128), device="cuda", generator=g)).bfloat16()
    tok = torch.tensor([[7]], device="cuda")
    with torch.no_grad():
        got = RWKV7.forward(params, tok, state)
        monkeypatch.setattr(ops, "rwkv7_decode", lambda *a: None)
        want = RWKV7.forward(params, tok, state)
    for a, b in zip(got, want):
        assert torch.equal(torch.isfinite(a), torch.isfinite(b))


@pytest.mark.parametrize("B,T,C", [(250, 1, 320), (31, 8, 2112), (129, 1, 4096)])
def test_recurrence_of_several_sequences_a_workgroup(B, T, C, monkeypatch):
    """More heads than the GPU holds workgroups of: two to nine sequences one after the other, the last workgroup with fewer."""
    test_native_decode_step(B, T, C, True, monkeypatch)
