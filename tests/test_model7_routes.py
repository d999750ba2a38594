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


def frozen(params, keep):
    """Only the parameters that ``keep`` names get a gradient; returns them."""
    out = {}
    for name, p in leaves(params):
        p.requires_grad_(bool(keep(name)))
        if keep(name):
            out[name] = p
    return out


KEEP = {"all but the embedding": lambda n: not n.startswith("emb"), "blocks": lambda n: n.startswith("blocks"),
        "one vector": lambda n: n == "blocks.att.w0", "ln0": lambda n: n.startswith("ln0"),
        "after the blocks": lambda n: n.split(".")[0] in ("ln_out", "head")}


@pytest.mark.parametrize("keep", list(KEEP))
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("T,B", [(1, 2), (3, 2), (8, 9), (20, 2)])
def test_every_trainable_parameter_gets_its_gradient(monkeypatch, T, B, dtype, keep):
    """Whatever is frozen: the derivative is asked for by any tensor that the results depend on, not by the embedding alone.  The
    new state is written whole on every route."""
    stub_library.install(monkeypatch)
    params = model(dtype)
    trainable = frozen(params, KEEP[keep])
    logits, new_state = call(params, T, B)
    assert not new_state.isnan().any() and not logits.isnan().any()
    assert logits.requires_grad
    if keep in ("all but the embedding", "blocks", "ln0"):
        assert new_state.requires_grad
    (logits.float().sum() + new_state.float().sum()).backward()
    # a first layer has no value residual, but later ones share the stacked parameter
    assert [n for n, p in trainable.items() if p.grad is None] == []


@pytest.mark.parametrize("T", [3, 20])
def test_frozen_embedding_with_another_recurrence(monkeypatch, T):
    from jaxrwkv_amd.model7 import RWKV7
    from jaxrwkv_amd.rwkv7 import HipRWKV
    stub_library.install(monkeypatch)

    class Own(HipRWKV):
        pass

    monkeypatch.setattr(RWKV7, "inner", Own)
    params = model(torch.bfloat16)
    trainable = frozen(params, KEEP["blocks"])
    logits, new_state = call(params, T)
    assert not new_state.isnan().any()
    (logits.float().sum() + new_state.float().sum()).backward()
    assert [n for n, p in trainable.items() if p.grad is None] == []


def test_no_derivative_no_graph(monkeypatch):
    """Training the head alone leaves the blocks on the inference route; without autograd decode steps are native."""
    from jaxrwkv_amd import blocks7, ops
    stub_library.install(monkeypatch)
    params = model(torch.bfloat16)
    frozen(params, KEEP["after the blocks"])
    kept = []
    run = blocks7._run
    monkeypatch.setattr(blocks7, "_run", lambda *a: kept.append(a[-1]) or run(*a))
    call(params, 20)
    assert kept == [None]
    native = []
    monkeypatch.setattr(ops, "rwkv7_decode", lambda *a: native.append(1) or ("logits", "state"))
    call(params, 1)
    assert not native
    with torch.no_grad():
        assert call(params, 1) == ("logits", "state")


def test_a_shift_row_is_not_dropped_under_autograd(monkeypatch):
    from jaxrwkv_amd import ops
    stub_library.install(monkeypatch)
    p = model(torch.float32)["blocks"]
    ln = {k: v[0].requires_grad_() for k, v in p["ln1"].items()}
    out = torch.zeros((2, C))
    with pytest.raises(ValueError):
        ops.rwkv7_ln_shiftmix(torch.randn(2, 3, C), None, ln, torch.zeros(2, C), None, None, [p["ffn"]["x_k"][0]], shift_out=out)


TANGENT = {"state": "state", "embedding": "emb.weight", "block": "blocks.att.x_r"}


@pytest.mark.parametrize("where", list(TANGENT))
@pytest.mark.parametrize("T", [1, 20])
@pytest.mark.parametrize("grad", [False, True])
def test_forward_mode_is_refused_and_not_dropped(monkeypatch, where, T, grad):
    """The recurrence has no forward-mode derivative: a tangent that reaches it is an error."""
    from torch.autograd import forward_ad
    stub_library.install(monkeypatch)
    params = model(torch.bfloat16)
    state = torch.zeros((2, L, 66, C), dtype=torch.bfloat16)
    with forward_ad.dual_level(), torch.set_grad_enabled(grad):
        dual = lambda t: forward_ad.make_dual(t, torch.ones_like(t))
        if where == "state":
            state = dual(state)
        elif where == "embedding":
            params["emb"]["weight"] = dual(params["emb"]["weight"])
        else:
            params["blocks"]["att"]["x_r"] = dual(params["blocks"]["att"]["x_r"])
        with pytest.raises(RuntimeError, match="jvp"):
            call(params, T, state=state)


@pytest.mark.parametrize("T", [1, 20])
def test_forward_mode_after_the_blocks(monkeypatch, T):
    """What follows the recurrence is torch's: its tangents are right."""
    from torch.autograd import forward_ad
    stub_library.install(monkeypatch)
    params = model(torch.float32)
    with forward_ad.dual_level():
        for name in ("ln_out", "head"):
            w = params[name]["weight"]
            params[name]["weight"] = forward_ad.make_dual(w, w)
        logits, _ = call(params, T)
        value, tangent = forward_ad.unpack_dual(logits)
    # logits are linear in head and in ln_out's weight (its bias is zero): each tangent is the value itself
    torch.testing.assert_close(tangent, 2 * value, rtol=1e-4, atol=1e-6)


@pytest.mark.parametrize("op", ["wkv4", "wkv6", "wkv7"])
def test_operators_refuse_tangents(monkeypatch, op):
    from torch.autograd import forward_ad
    from jaxrwkv_amd import ops
    stub_library.install(monkeypatch)
    tok = lambda: torch.randn(2, 20, 1, 64)
    args = {"wkv4": [torch.randn(64), torch.randn(64), torch.randn(2, 20, 64), torch.randn(2, 20, 64), torch.zeros(2, 3, 64)],
            "wkv6": [tok(), tok(), tok(), tok(), torch.randn(1, 64), torch.zeros(2, 1, 64, 64)],
            "wkv7": [tok() for _ in range(6)] + [torch.zeros(2, 1, 64, 64)]}[op]
    for i in range(len(args)):
        with forward_ad.dual_level():
            with pytest.raises(RuntimeError, match="jvp"):
                getattr(ops, op)(*args[:i], forward_ad.make_dual(args[i], torch.ones_like(args[i])), *args[i + 1:])


@pytest.mark.parametrize("T,grad", [(3, True), (20, False), (20, True)])
def test_state_in_another_memory_order(monkeypatch, T, grad):
    """A model state whose channels do not lie next to each other: every row of the new state is written, and nothing beside it.  The
    stub fills what a kernel is told to: C elements from the pointer on."""
    stub = stub_library.install(monkeypatch)
    params = model(torch.float32)
    state = torch.randn(2, L, C, 66).transpose(2, 3)
    if grad:
        frozen(params, KEEP["blocks"])
    seen = []
    call_ = stub_library.fill

    def fill(tensors):
        seen.extend(t for t in tensors if t.shape == (2, C))
        call_(tensors)

    monkeypatch.setattr(stub_library, "fill", fill)
    _, new_state = call(params, T, state=state)
    assert not new_state.isnan().any()
    assert seen and all(t.stride(1) == 1 for t in seen)          # shift rows: what the kernels take is a row of neighbours


@pytest.mark.parametrize("T", [3, 20])
def test_wide_models_keep_the_fused_steps(monkeypatch, T):
    """Channels that one workgroup of the fused head cannot span: norm and residual are torch's, everything else stays fused."""
    from jaxrwkv_amd import ops
    stub = stub_library.install(monkeypatch)
    monkeypatch.setattr(ops, "LN_SHIFTMIX_MAX_C", C - 8)
    with torch.no_grad():
        _, new_state = call(model(torch.bfloat16), T)
    assert not new_state.isnan().any()
    assert "hiprwkv_rwkv7_ln_shiftmix" not in stub.calls and "hiprwkv_gemm" not in stub.calls
    for name, n in (("shiftmix", 2 * L), ("pre", L), ("postmix", L), ("relusq", L)):
        assert stub.calls.count("hiprwkv_rwkv7_" + name) == n, name


@pytest.mark.parametrize("grad", [False, True])
@pytest.mark.parametrize("T", [1, 3, 20])
def test_a_subclass_with_mixing_methods_of_its_own(monkeypatch, T, grad):
    """They are called for every layer, with the norm's result and tensors for length and new_starts."""
    from jaxrwkv_amd.model7 import RWKV7
    stub_library.install(monkeypatch)
    seen = []

    class Model(RWKV7):
        @classmethod
        def time_mixing_seq(cls, x, shift_row, wkv_state, v_first, att, length, last_idx, new_starts, layer_id, wkv_out=None):
            assert v_first.shape == x.shape == (2, T, C) and length.shape == (2,) and new_starts.shape == (2, T)
            seen.append(("time", layer_id))
            out, *rest = super().time_mixing_seq(x, shift_row, wkv_state, v_first, att, length, last_idx, new_starts, layer_id, wkv_out)
            return (0 * out, *rest)

        @classmethod
        def channel_mixing_seq(cls, x, state_row, ffn, last_idx, new_starts):
            assert last_idx.tolist() == [T - 1] * 2
            seen.append(("channel", state_row.shape))
            return torch.ones_like(x), x[:, -1]

    params = model(torch.bfloat16)
    frozen(params, KEEP["all but the embedding"] if grad else (lambda n: False))
    tok = torch.arange(2 * T).reshape(2, T) % V
    logits, new_state = Model.forward(params, tok, RWKV7.default_state(params, 2))
    assert seen == [x for i in range(L) for x in (("time", i), ("channel", (2, C)))]
    assert not new_state.isnan().any() and logits.shape == (2, T, V)


def test_layer_of():
    from jaxrwkv_amd.model7 import layer_of, unstack
    params = model(torch.float32)["blocks"]
    for i, tree in enumerate(unstack(params, L)):
        for (n, a), (m, b) in zip(leaves(layer_of(params, i)), leaves(tree)):
            assert n == m and torch.equal(a, b)


@pytest.mark.parametrize("T", [3, 20])
def test_norms_held_in_fp32_stay_so(monkeypatch, T):
    """fp32 norms in a bf16 model: the fused head takes one type, and rounding the parameter to it would lose what the model has."""
    stub = stub_library.install(monkeypatch)
    params = model(torch.bfloat16)
    for ln in (params["ln0"], params["ln_out"], params["blocks"]["ln1"], params["blocks"]["ln2"]):
        for k in ln:
            ln[k] = ln[k].float()
    with torch.no_grad():
        call(params, T)
    assert "hiprwkv_rwkv7_ln_shiftmix" not in stub.calls and "hiprwkv_rwkv7_shiftmix" in stub.calls
    stub.calls.clear()
    params["ln_out"]["weight"] = params["ln_out"]["weight"].bfloat16()
    params["blocks"]["ln2"] = {k: v.bfloat16() for k, v in params["blocks"]["ln2"].items()}
    with torch.no_grad():
        call(params, T)                              # one norm's bias or one norm alone
    assert "hiprwkv_rwkv7_ln_shiftmix" not in stub.calls


@pytest.mark.parametrize("T", [3, 20])
@pytest.mark.parametrize("name", ["ln0", "ln1"])
def test_norms_anywhere_in_memory(monkeypatch, T, name):
    """A norm's parameter that does not lie on a 16-byte boundary (a slice of one flat array) is copied for the kernels."""
    from jaxrwkv_amd import blocks7
    stub_library.install(monkeypatch)
    monkeypatch.setattr(blocks7, "covers", lambda *a: False)
    params = model(torch.float32)
    tree = params if name == "ln0" else params["blocks"]
    w = tree[name]["weight"]
    tree[name]["weight"] = torch.cat([torch.zeros(1), w.flatten()])[1:].view(w.shape)
    from jaxrwkv_amd import ops
    seen = []
    fwd = ops._ln_shiftmix_fwd
    monkeypatch.setattr(ops, "_ln_shiftmix_fwd", lambda *a: seen.append(a[2].data_ptr() % 16 + a[3].data_ptr() % 16) or fwd(*a))
    with torch.no_grad():
        call(params, T)
    assert seen and not any(seen)


def _flat(w):
    return torch.cat([torch.zeros(1, dtype=w.dtype), w.flatten()])[1:].view(w.shape)


BAD = {"a vector of another size": ("x_k", lambda w: w[:, :32].contiguous()), "a factor of another size": ("w1", lambda w: w[:, :32].contiguous()),
       "a second factor of another size": ("g2", lambda w: w[:, :, :32].contiguous()),
       "one layer less": ("a0", lambda w: w[:1].contiguous()), "off a 16-byte boundary": ("v1", _flat),
       "a vector of another shape": ("x_v", lambda w: w.reshape(2 * L, -1)), "on another device": ("k_a", lambda w: w.to("meta"))}


@pytest.mark.parametrize("bad", list(BAD))
def test_the_stack_operator_takes_what_its_kernels_can_read(monkeypatch, bad):
    from jaxrwkv_amd import blocks7
    stub_library.install(monkeypatch)
    params = model(torch.bfloat16)
    x, state = torch.zeros((2, 20, C), dtype=torch.bfloat16), torch.zeros((2, L, 66, C), dtype=torch.bfloat16)
    assert blocks7.covers(blocks7.gather(params["blocks"]), x, state)
    name, change = BAD[bad]
    params["blocks"]["att"][name] = change(params["blocks"]["att"][name])
    assert not blocks7.covers(blocks7.gather(params["blocks"]), x, state)
    if bad == "a vector of another shape":                      # torch refuses it
        with pytest.raises(RuntimeError):
            call(params, 20)
    if bad == "off a 16-byte boundary":                         # torch's products take it
        with torch.no_grad():
            assert not call(params, 20)[1].isnan().any()


def test_fused_steps_look_at_their_operands(monkeypatch):
    from jaxrwkv_amd import ops
    stub_library.install(monkeypatch)
    n = lambda *s: torch.zeros(s)
    ln = {"weight": n(C), "bias": n(C)}
    head = lambda dx=n(2, 20, C), ns=None, length=None: ops.rwkv7_ln_shiftmix(n(2, 20, C), dx, ln, n(2, C), ns, length, [n(C)])
    head(ns=torch.zeros(20, dtype=torch.bool), length=3)        # broadcast over the batch as in the other operators
    for kw in (dict(dx=n(2, 19, C)), dict(ns=torch.zeros((2, 19), dtype=torch.bool)), dict(length=torch.ones(3))):
        with pytest.raises(AssertionError):
            head(**kw)
    tok, par = (n(2, 20, 1, 64) for _ in range(6)), [n(64) for _ in range(5)]
    tok = list(tok)
    ops.rwkv7_pre(*tok, *par)
    for i in range(6):
        with pytest.raises(AssertionError):
            ops.rwkv7_pre(*tok[:i], n(2, 19, 1, 64), *tok[i + 1:], *par)


@pytest.mark.parametrize("T", [3, 20])
def test_the_caller_may_reuse_length_before_the_backward(monkeypatch, T):
    stub_library.install(monkeypatch)
    params = model(torch.float32)
    frozen(params, KEEP["blocks"])
    length = torch.tensor([1, 2], dtype=torch.int32)
    logits, new_state = call(params, T, length=length)
    length.fill_(0)
    (logits.sum() + new_state.sum()).backward()


def _count_mm(monkeypatch):
    from jaxrwkv_amd import blocks7
    count, mm, gemm = [], torch.mm, blocks7._gemm
    monkeypatch.setattr(torch, "mm", lambda *a, **k: count.append(1) or mm(*a, **k))
    monkeypatch.setattr(blocks7, "_gemm", lambda jobs: count.extend(jobs) or gemm(jobs))
    return count


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_nothing_is_made_for_frozen_parameters(monkeypatch, dtype):
    """Products, cotangent arrays and saved activations follow what is trainable: the state alone, one vector, one matrix, all."""
    stub_library.install(monkeypatch)
    cost = {}
    subsets = {"state": lambda n: False, "vector": lambda n: n == "blocks.att.x_a", "matrix": lambda n: n == "blocks.ffn.key.weight",
               "all": lambda n: n.startswith("blocks")}
    for what, keep in subsets.items():
        with monkeypatch.context() as m:
            params = model(dtype)
            state = torch.zeros((2, L, 66, C), dtype=dtype).requires_grad_(what == "state")
            trainable = frozen(params, keep)
            saved = []
            with torch.autograd.graph.saved_tensors_hooks(lambda t: saved.append(t.numel()) or t, lambda t: t):
                logits, new_state = call(params, 20, state=state)
            made, like = [], torch.empty_like
            products = _count_mm(m)
            m.setattr(torch, "empty_like", lambda t, **k: made.append(tuple(t.shape)) or like(t, **k))
            ins = list(trainable.values()) or [state]
            grads = torch.autograd.grad((logits, new_state), ins, (torch.ones_like(logits), torch.ones_like(new_state)))
            assert not any(g.isnan().any() for g in grads)
            stacked = {tuple(p.shape) for _, p in leaves(params["blocks"])}
            cost[what] = (len(products), sum(saved), sum(s in stacked and len(s) == 3 for s in made))
    lora = 4 * L - 1 if dtype == torch.bfloat16 else 0             # the low-rank products are torch's own in fp32 (@, not counted)
    weights = 6 * L + 2 * lora
    assert cost["state"][0] == cost["vector"][0] == cost["all"][0] - weights - (2 * (4 * L - 1) if dtype == torch.float32 else 0)
    assert cost["matrix"][0] == cost["state"][0] + L
    assert cost["state"][1] < cost["all"][1] and cost["matrix"][1] < cost["all"][1]
    assert cost["state"][2] == cost["vector"][2] == 0 and cost["matrix"][2] <= 1


def test_native_step_leaves_a_state_elsewhere_alone(monkeypatch):
    """The native step takes the state by its pointer; a state on another device goes to the separate steps, which refuse it."""
    from jaxrwkv_amd import ops
    from jaxrwkv_amd.model7 import RWKV7
    stub_library.install(monkeypatch)
    params = model(torch.bfloat16)
    x, state = torch.zeros(2, 1, C, dtype=torch.bfloat16), RWKV7.default_state(params, 2)
    monkeypatch.setattr(ops, "_p", lambda t: None if t is None else t.data_ptr())
    monkeypatch.setattr(ops.ctypes, "byref", lambda a: torch.zeros(1, dtype=torch.bfloat16))
    assert ops.rwkv7_decode(params, x, state, None, None) is not None
    assert ops.rwkv7_decode(params, x, state.to("meta"), None, None) is None


@pytest.mark.parametrize("T", [3, 20])
def test_tokens_in_host_memory(monkeypatch, T):
    """Tokens may index the embedding from the host; ``length`` and ``new_starts`` go to the kernels' device all the same."""
    from jaxrwkv_amd import blocks7, ops
    from jaxrwkv_amd.model7 import tree_map
    stub_library.install(monkeypatch)
    got = []

    def route(*args):
        got.append([a.device.type for a in args if torch.is_tensor(a)])
        return (torch.zeros((2, T, C), dtype=torch.bfloat16, device="meta"),) * 3
    monkeypatch.setattr(ops, "autocast_elsewhere", lambda x: False)          # knows no such device
    monkeypatch.setattr(blocks7, "run", route)
    monkeypatch.setattr(ops, "rwkv7_decode", route)
    call(tree_map(lambda t: t.to("meta"), model(torch.bfloat16)), T, length=torch.tensor([2, 3]), new_starts=torch.zeros((2, T), dtype=torch.bool))
    assert got == [["meta"] * 4]


@pytest.mark.parametrize("C", [64, 4160])
@pytest.mark.parametrize("T", [3, 20])
def test_saved_tensors_may_come_back_in_another_memory_order(monkeypatch, T, C):
    """A saved-tensor hook gives the values back, not the strides: those of a state's row are not kept from the forward."""
    from jaxrwkv_amd.model7 import RWKV7, randomize_weights
    stub_library.install(monkeypatch)
    params = randomize_weights(1, 1, C, V, dtype=torch.float32, device="cpu", zero_init=False)
    for _, p in leaves(params):
        p.requires_grad_()
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t.detach().clone(memory_format=torch.contiguous_format), lambda t: t):
        logits, new_state = call(params, T)
    (logits.sum() + new_state.sum()).backward()


@pytest.mark.parametrize("T", [3, 20])
def test_one_layer_has_no_value_residual(monkeypatch, T):
    from jaxrwkv_amd.model7 import randomize_weights
    stub_library.install(monkeypatch)
    params = randomize_weights(1, 1, C, V, dtype=torch.bfloat16, device="cpu", zero_init=False)
    ps = {n: p.requires_grad_() for n, p in leaves(params)}
    logits, new_state = call(params, T)
    grads = torch.autograd.grad(logits.float().sum() + new_state.float().sum(), ps.values(), allow_unused=True)
    assert [n for n, g in zip(ps, grads) if g is None] == ["blocks.att.v0", "blocks.att.v1", "blocks.att.v2"]
