"""What is timed: the calls that a program built on this package makes, over the range of sizes it makes them at.

Two kinds of user are behind the cases.  One plugs ``HipRWKV.inner_loop`` into a model of their own (the op cases:
inference over whole sequences, and training steps that return every cotangent).  The other runs the RWKV-7 model through
``RWKV7.forward`` (prompts, decode steps, training steps).  Sizes are the benchmark's and the tests' shapes (the 0.1B
shape: 12 layers, 768 channels; the 1.5B shape: 24 layers, 2048 channels; the op shapes of ``bench.py``) and ordinary ones
between and below them, ragged lengths and resets included.
"""
import math

import torch

from jaxrwkv_amd import rwkv4, rwkv6, rwkv7
from jaxrwkv_amd.model7 import RWKV7

N = 64                       # head size of every RWKV-6 / RWKV-7 model
VOCAB = 65536
DTYPES = {"bf16": torch.bfloat16, "fp32": torch.float32}
MODEL_SHAPES = ((12, 768), (24, 1024), (24, 2048))          # inference
TRAIN_SHAPES = ((12, 768), (8, 1024), (6, 512))


def _op(name, kind, B, T, H, io, p_reset):
    return {"name": name, "kind": kind, "B": B, "T": T, "H": H, "io": io, "p_reset": p_reset}


def _model(name, kind, L, C, B, T, p_reset):
    return {"name": name, "kind": kind, "L": L, "C": C, "B": B, "T": T, "p_reset": p_reset}


def listed():
    return [
        # the op inside a large batched forward pass: packed documents (resets), ragged lengths
        _op("wkv7_fwd_large", "wkv7_fwd", 8, 4096, 32, "bf16", 1 / 1024),
        # the same in a training step: y and the state's cotangents go in, all seven cotangents come out
        _op("wkv7_train_large", "wkv7_train", 8, 4096, 32, "bf16", 1 / 1024),
        # one user's prompt, one layer of a 2048-channel model: a single long sequence of odd length, 32 heads
        _op("wkv7_fwd_prompt", "wkv7_fwd", 1, 2047, 32, "bf16", 0.0),
        # fine-tuning a small model in fp32: few sequences of odd length
        _op("wkv7_train_fp32", "wkv7_train", 3, 777, 12, "fp32", 1 / 256),
        # RWKV-6 training step over packed documents
        _op("wkv6_train_large", "wkv6_train", 16, 2048, 32, "bf16", 1 / 512),
        # RWKV-6 over a few prompts of odd length
        _op("wkv6_fwd_prompts", "wkv6_fwd", 3, 1001, 12, "bf16", 0.0),
        # RWKV-4 inference over a large batch of ragged sequences, 2560 channels
        {"name": "wkv4_fwd_large", "kind": "wkv4_fwd", "B": 32, "T": 4096, "C": 2560, "io": "fp32", "p_reset": 0.0},
        # RWKV-4 training step of a small model
        {"name": "wkv4_train_small", "kind": "wkv4_train", "B": 4, "T": 1000, "C": 768, "io": "bf16", "p_reset": 1 / 512},
        # chat with the 0.1B shape: one token for one user, all latency
        _model("model_decode_one", "model_fwd", 12, 768, 1, 1, 0.0),
        # serving the 1.5B shape: one token for each of 256 users
        _model("model_decode_256", "model_fwd", 24, 2048, 256, 1, 0.0),
        # serving the 1.5B shape: four prompts of different lengths
        _model("model_prefill", "model_fwd", 24, 2048, 4, 1021, 0.0),
        # a training step of the 0.1B shape: forward and every parameter's gradient
        _model("model_train", "model_train", 12, 768, 4, 512, 1 / 512),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["wkv7_fwd", "wkv7_train", "wkv6_fwd", "wkv6_train", "wkv4_fwd", "wkv4_train", "model_decode",
                       "model_prefill", "model_train"])
    p_reset = rng.choice([0.0, 1 / 1024, 1 / 128])
    if kind in ("wkv7_fwd", "wkv7_train", "wkv6_fwd", "wkv6_train"):
        io = rng.choice(["bf16", "bf16", "bf16", "fp32"])
        H = rng.choice([12, 16, 32])
        B = _log_int(rng, 1, 16)
        # no larger than the listed case of its kind; fp32 rows are twice as long and the fp32 kernels twice as slow
        tokens = 8 * 4096 * 32 // H // B // (2 if io == "fp32" else 1)
        T = _log_int(rng, 16, min(4096, tokens))
        return {"kind": kind, "B": B, "T": T, "H": H, "io": io, "p_reset": p_reset}
    if kind in ("wkv4_fwd", "wkv4_train"):
        C = rng.choice([512, 768, 1024, 2560])
        B = _log_int(rng, 1, 32 if kind == "wkv4_fwd" else 8)
        T = _log_int(rng, 16, 4096)
        return {"kind": kind, "B": B, "T": T, "C": C, "io": rng.choice(["bf16", "fp32"]), "p_reset": p_reset}
    if kind == "model_decode":
        L, C = rng.choice(MODEL_SHAPES)
        return {"kind": "model_fwd", "L": L, "C": C, "B": _log_int(rng, 1, 256), "T": 1, "p_reset": 0.0}
    if kind == "model_prefill":
        L, C = rng.choice(MODEL_SHAPES)
        B = _log_int(rng, 1, 8)
        return {"kind": "model_fwd", "L": L, "C": C, "B": B, "T": _log_int(rng, 16, 4 * 1021 // B), "p_reset": p_reset}
    L, C = rng.choice(TRAIN_SHAPES)
    B = _log_int(rng, 1, 4)
    return {"kind": "model_train", "L": L, "C": C, "B": B, "T": _log_int(rng, 16, 2048 // B), "p_reset": p_reset}


# ------------------------------------------------------------------------------------------------------- inputs
class _Gen:
    """Draws on the GPU from one seed."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda")
        self.g.manual_seed(seed)

    def normal(self, *shape, mean=0.0, std=1.0, dtype=torch.float32):
        return (mean + std * torch.randn(shape, generator=self.g, device="cuda", dtype=torch.float32)).to(dtype)

    def lengths(self, lo, hi, B):
        return torch.randint(lo, hi + 1, (B,), generator=self.g, device="cuda", dtype=torch.int32)

    def resets(self, B, T, p):
        return torch.rand((B, T), generator=self.g, device="cuda") < p


def _prepare_op(case, g):
    B, T = case["B"], case["T"]
    io = DTYPES[case["io"]]
    train = case["kind"].endswith("_train")
    length = g.lengths(max(1, T // 2), T, B) if B > 1 else torch.full((B,), T, dtype=torch.int32, device="cuda")
    new_starts = g.resets(B, T, case["p_reset"])
    if case["kind"].startswith("wkv4"):
        C = case["C"]
        fn = rwkv4.HipRWKV.inner_loop
        s = torch.zeros((B, 3, C), dtype=io, device="cuda")
        s[:, 2] = -1e38                                        # the state before the first token
        args = [g.normal(B, T, C, dtype=io).sigmoid(), g.normal(B, T, C, dtype=io), g.normal(B, T, C, dtype=io),
                g.normal(C, dtype=io), g.normal(C, std=0.5, dtype=io), s]          # r, k, v, w, time_first, s
        cot = [g.normal(B, T, C, dtype=io)] if train else []
    else:
        H = case["H"]
        tok = lambda **kw: g.normal(B, T, H, N, dtype=io, **kw)
        s = g.normal(B, H, N, N, std=0.1)
        if case["kind"].startswith("wkv7"):
            fn = rwkv7.HipRWKV.inner_loop
            kappa = torch.nn.functional.normalize(g.normal(B, T, H, N), dim=-1)
            b = (kappa * g.normal(B, T, H, N).sigmoid()).to(io)
            args = [tok(), tok(mean=-0.5, std=0.5), tok(), tok(), (-kappa).to(io), b, s]    # r, w, k, v, a, b, s
            del kappa
        else:
            fn = rwkv6.HipRWKV.inner_loop
            w = -torch.exp(g.normal(B, T, H, N, mean=-0.5, std=0.5))
            args = [tok(), tok(), tok(), w.to(io), g.normal(H, N, std=0.5, dtype=io), s]    # r, k, v, w, u, s
            del w
        cot = [g.normal(B, H, N, N, dtype=io), tok()] if train else []
    if train:
        leaves = args if not case["kind"].startswith("wkv4") else args[:5]
        for x in leaves:
            x.requires_grad_()
    else:
        leaves = []
    return {"case": case, "fn": fn, "args": args, "leaves": leaves, "cot": cot, "length": length, "new_starts": new_starts}


def _model_weights(L, C, g):
    """A parameter tree with the names and shapes of the RWKV-7 model and the sizes that trained weights have:
    matrices that keep a normalised input's size, mixing vectors in [0, 1], decays from slow to fast over a head."""
    bf = torch.bfloat16
    H = C // N
    mat = lambda rows, cols, gain: g.normal(L, rows, cols, std=gain / math.sqrt(cols), dtype=bf)       # used as x @ W.T
    lora = lambda rows, cols, gain: g.normal(L, rows, cols, std=gain / math.sqrt(rows), dtype=bf)      # used as x @ W
    residual = 0.5 / math.sqrt(2 * L)                          # each block adds a small part to the residual stream
    unit = lambda: torch.rand((L, C), generator=g.g, device="cuda").to(bf)
    norm = lambda *shape: {"weight": g.normal(*shape, mean=1.0, std=0.1, dtype=bf), "bias": g.normal(*shape, std=0.02, dtype=bf)}
    rank = lambda scale, power: max(32, int(round(scale * C ** power / 32) * 32))
    d_decay, d_mv, d_gate = rank(1.8, 0.5), rank(1.3, 0.5), rank(0.6, 0.8)
    att = {n: unit() for n in ("x_r", "x_w", "x_k", "x_v", "x_a", "x_g")}
    att.update(
        w0=(-6.0 + 6.0 * torch.rand((L, C), generator=g.g, device="cuda") ** 1.5).to(bf), w1=lora(C, d_decay, 0.5),
        w2=lora(d_decay, C, 0.5), a0=g.normal(L, C, std=0.3, dtype=bf), a1=lora(C, d_decay, 0.5), a2=lora(d_decay, C, 0.5),
        v0=g.normal(L, C, mean=0.7, std=0.2, dtype=bf), v1=lora(C, d_mv, 0.5), v2=lora(d_mv, C, 0.5),
        g1=lora(C, d_gate, 1.0), g2=lora(d_gate, C, 1.0), k_k=g.normal(L, C, mean=0.7, std=0.05, dtype=bf),
        k_a=g.normal(L, C, mean=1.0, std=0.05, dtype=bf), r_k=g.normal(L, H, N, std=0.1, dtype=bf),
        receptance={"weight": mat(C, C, 0.7)}, key={"weight": mat(C, C, 0.7)}, value={"weight": mat(C, C, 0.7)},
        output={"weight": mat(C, C, residual)}, ln_x=norm(L, C))
    ffn = {"x_k": unit(), "key": {"weight": mat(4 * C, C, 0.7)}, "value": {"weight": mat(C, 4 * C, residual)}}
    return {"blocks": {"att": att, "ffn": ffn, "ln1": norm(L, C), "ln2": norm(L, C)},
            "emb": {"weight": g.normal(VOCAB, C, std=0.5, dtype=bf)},
            "head": {"weight": g.normal(VOCAB, C, std=1.0 / math.sqrt(C), dtype=bf)}, "ln0": norm(C), "ln_out": norm(C)}


def _leaves(tree):
    for v in tree.values():
        if isinstance(v, dict):
            yield from _leaves(v)
        else:
            yield v


def _prepare_model(case, g):
    B, T = case["B"], case["T"]
    params = _model_weights(case["L"], case["C"], g)
    state = RWKV7.default_state(params, B)
    tokens = torch.randint(0, VOCAB, (B, T), generator=g.g, device="cuda")
    st = {"case": case, "params": params, "tokens": tokens, "state": state, "leaves": [], "cot": None, "length": None,
          "new_starts": None}
    if case["kind"] == "model_train":
        st["leaves"] = [p.requires_grad_() for p in _leaves(params)]
        # the loss is the caller's own; its gradient with respect to the logits is what reaches the model
        st["cot"] = g.normal(B, T, VOCAB, std=1.0 / (B * T), dtype=torch.bfloat16)
        st["new_starts"] = g.resets(B, T, case["p_reset"])
    elif T == 1:
        state.copy_(g.normal(*state.shape, std=0.3, dtype=torch.bfloat16))          # users in mid-conversation
    else:
        st["length"] = g.lengths(max(1, T // 2), T, B) if B > 1 else None
        st["new_starts"] = g.resets(B, T, case["p_reset"]) if case["p_reset"] else None
    return st


def prepare(case, seed):
    g = _Gen(seed)
    return _prepare_model(case, g) if case["kind"].startswith("model") else _prepare_op(case, g)


# --------------------------------------------------------------------------------------------------------- pass
def run(state):
    kind = state["case"]["kind"]
    if kind == "model_fwd":
        with torch.no_grad():
            return RWKV7.forward(state["params"], state["tokens"], state["state"], length=state["length"],
                                 new_starts=state["new_starts"])
    if kind == "model_train":
        logits, new_state = RWKV7.forward(state["params"], state["tokens"], state["state"], length=state["length"],
                                          new_starts=state["new_starts"])
        grads = torch.autograd.grad(logits, state["leaves"], state["cot"], allow_unused=True)
        return [logits.detach(), new_state.detach()] + [x for x in grads if x is not None]
    new_s, y = state["fn"](*state["args"], state["length"], state["new_starts"])
    if kind.endswith("_fwd"):
        return new_s, y
    outs = (y,) if kind == "wkv4_train" else (new_s, y)
    return [new_s.detach(), y.detach()] + list(torch.autograd.grad(outs, state["leaves"], state["cot"]))


# --------------------------------------------------------------------------------------- what a pass cannot do without
def _model_params(L, C):
    rank = lambda scale, power: max(32, int(round(scale * C ** power / 32) * 32))
    lora = 2 * C * (2 * rank(1.8, 0.5) + rank(1.3, 0.5) + rank(0.6, 0.8))
    return L * (4 * C * C + 8 * C * C + lora + 20 * C)


def work(case):
    B, T, kind = case["B"], case["T"], case["kind"]
    if kind.startswith("model"):
        L, C = case["L"], case["C"]
        body, head = _model_params(L, C), VOCAB * C
        tok = B * T
        state = 2 * B * L * (2 + N) * C * 2
        wkv = 9 * N * C * tok * L                                  # the recurrence's own multiply-adds, per channel
        flops = 2 * tok * (body + head) + wkv
        bytes_ = 2 * (body + head) + 2 * tok * C + state + 2 * tok * VOCAB
        if kind == "model_train":
            flops, bytes_ = 3 * flops, 2 * bytes_ + 2 * (body + 2 * head)
        return {"bytes": float(bytes_), "flops": float(flops)}
    e = 2 if case["io"] == "bf16" else 4
    if kind.startswith("wkv4"):
        n = B * T * case["C"]
        if kind == "wkv4_fwd":                                     # r, k, v -> out
            return {"bytes": float(4 * n * e), "flops": float(12 * n)}
        return {"bytes": float((4 + 4 + 3) * n * e), "flops": float(40 * n)}      # and r, k, v, gy -> gr, gk, gv
    rows = B * T * case["H"]
    state = B * case["H"] * N * N
    if kind == "wkv7_fwd":
        return {"bytes": float(7 * rows * N * e + state * (4 + e)), "flops": float(9 * N * N * rows)}
    if kind == "wkv7_train":                                       # 6 + 7 inputs, 1 + 6 outputs
        return {"bytes": float(20 * rows * N * e + state * (12 + 2 * e)), "flops": float(27 * N * N * rows)}
    if kind == "wkv6_fwd":
        return {"bytes": float(5 * rows * N * e + state * (4 + e)), "flops": float(5 * N * N * rows)}
    return {"bytes": float(14 * rows * N * e + state * (12 + 2 * e)), "flops": float(15 * N * N * rows)}


def tolerance(case):
    """Four times the differences measured between two formulations of the same pass: the model with fused and with
    separate element-wise steps (logits and state 1e-2; gradients, the worst parameter, 3.5e-2, where twice that is
    stated because separate steps round more often), the op on the matrix cores and on the vector units (bf16 1.3e-3,
    fp32 4.8e-6), RWKV-4 with bf16 and with fp32 inputs of the same values (3.9e-3)."""
    if case["kind"] == "model_train":
        return {"rel": 8e-2}
    if case["kind"] == "model_fwd":
        return {"rel": 4e-2}
    if case["io"] == "fp32":
        return {"rel": 2e-5}
    return {"rel": 1.5e-2 if case["kind"].startswith("wkv4") else 6e-3}
