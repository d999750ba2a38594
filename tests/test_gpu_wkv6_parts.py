"""The WKV6 bf16 forward with its sequences cut into parts (few sequences and heads) against the oracle and against the same
kernel over the whole sequence, to which it falls back without a workspace.

The chunks and their operands are the whole sequence's; a part adds one fp32 multiply-add per state element.  The bounds against
the oracle are those of the whole sequence (test_gpu_wkv6_chunked); the rms errors of the two are compared as well: the same
fp16 roundings of a state that differs by a few 2^-24.  Measured against 64 bits over three shapes and log decays of 1, 2^-6, 2^-10 and 0
times the usual: state 0.9e-4 / 2.0e-4 / 2.0e-4 / 2e-7 relative to the result, y 1.66e-3 to 1.70e-3, in parts the same to three digits (without
decay 0.5 to 0.7 times the state's).  A twentieth more is allowed."""
import numpy as np
import pytest
import torch

from oracle import wkv6 as o6
from tests.gpu_util import dev
from tests.inputs import bf16_round, wkv6_inputs
from tests.test_gpu_wkv6_chunked import check, run

pytestmark = pytest.mark.gpu


def lib():
    from jaxrwkv_amd import _lib
    return _lib.load()


def split(B, T, H):
    return lib().hiprwkv_wkv6_fwd_workspace_bytes(1, B, T, H, 64) // (16384 + 272) // (B * H) + 1


def whole(monkeypatch, *a, **k):
    with monkeypatch.context() as m:
        m.setattr(lib(), "hiprwkv_wkv6_fwd_workspace_bytes", lambda *_: 0)
        return run(*a, **k)


def rms(a):
    return float(np.sqrt(np.mean(np.square(a))))


@pytest.mark.parametrize("B,T,H,seed,p", [(1, 1000, 1, 0, 0.0), (1, 1009, 2, 1, 0.01), (2, 1025, 3, 2, 0.002), (3, 2047, 12, 3, 0.001)])
@pytest.mark.parametrize("compat", [True, False])
@pytest.mark.parametrize("state_dtype", [torch.float32, torch.bfloat16])
def test_against_the_oracle(B, T, H, seed, p, compat, state_dtype):
    P = split(B, T, H)
    assert P >= 2
    x = wkv6_inputs(B, T, H, 64, seed=seed, bf16=True, p_reset=p)
    chunks = -(-(-(-T // 16)) // P)
    x["length"][0] = 16 * chunks                       # the last token of the first part
    x["new_starts"][-1, 16 * chunks] = True            # a reset at the first token of the second
    if state_dtype == torch.bfloat16:
        x["s"] = bf16_round(x["s"])
        ref_s, ref_y = o6.wkv6_base(*(x[n] for n in ("r", "k", "v", "w", "u", "s", "length", "new_starts")), compat=compat)
        new_s, y = run(x, compat, state_dtype)
        assert (np.abs(new_s - ref_s) <= 2.0 ** -7 * np.abs(ref_s) + 2e-3 * rms(ref_s)).all()
    else:
        check(x, compat, *run(x, compat))


@pytest.mark.parametrize("L", [0, 1, 15, 500, 1017])
def test_lengths(L):
    x = wkv6_inputs(1, 1017, 2, 64, seed=L, bf16=True, p_reset=0.003)
    x["length"][:] = L
    for compat in (True, False):
        check(x, compat, *run(x, compat))


@pytest.mark.parametrize("decay", [1.0, 2.0 ** -6, 2.0 ** -10, 0.0])
@pytest.mark.parametrize("B,T,H", [(1, 2048, 2), (2, 1777, 12)])
def test_state_carried_over_the_parts(B, T, H, decay, monkeypatch):
    x = wkv6_inputs(B, T, H, 64, seed=5, bf16=True, resets=False)
    x["w"] = x["w"] * decay
    ref = o6.wkv6_base(*(x[n] for n in ("r", "k", "v", "w", "u", "s", "length", "new_starts")), compat=True)
    assert split(B, T, H) >= 2
    got, base = run(x, True), whole(monkeypatch, x, True)
    for g, w, e in zip(got, base, ref):
        assert rms(g - e) <= 1.05 * rms(w - e) + 1e-6 * rms(e)


def test_one_decay_for_all_tokens(monkeypatch):
    from jaxrwkv_amd import ops
    x = wkv6_inputs(1, 1200, 2, 64, seed=9, bf16=True, p_reset=0.002)
    t = [dev(x[n], torch.bfloat16) for n in ("r", "k", "v")]
    w, u, s = dev(x["w"][0, 0], torch.bfloat16), dev(x["u"], torch.bfloat16), dev(x["s"])
    ns = dev(x["new_starts"])
    a = ops.wkv6_fwd(*t, w, u, s, None, ns)
    b = ops.wkv6_fwd(*t, w.expand(1, 1200, 2, 64).contiguous(), u, s, None, ns)
    assert all(torch.equal(p, q) for p, q in zip(a, b))


def test_values_that_are_not_finite_end_at_a_reset(monkeypatch):
    x = wkv6_inputs(1, 1200, 1, 64, seed=7, bf16=True, resets=False, lengths=False)
    x["v"][:, 5] = 3e38
    x["new_starts"][:, 700] = True
    got, base = run(x, True), whole(monkeypatch, x, True)
    for g, w in zip(got, base):
        assert (np.isfinite(g) == np.isfinite(w)).all()
    # to the end of the reset's chunk (zeroed operands times NaN), as in the whole sequence
    assert not np.isfinite(got[1][:, 5:700]).all() and np.isfinite(got[1][:, 704:]).all() and np.isfinite(got[0]).all()
    # a growing decay of a state that stays zero: no inf * 0.  A chunk's exp(8) |r| stays inside fp16, a part's exp(128) beyond fp32
    z = wkv6_inputs(1, 2047, 32, 64, seed=8, bf16=True, resets=False, lengths=False)
    assert split(1, 2047, 32) == 8
    z["k"][..., 3] = 0.0
    z["s"][:, :, 3] = 0.0
    z["w"][..., 3] = 0.5
    got, base = run(z, True), whole(monkeypatch, z, True)
    for g, w in zip(got, base):
        assert np.isfinite(w).all() and np.isfinite(g).all()
