"""The WKV7 bf16 forward with its sequences cut into parts (few sequences and heads) against the oracle and against the same
kernel over the whole sequence, to which it falls back without a workspace.

The parts add one product per part in fp32 to the whole sequence's arithmetic; the operand rounding (fp16, 2^-11) is the same and
sets the error of both.  The bounds against the oracle are those of the whole sequence (test_gpu_wkv7_chunked); where the
state is carried over many parts (slow decay) the rms errors of the two are compared.  Measured against 64 bits at log decays of
-0.5, -2.5, -5 and -8 over five shapes of 700 to 4096 tokens, relative to the result: state 1.2e-4 / 2.1e-4 / 2.9e-4 / 3.7e-4 whole, in
parts 0.991 to 1.004 times that; y 1.66e-3 to 1.72e-3, the same to three digits.  A twentieth more is allowed."""
import numpy as np
import pytest
import torch

from oracle import wkv7 as o7
from tests.inputs import bf16_round, wkv7_inputs
from tests.test_gpu_wkv7_chunked import check, run

pytestmark = pytest.mark.gpu


def lib():
    from jaxrwkv_amd import _lib
    return _lib.load()


def split(B, T, H):
    return lib().hiprwkv_wkv7_fwd_workspace_bytes(1, B, T, H, 64) // (32768 + 32) // (B * H) + 1


def whole(monkeypatch, *a, **k):
    with monkeypatch.context() as m:
        m.setattr(lib(), "hiprwkv_wkv7_fwd_workspace_bytes", lambda *_: 0)
        return run(*a, **k)


@pytest.mark.parametrize("B,T,H,seed,p", [(1, 1000, 1, 0, 0.0), (1, 1009, 2, 1, 0.01), (2, 1025, 3, 2, 0.002), (3, 2047, 12, 3, 0.001)])
@pytest.mark.parametrize("compat", [True, False])
def test_against_the_oracle(B, T, H, seed, p, compat):
    P = split(B, T, H)
    assert P >= 2
    x = wkv7_inputs(B, T, H, 64, seed=seed, bf16=True, p_reset=p, min_len_frac=0.0)
    chunks = -(-(-(-T // 16)) // P)
    x["length"][0] = 16 * chunks                       # the last token of the first part
    x["new_starts"][-1, 16 * chunks] = True            # a reset at the first token of the second
    for want_sa in (False, True):
        check(x, compat, *run(x, compat, want_sa=want_sa))


@pytest.mark.parametrize("L", [0, 1, 15, 500, 1017])
def test_lengths(L):
    x = wkv7_inputs(1, 1017, 2, 64, seed=L, bf16=True, p_reset=0.003)
    x["length"][:] = L
    for compat in (True, False):
        check(x, compat, *run(x, compat))


def rms(a):
    return float(np.sqrt(np.mean(np.square(a))))


@pytest.mark.parametrize("decay", [-2.5, -5.0, -8.0])
@pytest.mark.parametrize("B,T,H", [(1, 2048, 2), (2, 1777, 12)])
def test_state_carried_over_the_parts(B, T, H, decay, monkeypatch):
    x = wkv7_inputs(B, T, H, 64, seed=5, bf16=True, resets=False)
    x["w"] = bf16_round(x["w"] + 0.5 + decay).astype(np.float64)
    ref = o7.wkv7_base(x["r"], x["w"], x["k"], x["v"], x["a"], x["b"], x["s"], x["length"], x["new_starts"], compat=True, return_sa=True)
    assert split(B, T, H) >= 2
    got, base = run(x, True), whole(monkeypatch, x, True)
    for g, w, e in zip(got, base, ref):
        assert rms(g - e) <= 1.05 * rms(w - e) + 1e-6 * rms(e)


def test_summaries_that_amplify_are_not_used(monkeypatch):
    """b = +0.03 a with a along one key for the second part's tokens, no decay to speak of: its state map grows by 1.03^160 = 100
    along that key.  The state entering that part is the first part's own, so the parts after it, which run its chunks again
    themselves, give the whole sequence's bits; with a summary that is used (the same without growth) the state's differ."""
    x = wkv7_inputs(1, 1200, 2, 64, seed=6, bf16=True, resets=False, lengths=False)
    P = split(1, 1200, 2)
    n = 16 * -(-75 // P)                                # tokens of a part
    assert P >= 4 and n >= 128
    x["w"][:] = -9.0
    for gain in (0.03, -0.03):
        x["a"][:, n:2 * n] = 0.0
        x["a"][:, n:2 * n, :, 5] = 1.0
        x["b"][:, n:2 * n] = bf16_round(gain * x["a"][:, n:2 * n])
        got, base = run(x, True), whole(monkeypatch, x, True)
        ref = o7.wkv7_base(x["r"], x["w"], x["k"], x["v"], x["a"], x["b"], x["s"], x["length"], x["new_starts"], compat=True, return_sa=True)
        assert np.array_equal(got[0], base[0]) == (gain > 0)
        for g, w, e in zip(got, base, ref):
            assert np.isfinite(g).all()
            assert np.array_equal(g, w) if gain > 0 else rms(g - e) <= 1.05 * rms(w - e) + 1e-6 * rms(e)
    big = wkv7_inputs(1, 1200, 1, 64, seed=7, bf16=True, resets=False, lengths=False)
    big["v"][:, 5] = 3e38                               # beyond the fp16 operands: the whole sequence turns non-finite, and so do the parts
    assert np.isnan(run(big, True)[0]).any() and np.isnan(whole(monkeypatch, big, True)[0]).any()


def test_numeric_events_are_those_of_the_whole_sequence(monkeypatch):
    """Every chunk and every carried state counts once, also where parts run the chunks before them again."""
    from jaxrwkv_amd import ops

    def events(x, f):
        before = ops.numeric_events()
        f(x, True)
        return ops.numeric_events() - before

    x = wkv7_inputs(1, 1200, 1, 64, seed=7, bf16=True, resets=False, lengths=False)
    x["w"][:, 700:716] = 3.0                            # e^-20 a token: a capped chunk
    capped = events(x, lambda *a: whole(monkeypatch, *a))
    assert split(1, 1200, 1) >= 4 and capped > 0 and events(x, run) == capped
    x["v"][:, 5] = 3e38                                 # no summary is usable, and the state turns non-finite
    both = events(x, lambda *a: whole(monkeypatch, *a))
    assert both > capped and events(x, run) == both


def test_a_broken_handshake_poisons_every_part(monkeypatch):
    from jaxrwkv_amd import _lib, ops
    monkeypatch.setenv("HIPRWKV_ENABLE_DEBUG_FLAGS", "1")
    x = wkv7_inputs(1, 1000, 1, 64, seed=8, bf16=True)
    from tests.gpu_util import dev
    t = [dev(x[n], torch.bfloat16) for n in ("r", "w", "k", "v", "a", "b")]
    try:
        new_s, y, sa = ops.wkv7_fwd(*t, dev(x["s"]), want_sa=True, debug_flags=0x100)
    except _lib.HipRwkvError:
        pytest.skip("the debug flag is read once per process and another test came first without it")
    assert torch.isnan(new_s).all() and torch.isnan(y).all() and torch.isnan(sa).all()
