"""The failure path of the hand-shake where sequences run in parts: with HIPRWKV_DEBUG_DROP_PUBLISH no workgroup publishes its last chunk,
so every wait runs out, every wave ends normally, and NaN stands in every row that some workgroup owns, at the boundaries between
the parts too.  Summaries made by such a workgroup are not used."""
import os

import pytest
import torch

os.environ["HIPRWKV_ENABLE_DEBUG_FLAGS"] = "1"      # read at the first call that carries the flag

pytestmark = pytest.mark.gpu

# sweep A whole and in parts (bf16: by the rule for these sizes; fp32 runs it in parts at both)
SIZES = [(1, 500, 3), (2, 1000, 12)]


def inputs(B, T, H, dtype):
    g = torch.Generator("cuda").manual_seed(T)
    n = lambda *s: torch.randn(s, device="cuda", generator=g)
    r, k, v, dy = (n(B, T, H, 64).to(dtype) for _ in range(4))
    kap = torch.nn.functional.normalize(n(B, T, H, 64), dim=-1)
    w, a, b = (-0.5 + 0.5 * n(B, T, H, 64)).to(dtype), (-kap).to(dtype), (kap * torch.sigmoid(n(B, T, H, 64))).to(dtype)
    return (r, w, k, v, a, b, 0.1 * n(B, H, 64, 64), None, None), dy, n(B, H, 64, 64)


def parts_of(io, B, T, H):
    from jaxrwkv_amd import _lib
    return _lib.load().hiprwkv_wkv7_ends_bytes(io, B, T, H, 64) // (4096 * 4 * B * H) + 1


def all_nan(*tensors):
    return all(bool(torch.isnan(t.float()).all()) for t in tensors)


def finite(*tensors):
    return all(bool(torch.isfinite(t.float()).all()) for t in tensors)


@pytest.mark.parametrize("B,T,H", SIZES)
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_backward(B, T, H, dtype):
    from jaxrwkv_amd import _lib, ops
    args, dy, ds = inputs(B, T, H, dtype)
    n = parts_of(0 if dtype == torch.float32 else 1, B, T, H)
    assert n >= 2
    _, _, sa, ends = ops._wkv7_fwd(*args, want_sa=True, want_ends=True)
    good = ops.wkv7_bwd(*args, dy, sa, ds, ends=ends)
    before = ops.handshake_failures()
    bad = ops.wkv7_bwd(*args, dy, sa, ds, ends=ends, debug_flags=_lib.DEBUG_DROP_PUBLISH)
    # sweeps B and C a failure a part, sweep A one a sequence and head or, in parts, as many and those of the summaries
    assert ops.handshake_failures() - before >= B * H * (2 * n + 1)
    assert finite(*good) and all_nan(*bad)
    before = ops.handshake_failures()
    again = ops.wkv7_bwd(*args, dy, sa, ds, ends=ends)
    assert ops.handshake_failures() == before
    assert all(torch.equal(x, y) for x, y in zip(again, good))


@pytest.mark.parametrize("B,T,H", SIZES)
def test_forward_fp32_and_a_backward_from_its_boundaries(B, T, H):
    from jaxrwkv_amd import _lib, ops
    args, dy, ds = inputs(B, T, H, torch.float32)
    n = parts_of(0, B, T, H)
    step = 16 * -(-(-(-T // 16)) // n)                       # tokens of a part
    good = ops._wkv7_fwd(*args, want_sa=True, want_ends=True)
    before = ops.handshake_failures()
    bad = ops._wkv7_fwd(*args, want_sa=True, want_ends=True, debug_flags=_lib.DEBUG_DROP_PUBLISH)
    assert ops.handshake_failures() - before >= B * H
    assert all_nan(*bad[:3]) and all_nan(bad[3].view(torch.float32)) and finite(good[3].view(torch.float32))
    # every part but the first starts from such a state, and the decay's cotangents of every part but the last from its carry
    gr, gw, gk, gv, ga, gb, gs = ops.wkv7_bwd(*args, dy, good[2], ds, ends=bad[3])
    assert all_nan(gr[:, step:], ga[:, step:], gw[:, :step * (n - 1)])
    assert finite(gr[:, :step], ga[:, :step], gk, gv, gb, gs)
    # an unreadable residual (a forward that failed) leaves nothing but the first token's da, which the given state makes
    gr, gw, gk, gv, ga, gb, gs = ops.wkv7_bwd(*args, dy, bad[2], ds, ends=bad[3])
    assert all_nan(gr, ga[:, 1:], gw)


def test_backward_bf16_of_a_failed_forward():
    """Its residual is NaN, and with it the records that the parts start from."""
    from jaxrwkv_amd import _lib, ops
    args, dy, ds = inputs(1, 500, 3, torch.bfloat16)
    bad = ops._wkv7_fwd(*args, want_sa=True, want_ends=True, debug_flags=_lib.DEBUG_DROP_PUBLISH)
    assert all_nan(*bad[:3])
    gr, gw, gk, gv, ga, gb, gs = ops.wkv7_bwd(*args, dy, bad[2], ds, ends=bad[3])
    assert all_nan(gr, ga[:, 1:], gw)
