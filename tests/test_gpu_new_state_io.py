"""HIPRWKV_NEW_STATE_IO: the forward kernels round the new state to the I/O type themselves.  The bits are those of the fp32 state rounded
afterwards, on every kernel that a call may take."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def operands(B, T, H, seed, n):
    g = torch.Generator("cuda").manual_seed(seed)
    tok = lambda: torch.randn((B, T, H, 64), device="cuda", generator=g).bfloat16()
    s = 0.1 * torch.randn((B, H, 64, 64), device="cuda", generator=g)
    length = torch.randint(0, T + 1, (B,), device="cuda", generator=g, dtype=torch.int32)
    ns = torch.rand((B, T), device="cuda", generator=g) < 0.05
    return [tok() for _ in range(n)], s, length, ns


# the small-T kernel, one chunk and a ragged one, a sequence in parts, more workgroups than CUs
SHAPES = [(3, 1, 2), (3, 8, 2), (2, 16, 1), (3, 41, 2), (1, 2047, 4), (33, 20, 8)]


@pytest.mark.parametrize("force_seq", [False, True])
@pytest.mark.parametrize("B,T,H", SHAPES)
def test_wkv7(B, T, H, force_seq):
    from jaxrwkv_amd import ops
    (r, w, k, v, a, b), s, length, ns = operands(B, T, H, T, 6)
    a = torch.nn.functional.normalize(a.float(), dim=-1).bfloat16()
    want, y = ops.wkv7(r, w, k, v, -a, 0.5 * a, s, length, ns, force_seq=force_seq)
    got, y2 = ops.wkv7(r, w, k, v, -a, 0.5 * a, s, length, ns, force_seq=force_seq, state_io=True)
    assert want.dtype == torch.float32 and got.dtype == torch.bfloat16
    assert torch.equal(got, want.bfloat16()) and torch.equal(y, y2)


@pytest.mark.parametrize("force_seq", [False, True])
@pytest.mark.parametrize("B,T,H", SHAPES)
def test_wkv6(B, T, H, force_seq):
    from jaxrwkv_amd import ops
    (r, k, v, w), s, length, ns = operands(B, T, H, T, 4)
    w, u = -torch.exp(w.float() - 0.5).bfloat16(), r[0, 0]
    want, y = ops.wkv6(r, k, v, w, u, s, length, ns, force_seq=force_seq)
    got, y2 = ops.wkv6(r, k, v, w, u, s, length, ns, force_seq=force_seq, state_io=True)
    assert want.dtype == torch.float32 and got.dtype == torch.bfloat16
    assert torch.equal(got, want.bfloat16()) and torch.equal(y, y2)


def test_other_types_are_as_before():
    """A wider I/O type than the state's, equal types, and a call with autograd: the state comes in its own type."""
    from jaxrwkv_amd import ops
    (r, w, k, v, a, b), s, length, ns = operands(2, 20, 2, 1, 6)
    args = (r, w, k, v, a, b)
    assert ops.wkv7(*(x.float() for x in args), s.bfloat16(), length, ns, state_io=True)[0].dtype == torch.bfloat16
    assert ops.wkv7(*args, s.bfloat16(), length, ns, state_io=True)[0].dtype == torch.bfloat16
    assert ops.wkv7(*(x.float() for x in args), s, length, ns, state_io=True)[0].dtype == torch.float32
    assert ops.wkv7(*args, s.requires_grad_(), length, ns, state_io=True)[0].dtype == torch.float32


def test_what_is_refused():
    from jaxrwkv_amd import _lib, ops
    lib = _lib.load()
    (r, w, k, v, a, b), s, length, ns = operands(1, 16, 1, 2, 6)
    p = [x.data_ptr() for x in (w, r, k, v, a, b)]
    y = torch.empty_like(r)
    stream = ops._stream()
    call = lambda new_s: lib.hiprwkv_wkv7_fwd_parts(stream, _lib.BF16, _lib.F32, 1, 16, 1, 64, *p, s.data_ptr(), None, None, y.data_ptr(),
                                                    None, new_s.data_ptr(), None, 0, _lib.NEW_STATE_IO)
    assert call(s) != 0                                  # one array of two types
    assert call(torch.empty_like(s)) == 0
    assert lib.hiprwkv_wkv7_step(stream, _lib.BF16, _lib.F32, 1, 1, 1, 64, *p, s.data_ptr(), 4096, None, None, y.data_ptr(),
                                 torch.empty_like(s).data_ptr(), 4096, _lib.NEW_STATE_IO) != 0
