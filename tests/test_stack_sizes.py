"""What the native stack keeps and borrows, by the library's own size functions (no GPU needed): arrays that nothing reads are not held."""
import ctypes

import pytest

B, T, L, C, F, D = 2, 1024, 6, 1024, 4096, (64, 64, 32, 160)
N = B * T * C * 2                                  # a (rows, C) array
SLACK = 64 * 2048                                  # arrays start on 1 KiB boundaries and up to 896 bytes past them


def args(L=L, saved=False):
    from jaxrwkv_amd import _lib
    A = _lib.Rwkv7StackArgs(B=B, T=T, L=L, C=C, H=C // 64, F=F, d_decay=D[0], d_aaa=D[1], d_mv=D[2], d_gate=D[3])
    A.saved = 16 if saved else None                # looked at as a flag
    return _lib.load(), A


def test_forward_without_a_backward():
    """The stream twice, six interpolations, r k v, the gate, w k a b v, the recurrence's and the group norm's results, the
    channel mix's input, the first layer's v and a product's result: 22; of the low-rank terms the gate alone is read again."""
    lib, A = args()
    own = lib.hiprwkv_wkv7_fwd_workspace_bytes(1, B, T, C // 64, 64)
    got = lib.hiprwkv_rwkv7_stack_workspace_bytes(ctypes.byref(A), 0)
    assert 22 * N < got - own <= 22 * N + B * T * (F + sum(D)) * 2 + SLACK


def test_backward():
    """17 arrays of the rows, three low-rank cotangents and the recurrence's state beside gff, whose memory gy and gyw use
    again, as the six interpolations' cotangents use the recurrence's."""
    lib, A = args(saved=True)
    H = C // 64
    own = lib.hiprwkv_wkv7_bwd_ends_workspace_bytes(1, B, T, H, 64) + lib.hiprwkv_wkv7_ends_bytes(1, B, T, H, 64)
    sums = max(lib.hiprwkv_rwkv7_ln_shiftmix_bwd_workspace_bytes(B, T, C, 6), lib.hiprwkv_rwkv7_postmix_bwd2_workspace_bytes(B * T, H, 64),
               lib.hiprwkv_rwkv7_pre_bwd_workspace_bytes(B * T, H, 64))
    got = lib.hiprwkv_rwkv7_stack_workspace_bytes(ctypes.byref(A), 1)
    assert 20 * N < got - own - sums <= 20 * N + (B * T * (F + sum(D)) + B * C * 64) * 2 + SLACK


@pytest.mark.parametrize("layers", [1, 2, 3, 6])
def test_layers(layers):
    """The first layer reads the call's x and has no value residual, the last one's result is the call's."""
    lib, A = args(layers, saved=True)
    size = [lib.hiprwkv_rwkv7_stack_saved_layer_bytes(ctypes.byref(A), i) for i in range(layers)]
    assert lib.hiprwkv_rwkv7_stack_saved_bytes(ctypes.byref(A)) == max(size)
    if layers > 2:
        whole, hid = size[1], B * T * D[2] * 2
        assert size[1:-1] == [whole] * (layers - 2)
        assert whole <= 24 * N + B * T * (2 * F + sum(D)) * 2 + 16 * B * T + SLACK      # and no array of the recurrence's parts
        assert abs(whole - size[0] - 3 * N - hid) <= SLACK and abs(whole - size[-1] - N) <= SLACK
    assert lib.hiprwkv_rwkv7_stack_saved_layer_bytes(ctypes.byref(A), layers) == 0 == lib.hiprwkv_rwkv7_stack_saved_layer_bytes(ctypes.byref(A), -1)
