"""Error returns of the entry points with boundaries, of the low-rank products with the gates and of the stack: refused before a launch
(made-up addresses, no GPU)."""
import ctypes

import pytest

OK, BAD, NULL = 0x10000, 0x10008, None
B, T, H = 1, 1000, 2
FORCE_SEQ = 2


def lib():
    from jaxrwkv_amd import _lib
    assert _lib.FORCE_SEQ == FORCE_SEQ
    return _lib.load()


def refused(rc, code, text):
    assert rc == code and text in lib().hiprwkv_last_error(), (rc, lib().hiprwkv_last_error())


def fwd(io=1, sa=OK, ends=OK, ws=NULL, nbytes=0, flags=0, first=OK):
    return lib().hiprwkv_wkv7_fwd_ends(NULL, io, 0, B, T, H, 64, first, OK, OK, OK, OK, OK, OK, NULL, NULL, OK, sa, OK, ends, ws, nbytes, flags)


def bwd(io=1, ends=OK, ws=OK, nbytes=0, flags=0, first=OK):
    return lib().hiprwkv_wkv7_bwd_ends(NULL, io, 0, B, T, H, 64, first, *[OK] * 6, NULL, NULL, OK, OK, NULL, ends, *[OK] * 7, ws, nbytes, flags)


@pytest.mark.parametrize("io", [0, 1])
def test_boundaries(io):
    n = lib().hiprwkv_wkv7_ends_bytes(io, B, T, H, 64)
    assert n > 0 and lib().hiprwkv_wkv7_ends_bytes(io, B, 8, H, 64) == 0 == lib().hiprwkv_wkv7_ends_bytes(io, B, T, H, 32)
    for kw in (dict(ends=BAD), dict(sa=NULL), dict(flags=FORCE_SEQ)):
        refused(fwd(io, **kw), -1, b"ends")
    refused(fwd(io, sa=BAD), -1, b"sa must be")
    refused(fwd(io, ws=BAD, nbytes=1 << 30), -1, b"workspace must be")
    refused(fwd(io, first=BAD), -1, b"aligned")
    refused(fwd(io, first=NULL), -1, b"null")
    need = lib().hiprwkv_wkv7_fwd_workspace_bytes(io, B, T, H, 64)
    assert need > 0
    refused(fwd(io, ws=OK, nbytes=need - 1), -3, b"workspace has")
    most = lib().hiprwkv_wkv7_bwd_ends_workspace_bytes(io, B, T, H, 64)
    assert most > lib().hiprwkv_wkv7_bwd_workspace_bytes(B, T, H, 64)
    for kw in (dict(ends=BAD), dict(flags=FORCE_SEQ)):
        refused(bwd(io, nbytes=most, **kw), -1, b"ends")
    refused(bwd(io, nbytes=most - 1), -3, b"workspace has")
    refused(bwd(io, nbytes=most, ws=BAD), -1, b"aligned")
    refused(bwd(io, nbytes=most, ws=NULL), -1, b"null")
    refused(bwd(io, nbytes=most, first=NULL), -1, b"null")


def lora(io=1, rows=32, N=64, d=(32, 32, 32, 32), hid=OK, w2=OK, out=OK, g=OK, vf=OK, v=OK, w=OK, arrays=True):
    arr = lambda p: (ctypes.c_void_p * 4)(OK, OK, p, OK)
    return lib().hiprwkv_rwkv7_lora_pre(NULL, io, rows, H, N, arr(hid) if arrays else NULL, arr(w2), (ctypes.c_int64 * 4)(*d), OK, v, vf, OK, OK, OK,
                                        OK, OK, NULL if out is NULL else arr(out), g, w, OK, OK, OK, OK)


def test_lora_pre():
    refused(lora(arrays=False), -1, b"null pointer array")
    refused(lora(io=0), -1, b"HIPRWKV_BF16")
    refused(lora(N=32), -1, b"N=32")
    refused(lora(d=(32, 20, 32, 32)), -1, b"multiples of 8")
    refused(lora(d=(32, 0, 32, 32)), -1, b"positive")
    refused(lora(d=(32, 32, 32, 1 << 40)), -1, b"4 GiB")
    refused(lora(d=(1 << 60, 32, 32, 32)), -1, b"4 GiB")
    refused(lora(rows=1 << 32), -1, b"rows")
    for kw in (dict(hid=BAD), dict(w2=BAD), dict(out=BAD), dict(w=BAD), dict(out=NULL, g=BAD), dict(hid=NULL), dict(v=NULL)):
        assert lora(**kw) == -1


def stack(**kw):
    from jaxrwkv_amd import _lib
    backward = kw.pop("backward", False)
    A = _lib.Rwkv7StackArgs(B=1, T=32, L=2, C=128, H=2, F=512, d_decay=32, d_aaa=32, d_mv=32, d_gate=32)
    for n in "x state s xs dx g_xs g_dx g_x workspace".split():
        setattr(A, n, OK)
    A.new_state, A.new_s, A.workspace_bytes = 2 * OK, 2 * OK, 1 << 40
    A.param[:] = A.grad[:] = [OK] * 33
    saved = (ctypes.c_void_p * 2)(OK, kw.pop("saved", OK))
    A.saved = ctypes.addressof(saved) if backward else None
    for n, v in kw.items():
        if n in ("param", "grad"):
            getattr(A, n)[v[0]] = v[1]
        elif n == "no_saved":
            A.saved = None
        else:
            setattr(A, n, v)
    return (lib().hiprwkv_rwkv7_stack_bwd if backward else lib().hiprwkv_rwkv7_stack_fwd)(NULL, ctypes.byref(A))


@pytest.mark.parametrize("backward", [False, True])
def test_stack(backward):
    f = lib().hiprwkv_rwkv7_stack_bwd if backward else lib().hiprwkv_rwkv7_stack_fwd
    refused(f(NULL, None), -1, b"null arguments")
    for kw in (dict(B=0), dict(T=-1), dict(C=192), dict(H=65, C=65 * 64), dict(F=500), dict(d_mv=4), dict(d_gate=1 << 24), dict(B=1 << 20, T=1 << 12)):
        refused(stack(backward=backward, **kw), -1, b"sizes must be")
    refused(stack(backward=backward, flags=4), -1, b"flag")
    for kw in (dict(x=BAD), dict(state=NULL), dict(s=BAD), dict(workspace=NULL), dict(param=(3, NULL)), dict(param=(32, BAD)), dict(g_s=BAD)):
        refused(stack(backward=backward, **kw), -1, b"null or misaligned")
    refused(stack(backward=backward, workspace_bytes=1024), -3, b"workspace has")


def test_stack_by_direction():
    refused(stack(new_state=OK), -1, b"different arrays")
    refused(stack(new_s=OK), -1, b"different arrays")
    refused(stack(dx=NULL), -1, b"null or misaligned")
    for kw in (dict(no_saved=True), dict(saved=BAD), dict(saved=NULL), dict(g_x=NULL), dict(grad=(5, NULL)), dict(grad=(12, NULL))):
        refused(stack(backward=True, **kw), -1, b"null or misaligned")
