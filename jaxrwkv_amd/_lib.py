"""ctypes binding of ``libhiprwkv.so`` (the C ABI declared in ``include/hiprwkv.h``).

There is no fallback: if the library has not been built, or a call fails, an exception is raised.
"""
import ctypes
import os

HERE = os.path.dirname(os.path.abspath(__file__))
LIB_PATH = os.path.join(HERE, "libhiprwkv.so")

F32, BF16 = 0, 1
COMPAT_ASSOC = 1
FORCE_SEQ = 2
NO_SMALL_T = 4
W_PER_HEAD = 0x10
CKPT_READY = 0x20
LENGTH_I32 = 0x40
W_RAW = 0x80
NEW_STATE_IO = 0x200             # the forwards of WKV7 and WKV6 alone
DEBUG_DROP_PUBLISH = 0x100      # refused unless the process runs with HIPRWKV_ENABLE_DEBUG_FLAGS=1
PUBLIC_FLAGS = COMPAT_ASSOC | FORCE_SEQ | NO_SMALL_T | W_PER_HEAD | CKPT_READY | LENGTH_I32 | W_RAW

_vp, _i64, _int, _u32, _sz = ctypes.c_void_p, ctypes.c_int64, ctypes.c_int, ctypes.c_uint, ctypes.c_size_t



class Rwkv7DecodeArgs(ctypes.Structure):
    """``hiprwkv_rwkv7_decode_args``"""
    _fields_ = ([(n, _i64) for n in "B T L C H F vocab d_decay d_aaa d_mv d_gate".split()]
                + [(n, _vp) for n in ("x state new_state length new_starts ln0_w ln0_b ln_out_w ln_out_b head ln1_w ln1_b "
                                      "ln2_w ln2_b x_r x_w x_k x_v x_a x_g w0 w1 w2 a0 a1 a2 v0 v1 v2 g1 g2 k_k k_a r_k "
                                      "receptance key value output lnx_w lnx_b ffn_x_k ffn_key ffn_value xn logits "
                                      "workspace").split()]
                + [("workspace_bytes", ctypes.c_uint64), ("flags", ctypes.c_uint64)])


class GemmJob(ctypes.Structure):
    """``hiprwkv_gemm_job``"""
    _fields_ = ([(n, _vp) for n in ("x", "w", "aux", "out")]
                + [(n, ctypes.c_int32) for n in ("M", "N", "K", "km", "kn", "act", "tile0", "pad")])


class Rwkv7StackArgs(ctypes.Structure):
    """``hiprwkv_rwkv7_stack_args``; ``param`` and ``grad`` in the order of blocks7.NAMES"""
    _fields_ = ([(n, _i64) for n in "B T L C H F d_decay d_aaa d_mv d_gate".split()]
                + [(n, _vp) for n in "x state s new_state new_s length new_starts xs dx saved workspace".split()]
                + [("workspace_bytes", ctypes.c_uint64), ("flags", ctypes.c_uint64)]
                + [(n, _vp) for n in "g_xs g_dx g_shift g_s g_x".split()] + [("param", _vp * 33), ("grad", _vp * 33)])


# name -> (restype, argtypes); mirrors include/hiprwkv.h declaration by declaration
SIGNATURES = {
    "hiprwkv_last_error": (ctypes.c_char_p, []),
    "hiprwkv_version": (_int, []),
    "hiprwkv_handshake_failures": (_int, [_vp, ctypes.POINTER(ctypes.c_uint)]),
    "hiprwkv_numeric_events": (_int, [_vp, ctypes.POINTER(ctypes.c_uint)]),
    "hiprwkv_wkv7_fwd": (_int, [_vp, _int, _int, _i64, _i64, _i64, _i64] + [_vp] * 7 + [_vp, _vp] + [_vp, _vp, _vp, _u32]),
    "hiprwkv_wkv7_fwd_workspace_bytes": (_sz, [_int] + [_i64] * 4),
    "hiprwkv_wkv7_fwd_parts": (_int, [_vp, _int, _int, _i64, _i64, _i64, _i64] + [_vp] * 7 + [_vp, _vp] + [_vp] * 4 + [_sz, _u32]),
    "hiprwkv_wkv7_ends_bytes": (_sz, [_int] + [_i64] * 4),
    "hiprwkv_wkv7_fwd_ends": (_int, [_vp, _int, _int, _i64, _i64, _i64, _i64] + [_vp] * 7 + [_vp, _vp] + [_vp] * 5 + [_sz, _u32]),
    "hiprwkv_wkv7_step": (_int, [_vp, _int, _int, _i64, _i64, _i64, _i64] + [_vp] * 6 + [_vp, _i64] + [_vp, _vp]
                          + [_vp, _vp, _i64, _u32]),
    "hiprwkv_wkv7_bwd_workspace_bytes": (_sz, [_i64] * 4),
    "hiprwkv_wkv7_bwd": (_int, [_vp, _int, _int, _i64, _i64, _i64, _i64] + [_vp] * 7 + [_vp, _vp] + [_vp] * 3
                         + [_vp] * 7 + [_vp, _sz, _u32]),
    "hiprwkv_wkv7_bwd_ends_workspace_bytes": (_sz, [_int] + [_i64] * 4),
    "hiprwkv_wkv7_bwd_ends": (_int, [_vp, _int, _int, _i64, _i64, _i64, _i64] + [_vp] * 7 + [_vp, _vp] + [_vp] * 4
                              + [_vp] * 7 + [_vp, _sz, _u32]),
    "hiprwkv_wkv6_fwd": (_int, [_vp, _int, _int, _i64, _i64, _i64, _i64] + [_vp] * 6 + [_vp, _vp] + [_vp, _vp, _u32]),
    "hiprwkv_wkv6_fwd_workspace_bytes": (_sz, [_int] + [_i64] * 4),
    "hiprwkv_wkv6_fwd_parts": (_int, [_vp, _int, _int, _i64, _i64, _i64, _i64] + [_vp] * 6 + [_vp, _vp] + [_vp] * 3 + [_sz, _u32]),
    "hiprwkv_wkv6_step": (_int, [_vp, _int, _int, _i64, _i64, _i64, _i64] + [_vp] * 5 + [_vp, _i64] + [_vp, _vp]
                          + [_vp, _vp, _i64, _u32]),
    "hiprwkv_wkv6_bwd_workspace_bytes": (_sz, [_i64] * 4),
    "hiprwkv_wkv6_bwd": (_int, [_vp, _int, _int, _i64, _i64, _i64, _i64] + [_vp] * 6 + [_vp, _vp] + [_vp, _vp]
                         + [_vp] * 6 + [_vp, _sz, _u32]),
    "hiprwkv_wkv4_fwd": (_int, [_vp, _int, _i64, _i64, _i64] + [_vp] * 5 + [_vp, _vp] + [_vp, _vp, _u32]),
    "hiprwkv_wkv4_fwd_ckpt": (_int, [_vp, _int, _i64, _i64, _i64] + [_vp] * 5 + [_vp, _vp] + [_vp, _vp, _vp,
                                     ctypes.c_size_t, _u32]),
    "hiprwkv_wkv4_bwd_workspace_bytes": (_sz, [_i64] * 3),
    "hiprwkv_wkv4_bwd": (_int, [_vp, _int, _i64, _i64, _i64] + [_vp] * 6 + [_vp, _vp] + [_vp] + [_vp] * 5
                         + [_vp, _sz, _u32]),
    "hiprwkv_wkv4_bwd_noalloc_max_bytes": (_sz, []),
    "hiprwkv_wkv4_bwd_noalloc": (_int, [_vp, _int, _i64, _i64, _i64] + [_vp] * 6 + [_vp, _vp] + [_vp] + [_vp] * 5 + [_u32]),
    "hiprwkv_wkv4_mix_workspace_bytes": (_sz, [_i64] * 3),
    "hiprwkv_wkv4_mix": (_int, [_vp, _int, _i64, _i64, _i64] + [_vp] * 10 + [_vp, _sz, _vp, _sz, _u32]),
    "hiprwkv_wkv4_mix_bwd_workspace_bytes": (_sz, [_i64] * 3),
    "hiprwkv_wkv4_mix_bwd": (_int, [_vp, _int, _i64, _i64, _i64] + [_vp] * 10 + [_vp, _sz] + [_vp] * 6 + [_vp, _sz, _u32]),
    "hiprwkv_rwkv7_shiftmix": (_int, [_vp, _int, _i64, _i64, _i64, _int, _vp, _vp, _i64, _vp, _vp, _vp]),
    "hiprwkv_rwkv7_shiftmix_bwd": (_int, [_vp, _int, _i64, _i64, _i64, _int, _vp, _vp, _i64, _vp, _vp, _vp, _vp, _vp, _i64, _vp]),
    "hiprwkv_rwkv7_decay": (_int, [_vp, _int, _i64, _i64, _vp, _vp, _vp]),
    "hiprwkv_rwkv7_decay_bwd": (_int, [_vp, _int, _i64, _i64, _vp, _vp, _vp, _vp, _vp]),
    "hiprwkv_rwkv7_agate": (_int, [_vp, _int, _i64, _i64, _vp, _vp, _vp]),
    "hiprwkv_rwkv7_agate_bwd": (_int, [_vp, _int, _i64, _i64, _vp, _vp, _vp, _vp, _vp]),
    "hiprwkv_rwkv7_relusq": (_int, [_vp, _int, _i64, _vp, _vp]),
    "hiprwkv_rwkv7_relusq_bwd": (_int, [_vp, _int, _i64, _vp, _vp, _vp]),
    "hiprwkv_rwkv7_vmix": (_int, [_vp, _int, _i64, _i64, _vp, _vp, _vp, _vp, _vp]),
    "hiprwkv_rwkv7_vmix_bwd": (_int, [_vp, _int, _i64, _i64, _vp, _vp, _vp, _vp, _vp, _vp, _vp, _vp, _vp]),
    "hiprwkv_rwkv7_ln_shiftmix": (_int, [_vp, _int, _i64, _i64, _i64, _int] + [_vp] * 4 + [ctypes.c_float, _vp, _i64]
                                  + [_vp] * 6 + [_i64, _vp]),
    "hiprwkv_rwkv7_ln_shiftmix_bwd_workspace_bytes": (_sz, [_i64] * 3 + [_int]),
    "hiprwkv_rwkv7_ln_shiftmix_bwd": (_int, [_vp, _int, _i64, _i64, _i64, _int] + [_vp] * 5 + [_i64] + [_vp] * 10 + [_sz]),
    "hiprwkv_rwkv7_lora_pre": (_int, [_vp, _int, _i64, _i64, _i64] + [_vp] * 18),
    "hiprwkv_rwkv7_pre": (_int, [_vp, _int, _i64, _i64, _i64] + [_vp] * 16),
    "hiprwkv_rwkv7_pre_bwd_workspace_bytes": (_sz, [_i64] * 3),
    "hiprwkv_rwkv7_pre_bwd": (_int, [_vp, _int, _i64, _i64, _i64] + [_vp] * 29 + [_sz]),
    "hiprwkv_rwkv7_postmix_bwd2_workspace_bytes": (_sz, [_i64] * 3),
    "hiprwkv_rwkv7_postmix_bwd2": (_int, [_vp, _int, _i64, _i64, _i64] + [_vp] * 8 + [ctypes.c_float] + [_vp] * 8 + [_sz]),
    "hiprwkv_gemm": (_int, [_vp, _int, ctypes.POINTER(GemmJob)]),
    "hiprwkv_rwkv7_decode_workspace_bytes": (_sz, [ctypes.POINTER(Rwkv7DecodeArgs)]),
    "hiprwkv_rwkv7_decode": (_int, [_vp, ctypes.POINTER(Rwkv7DecodeArgs)]),
    "hiprwkv_rwkv7_stack_saved_bytes": (_sz, [ctypes.POINTER(Rwkv7StackArgs)]),
    "hiprwkv_rwkv7_stack_saved_layer_bytes": (_sz, [ctypes.POINTER(Rwkv7StackArgs), _i64]),
    "hiprwkv_rwkv7_stack_workspace_bytes": (_sz, [ctypes.POINTER(Rwkv7StackArgs), _int]),
    "hiprwkv_rwkv7_stack_fwd": (_int, [_vp, ctypes.POINTER(Rwkv7StackArgs)]),
    "hiprwkv_rwkv7_stack_bwd": (_int, [_vp, ctypes.POINTER(Rwkv7StackArgs)]),
    "hiprwkv_rwkv7_premix": (_int, [_vp, _int, _i64, _i64, _i64] + [_vp] * 7),
    "hiprwkv_rwkv7_postmix": (_int, [_vp, _int, _i64, _i64, _i64] + [_vp] * 8 + [ctypes.c_float, _vp]),
    "hiprwkv_rwkv7_premix_bwd": (_int, [_vp, _int, _i64, _i64, _i64] + [_vp] * 11),
    "hiprwkv_rwkv7_postmix_bwd": (_int, [_vp, _int, _i64, _i64, _i64] + [_vp] * 8 + [ctypes.c_float] + [_vp] * 9),
}

_lib = None


class HipRwkvError(RuntimeError):
    pass


def load():
    """Loads the library once and types every entry point; raises if it is missing."""
    global _lib
    if _lib is not None:
        return _lib
    if not os.path.exists(LIB_PATH):
        raise HipRwkvError(
            f"{LIB_PATH} is missing: build it with `python -m jaxrwkv_amd.build` (there is no CPU fallback)")
    lib = ctypes.CDLL(LIB_PATH)
    for name, (res, args) in SIGNATURES.items():
        fn = getattr(lib, name)
        fn.restype = res
        fn.argtypes = args
    _lib = lib
    return lib


def check(rc, what):
    if rc != 0:
        msg = load().hiprwkv_last_error().decode()
        raise HipRwkvError(f"{what} failed with code {rc}: {msg}")
