/*
 * hiprwkv -- C ABI of the MI355X (gfx950) WKV recurrence library.
 *
 * Every entry point only enqueues work on the caller's HIP stream: it does not
 * allocate, free or synchronise, so it can be called from an XLA custom-call
 * handler thread.  All pointers are device pointers, 16-byte aligned.  Entry points return
 * HIPRWKV_OK or a negative HIPRWKV_E* code; hiprwkv_last_error() then returns a
 * thread-local message.
 *
 * Operand order follows the reference's jax.ffi targets, whose native
 * implementation (package `jaxrwkvkernel`, CUDA only) is not part of the
 * reference tree; each declaration cites the Python call site it replaces.
 *
 * Shapes: B sequences (the reference's vmap axis), T tokens, H heads, N head size.
 *   WKV7/WKV6 token tensors  (B,T,H,N) row-major, io_dtype
 *   WKV7 state               (B,H,N,N) state_dtype, s[b,h,i,j]: value row i, key column j
 *   WKV6 state               (B,H,N,N) state_dtype, s[b,h,i,j]: key row i, value column j
 *   WKV4 token tensors       (B,T,C), state (B,3,C) = (aa,bb,pp)
 *   length                   (B,) uint32, may be NULL (= T)
 *   new_starts               (B,T) one byte per token (0/1), may be NULL (= none)
 * The recurrence always runs in fp32 whatever the io/state dtypes are.
 *
 * Placement of the token tensors.  The kernels touch the rows of all token tensors of a call at the same
 * (token, head) together.  When the tensors' base addresses are congruent modulo 1 KiB (two large allocations
 * of a caching allocator usually are: both start on 2 MiB boundaries) those rows compete for the same part of
 * the memory system.  Measured on MI355X, WKV7 at B8 T4096 H32 bf16, forward with its residual / forward +
 * backward: 303 / 1619 us with every tensor on a 2 MiB boundary; 284 / 1535 us with only the outputs, the
 * gradients and the workspace arrays moved; 265 / 1469 us with each tensor, the inputs included, at its own
 * multiple of 128 bytes past a 1 KiB boundary (0, 128, ..., 896).  Offsets that are multiples of 1 KiB change
 * nothing.  A caller that owns the placement of its operands should stagger them that way; the library does
 * it for the arrays inside `workspace`, and the Python operators do it for every tensor they allocate.
 */
#ifndef HIPRWKV_H_
#define HIPRWKV_H_

#include <stddef.h>
#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

#define HIPRWKV_OK 0
#define HIPRWKV_EINVAL (-1)   /* bad argument (shape, dtype, NULL pointer) */
#define HIPRWKV_ELAUNCH (-2)  /* hipLaunchKernel reported an error */
#define HIPRWKV_ENOSPACE (-3) /* workspace too small */

#define HIPRWKV_F32 0
#define HIPRWKV_BF16 1

/* flags */
/* Reproduce AssociativeScanRWKV where it differs from the sequential loop:
 * WKV7 y[t] = 0 when new_starts[t+1] (rwkv7.py:331-333,344); returned state is the
 * one entering position `length` (rwkv7.py:345, rwkv6.py:301, rwkv4.py:300). */
#define HIPRWKV_COMPAT_ASSOC 1u
/* Force the sequential fp32 VALU kernel even where a chunked MFMA kernel exists. */
#define HIPRWKV_FORCE_SEQ 2u
/* hiprwkv_wkv7_fwd and hiprwkv_wkv6_fwd run sequences of at most HIPRWKV_SMALL_T tokens (decode steps) on a kernel
 * that streams the state once and has no per-launch set-up; this flag sends them to the general kernels instead. */
#define HIPRWKV_NO_SMALL_T 4u
#define HIPRWKV_SMALL_T 8
/* hiprwkv_wkv6_fwd / hiprwkv_wkv6_bwd: `w` is (H, N), one log decay per head channel shared by every token and
 * sequence (RWKV-5, rwkv5.py:194 / rwkv5_2.py:198), instead of (B, T, H, N).  The backward still writes the decay
 * cotangent per token, (B, T, H, N); the caller sums it over B and T. */
#define HIPRWKV_W_PER_HEAD 0x10u
/* hiprwkv_wkv4_bwd: the workspace already holds the checkpoints that hiprwkv_wkv4_fwd_ckpt wrote for the same
 * inputs; the backward then skips its own first pass over k and v. */
#define HIPRWKV_CKPT_READY 0x20u
/* `length` holds int32 values, and a negative one counts as 0 (without the flag: uint32). */
#define HIPRWKV_LENGTH_I32 0x40u
/* hiprwkv_wkv4_*: `w` is the parameter time_decay itself; the op's decay is -exp(w), rounded to io_dtype
 * (rwkv4.py:312), and the cotangent returned is the one of w. */
#define HIPRWKV_W_RAW 0x80u
/* Test hook for the chunked kernels' bounded hand-shake: the producer wave of the last chunk does not publish it, the
 * consumer waves' wait runs out (a few milliseconds), every wave still ends normally, the outputs of every
 * (sequence, head) are NaN and hiprwkv_handshake_failures() has advanced by B*H per kernel. */
#define HIPRWKV_DEBUG_DROP_PUBLISH 0x100u
/* hiprwkv_wkv7_fwd*, hiprwkv_wkv6_fwd*: new_s is written in io_dtype (rounded once from the fp32 state of the kernel) instead of
 * state_dtype, which then is s's type alone; s and new_s have to be different arrays where the two types differ. */
#define HIPRWKV_NEW_STATE_IO 0x200u
/* Every flag a production caller may pass, but for HIPRWKV_NEW_STATE_IO, which only the entry points above take.  Entry points refuse other bits, and refuse HIPRWKV_DEBUG_DROP_PUBLISH
 * unless the process runs with HIPRWKV_ENABLE_DEBUG_FLAGS=1 in its environment. */
#define HIPRWKV_PUBLIC_FLAGS (HIPRWKV_COMPAT_ASSOC | HIPRWKV_FORCE_SEQ | HIPRWKV_NO_SMALL_T | HIPRWKV_W_PER_HEAD | HIPRWKV_CKPT_READY | HIPRWKV_LENGTH_I32 | HIPRWKV_W_RAW)

typedef void* hiprwkv_stream; /* a hipStream_t */

const char* hiprwkv_last_error(void);
int hiprwkv_version(void);

/* The chunked kernels pass work between waves of a workgroup through a hand-shake with a bounded wait (a broken
 * hand-shake must not hang the GPU).  A workgroup whose wait runs out overwrites all its outputs for that
 * (sequence, head) with NaN and adds one to a per-device counter; this call copies the counter of the current
 * device to *count (host memory).  Unlike every other entry point it synchronises `stream`.  No counterpart in
 * the reference; for health checks and tests. */
int hiprwkv_handshake_failures(hiprwkv_stream stream, unsigned* count);

/* Numeric events of the chunked matrix-core kernels since the process started, per device, copied to *count (host
 * memory; synchronises `stream`).  Two things are counted, once per wave that meets them:
 *  - a key channel whose log decay summed over a 16-token chunk is below -80 (a decay of e^-5 per token sustained over
 *    the chunk; RWKV-7's own w <= -0.5 keeps it above -10): the chunked kernels, fp32 I/O included, scale that
 *    channel's steps of the chunk to a total of -80, so its result is no longer exact.  Every sweep of a backward
 *    call that meets such a chunk counts it again.  HIPRWKV_FORCE_SEQ has no such floor.
 *  - inf or NaN in the carried state of the bf16-I/O forward kernels (WKV7, WKV6) after the last token: their matrix
 *    operands are IEEE half, so |state|, |sa|, |v| or a decay-scaled input beyond 65504 overflow; y and the state
 *    are then inf/NaN from that token on (until a reset starts a new state: an overflow whose state a later reset
 *    discards shows in y alone).
 * Magnitudes far below 1 lose precision silently instead: the half operands have 11 significant bits down to 6e-5
 * and fewer below, so v (and with it the state and sa) scaled by 1e-5 doubles the error of y and 1e-7 brings it to
 * 4 %; the op is linear in (v, s), so a caller with such values scales them by a power of two around the call.
 * No counterpart in the reference; for health checks and tests. */
int hiprwkv_numeric_events(hiprwkv_stream stream, unsigned* count);

/* ---- WKV7 ------------------------------------------------------------------
 * Replaces ffi target "wkv7-fwd-{fp32,bf16}": operands w,r,k,v,a,b,s,length,new_starts
 * -> out, s_restore, sa_restore, new_s  (rwkv7.py:372-375).  `w` is the raw decay
 * argument; the op applies exp(-exp(w)) (rwkv7.py:201).  `sa` (B,T,H,N) is
 * the residual S_{t-1} a_t kept for the backward pass (the reference's sa_restore):
 * fp32 beside fp32 I/O, IEEE half (2 bytes per element) beside bf16 I/O; the caller hands
 * the same buffer to hiprwkv_wkv7_bwd.  Pass NULL for inference.  No state checkpoints
 * (s_restore) are needed. */
int hiprwkv_wkv7_fwd(hiprwkv_stream stream, int io_dtype, int state_dtype,
                     int64_t B, int64_t T, int64_t H, int64_t N,
                     const void* w, const void* r, const void* k, const void* v,
                     const void* a, const void* b, const void* s,
                     const uint32_t* length, const uint8_t* new_starts,
                     void* out, void* sa, void* new_s, unsigned flags);

/* The same with `workspace` (hiprwkv_wkv7_fwd_workspace_bytes, 0 where it is of no use; NULL: as hiprwkv_wkv7_fwd).  Where
 * B*H leaves most of the GPU idle, sequences are cut into parts whose summaries (state maps) are made first.  A
 * part whose hand-shake fails counts as one of its own in hiprwkv_handshake_failures and makes its own rows NaN. */
size_t hiprwkv_wkv7_fwd_workspace_bytes(int io_dtype, int64_t B, int64_t T, int64_t H, int64_t N);
int hiprwkv_wkv7_fwd_parts(hiprwkv_stream stream, int io_dtype, int state_dtype,
                           int64_t B, int64_t T, int64_t H, int64_t N,
                           const void* w, const void* r, const void* k, const void* v,
                           const void* a, const void* b, const void* s,
                           const uint32_t* length, const uint8_t* new_starts,
                           void* out, void* sa, void* new_s, void* workspace, size_t workspace_bytes, unsigned flags);

/* The same for a call with a backward to come: `ends` (hiprwkv_wkv7_ends_bytes, 0 where it is of no use, 16-byte aligned; NULL: none
 * wanted; not with HIPRWKV_FORCE_SEQ) goes on to hiprwkv_wkv7_bwd_ends, which then cuts the sequence into parts that run at the
 * same time.  It holds what is needed of the states there, put in by this call (HIPRWKV_F32) or by the backward itself. */
size_t hiprwkv_wkv7_ends_bytes(int io_dtype, int64_t B, int64_t T, int64_t H, int64_t N);
int hiprwkv_wkv7_fwd_ends(hiprwkv_stream stream, int io_dtype, int state_dtype,
                          int64_t B, int64_t T, int64_t H, int64_t N,
                          const void* w, const void* r, const void* k, const void* v,
                          const void* a, const void* b, const void* s,
                          const uint32_t* length, const uint8_t* new_starts,
                          void* out, void* sa, void* new_s, void* ends, void* workspace, size_t workspace_bytes, unsigned flags);

/* A decode step (T <= HIPRWKV_SMALL_T tokens per sequence) on a state that lives inside the packed model state of the
 * reference: there a sequence's state is (L, 2+N, C) and layer l's rows 2.. are the (H,N,N) WKV state, flat
 * (rwkv7.py:176-180 default_state, :254-260 the slice and reshape around inner_loop), so with a batch axis in front
 * the states of consecutive sequences are H*N*N contiguous elements each, L*(2+N)*C elements apart.  `s` and `new_s`
 * point at the first sequence's state, `*_batch_stride` is that distance in elements (>= H*N*N, a multiple of 16
 * bytes); everything else is as in hiprwkv_wkv7_fwd without `sa`.  Every element of a state is read once, before
 * anything is written, by the thread that writes it: `new_s` may be `s` (same stride) for an update in place. */
int hiprwkv_wkv7_step(hiprwkv_stream stream, int io_dtype, int state_dtype,
                      int64_t B, int64_t T, int64_t H, int64_t N,
                      const void* w, const void* r, const void* k, const void* v,
                      const void* a, const void* b, const void* s, int64_t s_batch_stride,
                      const uint32_t* length, const uint8_t* new_starts,
                      void* out, void* new_s, int64_t new_s_batch_stride, unsigned flags);

/* Bytes of scratch hiprwkv_wkv7_bwd needs for this shape: three fp32 (B,T,H,N) arrays plus 1 KiB each (see "Placement"). */
size_t hiprwkv_wkv7_bwd_workspace_bytes(int64_t B, int64_t T, int64_t H, int64_t N);

/* Replaces ffi target "wkv7-bwd-{fp32,bf16}": operands w,r,k,v,a,b,s,length,new_starts,
 * gy,s_restore,sa_restore,gs_out -> gw,gr,gk,gv,ga,gb,gs  (rwkv7.py:406-408).
 * Unlike the reference's native op it honours new_starts, takes the cotangent of the
 * returned state (gs_out, may be NULL = 0) and returns the one of the input state.
 * Three sweeps over the sequence on the matrix cores: bf16 hi+lo operand pairs beside bf16
 * I/O (the cotangent of `sa` passes between them as 16-bit fixed point with a power-of-two
 * scale per 16 x 16 tile: 16 bits whatever the size of the cotangents), fp32 operands and an
 * fp32 workspace (no rounding below fp32) beside fp32 I/O; HIPRWKV_FORCE_SEQ runs the
 * sequential fp32 sweeps instead. */
int hiprwkv_wkv7_bwd(hiprwkv_stream stream, int io_dtype, int state_dtype,
                     int64_t B, int64_t T, int64_t H, int64_t N,
                     const void* w, const void* r, const void* k, const void* v,
                     const void* a, const void* b, const void* s,
                     const uint32_t* length, const uint8_t* new_starts,
                     const void* gy, const void* sa, const void* gs_out,
                     void* gw, void* gr, void* gk, void* gv, void* ga, void* gb, void* gs,
                     void* workspace, size_t workspace_bytes, unsigned flags);

/* The same with the `ends` of hiprwkv_wkv7_fwd_ends (NULL: as hiprwkv_wkv7_bwd) and a workspace of
 * hiprwkv_wkv7_bwd_ends_workspace_bytes: few sequences and heads run in parts. */
size_t hiprwkv_wkv7_bwd_ends_workspace_bytes(int io_dtype, int64_t B, int64_t T, int64_t H, int64_t N);
int hiprwkv_wkv7_bwd_ends(hiprwkv_stream stream, int io_dtype, int state_dtype,
                          int64_t B, int64_t T, int64_t H, int64_t N,
                          const void* w, const void* r, const void* k, const void* v,
                          const void* a, const void* b, const void* s,
                          const uint32_t* length, const uint8_t* new_starts,
                          const void* gy, const void* sa, const void* gs_out, void* ends,
                          void* gw, void* gr, void* gk, void* gv, void* ga, void* gb, void* gs,
                          void* workspace, size_t workspace_bytes, unsigned flags);

/* ---- WKV6 ------------------------------------------------------------------
 * The reference has no native WKV6 op (README.md:93-99); the operand order follows
 * inner_loop(r,k,v,w,time_first,s,length,new_starts) (rwkv6.py:175).  `w` is the log
 * decay -exp(raw) (rwkv6.py:217-218), `u` = time_faaaa (H,N) io_dtype. */
int hiprwkv_wkv6_fwd(hiprwkv_stream stream, int io_dtype, int state_dtype,
                     int64_t B, int64_t T, int64_t H, int64_t N,
                     const void* r, const void* k, const void* v, const void* w,
                     const void* u, const void* s,
                     const uint32_t* length, const uint8_t* new_starts,
                     void* out, void* new_s, unsigned flags);
/* The same with `workspace`, as hiprwkv_wkv7_fwd_parts. */
size_t hiprwkv_wkv6_fwd_workspace_bytes(int io_dtype, int64_t B, int64_t T, int64_t H, int64_t N);
int hiprwkv_wkv6_fwd_parts(hiprwkv_stream stream, int io_dtype, int state_dtype,
                     int64_t B, int64_t T, int64_t H, int64_t N,
                     const void* r, const void* k, const void* v, const void* w,
                     const void* u, const void* s,
                     const uint32_t* length, const uint8_t* new_starts,
                     void* out, void* new_s, void* workspace, size_t workspace_bytes, unsigned flags);

/* hiprwkv_wkv6_fwd for a decode step (T <= HIPRWKV_SMALL_T) on a state inside the reference's packed model state
 * (rwkv6.py:148-153 default_state: (L, 2+N, C) per sequence; :221-224 the slice state[1:] of the time-mixing part,
 * reshaped to (H,N,N) around inner_loop and written back): `s` and `new_s` point at the first sequence's state, the
 * states of consecutive sequences are `*_batch_stride` elements apart (>= H*N*N, a multiple of 16 bytes); `new_s` may
 * be `s` for an update in place.  Same conventions as hiprwkv_wkv7_step. */
int hiprwkv_wkv6_step(hiprwkv_stream stream, int io_dtype, int state_dtype,
                      int64_t B, int64_t T, int64_t H, int64_t N,
                      const void* r, const void* k, const void* v, const void* w,
                      const void* u, const void* s, int64_t s_batch_stride,
                      const uint32_t* length, const uint8_t* new_starts,
                      void* out, void* new_s, int64_t new_s_batch_stride, unsigned flags);

size_t hiprwkv_wkv6_bwd_workspace_bytes(int64_t B, int64_t T, int64_t H, int64_t N);

/* Cotangents of wkv6_fwd: gr,gk,gv,gw (B,T,H,N) io_dtype; gu (B,H,N) fp32, to be summed
 * over B by the caller (as the reference does for the WKV4 parameters, rwkv4.py:351);
 * gs (B,H,N,N) state_dtype.  Forward and backward run on the matrix cores for both I/O
 * dtypes (fp32 operands beside fp32 I/O); HIPRWKV_FORCE_SEQ selects the sequential kernels. */
int hiprwkv_wkv6_bwd(hiprwkv_stream stream, int io_dtype, int state_dtype,
                     int64_t B, int64_t T, int64_t H, int64_t N,
                     const void* r, const void* k, const void* v, const void* w,
                     const void* u, const void* s,
                     const uint32_t* length, const uint8_t* new_starts,
                     const void* gy, const void* gs_out,
                     void* gr, void* gk, void* gv, void* gw, float* gu, void* gs,
                     void* workspace, size_t workspace_bytes, unsigned flags);

/* ---- WKV4 ------------------------------------------------------------------
 * Replaces ffi target "wkv4-fwd-{fp32,bf16}": operands w,time_first,k,v,s,length,new_starts
 * -> new_s, out  (rwkv4.py:320-321).  `w` = -exp(time_decay) (rwkv4.py:312) and `u` are (C,)
 * io_dtype; the receptance is applied by the caller (rwkv4.py:406).  C <= 2^23.  The output is
 * num * (1/den) with a 1-ulp reciprocal where the reference divides (difference ~1e-7 relative). */
int hiprwkv_wkv4_fwd(hiprwkv_stream stream, int io_dtype,
                     int64_t B, int64_t T, int64_t C,
                     const void* w, const void* u, const void* k, const void* v, const void* s,
                     const uint32_t* length, const uint8_t* new_starts,
                     void* new_s, void* out, unsigned flags);

size_t hiprwkv_wkv4_bwd_workspace_bytes(int64_t B, int64_t T, int64_t C);

/* hiprwkv_wkv4_fwd for a caller that will run the backward pass (the forward rule of the custom VJP, rwkv4.py:379-383):
 * same results, and the state entering every 16th step goes to `workspace` (hiprwkv_wkv4_bwd_workspace_bytes), which
 * hiprwkv_wkv4_bwd then takes with HIPRWKV_CKPT_READY.  Saves that pass its re-read of k and v. */
int hiprwkv_wkv4_fwd_ckpt(hiprwkv_stream stream, int io_dtype,
                          int64_t B, int64_t T, int64_t C,
                          const void* w, const void* u, const void* k, const void* v, const void* s,
                          const uint32_t* length, const uint8_t* new_starts,
                          void* new_s, void* out, void* workspace, size_t workspace_bytes, unsigned flags);

/* Replaces ffi target "wkv4-bwd-{fp32,bf16}": operands w,u,k,v,gy,s,length,new_starts,gs_new
 * -> gw (B,C), gu (B,C), gk, gv, gs  (rwkv4.py:347-349); gw and gu are per sequence in fp32 and are summed
 * over B by the caller (rwkv4.py:351).  gy is the cotangent of the un-gated output.  Unlike the reference's
 * native op it honours gs_new (may be NULL = 0), returns gs, and cuts the chain at new_starts.  C <= 2^23. */
int hiprwkv_wkv4_bwd(hiprwkv_stream stream, int io_dtype,
                     int64_t B, int64_t T, int64_t C,
                     const void* w, const void* u, const void* k, const void* v, const void* gy, const void* s,
                     const uint32_t* length, const uint8_t* new_starts, const void* gs_new,
                     float* gw, float* gu, void* gk, void* gv, void* gs,
                     void* workspace, size_t workspace_bytes, unsigned flags);

/* hiprwkv_wkv4_bwd for callers that cannot allocate device memory (code under HIP graph capture, serving loops,
 * harnesses that forbid hipMalloc): the same kernels, with the checkpoint workspace in a 16 MiB array that is part
 * of the library's device image (one copy per GPU, held until the process ends) instead of a caller's buffer.  It has
 * no counterpart in the reference.  Calls nothing that allocates.  Shapes whose checkpoints
 * (hiprwkv_wkv4_bwd_workspace_bytes) exceed hiprwkv_wkv4_bwd_noalloc_max_bytes() are refused with HIPRWKV_ENOSPACE.
 * Every call on a GPU shares that GPU's array: calls that overlap in time on one GPU (different streams) race; calls
 * on one stream, or ordered by events, do not.  Nothing in the array needs clearing between calls (each call writes
 * every checkpoint before it reads it). */
size_t hiprwkv_wkv4_bwd_noalloc_max_bytes(void);
int hiprwkv_wkv4_bwd_noalloc(hiprwkv_stream stream, int io_dtype,
                             int64_t B, int64_t T, int64_t C,
                             const void* w, const void* u, const void* k, const void* v, const void* gy, const void* s,
                             const uint32_t* length, const uint8_t* new_starts, const void* gs_new,
                             float* gw, float* gu, void* gk, void* gv, void* gs, unsigned flags);

/* inner_loop of RWKV-4 around the op (rwkv4.py:402-406): out = r . wkv, wkv rounded to io_dtype first; r NULL: the op alone.
 * Where B and C leave most of the GPU idle the sequences are cut into parts whose summaries are made first, in
 * `workspace` (hiprwkv_wkv4_mix_workspace_bytes, may be 0).  ckpt as in hiprwkv_wkv4_fwd_ckpt, or NULL. */
size_t hiprwkv_wkv4_mix_workspace_bytes(int64_t B, int64_t T, int64_t C);
int hiprwkv_wkv4_mix(hiprwkv_stream stream, int io_dtype, int64_t B, int64_t T, int64_t C,
                     const void* w, const void* u, const void* k, const void* v, const void* r, const void* s,
                     const uint32_t* length, const uint8_t* new_starts, void* new_s, void* out,
                     void* ckpt, size_t ckpt_bytes, void* workspace, size_t workspace_bytes, unsigned flags);
/* Its cotangents for gout, the one of out: gw and gu (C,) io_dtype summed over the sequences, gk, gv, gr (B,T,C), gs.  ckpt:
 * hiprwkv_wkv4_bwd_workspace_bytes, filled by hiprwkv_wkv4_mix when HIPRWKV_CKPT_READY is set.  r and gr both NULL: the op
 * alone. */
size_t hiprwkv_wkv4_mix_bwd_workspace_bytes(int64_t B, int64_t T, int64_t C);
int hiprwkv_wkv4_mix_bwd(hiprwkv_stream stream, int io_dtype, int64_t B, int64_t T, int64_t C,
                         const void* w, const void* u, const void* k, const void* v, const void* r, const void* gout,
                         const void* s, const uint32_t* length, const uint8_t* new_starts, const void* gs_new,
                         void* ckpt, size_t ckpt_bytes, void* gw, void* gu, void* gk, void* gv, void* gr, void* gs,
                         void* workspace, size_t workspace_bytes, unsigned flags);

/* ---- RWKV-7 token shift and interpolation ---------------------------------------------------
 * The head of time_mixing_seq and channel_mixing_seq (rwkv7.py:226-235 and :192-195), which the reference computes in
 * jnp; no counterpart among its ffi targets:
 *     sx_t = (new_starts[t] ? 0 : x_{t-1}) - x_t ,  out_i = x + sx . mix_i ,  i < n_out   (6: x_r x_w x_k x_v x_a x_g; 1: x_k)
 * x and every out_i are (B,T,C) io_dtype; `prev` is the token before t = 0 of every sequence, C elements each,
 * `prev_batch_stride` elements apart (>= C, a multiple of 16 bytes: the layer's shift row inside the packed model
 * state, rwkv7.py:254, :284); `mix` and `out` are host arrays of n_out device pointers, mix[i] a (C,) io_dtype
 * parameter.  C must be a multiple of 8.  new_starts (B,T) bytes or NULL. */
int hiprwkv_rwkv7_shiftmix(hiprwkv_stream stream, int io_dtype, int64_t B, int64_t T, int64_t C, int n_out,
                           const void* x, const void* prev, int64_t prev_batch_stride, const uint8_t* new_starts,
                           const void* const* mix, void* const* out);
/* Cotangents for cotangents g[i] (B,T,C) of the outputs: dx (B,T,C) and dprev (C elements per sequence,
 * `dprev_batch_stride` apart) in io_dtype, dmix (n_out, C) fp32, summed over sequences and tokens (zeroed by the call). */
int hiprwkv_rwkv7_shiftmix_bwd(hiprwkv_stream stream, int io_dtype, int64_t B, int64_t T, int64_t C, int n_out,
                               const void* x, const void* prev, int64_t prev_batch_stride, const uint8_t* new_starts,
                               const void* const* mix, const void* const* g, void* dx, void* dprev,
                               int64_t dprev_batch_stride, float* dmix);

/* ---- RWKV-7 decay, value mix and gate between the projections and the op -------------------
 * Element-wise steps of time_mixing_seq that the reference computes in jnp (rwkv7.py:237, :241-242, :244); no
 * counterpart among its ffi targets.  Token tensors (rows, C) io_dtype, parameters w0, v0, a0 (C,) io_dtype, C a
 * multiple of 8; the parameter cotangents dw0, dv0, da0 are (C,) fp32 sums over the rows (zeroed by the call).
 *     decay:  w  = -softplus(-(w0 + x)) - 0.5          x = tanh(xw w1) w2
 *     vmix :  v' = v + (v_first - v) sigmoid(v0 + x)   x = (xv v1) v2      (layers after the first)
 *     agate:  a  = sigmoid(a0 + x)                     x = (xa a1) a2 */
int hiprwkv_rwkv7_decay(hiprwkv_stream stream, int io_dtype, int64_t rows, int64_t C, const void* x, const void* w0, void* w);
int hiprwkv_rwkv7_decay_bwd(hiprwkv_stream stream, int io_dtype, int64_t rows, int64_t C, const void* x, const void* w0,
                            const void* g, void* dx, float* dw0);
int hiprwkv_rwkv7_agate(hiprwkv_stream stream, int io_dtype, int64_t rows, int64_t C, const void* x, const void* a0, void* a);
int hiprwkv_rwkv7_agate_bwd(hiprwkv_stream stream, int io_dtype, int64_t rows, int64_t C, const void* x, const void* a0,
                            const void* g, void* dx, float* da0);
/* Channel mixing's activation, rwkv7.py:196: out = relu(x)^2 over n elements (n a multiple of 8); dx = 2 g relu(x). */
int hiprwkv_rwkv7_relusq(hiprwkv_stream stream, int io_dtype, int64_t n, const void* x, void* out);
int hiprwkv_rwkv7_relusq_bwd(hiprwkv_stream stream, int io_dtype, int64_t n, const void* x, const void* g, void* dx);
int hiprwkv_rwkv7_vmix(hiprwkv_stream stream, int io_dtype, int64_t rows, int64_t C, const void* v, const void* v_first,
                       const void* x, const void* v0, void* out);
int hiprwkv_rwkv7_vmix_bwd(hiprwkv_stream stream, int io_dtype, int64_t rows, int64_t C, const void* v, const void* v_first,
                           const void* x, const void* v0, const void* g, void* dv, void* dv_first, void* dx, float* dv0);

/* ---- RWKV-7 sub-block head: residual addition, LayerNorm, token shift, interpolation --------------------
 * rwkv7.py:8-12 and :226-235 / :192-195 in one pass:
 *     xs = x + dx ,  xn = layer_norm(xs; ln_w, ln_b, eps) ,  sx_t = (new_starts[t] ? 0 : xn_{t-1}) - xn_t ,
 *     out_i = xn + sx . mix_i ,  i < n_out  (6, 1; 0: out_0 = xn)
 * Every tensor io_dtype; xs and xn are rounded to it.  dx may be NULL (xs is then x and is not written).  `prev` as in
 * hiprwkv_rwkv7_shiftmix (unused for n_out = 0).  shift (may be NULL): row b, `shift_batch_stride` elements after row
 * b - 1, receives xn of token (length[b] - 1) mod T; length (B,) int32 or NULL (= T).  stats (may be NULL): (B*T, 2) fp32
 * mean and 1/std of xs for the backward pass.  C a multiple of 8, at most 4096. */
int hiprwkv_rwkv7_ln_shiftmix(hiprwkv_stream stream, int io_dtype, int64_t B, int64_t T, int64_t C, int n_out,
                              const void* x, const void* dx, const void* ln_w, const void* ln_b, float eps,
                              const void* prev, int64_t prev_batch_stride, const uint8_t* new_starts,
                              const int32_t* length, const void* const* mix, void* const* out, void* xs, void* shift,
                              int64_t shift_batch_stride, float* stats);
size_t hiprwkv_rwkv7_ln_shiftmix_bwd_workspace_bytes(int64_t B, int64_t T, int64_t C, int n_out);
/* Cotangents for g[i] (B,T,C) of the outputs, gx (B,T,C, may be NULL) of xs and gshift (B,C, may be NULL) of the shift rows:
 * dxs (B,T,C), the cotangent of x and of dx; dprev (B,C, may be NULL); dparam: n_out + 2 arrays (C,) io_dtype, the mix
 * vectors' then ln_w's and ln_b's.  xs and stats are the forward's. */
int hiprwkv_rwkv7_ln_shiftmix_bwd(hiprwkv_stream stream, int io_dtype, int64_t B, int64_t T, int64_t C, int n_out,
                                  const void* xs, const float* stats, const void* ln_w, const void* ln_b,
                                  const void* prev, int64_t prev_batch_stride, const uint8_t* new_starts,
                                  const int32_t* length, const void* const* mix, const void* const* g, const void* gx,
                                  const void* gshift, void* dxs, void* dprev, void* const* dparam, void* workspace,
                                  size_t workspace_bytes);

/* ---- RWKV-7: everything element-wise between the projections and the WKV op ----------------------------
 * hiprwkv_rwkv7_decay, _vmix, _agate and _premix in one pass, with their results: token tensors (rows, H, 64),
 * parameters (H, 64), all io_dtype.  v_first NULL: no value residual (v, xv, v0, v_out unused). */
int hiprwkv_rwkv7_pre(hiprwkv_stream stream, int io_dtype, int64_t rows, int64_t H, int64_t N, const void* xw,
                      const void* k, const void* xa, const void* v, const void* v_first, const void* xv, const void* w0,
                      const void* a0, const void* v0, const void* k_k, const void* k_a, void* w, void* k_out,
                      void* v_out, void* a_out, void* b_out);
/* The same with the low-rank terms made on the way, HIPRWKV_BF16 only: term i = hid[i] (rows, d[i]) times w2[i] (d[i], H*64), rounded, in
 * the order xw, xa, g, xv; all go to out[i], or, with out NULL, g alone to g.  d multiples of 8; without v_first three terms. */
int hiprwkv_rwkv7_lora_pre(hiprwkv_stream stream, int io_dtype, int64_t rows, int64_t H, int64_t N, const void* const* hid,
                           const void* const* w2, const int64_t* d, const void* k, const void* v, const void* v_first, const void* w0,
                           const void* a0, const void* v0, const void* k_k, const void* k_a, void* const* out, void* g, void* w,
                           void* k_out, void* v_out, void* a_out, void* b_out);
size_t hiprwkv_rwkv7_pre_bwd_workspace_bytes(int64_t rows, int64_t H, int64_t N);
/* From the cotangents of w, k_out, v_out, a_out, b_out to those of the inputs; dparam: (H, 64) io_dtype arrays of w0, a0,
 * k_k, k_a and, with v_first, v0.  gk_out2, gv_out2 (may be NULL) are added to gk_out and gv_out; dr (may be NULL) = gr + gr2:
 * r, k_out and v_out have a second use after the op. */
int hiprwkv_rwkv7_pre_bwd(hiprwkv_stream stream, int io_dtype, int64_t rows, int64_t H, int64_t N, const void* xw,
                          const void* k, const void* xa, const void* v, const void* v_first, const void* xv,
                          const void* w0, const void* a0, const void* v0, const void* k_k, const void* k_a,
                          const void* gw, const void* gk_out, const void* gv_out, const void* ga_out,
                          const void* gb_out, const void* gk_out2, const void* gv_out2, const void* gr, const void* gr2,
                          void* dr, void* dxw, void* dk, void* dv, void* dv_first, void* dxv, void* dxa,
                          void* const* dparam, void* workspace, size_t workspace_bytes);

/* ---- Several narrow products in one launch -------------------------------------------------------------
 * bf16, fp32 accumulation, the sum rounded to bf16 before f: out[m][n] = f(sum_k x(m, k) w(n, k)), out (M, N) row-major.  x is (M, K) row-major, with km its
 * transpose (K, M); w is (N, K), with kn (K, N).  For the low-rank factors of RWKV-7's decay, gates and value residual
 * (rwkv7.py:237-245) and their cotangents.  f: without aux 0 none, 1 tanh, 2 sigmoid, 3 relu(.)^2; with aux, an (M, N) array:
 * 0 + aux, 1 times 1 - aux^2, 2 times aux (1 - aux) (the derivatives in terms of the activations' values).  Sizes that are
 * contiguous in memory must be multiples of 8. */
#define HIPRWKV_GEMM_MAX_JOBS 8
typedef struct hiprwkv_gemm_job {
  const void *x, *w, *aux;
  void* out;
  int32_t M, N, K, km, kn, act;
  int32_t tile0, pad;      /* used by the library */
} hiprwkv_gemm_job;
int hiprwkv_gemm(hiprwkv_stream stream, int n_jobs, const hiprwkv_gemm_job* jobs);

/* ---- RWKV-7: a decode step of the whole model ---------------------------------------------------------
 * rwkv7.py:190-198, :223-291 for at most HIPRWKV_SMALL_T tokens per sequence and HIPRWKV_DECODE_MAX_ROWS tokens in all, bf16
 * throughout, from the embedded tokens to the last norm (and, where `logits` is given, through the head).  Parameters are
 * the reference's arrays stacked over the L layers, contiguous: vectors (L, C), r_k (L, H, 64), receptance / key / value /
 * output (L, C, C) and ffn_key (L, F, C), ffn_value (L, C, F) used as x W^T, the low-rank factors (L, C, d) and (L, d, C)
 * used as x W; head (vocab, C).  state and new_state are (B, L, 2 + 64, C) and different arrays; length (B,) int32 or
 * NULL (= T), new_starts (B, T) or NULL.  C = 64 H at most 4096; d_* and F multiples of 32; vocab a multiple of 16.
 * x (B*T, C) in, xn (B*T, C) out, logits (B*T, vocab) out or NULL.  flags: HIPRWKV_COMPAT_ASSOC. */
#define HIPRWKV_DECODE_MAX_ROWS 256
typedef struct hiprwkv_rwkv7_decode_args {
  int64_t B, T, L, C, H, F, vocab, d_decay, d_aaa, d_mv, d_gate;
  const void *x, *state;
  void *new_state;
  const int32_t* length;
  const uint8_t* new_starts;
  const void *ln0_w, *ln0_b, *ln_out_w, *ln_out_b, *head, *ln1_w, *ln1_b, *ln2_w, *ln2_b;
  const void *x_r, *x_w, *x_k, *x_v, *x_a, *x_g;
  const void *w0, *w1, *w2, *a0, *a1, *a2, *v0, *v1, *v2, *g1, *g2, *k_k, *k_a, *r_k;
  const void *receptance, *key, *value, *output, *lnx_w, *lnx_b, *ffn_x_k, *ffn_key, *ffn_value;
  void *xn, *logits, *workspace;
  uint64_t workspace_bytes;
  uint64_t flags;
} hiprwkv_rwkv7_decode_args;
size_t hiprwkv_rwkv7_decode_workspace_bytes(const hiprwkv_rwkv7_decode_args* args);
int hiprwkv_rwkv7_decode(hiprwkv_stream stream, const hiprwkv_rwkv7_decode_args* args);

/* ---- The stack of RWKV-7 blocks over whole sequences -------------------------------------
 * rwkv7.py:190-198, :223-291 without the norms around the stack, bf16, all tokens of B sequences through L layers.  C = 64 H, at most
 * 4096; F and the four inner sizes multiples of 8; no array of 2 GiB or more; parameters stacked over the layers, one contiguous array
 * each, in the orders of hiprwkv_rwkv7_decode_args.
 *   forward : from x (B,T,C) and the states the residual stream as a sum xs + dx.  state (B,L,2+64,C): rows 0 and 1 are the token-shift
 *             states, read there and written in new_state; s, new_s (L,B,64,C): the recurrence's, as arrays of their own.
 *             saved: L allocations for the backward, or null without one to come; of layer l hiprwkv_rwkv7_stack_saved_layer_bytes,
 *             of any hiprwkv_rwkv7_stack_saved_bytes.
 *   backward: from g_xs, g_dx and, where not null, the cotangents of the new shift states g_shift (2,L,B,C) and recurrence states g_s
 *             (L,B,64,C) to g_x and every parameter's (grad, same order as param; rows of layer 0 of v0, v1, v2 are left alone).  The
 *             forward's x, xs, state, s and saved go in again; there is no cotangent of the states. */
typedef struct hiprwkv_rwkv7_block_params {
  const void *x_r, *x_w, *x_k, *x_v, *x_a, *x_g;
  const void *w0, *w1, *w2, *a0, *a1, *a2, *v0, *v1, *v2, *g1, *g2, *k_k, *k_a, *r_k;
  const void *receptance, *key, *value, *output, *lnx_w, *lnx_b, *ffn_x_k, *ffn_key, *ffn_value, *ln1_w, *ln1_b, *ln2_w, *ln2_b;
} hiprwkv_rwkv7_block_params;
typedef struct hiprwkv_rwkv7_stack_args {
  int64_t B, T, L, C, H, F, d_decay, d_aaa, d_mv, d_gate;
  const void *x, *state, *s;
  void *new_state, *new_s;
  const int32_t* length;
  const uint8_t* new_starts;
  void *xs, *dx;
  void* const* saved;
  void* workspace;
  uint64_t workspace_bytes, flags;
  const void *g_xs, *g_dx, *g_shift, *g_s;
  void* g_x;
  hiprwkv_rwkv7_block_params param, grad;
} hiprwkv_rwkv7_stack_args;
size_t hiprwkv_rwkv7_stack_saved_bytes(const hiprwkv_rwkv7_stack_args* args);
size_t hiprwkv_rwkv7_stack_saved_layer_bytes(const hiprwkv_rwkv7_stack_args* args, int64_t layer);
size_t hiprwkv_rwkv7_stack_workspace_bytes(const hiprwkv_rwkv7_stack_args* args, int backward);
int hiprwkv_rwkv7_stack_fwd(hiprwkv_stream stream, const hiprwkv_rwkv7_stack_args* args);
int hiprwkv_rwkv7_stack_bwd(hiprwkv_stream stream, const hiprwkv_rwkv7_stack_args* args);

/* ---- RWKV-7 time-mixing stages around the op ------------------------------------------
 * The element-wise work the reference does in jnp on either side of inner_loop (rwkv7.py:248-252, 257 and :263-265),
 * fused into one pass each; it has no counterpart among the reference's ffi targets.  `rows` = number of tokens
 * (all batch axes flattened), tensors (rows, H, 64) io_dtype, parameters k_k, k_a, ln_w, ln_b, r_k (H, 64) io_dtype.
 *   premix : kk = normalize_head(k . k_k); k_out = k (1 + (a - 1) k_a); a_out = -kk; b_out = kk . a
 *   postmix: out = (group_norm_head(y, eps) . ln_w + ln_b + (sum_j r_j k_j r_k_j) v) . g      (k = premix's k_out) */
int hiprwkv_rwkv7_premix(hiprwkv_stream stream, int io_dtype, int64_t rows, int64_t H, int64_t N,
                         const void* k, const void* a, const void* k_k, const void* k_a,
                         void* k_out, void* a_out, void* b_out);
int hiprwkv_rwkv7_postmix(hiprwkv_stream stream, int io_dtype, int64_t rows, int64_t H, int64_t N,
                          const void* y, const void* r, const void* k, const void* v, const void* g,
                          const void* ln_w, const void* ln_b, const void* r_k, float eps, void* out);

/* Their backward passes (what jax.grad derives for rwkv7.py:248-252, 257 and :263-265).  The forward quantities are
 * recomputed from the same inputs; nothing is saved.  Cotangents of tensors are io_dtype (rows, H, 64); cotangents of
 * the per-head parameters (sums over all rows) are always fp32 (H, 64) and are overwritten, not accumulated into.
 *   premix_bwd : from the cotangents of k_out, a_out, b_out to those of k, a, k_k, k_a
 *   postmix_bwd: from the cotangent of out to those of y, r, k, v, g, ln_w, ln_b, r_k */
int hiprwkv_rwkv7_premix_bwd(hiprwkv_stream stream, int io_dtype, int64_t rows, int64_t H, int64_t N,
                             const void* k, const void* a, const void* k_k, const void* k_a,
                             const void* gk_out, const void* ga_out, const void* gb_out,
                             void* gk, void* ga, float* gk_k, float* gk_a);
int hiprwkv_rwkv7_postmix_bwd(hiprwkv_stream stream, int io_dtype, int64_t rows, int64_t H, int64_t N,
                              const void* y, const void* r, const void* k, const void* v, const void* g,
                              const void* ln_w, const void* ln_b, const void* r_k, float eps, const void* gout,
                              void* gy, void* gr, void* gk, void* gv, void* gg,
                              float* gln_w, float* gln_b, float* gr_k);

/* hiprwkv_rwkv7_postmix_bwd with the parameter cotangents as three (H, 64) io_dtype arrays, dparam = ln_w, ln_b, r_k, summed
 * through `workspace` instead of atomics. */
size_t hiprwkv_rwkv7_postmix_bwd2_workspace_bytes(int64_t rows, int64_t H, int64_t N);
int hiprwkv_rwkv7_postmix_bwd2(hiprwkv_stream stream, int io_dtype, int64_t rows, int64_t H, int64_t N,
                               const void* y, const void* r, const void* k, const void* v, const void* g,
                               const void* ln_w, const void* ln_b, const void* r_k, float eps, const void* gout,
                               void* gy, void* gr, void* gk, void* gv, void* gg, void* const* dparam, void* workspace,
                               size_t workspace_bytes);

#ifdef __cplusplus
}
#endif
#endif /* HIPRWKV_H_ */
