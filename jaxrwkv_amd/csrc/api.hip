// C ABI of libhiprwkv: argument checks, workspace carving, kernel selection.  Declarations: include/hiprwkv.h
#include "../../include/hiprwkv.h"

#include <stdarg.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include <algorithm>
#include <initializer_list>
#include <mutex>

#include "wkv_args.h"

using namespace hiprwkv;

namespace {

thread_local char g_err[512] = "";

int fail(int code, const char* fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_err, sizeof(g_err), fmt, ap);
  va_end(ap);
  return code;
}

bool dtype_ok(int d) { return d == HIPRWKV_F32 || d == HIPRWKV_BF16; }

size_t align256(size_t x) { return (x + 255) & ~(size_t)255; }

// Rows of different (B,T,H,N) arrays at the same (token, head) are accessed together; arrays whose base addresses are
// congruent modulo 1 KiB then compete for the same part of the memory system (measured on MI355X: the backward sweeps
// that read and write the workspace arrays lose 5-10 % when everything starts on a 2 MiB boundary, and offsets that
// are multiples of 1 KiB change nothing).  The workspace arrays therefore start at their own 128-byte step past the
// phase of the first operand.
constexpr size_t PHASE_BYTES = 128, PHASE_SPAN = 1024;
char* at_phase(char* p, const void* like, unsigned steps) {
  const uintptr_t want = (reinterpret_cast<uintptr_t>(like) + steps * PHASE_BYTES) % PHASE_SPAN / PHASE_BYTES * PHASE_BYTES;
  const uintptr_t at = reinterpret_cast<uintptr_t>(p);
  const uintptr_t up = (at + 15) & ~(uintptr_t)15;
  return reinterpret_cast<char*>(up + (want + PHASE_SPAN - up % PHASE_SPAN) % PHASE_SPAN);
}

int check_matrix_shape(const char* op, int io_dtype, int state_dtype, int64_t B, int64_t T, int64_t H, int64_t N) {
  if (!dtype_ok(io_dtype) || !dtype_ok(state_dtype)) return fail(HIPRWKV_EINVAL, "%s: dtype must be HIPRWKV_F32 or HIPRWKV_BF16", op);
  if (N != 64) return fail(HIPRWKV_EINVAL, "%s: head size N=%lld not supported (kernels are built for N=64)", op, (long long)N);
  if (B <= 0 || T <= 0 || H <= 0) return fail(HIPRWKV_EINVAL, "%s: B,T,H must be positive (got %lld,%lld,%lld)", op, (long long)B, (long long)T, (long long)H);
  if (B * H > 0x7fffffffLL) return fail(HIPRWKV_EINVAL, "%s: B*H exceeds the grid limit", op);
  return HIPRWKV_OK;
}

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

// Word 0 counts the workgroups of the chunked kernels whose bounded hand-shake wait ran out (they overwrite their
// outputs with NaN and add one here).  Word 1 counts numeric events of the chunked kernels: waves that had to cap a
// channel's decay over a chunk, and waves that found inf or NaN in a carried state (an fp16 operand overflowed).
// Every GPU holds its own copy of the words; their address is looked up once per device.
__device__ unsigned int g_status_words[2] = {0u, 0u};

constexpr int MAX_DEVICES = 64;
std::mutex g_sym_mu;
unsigned* g_status_ptr[MAX_DEVICES] = {};

// Workspace of hiprwkv_wkv4_bwd_noalloc: the checkpoint array of the WKV4 backward pass, (B, ceil(T/16), 3, C) fp32,
// for callers that cannot allocate.  Every GPU the library runs on holds its own 16 MiB copy until the process
// ends.  Host code never uses the array's name as an address: the device address is looked up once per device
// (scratch_base) and passed to the kernels like a caller's workspace.
constexpr size_t SCRATCH_BYTES = (size_t)16 << 20;
static __device__ __align__(256) __attribute__((used)) unsigned char scratch[SCRATCH_BYTES];
void* g_scratch_ptr[MAX_DEVICES] = {};

// Device address of the current device's scratch array; null (with the error text set) when the lookup fails.
void* scratch_base() {
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess || dev < 0 || dev >= MAX_DEVICES) {
    fail(HIPRWKV_ELAUNCH, "wkv4_bwd_noalloc: no usable current device (%s)", hipGetErrorString(e));
    return nullptr;
  }
  std::lock_guard<std::mutex> lock(g_sym_mu);
  if (g_scratch_ptr[dev] == nullptr) {
    void* p = nullptr;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || p == nullptr) {
      fail(HIPRWKV_ELAUNCH, "wkv4_bwd_noalloc: hipGetSymbolAddress failed (%s)", hipGetErrorString(e));
      return nullptr;
    }
    g_scratch_ptr[dev] = p;
  }
  return g_scratch_ptr[dev];
}

// Public flag bits are accepted everywhere; the test hook HIPRWKV_DEBUG_DROP_PUBLISH only in a process that sets the
// environment variable HIPRWKV_ENABLE_DEBUG_FLAGS=1, so that a stray bit cannot turn a production call's outputs
// into NaN.  Unknown bits are refused.
int check_flags(const char* op, unsigned flags, bool new_state_io = false) {
  const unsigned known = HIPRWKV_PUBLIC_FLAGS | HIPRWKV_DEBUG_DROP_PUBLISH | (new_state_io ? HIPRWKV_NEW_STATE_IO : 0u);
  if (flags & ~known) return fail(HIPRWKV_EINVAL, "%s: unknown flag bits 0x%x", op, flags & ~known);
  if (flags & HIPRWKV_DEBUG_DROP_PUBLISH) {
    static const bool enabled = [] { const char* e = getenv("HIPRWKV_ENABLE_DEBUG_FLAGS"); return e != nullptr && e[0] == '1'; }();
    if (!enabled)
      return fail(HIPRWKV_EINVAL, "%s: HIPRWKV_DEBUG_DROP_PUBLISH needs HIPRWKV_ENABLE_DEBUG_FLAGS=1 in the environment", op);
  }
  return HIPRWKV_OK;
}

// Address of the current device's failure counter, or null when it cannot be obtained (the kernels then skip the
// count; the NaN poisoning does not depend on it).
unsigned* status_word() {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= MAX_DEVICES) return nullptr;
  std::lock_guard<std::mutex> lock(g_sym_mu);
  if (g_status_ptr[dev] == nullptr) {
    void* p = nullptr;
    if (hipGetSymbolAddress(&p, HIP_SYMBOL(g_status_words)) != hipSuccess) return nullptr;
    g_status_ptr[dev] = static_cast<unsigned*>(p);
  }
  return g_status_ptr[dev];
}

}  // namespace

extern "C" {

const char* hiprwkv_last_error(void) { return g_err; }
int hiprwkv_version(void) { return 107; }

int hiprwkv_handshake_failures(hiprwkv_stream stream, unsigned* count) {
  if (count == nullptr) return fail(HIPRWKV_EINVAL, "handshake_failures: null count pointer");
  unsigned* word = status_word();
  if (word == nullptr) return fail(HIPRWKV_ELAUNCH, "handshake_failures: the device counter is not reachable");
  hipStream_t st = static_cast<hipStream_t>(stream);
  hipError_t e = hipMemcpyAsync(count, word, sizeof(unsigned), hipMemcpyDeviceToHost, st);
  if (e == hipSuccess) e = hipStreamSynchronize(st);
  if (e != hipSuccess) return fail(HIPRWKV_ELAUNCH, "handshake_failures: %s", hipGetErrorString(e));
  return HIPRWKV_OK;
}

int hiprwkv_numeric_events(hiprwkv_stream stream, unsigned* count) {
  if (count == nullptr) return fail(HIPRWKV_EINVAL, "numeric_events: null count pointer");
  unsigned* word = status_word();
  if (word == nullptr) return fail(HIPRWKV_ELAUNCH, "numeric_events: the device counter is not reachable");
  hipStream_t st = static_cast<hipStream_t>(stream);
  hipError_t e = hipMemcpyAsync(count, word + 1, sizeof(unsigned), hipMemcpyDeviceToHost, st);
  if (e == hipSuccess) e = hipStreamSynchronize(st);
  if (e != hipSuccess) return fail(HIPRWKV_ELAUNCH, "numeric_events: %s", hipGetErrorString(e));
  return HIPRWKV_OK;
}

int hiprwkv_wkv7_fwd(hiprwkv_stream stream, int io_dtype, int state_dtype, int64_t B, int64_t T, int64_t H, int64_t N,
                     const void* w, const void* r, const void* k, const void* v, const void* a, const void* b,
                     const void* s, const uint32_t* length, const uint8_t* new_starts, void* out, void* sa,
                     void* new_s, unsigned flags) {
  return hiprwkv_wkv7_fwd_parts(stream, io_dtype, state_dtype, B, T, H, N, w, r, k, v, a, b, s, length, new_starts, out, sa, new_s,
                                nullptr, 0, flags);
}

// whether sequences of this shape may run in parts
static bool wkv7_in_parts(int io_dtype, int64_t B, int64_t T, int64_t H, int64_t N) {
  return (io_dtype == HIPRWKV_BF16 || io_dtype == HIPRWKV_F32) && N == 64 && B > 0 && T > HIPRWKV_SMALL_T && H > 0 && B * H <= 0x7fffffffLL;
}

size_t hiprwkv_wkv7_fwd_workspace_bytes(int io_dtype, int64_t B, int64_t T, int64_t H, int64_t N) {
  if (!wkv7_in_parts(io_dtype, B, T, H, N)) return 0;
  return wkv7_fwd_parts_bytes(B * H, T, io_dtype == HIPRWKV_F32);
}

int hiprwkv_wkv7_fwd_parts(hiprwkv_stream stream, int io_dtype, int state_dtype, int64_t B, int64_t T, int64_t H, int64_t N,
                           const void* w, const void* r, const void* k, const void* v, const void* a, const void* b,
                           const void* s, const uint32_t* length, const uint8_t* new_starts, void* out, void* sa,
                           void* new_s, void* workspace, size_t workspace_bytes, unsigned flags) {
  return hiprwkv_wkv7_fwd_ends(stream, io_dtype, state_dtype, B, T, H, N, w, r, k, v, a, b, s, length, new_starts, out, sa, new_s,
                               nullptr, workspace, workspace_bytes, flags);
}

size_t hiprwkv_wkv7_ends_bytes(int io_dtype, int64_t B, int64_t T, int64_t H, int64_t N) {
  if (!wkv7_in_parts(io_dtype, B, T, H, N)) return 0;
  const bool f32 = io_dtype == HIPRWKV_F32;
  return wkv7_ends_bytes(B * H, wkv7_bwd_parts(B * H, T, f32), f32);
}

int hiprwkv_wkv7_fwd_ends(hiprwkv_stream stream, int io_dtype, int state_dtype, int64_t B, int64_t T, int64_t H, int64_t N,
                          const void* w, const void* r, const void* k, const void* v, const void* a, const void* b,
                          const void* s, const uint32_t* length, const uint8_t* new_starts, void* out, void* sa,
                          void* new_s, void* ends, void* workspace, size_t workspace_bytes, unsigned flags) {
  int rc = check_matrix_shape("wkv7_fwd", io_dtype, state_dtype, B, T, H, N);
  if (rc) return rc;
  if ((rc = check_flags("wkv7_fwd", flags, true)) != HIPRWKV_OK) return rc;
  if ((flags & HIPRWKV_NEW_STATE_IO) && io_dtype != state_dtype && s == new_s)
    return fail(HIPRWKV_EINVAL, "wkv7_fwd: s and new_s must be different arrays where their types differ");
  const void* req[] = {w, r, k, v, a, b, s, out, new_s};
  for (const void* p : req) {
    if (p == nullptr) return fail(HIPRWKV_EINVAL, "wkv7_fwd: null tensor pointer");
    if (!aligned16(p)) return fail(HIPRWKV_EINVAL, "wkv7_fwd: tensor pointers must be 16-byte aligned");
  }
  if (sa && !aligned16(sa)) return fail(HIPRWKV_EINVAL, "wkv7_fwd: sa must be 16-byte aligned");
  if (ends && (!aligned16(ends) || !sa || (flags & HIPRWKV_FORCE_SEQ)))
    return fail(HIPRWKV_EINVAL, "wkv7_fwd: ends must be 16-byte aligned and goes with sa, without HIPRWKV_FORCE_SEQ");
  if (workspace && !aligned16(workspace)) return fail(HIPRWKV_EINVAL, "wkv7_fwd: workspace must be 16-byte aligned");
  const size_t need = workspace != nullptr ? hiprwkv_wkv7_fwd_workspace_bytes(io_dtype, B, T, H, N) : 0;
  if (workspace_bytes < need)
    return fail(HIPRWKV_ENOSPACE, "wkv7_fwd: workspace has %zu bytes, %zu needed", workspace_bytes, need);
  Wkv7Args A;
  memset(&A, 0, sizeof(A));
  A.B = B; A.T = T; A.H = H;
  A.w = w; A.r = r; A.k = k; A.v = v; A.a = a; A.b = b; A.s = s;
  A.length = length; A.ns = new_starts;
  A.out = out; A.sa = sa; A.new_s = new_s;
  A.io_f32 = io_dtype == HIPRWKV_F32; A.st_f32 = state_dtype == HIPRWKV_F32; A.new_st_f32 = (flags & HIPRWKV_NEW_STATE_IO) ? A.io_f32 : A.st_f32;
  A.flags = flags;
  A.status = status_word();
  A.parts = need != 0 ? workspace : nullptr;
  if (A.io_f32 && ends != nullptr && hiprwkv_wkv7_ends_bytes(io_dtype, B, T, H, N) != 0) {      // in bf16 the backward fills it
    const Wkv7BwdSplit S = wkv7_bwd_parts(B * H, T, true);
    A.ends = static_cast<float*>(ends); A.n_end = S.n_end; A.end_chunks = S.end_chunks;
  }
  // T <= 8 (decode) runs on the small-T kernel; otherwise the chunked matrix-core kernels (fp16 operands for bf16
  // I/O, fp32 operands for fp32 I/O); HIPRWKV_FORCE_SEQ selects the sequential kernel
  const bool small_t = T <= HIPRWKV_SMALL_T && !(flags & HIPRWKV_NO_SMALL_T);
  const bool chunked = !(flags & HIPRWKV_FORCE_SEQ);
  hipStream_t st = static_cast<hipStream_t>(stream);
  hipError_t e = small_t ? launch_wkv7_small_t_fwd(A, st)
               : !chunked ? launch_wkv7_seq_fwd(A, st)
               : A.io_f32 ? launch_wkv7_chunk_fwd_f32(A, st) : launch_wkv7_chunk_fwd(A, st);
  if (e != hipSuccess) return fail(HIPRWKV_ELAUNCH, "wkv7_fwd: %s", hipGetErrorString(e));
  return HIPRWKV_OK;
}

int hiprwkv_wkv7_step(hiprwkv_stream stream, int io_dtype, int state_dtype, int64_t B, int64_t T, int64_t H, int64_t N,
                      const void* w, const void* r, const void* k, const void* v, const void* a, const void* b,
                      const void* s, int64_t s_batch_stride, const uint32_t* length, const uint8_t* new_starts,
                      void* out, void* new_s, int64_t new_s_batch_stride, unsigned flags) {
  int rc = check_matrix_shape("wkv7_step", io_dtype, state_dtype, B, T, H, N);
  if (rc) return rc;
  if ((rc = check_flags("wkv7_step", flags)) != HIPRWKV_OK) return rc;
  if (T > HIPRWKV_SMALL_T) return fail(HIPRWKV_EINVAL, "wkv7_step: T=%lld, at most %d tokens per call", (long long)T, HIPRWKV_SMALL_T);
  const void* req[] = {w, r, k, v, a, b, s, out, new_s};
  for (const void* p : req) {
    if (p == nullptr) return fail(HIPRWKV_EINVAL, "wkv7_step: null tensor pointer");
    if (!aligned16(p)) return fail(HIPRWKV_EINVAL, "wkv7_step: tensor pointers must be 16-byte aligned");
  }
  const int64_t dense = H * N * N;
  const int64_t elem = state_dtype == HIPRWKV_F32 ? 4 : 2;
  for (int64_t stride : {s_batch_stride, new_s_batch_stride}) {
    if (stride < dense) return fail(HIPRWKV_EINVAL, "wkv7_step: state batch stride %lld is less than H*N*N = %lld", (long long)stride, (long long)dense);
    if ((stride * elem) % 16 != 0) return fail(HIPRWKV_EINVAL, "wkv7_step: state batch stride must be a multiple of 16 bytes");
  }
  Wkv7Args A;
  memset(&A, 0, sizeof(A));
  A.B = B; A.T = T; A.H = H;
  A.w = w; A.r = r; A.k = k; A.v = v; A.a = a; A.b = b; A.s = s;
  A.length = length; A.ns = new_starts;
  A.out = out; A.new_s = new_s;
  A.io_f32 = io_dtype == HIPRWKV_F32; A.st_f32 = A.new_st_f32 = state_dtype == HIPRWKV_F32;
  A.flags = flags;
  A.s_bstride = s_batch_stride; A.new_s_bstride = new_s_batch_stride;
  const hipError_t e = launch_wkv7_small_t_fwd(A, static_cast<hipStream_t>(stream));
  if (e != hipSuccess) return fail(HIPRWKV_ELAUNCH, "wkv7_step: %s", hipGetErrorString(e));
  return HIPRWKV_OK;
}

size_t hiprwkv_wkv7_bwd_workspace_bytes(int64_t B, int64_t T, int64_t H, int64_t N) {
  // three fp32 arrays with one value per token and key; the second one is kept per chunk of 16 tokens (f_record)
  const size_t tokens = (size_t)((T + 15) / 16) * 16;
  return 3 * (align256((size_t)B * tokens * H * N * sizeof(float)) + PHASE_SPAN);
}

int hiprwkv_wkv7_bwd(hiprwkv_stream stream, int io_dtype, int state_dtype, int64_t B, int64_t T, int64_t H, int64_t N,
                     const void* w, const void* r, const void* k, const void* v, const void* a, const void* b,
                     const void* s, const uint32_t* length, const uint8_t* new_starts, const void* gy, const void* sa,
                     const void* gs_out, void* gw, void* gr, void* gk, void* gv, void* ga, void* gb, void* gs,
                     void* workspace, size_t workspace_bytes, unsigned flags) {
  return hiprwkv_wkv7_bwd_ends(stream, io_dtype, state_dtype, B, T, H, N, w, r, k, v, a, b, s, length, new_starts, gy, sa, gs_out,
                               nullptr, gw, gr, gk, gv, ga, gb, gs, workspace, workspace_bytes, flags);
}

size_t hiprwkv_wkv7_bwd_ends_workspace_bytes(int io_dtype, int64_t B, int64_t T, int64_t H, int64_t N) {
  const size_t base = hiprwkv_wkv7_bwd_workspace_bytes(B, T, H, N);
  if (hiprwkv_wkv7_ends_bytes(io_dtype, B, T, H, N) == 0) return base;
  const Wkv7BwdSplit S = wkv7_bwd_parts(B * H, T, io_dtype == HIPRWKV_F32);
  return base + 16 + wkv7_ends_bytes(B * H, S, true) + wkv7_bwd_sums_bytes(B * H, S);      // the cotangents are matrices in both types
}

int hiprwkv_wkv7_bwd_ends(hiprwkv_stream stream, int io_dtype, int state_dtype, int64_t B, int64_t T, int64_t H, int64_t N,
                          const void* w, const void* r, const void* k, const void* v, const void* a, const void* b,
                          const void* s, const uint32_t* length, const uint8_t* new_starts, const void* gy, const void* sa,
                          const void* gs_out, void* ends, void* gw, void* gr, void* gk, void* gv, void* ga, void* gb,
                          void* gs, void* workspace, size_t workspace_bytes, unsigned flags) {
  int rc = check_matrix_shape("wkv7_bwd", io_dtype, state_dtype, B, T, H, N);
  if (rc) return rc;
  if ((rc = check_flags("wkv7_bwd", flags)) != HIPRWKV_OK) return rc;
  const void* req[] = {w, r, k, v, a, b, s, gy, sa, gw, gr, gk, gv, ga, gb, gs, workspace};
  for (const void* p : req) {
    if (p == nullptr) return fail(HIPRWKV_EINVAL, "wkv7_bwd: null tensor pointer");
    if (!aligned16(p)) return fail(HIPRWKV_EINVAL, "wkv7_bwd: tensor pointers must be 16-byte aligned");
  }
  if (ends && (!aligned16(ends) || (flags & HIPRWKV_FORCE_SEQ)))
    return fail(HIPRWKV_EINVAL, "wkv7_bwd: ends must be 16-byte aligned and does not go with HIPRWKV_FORCE_SEQ");
  const size_t base = hiprwkv_wkv7_bwd_workspace_bytes(B, T, H, N);
  const size_t need = ends != nullptr ? hiprwkv_wkv7_bwd_ends_workspace_bytes(io_dtype, B, T, H, N) : base;
  if (workspace_bytes < need)
    return fail(HIPRWKV_ENOSPACE, "wkv7_bwd: workspace has %zu bytes, %zu needed", workspace_bytes, need);
  Wkv7Args A;
  memset(&A, 0, sizeof(A));
  A.B = B; A.T = T; A.H = H;
  A.w = w; A.r = r; A.k = k; A.v = v; A.a = a; A.b = b; A.s = s;
  A.length = length; A.ns = new_starts;
  A.io_f32 = io_dtype == HIPRWKV_F32; A.st_f32 = state_dtype == HIPRWKV_F32;
  A.flags = flags;
  A.status = status_word();
  A.gy = gy; A.sa_in = sa; A.gs_out = gs_out;
  A.gw = gw; A.gr = gr; A.gk = gk; A.gv = gv; A.ga = ga; A.gb = gb; A.gs = gs;
  const size_t one = base / 3 - PHASE_SPAN;
  char* ws = static_cast<char*>(workspace);
  A.n_end = 1; A.end_chunks = (int)((T + 15) / 16);
  if (ends != nullptr && hiprwkv_wkv7_ends_bytes(io_dtype, B, T, H, N) != 0) {
    const Wkv7BwdSplit S = wkv7_bwd_parts(B * H, T, io_dtype == HIPRWKV_F32);
    A.n_end = S.n_end; A.end_chunks = S.end_chunks;
    A.ends = static_cast<float*>(ends);
    char* const more = ws + (base + 15) / 16 * 16;
    A.gends = reinterpret_cast<float*>(more);
    if (S.a_parts) { A.parts = more + wkv7_ends_bytes(B * H, S, true); A.n_part = S.n_end; A.part_chunks = S.end_chunks; }
  }
  A.dsa = reinterpret_cast<float*>(at_phase(ws, r, 3));
  A.e2 = reinterpret_cast<float*>(at_phase(reinterpret_cast<char*>(A.dsa) + one, r, 5));
  A.e3 = reinterpret_cast<float*>(at_phase(reinterpret_cast<char*>(A.e2) + one, r, 7));
  // Three sweeps: A (reverse) -> gv, dsa, gs; B (forward) -> gr, ga, e2, e3 (the chunked B: their sum shifted by a
  // token, in e2); C (reverse) -> gk, gb, gw.
  // All three run on the chunked matrix-core kernels (bf16 pairs for bf16 I/O, fp32 operands for fp32 I/O);
  // HIPRWKV_FORCE_SEQ selects the sequential kernels.
  const bool chunked = !(flags & HIPRWKV_FORCE_SEQ);
  const bool f32 = A.io_f32 != 0;
  hipStream_t st = static_cast<hipStream_t>(stream);
  hipError_t e = !chunked ? launch_wkv7_seq_bwd_a(A, st) : f32 ? launch_wkv7_chunk_bwd_a_f32(A, st) : launch_wkv7_chunk_bwd_a(A, st);
  if (e == hipSuccess)
    e = !chunked ? launch_wkv7_seq_bwd_b(A, st) : f32 ? launch_wkv7_chunk_bwd_b_f32(A, st) : launch_wkv7_chunk_bwd_b(A, st);
  if (e == hipSuccess)
    e = !chunked ? launch_wkv7_seq_bwd_c(A, st) : f32 ? launch_wkv7_chunk_bwd_c_f32(A, st) : launch_wkv7_chunk_bwd_c(A, st);
  if (e != hipSuccess) return fail(HIPRWKV_ELAUNCH, "wkv7_bwd: %s", hipGetErrorString(e));
  return HIPRWKV_OK;
}

int hiprwkv_wkv6_fwd(hiprwkv_stream stream, int io_dtype, int state_dtype, int64_t B, int64_t T, int64_t H, int64_t N,
                     const void* r, const void* k, const void* v, const void* w, const void* u, const void* s,
                     const uint32_t* length, const uint8_t* new_starts, void* out, void* new_s, unsigned flags) {
  return hiprwkv_wkv6_fwd_parts(stream, io_dtype, state_dtype, B, T, H, N, r, k, v, w, u, s, length, new_starts, out, new_s, nullptr, 0,
                                flags);
}

size_t hiprwkv_wkv6_fwd_workspace_bytes(int io_dtype, int64_t B, int64_t T, int64_t H, int64_t N) {
  if (io_dtype != HIPRWKV_BF16 || N != 64 || B <= 0 || T <= HIPRWKV_SMALL_T || H <= 0 || B * H > 0x7fffffffLL) return 0;
  return wkv6_fwd_parts_bytes(B * H, T);
}

int hiprwkv_wkv6_fwd_parts(hiprwkv_stream stream, int io_dtype, int state_dtype, int64_t B, int64_t T, int64_t H, int64_t N,
                           const void* r, const void* k, const void* v, const void* w, const void* u, const void* s,
                           const uint32_t* length, const uint8_t* new_starts, void* out, void* new_s, void* workspace,
                           size_t workspace_bytes, unsigned flags) {
  int rc = check_matrix_shape("wkv6_fwd", io_dtype, state_dtype, B, T, H, N);
  if (rc) return rc;
  if ((rc = check_flags("wkv6_fwd", flags, true)) != HIPRWKV_OK) return rc;
  if ((flags & HIPRWKV_NEW_STATE_IO) && io_dtype != state_dtype && s == new_s)
    return fail(HIPRWKV_EINVAL, "wkv6_fwd: s and new_s must be different arrays where their types differ");
  const void* req[] = {r, k, v, w, u, s, out, new_s};
  for (const void* p : req) {
    if (p == nullptr) return fail(HIPRWKV_EINVAL, "wkv6_fwd: null tensor pointer");
    if (!aligned16(p)) return fail(HIPRWKV_EINVAL, "wkv6_fwd: tensor pointers must be 16-byte aligned");
  }
  if (workspace && !aligned16(workspace)) return fail(HIPRWKV_EINVAL, "wkv6_fwd: workspace must be 16-byte aligned");
  const size_t need = workspace != nullptr ? hiprwkv_wkv6_fwd_workspace_bytes(io_dtype, B, T, H, N) : 0;
  if (workspace_bytes < need)
    return fail(HIPRWKV_ENOSPACE, "wkv6_fwd: workspace has %zu bytes, %zu needed", workspace_bytes, need);
  Wkv6Args A;
  memset(&A, 0, sizeof(A));
  A.B = B; A.T = T; A.H = H;
  A.r = r; A.k = k; A.v = v; A.w = w; A.u = u; A.s = s;
  A.length = length; A.ns = new_starts;
  A.out = out; A.new_s = new_s;
  A.io_f32 = io_dtype == HIPRWKV_F32; A.st_f32 = state_dtype == HIPRWKV_F32; A.new_st_f32 = (flags & HIPRWKV_NEW_STATE_IO) ? A.io_f32 : A.st_f32;
  A.flags = flags;
  A.parts = need != 0 ? workspace : nullptr;
  A.status = status_word();
  // chunked matrix-core kernels (fp16 operands for bf16 I/O, fp32 operands for fp32 I/O) unless HIPRWKV_FORCE_SEQ
  const bool chunked = !(flags & HIPRWKV_FORCE_SEQ);
  const bool small_t = T <= HIPRWKV_SMALL_T && !(flags & HIPRWKV_NO_SMALL_T);
  hipStream_t st = static_cast<hipStream_t>(stream);
  hipError_t e = small_t ? launch_wkv6_small_t_fwd(A, st)
               : !chunked ? launch_wkv6_seq_fwd(A, st)
               : A.io_f32 ? launch_wkv6_chunk_fwd_f32(A, st) : launch_wkv6_chunk_fwd(A, st);
  if (e != hipSuccess) return fail(HIPRWKV_ELAUNCH, "wkv6_fwd: %s", hipGetErrorString(e));
  return HIPRWKV_OK;
}

int hiprwkv_wkv6_step(hiprwkv_stream stream, int io_dtype, int state_dtype, int64_t B, int64_t T, int64_t H, int64_t N,
                      const void* r, const void* k, const void* v, const void* w, const void* u, const void* s,
                      int64_t s_batch_stride, const uint32_t* length, const uint8_t* new_starts, void* out, void* new_s,
                      int64_t new_s_batch_stride, unsigned flags) {
  int rc = check_matrix_shape("wkv6_step", io_dtype, state_dtype, B, T, H, N);
  if (rc) return rc;
  if ((rc = check_flags("wkv6_step", flags)) != HIPRWKV_OK) return rc;
  if (T > HIPRWKV_SMALL_T) return fail(HIPRWKV_EINVAL, "wkv6_step: T=%lld, at most %d tokens per call", (long long)T, HIPRWKV_SMALL_T);
  const void* req[] = {r, k, v, w, u, s, out, new_s};
  for (const void* p : req) {
    if (p == nullptr) return fail(HIPRWKV_EINVAL, "wkv6_step: null tensor pointer");
    if (!aligned16(p)) return fail(HIPRWKV_EINVAL, "wkv6_step: tensor pointers must be 16-byte aligned");
  }
  const int64_t dense = H * N * N;
  const int64_t elem = state_dtype == HIPRWKV_F32 ? 4 : 2;
  for (int64_t stride : {s_batch_stride, new_s_batch_stride}) {
    if (stride < dense) return fail(HIPRWKV_EINVAL, "wkv6_step: state batch stride %lld is less than H*N*N = %lld", (long long)stride, (long long)dense);
    if ((stride * elem) % 16 != 0) return fail(HIPRWKV_EINVAL, "wkv6_step: state batch stride must be a multiple of 16 bytes");
  }
  Wkv6Args A;
  memset(&A, 0, sizeof(A));
  A.B = B; A.T = T; A.H = H;
  A.r = r; A.k = k; A.v = v; A.w = w; A.u = u; A.s = s;
  A.length = length; A.ns = new_starts;
  A.out = out; A.new_s = new_s;
  A.io_f32 = io_dtype == HIPRWKV_F32; A.st_f32 = A.new_st_f32 = state_dtype == HIPRWKV_F32;
  A.flags = flags;
  A.s_bstride = s_batch_stride; A.new_s_bstride = new_s_batch_stride;
  const hipError_t e = launch_wkv6_small_t_fwd(A, static_cast<hipStream_t>(stream));
  if (e != hipSuccess) return fail(HIPRWKV_ELAUNCH, "wkv6_step: %s", hipGetErrorString(e));
  return HIPRWKV_OK;
}

size_t hiprwkv_wkv6_bwd_workspace_bytes(int64_t B, int64_t T, int64_t H, int64_t N) {
  return align256((size_t)B * T * H * N * sizeof(float)) + PHASE_SPAN + align256((size_t)B * H * N * sizeof(float));
}

int hiprwkv_wkv6_bwd(hiprwkv_stream stream, int io_dtype, int state_dtype, int64_t B, int64_t T, int64_t H, int64_t N,
                     const void* r, const void* k, const void* v, const void* w, const void* u, const void* s,
                     const uint32_t* length, const uint8_t* new_starts, const void* gy, const void* gs_out, void* gr,
                     void* gk, void* gv, void* gw, float* gu, void* gs, void* workspace, size_t workspace_bytes,
                     unsigned flags) {
  int rc = check_matrix_shape("wkv6_bwd", io_dtype, state_dtype, B, T, H, N);
  if (rc) return rc;
  if ((rc = check_flags("wkv6_bwd", flags)) != HIPRWKV_OK) return rc;
  const void* req[] = {r, k, v, w, u, s, gy, gr, gk, gv, gw, gu, gs, workspace};
  for (const void* p : req) {
    if (p == nullptr) return fail(HIPRWKV_EINVAL, "wkv6_bwd: null tensor pointer");
    if (!aligned16(p)) return fail(HIPRWKV_EINVAL, "wkv6_bwd: tensor pointers must be 16-byte aligned");
  }
  const size_t need = hiprwkv_wkv6_bwd_workspace_bytes(B, T, H, N);
  if (workspace_bytes < need)
    return fail(HIPRWKV_ENOSPACE, "wkv6_bwd: workspace has %zu bytes, %zu needed", workspace_bytes, need);
  Wkv6Args A;
  memset(&A, 0, sizeof(A));
  A.B = B; A.T = T; A.H = H;
  A.r = r; A.k = k; A.v = v; A.w = w; A.u = u; A.s = s;
  A.length = length; A.ns = new_starts;
  A.io_f32 = io_dtype == HIPRWKV_F32; A.st_f32 = state_dtype == HIPRWKV_F32;
  A.flags = flags;
  A.status = status_word();
  A.gy = gy; A.gs_out = gs_out;
  A.gr = gr; A.gk = gk; A.gv = gv; A.gw = gw; A.gu = gu; A.gs = gs;
  char* ws = static_cast<char*>(workspace);
  A.er = reinterpret_cast<float*>(at_phase(ws, r, 5));
  A.eI = reinterpret_cast<float*>(reinterpret_cast<char*>(A.er) + align256((size_t)B * T * H * N * sizeof(float)));
  // Two sweeps: F (forward) -> gr, gu, er, eI; R (reverse) -> gk, gv, gw, gs, on the chunked matrix-core kernels
  // (bf16 pairs for bf16 I/O, fp32 operands for fp32 I/O); HIPRWKV_FORCE_SEQ selects the sequential kernel.
  hipStream_t st = static_cast<hipStream_t>(stream);
  hipError_t e;
  if (flags & HIPRWKV_FORCE_SEQ) {
    e = launch_wkv6_seq_bwd(A, st);
  } else if (A.io_f32) {
    e = launch_wkv6_chunk_bwd_f_f32(A, st);
    if (e == hipSuccess) e = launch_wkv6_chunk_bwd_r_f32(A, st);
  } else {
    e = launch_wkv6_chunk_bwd_f(A, st);
    if (e == hipSuccess) e = launch_wkv6_chunk_bwd_r(A, st);
  }
  if (e != hipSuccess) return fail(HIPRWKV_ELAUNCH, "wkv6_bwd: %s", hipGetErrorString(e));
  return HIPRWKV_OK;
}

static int wkv4_fwd_impl(hiprwkv_stream stream, int io_dtype, int64_t B, int64_t T, int64_t C, const void* w,
                         const void* u, const void* k, const void* v, const void* s, const uint32_t* length,
                         const uint8_t* new_starts, void* new_s, void* out, float* ckpt, unsigned flags);

int hiprwkv_wkv4_fwd(hiprwkv_stream stream, int io_dtype, int64_t B, int64_t T, int64_t C, const void* w,
                     const void* u, const void* k, const void* v, const void* s, const uint32_t* length,
                     const uint8_t* new_starts, void* new_s, void* out, unsigned flags) {
  return wkv4_fwd_impl(stream, io_dtype, B, T, C, w, u, k, v, s, length, new_starts, new_s, out, nullptr, flags);
}

int hiprwkv_wkv4_fwd_ckpt(hiprwkv_stream stream, int io_dtype, int64_t B, int64_t T, int64_t C, const void* w,
                          const void* u, const void* k, const void* v, const void* s, const uint32_t* length,
                          const uint8_t* new_starts, void* new_s, void* out, void* workspace, size_t workspace_bytes,
                          unsigned flags) {
  if (workspace == nullptr || !aligned16(workspace))
    return fail(HIPRWKV_EINVAL, "wkv4_fwd_ckpt: workspace must be a 16-byte aligned device pointer");
  if (B <= 0 || T <= 0 || C <= 0) return fail(HIPRWKV_EINVAL, "wkv4_fwd_ckpt: B,T,C must be positive");
  const size_t need = hiprwkv_wkv4_bwd_workspace_bytes(B, T, C);
  if (workspace_bytes < need)
    return fail(HIPRWKV_ENOSPACE, "wkv4_fwd_ckpt: workspace has %zu bytes, %zu needed", workspace_bytes, need);
  return wkv4_fwd_impl(stream, io_dtype, B, T, C, w, u, k, v, s, length, new_starts, new_s, out,
                       static_cast<float*>(workspace), flags);
}

static int wkv4_fwd_impl(hiprwkv_stream stream, int io_dtype, int64_t B, int64_t T, int64_t C, const void* w,
                         const void* u, const void* k, const void* v, const void* s, const uint32_t* length,
                         const uint8_t* new_starts, void* new_s, void* out, float* ckpt, unsigned flags) {
  if (int rc = check_flags("wkv4_fwd", flags)) return rc;
  if (!dtype_ok(io_dtype)) return fail(HIPRWKV_EINVAL, "wkv4_fwd: dtype must be HIPRWKV_F32 or HIPRWKV_BF16");
  if (B <= 0 || T <= 0 || C <= 0) return fail(HIPRWKV_EINVAL, "wkv4_fwd: B,T,C must be positive");
  if (B * ((C + 63) / 64) > 0x7fffffffLL) return fail(HIPRWKV_EINVAL, "wkv4_fwd: B*C exceeds the grid limit");
  // the forward kernel addresses a block of 32 tokens with 32-bit byte offsets from the block's first token
  if (C > (1LL << 23)) return fail(HIPRWKV_EINVAL, "wkv4_fwd: C exceeds 2^23 channels");
  const void* req[] = {w, u, k, v, s, new_s, out};
  for (const void* p : req) {
    if (p == nullptr) return fail(HIPRWKV_EINVAL, "wkv4_fwd: null tensor pointer");
    if (!aligned16(p)) return fail(HIPRWKV_EINVAL, "wkv4_fwd: tensor pointers must be 16-byte aligned");
  }
  Wkv4Args A;
  memset(&A, 0, sizeof(A));
  A.B = B; A.T = T; A.C = C;
  A.w = w; A.u = u; A.k = k; A.v = v; A.s = s;
  A.length = length; A.ns = new_starts;
  A.new_s = new_s; A.out = out;
  A.ckpt = ckpt;
  A.nz = 1; A.part = (T + 15) / 16 * 16;
  A.io_f32 = io_dtype == HIPRWKV_F32;
  A.flags = flags;
  hipError_t e = launch_wkv4_fwd(A, static_cast<hipStream_t>(stream));
  if (e != hipSuccess) return fail(HIPRWKV_ELAUNCH, "wkv4_fwd: %s", hipGetErrorString(e));
  return HIPRWKV_OK;
}

size_t hiprwkv_wkv4_bwd_workspace_bytes(int64_t B, int64_t T, int64_t C) {
  return align256((size_t)B * ((T + 15) / 16) * 3 * C * sizeof(float));
}

int hiprwkv_wkv4_bwd(hiprwkv_stream stream, int io_dtype, int64_t B, int64_t T, int64_t C, const void* w,
                     const void* u, const void* k, const void* v, const void* gy, const void* s,
                     const uint32_t* length, const uint8_t* new_starts, const void* gs_new, float* gw, float* gu,
                     void* gk, void* gv, void* gs, void* workspace, size_t workspace_bytes, unsigned flags) {
  if (int rc = check_flags("wkv4_bwd", flags)) return rc;
  if (!dtype_ok(io_dtype)) return fail(HIPRWKV_EINVAL, "wkv4_bwd: dtype must be HIPRWKV_F32 or HIPRWKV_BF16");
  if (B <= 0 || T <= 0 || C <= 0) return fail(HIPRWKV_EINVAL, "wkv4_bwd: B,T,C must be positive");
  if (B * ((C + 63) / 64) > 0x7fffffffLL) return fail(HIPRWKV_EINVAL, "wkv4_bwd: B*C exceeds the grid limit");
  if (C > (1LL << 23)) return fail(HIPRWKV_EINVAL, "wkv4_bwd: C exceeds 2^23 channels");
  const void* req[] = {w, u, k, v, gy, s, gw, gu, gk, gv, gs, workspace};
  for (const void* p : req) {
    if (p == nullptr) return fail(HIPRWKV_EINVAL, "wkv4_bwd: null tensor pointer");
    if (!aligned16(p)) return fail(HIPRWKV_EINVAL, "wkv4_bwd: tensor pointers must be 16-byte aligned");
  }
  if (gs_new && !aligned16(gs_new)) return fail(HIPRWKV_EINVAL, "wkv4_bwd: tensor pointers must be 16-byte aligned");
  const size_t need = hiprwkv_wkv4_bwd_workspace_bytes(B, T, C);
  if (workspace_bytes < need)
    return fail(HIPRWKV_ENOSPACE, "wkv4_bwd: workspace has %zu bytes, %zu needed", workspace_bytes, need);
  Wkv4Args A;
  memset(&A, 0, sizeof(A));
  A.B = B; A.T = T; A.C = C;
  A.w = w; A.u = u; A.k = k; A.v = v; A.s = s;
  A.length = length; A.ns = new_starts;
  A.io_f32 = io_dtype == HIPRWKV_F32;
  A.flags = flags;
  A.gy = gy; A.gs_new = gs_new;
  A.gk = gk; A.gv = gv; A.gs = gs; A.gw = gw; A.gu = gu; A.gw_stride = C;
  A.nz = 1; A.part = (T + 15) / 16 * 16;
  A.ckpt = static_cast<float*>(workspace);
  hipError_t e = launch_wkv4_bwd(A, static_cast<hipStream_t>(stream));
  if (e != hipSuccess) return fail(HIPRWKV_ELAUNCH, "wkv4_bwd: %s", hipGetErrorString(e));
  return HIPRWKV_OK;
}

size_t hiprwkv_wkv4_bwd_noalloc_max_bytes(void) { return SCRATCH_BYTES; }

int hiprwkv_wkv4_bwd_noalloc(hiprwkv_stream stream, int io_dtype, int64_t B, int64_t T, int64_t C, const void* w,
                             const void* u, const void* k, const void* v, const void* gy, const void* s,
                             const uint32_t* length, const uint8_t* new_starts, const void* gs_new, float* gw,
                             float* gu, void* gk, void* gv, void* gs, unsigned flags) {
  if (B <= 0 || T <= 0 || C <= 0) return fail(HIPRWKV_EINVAL, "wkv4_bwd_noalloc: B,T,C must be positive");
  // the shared scratch array holds whatever the last call left: this entry point always writes its own checkpoints
  if (flags & HIPRWKV_CKPT_READY)
    return fail(HIPRWKV_EINVAL, "wkv4_bwd_noalloc: HIPRWKV_CKPT_READY is not accepted (the built-in scratch is shared between calls)");
  const size_t need = hiprwkv_wkv4_bwd_workspace_bytes(B, T, C);
  if (need > SCRATCH_BYTES)
    return fail(HIPRWKV_ENOSPACE,
                "wkv4_bwd_noalloc: B*ceil(T/16)*3*C*4 = %zu bytes of checkpoints exceed the built-in %zu-byte "
                "scratch; use hiprwkv_wkv4_bwd with a caller-provided workspace", need, SCRATCH_BYTES);
  void* ws = scratch_base();
  if (ws == nullptr) return HIPRWKV_ELAUNCH;
  return hiprwkv_wkv4_bwd(stream, io_dtype, B, T, C, w, u, k, v, gy, s, length, new_starts, gs_new, gw, gu, gk, gv,
                          gs, ws, SCRATCH_BYTES, flags);
}

namespace {
int check_shiftmix(const char* op, int io_dtype, int64_t B, int64_t T, int64_t C, int n_out, const void* x,
                   const void* prev, int64_t prev_bstride, const void* const* mix, const void* const* per_out) {
  if (!dtype_ok(io_dtype)) return fail(HIPRWKV_EINVAL, "%s: dtype must be HIPRWKV_F32 or HIPRWKV_BF16", op);
  if (B <= 0 || T <= 0 || C <= 0 || C % 8 != 0) return fail(HIPRWKV_EINVAL, "%s: B, T must be positive and C a positive multiple of 8", op);
  if (B * T * (C / 8) > 0x7fffffffLL * 256) return fail(HIPRWKV_EINVAL, "%s: too many elements for one launch", op);
  if (n_out != 1 && n_out != 6) return fail(HIPRWKV_EINVAL, "%s: n_out must be 1 (channel mixing) or 6 (time mixing)", op);
  if (mix == nullptr || per_out == nullptr) return fail(HIPRWKV_EINVAL, "%s: null pointer array", op);
  const int64_t elem = io_dtype == HIPRWKV_F32 ? 4 : 2;
  if (prev_bstride < C || (prev_bstride * elem) % 16 != 0)
    return fail(HIPRWKV_EINVAL, "%s: the batch stride of the shift row must be at least C and a multiple of 16 bytes", op);
  const void* req[] = {x, prev};
  for (const void* p : req) {
    if (p == nullptr) return fail(HIPRWKV_EINVAL, "%s: null tensor pointer", op);
    if (!aligned16(p)) return fail(HIPRWKV_EINVAL, "%s: tensor pointers must be 16-byte aligned", op);
  }
  for (int i = 0; i < n_out; ++i) {
    if (mix[i] == nullptr || per_out[i] == nullptr) return fail(HIPRWKV_EINVAL, "%s: null tensor pointer", op);
    if (!aligned16(mix[i]) || !aligned16(per_out[i])) return fail(HIPRWKV_EINVAL, "%s: tensor pointers must be 16-byte aligned", op);
  }
  return HIPRWKV_OK;
}
}  // namespace

int hiprwkv_rwkv7_shiftmix(hiprwkv_stream stream, int io_dtype, int64_t B, int64_t T, int64_t C, int n_out, const void* x,
                           const void* prev, int64_t prev_batch_stride, const uint8_t* new_starts,
                           const void* const* mix, void* const* out) {
  int rc = check_shiftmix("rwkv7_shiftmix", io_dtype, B, T, C, n_out, x, prev, prev_batch_stride, mix,
                          const_cast<const void* const*>(out));
  if (rc) return rc;
  hipError_t e = launch_rwkv7_shiftmix(io_dtype == HIPRWKV_F32, B, T, C, n_out, x, prev, prev_batch_stride, new_starts,
                                       mix, out, static_cast<hipStream_t>(stream));
  if (e != hipSuccess) return fail(HIPRWKV_ELAUNCH, "rwkv7_shiftmix: %s", hipGetErrorString(e));
  return HIPRWKV_OK;
}

int hiprwkv_rwkv7_shiftmix_bwd(hiprwkv_stream stream, int io_dtype, int64_t B, int64_t T, int64_t C, int n_out,
                               const void* x, const void* prev, int64_t prev_batch_stride, const uint8_t* new_starts,
                               const void* const* mix, const void* const* g, void* dx, void* dprev,
                               int64_t dprev_batch_stride, float* dmix) {
  int rc = check_shiftmix("rwkv7_shiftmix_bwd", io_dtype, B, T, C, n_out, x, prev, prev_batch_stride, mix, g);
  if (rc) return rc;
  const void* req[] = {dx, dprev, dmix};
  for (const void* p : req) {
    if (p == nullptr) return fail(HIPRWKV_EINVAL, "rwkv7_shiftmix_bwd: null tensor pointer");
    if (!aligned16(p)) return fail(HIPRWKV_EINVAL, "rwkv7_shiftmix_bwd: tensor pointers must be 16-byte aligned");
  }
  const int64_t elem = io_dtype == HIPRWKV_F32 ? 4 : 2;
  if (dprev_batch_stride < C || (dprev_batch_stride * elem) % 16 != 0)
    return fail(HIPRWKV_EINVAL, "rwkv7_shiftmix_bwd: the batch stride of dprev must be at least C and a multiple of 16 bytes");
  hipError_t e = launch_rwkv7_shiftmix_bwd(io_dtype == HIPRWKV_F32, B, T, C, n_out, x, prev, prev_batch_stride, new_starts,
                                           mix, g, dx, dprev, dprev_batch_stride, dmix, static_cast<hipStream_t>(stream));
  if (e != hipSuccess) return fail(HIPRWKV_ELAUNCH, "rwkv7_shiftmix_bwd: %s", hipGetErrorString(e));
  return HIPRWKV_OK;
}

namespace {
int check_gate(const char* op, int io_dtype, int64_t rows, int64_t C, std::initializer_list<const void*> ptrs) {
  if (!dtype_ok(io_dtype)) return fail(HIPRWKV_EINVAL, "%s: dtype must be HIPRWKV_F32 or HIPRWKV_BF16", op);
  if (rows <= 0 || C <= 0 || C % 8 != 0) return fail(HIPRWKV_EINVAL, "%s: rows must be positive and C a positive multiple of 8", op);
  if (rows * (C / 8) > 0x7fffffffLL * 256) return fail(HIPRWKV_EINVAL, "%s: too many elements for one launch", op);
  for (const void* p : ptrs) {
    if (p == nullptr) return fail(HIPRWKV_EINVAL, "%s: null tensor pointer", op);
    if (!aligned16(p)) return fail(HIPRWKV_EINVAL, "%s: tensor pointers must be 16-byte aligned", op);
  }
  return HIPRWKV_OK;
}
int gate_done(const char* op, hipError_t e) {
  if (e != hipSuccess) return fail(HIPRWKV_ELAUNCH, "%s: %s", op, hipGetErrorString(e));
  return HIPRWKV_OK;
}
}  // namespace

int hiprwkv_rwkv7_decay(hiprwkv_stream stream, int io_dtype, int64_t rows, int64_t C, const void* x, const void* w0, void* w) {
  if (int rc = check_gate("rwkv7_decay", io_dtype, rows, C, {x, w0, w})) return rc;
  return gate_done("rwkv7_decay", launch_rwkv7_decay(io_dtype == HIPRWKV_F32, 0, rows, C, x, w0, w, static_cast<hipStream_t>(stream)));
}
int hiprwkv_rwkv7_decay_bwd(hiprwkv_stream stream, int io_dtype, int64_t rows, int64_t C, const void* x, const void* w0,
                            const void* g, void* dx, float* dw0) {
  if (int rc = check_gate("rwkv7_decay_bwd", io_dtype, rows, C, {x, w0, g, dx, dw0})) return rc;
  return gate_done("rwkv7_decay_bwd", launch_rwkv7_decay_bwd(io_dtype == HIPRWKV_F32, 0, rows, C, x, w0, g, dx, dw0, static_cast<hipStream_t>(stream)));
}
int hiprwkv_rwkv7_agate(hiprwkv_stream stream, int io_dtype, int64_t rows, int64_t C, const void* x, const void* a0, void* a) {
  if (int rc = check_gate("rwkv7_agate", io_dtype, rows, C, {x, a0, a})) return rc;
  return gate_done("rwkv7_agate", launch_rwkv7_decay(io_dtype == HIPRWKV_F32, 1, rows, C, x, a0, a, static_cast<hipStream_t>(stream)));
}
int hiprwkv_rwkv7_agate_bwd(hiprwkv_stream stream, int io_dtype, int64_t rows, int64_t C, const void* x, const void* a0,
                            const void* g, void* dx, float* da0) {
  if (int rc = check_gate("rwkv7_agate_bwd", io_dtype, rows, C, {x, a0, g, dx, da0})) return rc;
  return gate_done("rwkv7_agate_bwd", launch_rwkv7_decay_bwd(io_dtype == HIPRWKV_F32, 1, rows, C, x, a0, g, dx, da0, static_cast<hipStream_t>(stream)));
}
int hiprwkv_rwkv7_relusq(hiprwkv_stream stream, int io_dtype, int64_t n, const void* x, void* out) {
  if (int rc = check_gate("rwkv7_relusq", io_dtype, 1, n, {x, out})) return rc;
  return gate_done("rwkv7_relusq", launch_rwkv7_relusq(io_dtype == HIPRWKV_F32, n, x, nullptr, out, static_cast<hipStream_t>(stream)));
}
int hiprwkv_rwkv7_relusq_bwd(hiprwkv_stream stream, int io_dtype, int64_t n, const void* x, const void* g, void* dx) {
  if (int rc = check_gate("rwkv7_relusq_bwd", io_dtype, 1, n, {x, g, dx})) return rc;
  return gate_done("rwkv7_relusq_bwd", launch_rwkv7_relusq(io_dtype == HIPRWKV_F32, n, x, g, dx, static_cast<hipStream_t>(stream)));
}
int hiprwkv_rwkv7_vmix(hiprwkv_stream stream, int io_dtype, int64_t rows, int64_t C, const void* v, const void* v_first,
                       const void* x, const void* v0, void* out) {
  if (int rc = check_gate("rwkv7_vmix", io_dtype, rows, C, {v, v_first, x, v0, out})) return rc;
  return gate_done("rwkv7_vmix", launch_rwkv7_vmix(io_dtype == HIPRWKV_F32, rows, C, v, v_first, x, v0, out, static_cast<hipStream_t>(stream)));
}
int hiprwkv_rwkv7_vmix_bwd(hiprwkv_stream stream, int io_dtype, int64_t rows, int64_t C, const void* v, const void* v_first,
                           const void* x, const void* v0, const void* g, void* dv, void* dv_first, void* dx, float* dv0) {
  if (int rc = check_gate("rwkv7_vmix_bwd", io_dtype, rows, C, {v, v_first, x, v0, g, dv, dv_first, dx, dv0})) return rc;
  return gate_done("rwkv7_vmix_bwd", launch_rwkv7_vmix_bwd(io_dtype == HIPRWKV_F32, rows, C, v, v_first, x, v0, g, dv, dv_first, dx, dv0, static_cast<hipStream_t>(stream)));
}

int hiprwkv_rwkv7_premix(hiprwkv_stream stream, int io_dtype, int64_t rows, int64_t H, int64_t N, const void* k,
                         const void* a, const void* k_k, const void* k_a, void* k_out, void* a_out, void* b_out) {
  if (!dtype_ok(io_dtype)) return fail(HIPRWKV_EINVAL, "rwkv7_premix: dtype must be HIPRWKV_F32 or HIPRWKV_BF16");
  if (N != 64) return fail(HIPRWKV_EINVAL, "rwkv7_premix: head size N=%lld not supported (64 only)", (long long)N);
  if (rows <= 0 || H <= 0 || (rows * H + 3) / 4 > 0x7fffffffLL) return fail(HIPRWKV_EINVAL, "rwkv7_premix: bad rows/H");
  const void* req[] = {k, a, k_k, k_a, k_out, a_out, b_out};
  for (const void* p : req) {
    if (p == nullptr) return fail(HIPRWKV_EINVAL, "rwkv7_premix: null tensor pointer");
    if (!aligned16(p)) return fail(HIPRWKV_EINVAL, "rwkv7_premix: tensor pointers must be 16-byte aligned");
  }
  hipError_t e = launch_rwkv7_premix(io_dtype == HIPRWKV_F32, rows, H, k, a, k_k, k_a, k_out, a_out, b_out,
                                     static_cast<hipStream_t>(stream));
  if (e != hipSuccess) return fail(HIPRWKV_ELAUNCH, "rwkv7_premix: %s", hipGetErrorString(e));
  return HIPRWKV_OK;
}

int hiprwkv_rwkv7_postmix(hiprwkv_stream stream, int io_dtype, int64_t rows, int64_t H, int64_t N, const void* y,
                          const void* r, const void* k, const void* v, const void* g, const void* ln_w,
                          const void* ln_b, const void* r_k, float eps, void* out) {
  if (!dtype_ok(io_dtype)) return fail(HIPRWKV_EINVAL, "rwkv7_postmix: dtype must be HIPRWKV_F32 or HIPRWKV_BF16");
  if (N != 64) return fail(HIPRWKV_EINVAL, "rwkv7_postmix: head size N=%lld not supported (64 only)", (long long)N);
  if (rows <= 0 || H <= 0 || (rows * H + 3) / 4 > 0x7fffffffLL) return fail(HIPRWKV_EINVAL, "rwkv7_postmix: bad rows/H");
  const void* req[] = {y, r, k, v, g, ln_w, ln_b, r_k, out};
  for (const void* p : req) {
    if (p == nullptr) return fail(HIPRWKV_EINVAL, "rwkv7_postmix: null tensor pointer");
    if (!aligned16(p)) return fail(HIPRWKV_EINVAL, "rwkv7_postmix: tensor pointers must be 16-byte aligned");
  }
  hipError_t e = launch_rwkv7_postmix(io_dtype == HIPRWKV_F32, rows, H, y, r, k, v, g, ln_w, ln_b, r_k, eps, out,
                                      static_cast<hipStream_t>(stream));
  if (e != hipSuccess) return fail(HIPRWKV_ELAUNCH, "rwkv7_postmix: %s", hipGetErrorString(e));
  return HIPRWKV_OK;
}

int hiprwkv_rwkv7_premix_bwd(hiprwkv_stream stream, int io_dtype, int64_t rows, int64_t H, int64_t N, const void* k,
                             const void* a, const void* k_k, const void* k_a, const void* gk_out, const void* ga_out,
                             const void* gb_out, void* gk, void* ga, float* gk_k, float* gk_a) {
  if (!dtype_ok(io_dtype)) return fail(HIPRWKV_EINVAL, "rwkv7_premix_bwd: dtype must be HIPRWKV_F32 or HIPRWKV_BF16");
  if (N != 64) return fail(HIPRWKV_EINVAL, "rwkv7_premix_bwd: head size N=%lld not supported (64 only)", (long long)N);
  if (rows <= 0 || H <= 0 || H > 65536 || (rows * H + 3) / 4 > 0x7fffffffLL)
    return fail(HIPRWKV_EINVAL, "rwkv7_premix_bwd: bad rows/H");
  const void* req[] = {k, a, k_k, k_a, gk_out, ga_out, gb_out, gk, ga, gk_k, gk_a};
  for (const void* p : req) {
    if (p == nullptr) return fail(HIPRWKV_EINVAL, "rwkv7_premix_bwd: null tensor pointer");
    if (!aligned16(p)) return fail(HIPRWKV_EINVAL, "rwkv7_premix_bwd: tensor pointers must be 16-byte aligned");
  }
  hipError_t e = launch_rwkv7_premix_bwd(io_dtype == HIPRWKV_F32, rows, H, k, a, k_k, k_a, gk_out, ga_out, gb_out, gk,
                                         ga, gk_k, gk_a, static_cast<hipStream_t>(stream));
  if (e != hipSuccess) return fail(HIPRWKV_ELAUNCH, "rwkv7_premix_bwd: %s", hipGetErrorString(e));
  return HIPRWKV_OK;
}

int hiprwkv_rwkv7_postmix_bwd(hiprwkv_stream stream, int io_dtype, int64_t rows, int64_t H, int64_t N, const void* y,
                              const void* r, const void* k, const void* v, const void* g, const void* ln_w,
                              const void* ln_b, const void* r_k, float eps, const void* gout, void* gy, void* gr,
                              void* gk, void* gv, void* gg, float* gln_w, float* gln_b, float* gr_k) {
  if (!dtype_ok(io_dtype)) return fail(HIPRWKV_EINVAL, "rwkv7_postmix_bwd: dtype must be HIPRWKV_F32 or HIPRWKV_BF16");
  if (N != 64) return fail(HIPRWKV_EINVAL, "rwkv7_postmix_bwd: head size N=%lld not supported (64 only)", (long long)N);
  if (rows <= 0 || H <= 0 || H > 65536 || (rows * H + 3) / 4 > 0x7fffffffLL)
    return fail(HIPRWKV_EINVAL, "rwkv7_postmix_bwd: bad rows/H");
  const void* req[] = {y, r, k, v, g, ln_w, ln_b, r_k, gout, gy, gr, gk, gv, gg, gln_w, gln_b, gr_k};
  for (const void* p : req) {
    if (p == nullptr) return fail(HIPRWKV_EINVAL, "rwkv7_postmix_bwd: null tensor pointer");
    if (!aligned16(p)) return fail(HIPRWKV_EINVAL, "rwkv7_postmix_bwd: tensor pointers must be 16-byte aligned");
  }
  hipError_t e = launch_rwkv7_postmix_bwd(io_dtype == HIPRWKV_F32, rows, H, y, r, k, v, g, ln_w, ln_b, r_k, eps, gout,
                                          gy, gr, gk, gv, gg, gln_w, gln_b, gr_k, nullptr, nullptr, static_cast<hipStream_t>(stream));
  if (e != hipSuccess) return fail(HIPRWKV_ELAUNCH, "rwkv7_postmix_bwd: %s", hipGetErrorString(e));
  return HIPRWKV_OK;
}

namespace {
int check_ln_mix(const char* op, int io_dtype, const LnMixArgs& A, int n_out, const void* const* per_out,
                 std::initializer_list<const void*> req, std::initializer_list<const void*> opt) {
  if (!dtype_ok(io_dtype)) return fail(HIPRWKV_EINVAL, "%s: dtype must be HIPRWKV_F32 or HIPRWKV_BF16", op);
  if (A.B <= 0 || A.T <= 0 || A.C <= 0 || A.C % 8 != 0 || A.C > 4096)
    return fail(HIPRWKV_EINVAL, "%s: B, T must be positive and C a positive multiple of 8 of at most 4096", op);
  if (A.B * A.T > 0x7fffffffLL) return fail(HIPRWKV_EINVAL, "%s: too many tokens for one launch", op);
  if (n_out != 0 && n_out != 1 && n_out != 6) return fail(HIPRWKV_EINVAL, "%s: n_out must be 0, 1 or 6", op);
  for (const void* p : req)
    if (p == nullptr || !aligned16(p)) return fail(HIPRWKV_EINVAL, "%s: null or misaligned tensor pointer (16 bytes)", op);
  for (const void* p : opt)
    if (p != nullptr && !aligned16(p)) return fail(HIPRWKV_EINVAL, "%s: tensor pointers must be 16-byte aligned", op);
  const int64_t elem = io_dtype == HIPRWKV_F32 ? 4 : 2;
  if (n_out != 0) {
    if (A.prev == nullptr || !aligned16(A.prev)) return fail(HIPRWKV_EINVAL, "%s: null or misaligned shift row", op);
    if (A.prev_bstride < A.C || (A.prev_bstride * elem) % 16 != 0)
      return fail(HIPRWKV_EINVAL, "%s: the batch stride of the shift row must be at least C and a multiple of 16 bytes", op);
  }
  if (A.shift != nullptr && (A.shift_bstride < A.C || (A.shift_bstride * elem) % 16 != 0))
    return fail(HIPRWKV_EINVAL, "%s: the batch stride of the new shift row must be at least C and a multiple of 16 bytes", op);
  for (int i = 0; i < n_out; ++i)
    if (A.mix[i] == nullptr || !aligned16(A.mix[i])) return fail(HIPRWKV_EINVAL, "%s: null or misaligned mix vector", op);
  for (int i = 0; i < (n_out ? n_out : 1); ++i)
    if (per_out[i] == nullptr || !aligned16(per_out[i])) return fail(HIPRWKV_EINVAL, "%s: null or misaligned tensor pointer", op);
  return HIPRWKV_OK;
}
}  // namespace

int hiprwkv_rwkv7_ln_shiftmix(hiprwkv_stream stream, int io_dtype, int64_t B, int64_t T, int64_t C, int n_out,
                              const void* x, const void* dx, const void* ln_w, const void* ln_b, float eps,
                              const void* prev, int64_t prev_batch_stride, const uint8_t* new_starts,
                              const int32_t* length, const void* const* mix, void* const* out, void* xs, void* shift,
                              int64_t shift_batch_stride, float* stats) {
  LnMixArgs A;
  memset(&A, 0, sizeof(A));
  A.B = B; A.T = T; A.C = C;
  A.x = x; A.dx = dx; A.ln_w = ln_w; A.ln_b = ln_b; A.eps = eps;
  A.prev = prev; A.prev_bstride = prev_batch_stride; A.ns = new_starts; A.length = length;
  A.xs = xs; A.shift = shift; A.shift_bstride = shift_batch_stride; A.stats = stats;
  if ((n_out != 0 && mix == nullptr) || out == nullptr) return fail(HIPRWKV_EINVAL, "rwkv7_ln_shiftmix: null pointer array");
  if (dx != nullptr && xs == nullptr) return fail(HIPRWKV_EINVAL, "rwkv7_ln_shiftmix: dx needs xs");
  for (int i = 0; i < n_out && i < 6; ++i) A.mix[i] = mix[i];
  for (int i = 0; i < (n_out ? n_out : 1) && i < 6; ++i) A.out[i] = out[i];
  if (int rc = check_ln_mix("rwkv7_ln_shiftmix", io_dtype, A, n_out, A.out, {x, ln_w, ln_b}, {dx, xs, shift, stats})) return rc;
  return gate_done("rwkv7_ln_shiftmix", launch_ln_shiftmix(io_dtype == HIPRWKV_F32, n_out, A, static_cast<hipStream_t>(stream)));
}

size_t hiprwkv_rwkv7_ln_shiftmix_bwd_workspace_bytes(int64_t B, int64_t T, int64_t C, int n_out) {
  if (B <= 0 || T <= 0 || C <= 0 || n_out < 0) return 0;
  const int64_t run = ln_shiftmix_bwd_run(B * T);
  return (size_t)((B * T + run - 1) / run) * (n_out + 2) * C * sizeof(float);
}

int hiprwkv_rwkv7_ln_shiftmix_bwd(hiprwkv_stream stream, int io_dtype, int64_t B, int64_t T, int64_t C, int n_out,
                                  const void* xs, const float* stats, const void* ln_w, const void* ln_b,
                                  const void* prev, int64_t prev_batch_stride, const uint8_t* new_starts,
                                  const int32_t* length, const void* const* mix, const void* const* g, const void* gx,
                                  const void* gshift, void* dxs, void* dprev, void* const* dparam, void* workspace,
                                  size_t workspace_bytes) {
  LnMixArgs A;
  memset(&A, 0, sizeof(A));
  A.B = B; A.T = T; A.C = C;
  A.xs = const_cast<void*>(xs); A.stats = const_cast<float*>(stats); A.ln_w = ln_w; A.ln_b = ln_b;
  A.prev = prev; A.prev_bstride = prev_batch_stride; A.ns = new_starts; A.length = length;
  A.gx = gx; A.gshift = gshift; A.dxs = dxs; A.dprev = dprev; A.part = static_cast<float*>(workspace);
  if ((n_out != 0 && mix == nullptr) || g == nullptr || dparam == nullptr)
    return fail(HIPRWKV_EINVAL, "rwkv7_ln_shiftmix_bwd: null pointer array");
  for (int i = 0; i < n_out && i < 6; ++i) A.mix[i] = mix[i];
  for (int i = 0; i < (n_out ? n_out : 1) && i < 6; ++i) A.g[i] = g[i];
  if (int rc = check_ln_mix("rwkv7_ln_shiftmix_bwd", io_dtype, A, n_out, A.g, {xs, stats, ln_w, ln_b, dxs, workspace}, {gx, gshift, dprev}))
    return rc;
  for (int i = 0; i < n_out + 2; ++i)
    if (dparam[i] == nullptr) return fail(HIPRWKV_EINVAL, "rwkv7_ln_shiftmix_bwd: null tensor pointer");
  const size_t need = hiprwkv_rwkv7_ln_shiftmix_bwd_workspace_bytes(B, T, C, n_out);
  if (workspace_bytes < need)
    return fail(HIPRWKV_ENOSPACE, "rwkv7_ln_shiftmix_bwd: workspace has %zu bytes, %zu needed", workspace_bytes, need);
  return gate_done("rwkv7_ln_shiftmix_bwd", launch_ln_shiftmix_bwd(io_dtype == HIPRWKV_F32, n_out, A, dparam, static_cast<hipStream_t>(stream)));
}

namespace {
int check_pre(const char* op, int io_dtype, int64_t N, const PreArgs& A, std::initializer_list<const void*> req,
              std::initializer_list<const void*> with_vf) {
  if (!dtype_ok(io_dtype)) return fail(HIPRWKV_EINVAL, "%s: dtype must be HIPRWKV_F32 or HIPRWKV_BF16", op);
  if (N != 64) return fail(HIPRWKV_EINVAL, "%s: head size N=%lld not supported (64 only)", op, (long long)N);
  if (A.rows <= 0 || A.H <= 0 || A.H > 65536 || (A.rows * A.H + 3) / 4 > 0x7fffffffLL) return fail(HIPRWKV_EINVAL, "%s: bad rows/H", op);
  for (const void* p : req)
    if (p == nullptr || !aligned16(p)) return fail(HIPRWKV_EINVAL, "%s: null or misaligned tensor pointer (16 bytes)", op);
  if (A.vf != nullptr)
    for (const void* p : with_vf)
      if (p == nullptr || !aligned16(p)) return fail(HIPRWKV_EINVAL, "%s: null or misaligned tensor pointer (16 bytes)", op);
  return HIPRWKV_OK;
}
}  // namespace

int hiprwkv_rwkv7_pre(hiprwkv_stream stream, int io_dtype, int64_t rows, int64_t H, int64_t N, const void* xw,
                      const void* k, const void* xa, const void* v, const void* v_first, const void* xv, const void* w0,
                      const void* a0, const void* v0, const void* k_k, const void* k_a, void* w, void* k_out,
                      void* v_out, void* a_out, void* b_out) {
  PreArgs A;
  memset(&A, 0, sizeof(A));
  A.rows = rows; A.H = H;
  A.xw = xw; A.k = k; A.xa = xa; A.v = v; A.vf = v_first; A.xv = xv;
  A.w0 = w0; A.a0 = a0; A.v0 = v0; A.k_k = k_k; A.k_a = k_a;
  A.w = w; A.k_out = k_out; A.v_out = v_out; A.a_out = a_out; A.b_out = b_out;
  if (int rc = check_pre("rwkv7_pre", io_dtype, N, A, {xw, k, xa, w0, a0, k_k, k_a, w, k_out, a_out, b_out}, {v, v_first, xv, v0, v_out}))
    return rc;
  return gate_done("rwkv7_pre", launch_rwkv7_pre(io_dtype == HIPRWKV_F32, A, static_cast<hipStream_t>(stream)));
}

int hiprwkv_rwkv7_lora_pre(hiprwkv_stream stream, int io_dtype, int64_t rows, int64_t H, int64_t N, const void* const* hid,
                           const void* const* w2, const int64_t* d, const void* k, const void* v, const void* v_first, const void* w0,
                           const void* a0, const void* v0, const void* k_k, const void* k_a, void* const* out, void* g, void* w,
                           void* k_out, void* v_out, void* a_out, void* b_out) {
  LoraPreArgs X;
  memset(&X, 0, sizeof(X));
  PreArgs& A = X.P;
  A.rows = rows; A.H = H;
  A.k = k; A.v = v; A.vf = v_first;
  A.w0 = w0; A.a0 = a0; A.v0 = v0; A.k_k = k_k; A.k_a = k_a;
  A.w = w; A.k_out = k_out; A.v_out = v_out; A.a_out = a_out; A.b_out = b_out;
  if (hid == nullptr || w2 == nullptr || d == nullptr) return fail(HIPRWKV_EINVAL, "rwkv7_lora_pre: null pointer array");
  if (io_dtype != HIPRWKV_BF16) return fail(HIPRWKV_EINVAL, "rwkv7_lora_pre: dtype must be HIPRWKV_BF16");
  if (int rc = check_pre("rwkv7_lora_pre", io_dtype, N, A, {k, w0, a0, k_k, k_a, out != nullptr ? out[2] : g, w, k_out, a_out, b_out}, {v, v_first, v0, v_out})) return rc;
  if ((rows + 63) / 64 * H > 0x7fffffffLL || rows > 0x7fffffffLL - 64) return fail(HIPRWKV_EINVAL, "rwkv7_lora_pre: too many rows");
  for (int i = 0; i < (v_first != nullptr ? 4 : 3); ++i) {
    if (d[i] <= 0 || d[i] % 8 != 0 || d[i] > 0x7fffffffLL || std::max(rows, H * N) * d[i] >= 0x7fffffffLL)
      return fail(HIPRWKV_EINVAL, "rwkv7_lora_pre: inner sizes must be positive multiples of 8, arrays below 4 GiB");
    for (const void* p : {hid[i], w2[i]})
      if (p == nullptr || !aligned16(p)) return fail(HIPRWKV_EINVAL, "rwkv7_lora_pre: null or misaligned tensor pointer (16 bytes)");
    if (out != nullptr && (out[i] == nullptr || !aligned16(out[i])))
      return fail(HIPRWKV_EINVAL, "rwkv7_lora_pre: null or misaligned tensor pointer (16 bytes)");
    X.hid[i] = hid[i]; X.w2[i] = w2[i]; X.d[i] = (int)d[i]; X.out[i] = out != nullptr ? out[i] : i == 2 ? g : nullptr;
  }
  return gate_done("rwkv7_lora_pre", launch_rwkv7_lora_pre(X, static_cast<hipStream_t>(stream)));
}

size_t hiprwkv_rwkv7_pre_bwd_workspace_bytes(int64_t rows, int64_t H, int64_t N) {
  return rows <= 0 || H <= 0 || N <= 0 ? 0 : (size_t)rwkv7_pre_bwd_rows(rows, H) * 5 * H * N * sizeof(float);
}

int hiprwkv_rwkv7_pre_bwd(hiprwkv_stream stream, int io_dtype, int64_t rows, int64_t H, int64_t N, const void* xw,
                          const void* k, const void* xa, const void* v, const void* v_first, const void* xv,
                          const void* w0, const void* a0, const void* v0, const void* k_k, const void* k_a,
                          const void* gw, const void* gk_out, const void* gv_out, const void* ga_out,
                          const void* gb_out, const void* gk_out2, const void* gv_out2, const void* gr, const void* gr2,
                          void* dr, void* dxw, void* dk, void* dv, void* dv_first, void* dxv, void* dxa,
                          void* const* dparam, void* workspace, size_t workspace_bytes) {
  PreArgs A;
  memset(&A, 0, sizeof(A));
  A.rows = rows; A.H = H;
  A.xw = xw; A.k = k; A.xa = xa; A.v = v; A.vf = v_first; A.xv = xv;
  A.w0 = w0; A.a0 = a0; A.v0 = v0; A.k_k = k_k; A.k_a = k_a;
  A.gw = gw; A.gk = gk_out; A.gv = gv_out; A.ga = ga_out; A.gb = gb_out;
  A.gk2 = gk_out2; A.gv2 = gv_out2; A.gr = gr; A.gr2 = gr2; A.dr = dr;
  for (const void* p : {gk_out2, gv_out2, gr, gr2, static_cast<const void*>(dr)})
    if (p != nullptr && !aligned16(p)) return fail(HIPRWKV_EINVAL, "rwkv7_pre_bwd: tensor pointers must be 16-byte aligned");
  if (dr != nullptr && (gr == nullptr || gr2 == nullptr)) return fail(HIPRWKV_EINVAL, "rwkv7_pre_bwd: dr needs gr and gr2");
  A.dxw = dxw; A.dk = dk; A.dv = dv; A.dvf = dv_first; A.dxv = dxv; A.dxa = dxa;
  A.part = static_cast<float*>(workspace);
  if (int rc = check_pre("rwkv7_pre_bwd", io_dtype, N, A,
                         {xw, k, xa, w0, a0, k_k, k_a, gw, gk_out, ga_out, gb_out, dxw, dk, dxa, workspace},
                         {v, v_first, xv, v0, gv_out, dv, dv_first, dxv}))
    return rc;
  if (dparam == nullptr) return fail(HIPRWKV_EINVAL, "rwkv7_pre_bwd: null pointer array");
  for (int i = 0; i < (v_first != nullptr ? 5 : 4); ++i)
    if (dparam[i] == nullptr) return fail(HIPRWKV_EINVAL, "rwkv7_pre_bwd: null tensor pointer");
  const size_t need = hiprwkv_rwkv7_pre_bwd_workspace_bytes(rows, H, N);
  if (workspace_bytes < need)
    return fail(HIPRWKV_ENOSPACE, "rwkv7_pre_bwd: workspace has %zu bytes, %zu needed", workspace_bytes, need);
  return gate_done("rwkv7_pre_bwd", launch_rwkv7_pre_bwd(io_dtype == HIPRWKV_F32, A, dparam, static_cast<hipStream_t>(stream)));
}

size_t hiprwkv_rwkv7_decode_workspace_bytes(const hiprwkv_rwkv7_decode_args* args) {
  return args == nullptr || args->B <= 0 || args->T <= 0 ? 0 : rwkv7_decode_workspace(*args);
}

int hiprwkv_rwkv7_decode(hiprwkv_stream stream, const hiprwkv_rwkv7_decode_args* args) {
  if (args == nullptr) return fail(HIPRWKV_EINVAL, "rwkv7_decode: null arguments");
  const hiprwkv_rwkv7_decode_args& D = *args;
  if (D.B <= 0 || D.T <= 0 || D.L <= 0 || D.T > HIPRWKV_SMALL_T || D.B * D.T > HIPRWKV_DECODE_MAX_ROWS)
    return fail(HIPRWKV_EINVAL, "rwkv7_decode: B, T, L must be positive, T at most %d and B*T at most %d", HIPRWKV_SMALL_T, HIPRWKV_DECODE_MAX_ROWS);
  if (D.H <= 0 || D.H > 64 || D.C != D.H * 64) return fail(HIPRWKV_EINVAL, "rwkv7_decode: C must be 64 H, positive and at most 4096");
  for (int64_t d : {D.F, D.d_decay, D.d_aaa, D.d_mv, D.d_gate})
    if (d <= 0 || d % 32 != 0) return fail(HIPRWKV_EINVAL, "rwkv7_decode: inner sizes must be positive multiples of 32");
  if (D.logits != nullptr && (D.vocab <= 0 || D.vocab % 16 != 0)) return fail(HIPRWKV_EINVAL, "rwkv7_decode: vocab must be a positive multiple of 16");
  if (D.flags & ~(uint64_t)HIPRWKV_COMPAT_ASSOC) return fail(HIPRWKV_EINVAL, "rwkv7_decode: unknown flag bits");
  const void* req[] = {D.x, D.state, D.new_state, D.ln0_w, D.ln0_b, D.ln_out_w, D.ln_out_b, D.ln1_w, D.ln1_b, D.ln2_w,
                       D.ln2_b, D.x_r, D.x_w, D.x_k, D.x_v, D.x_a, D.x_g, D.w0, D.w1, D.w2, D.a0, D.a1, D.a2, D.v0, D.v1,
                       D.v2, D.g1, D.g2, D.k_k, D.k_a, D.r_k, D.receptance, D.key, D.value, D.output, D.lnx_w, D.lnx_b,
                       D.ffn_x_k, D.ffn_key, D.ffn_value, D.xn, D.workspace};
  for (const void* p : req)
    if (p == nullptr || !aligned16(p)) return fail(HIPRWKV_EINVAL, "rwkv7_decode: null or misaligned tensor pointer (16 bytes)");
  if (D.logits != nullptr && (D.head == nullptr || !aligned16(D.head) || !aligned16(D.logits)))
    return fail(HIPRWKV_EINVAL, "rwkv7_decode: null or misaligned head or logits");
  if (D.state == D.new_state) return fail(HIPRWKV_EINVAL, "rwkv7_decode: state and new_state must be different arrays");
  const size_t need = rwkv7_decode_workspace(D);
  if (D.workspace_bytes < need)
    return fail(HIPRWKV_ENOSPACE, "rwkv7_decode: workspace has %llu bytes, %zu needed", (unsigned long long)D.workspace_bytes, need);
  return gate_done("rwkv7_decode", launch_rwkv7_decode(D, static_cast<hipStream_t>(stream)));
}

namespace {
bool stack_sizes_ok(const hiprwkv_rwkv7_stack_args& D) {
  for (int64_t n : {D.B, D.T, D.L, D.C, D.H, D.F, D.d_decay, D.d_aaa, D.d_mv, D.d_gate})
    if (n <= 0 || n > 0x7fffffffLL) return false;
  if (D.B * D.T > 0x7fffffffLL || D.H > 64 || D.C != D.H * 64) return false;
  for (int64_t n : {D.F, D.d_decay, D.d_aaa, D.d_mv, D.d_gate})
    if (n % 8 != 0 || std::max(n, D.C) * std::max(D.B * D.T, D.C) * 2 >= 0x7fffffffLL || n * 256 >= 0x7fffffffLL) return false;
  return D.B * D.T * 256 < 0x7fffffffLL;
}
int check_stack(const char* op, const hiprwkv_rwkv7_stack_args* args, bool backward) {
  if (args == nullptr) return fail(HIPRWKV_EINVAL, "%s: null arguments", op);
  const hiprwkv_rwkv7_stack_args& D = *args;
  if (!stack_sizes_ok(D)) return fail(HIPRWKV_EINVAL, "%s: sizes must be positive, C = 64 H at most 4096, inner sizes multiples of 8, arrays below 2 GiB", op);
  if (D.flags & ~(uint64_t)HIPRWKV_COMPAT_ASSOC) return fail(HIPRWKV_EINVAL, "%s: unknown flag bits", op);
  const void* req[] = {D.x, D.state, D.s, D.xs, D.workspace};
  const void* fwd[] = {D.new_state, D.new_s, D.dx};
  const void* bwd[] = {D.g_xs, D.g_dx, D.g_x};
  bool ok = true;
  for (const void* p : req) ok = ok && p != nullptr && aligned16(p);
  for (const void* p : backward ? bwd : fwd) ok = ok && p != nullptr && aligned16(p);
  for (const void* p : {D.g_shift, D.g_s}) ok = ok && (p == nullptr || aligned16(p));
  constexpr int n = sizeof(D.param) / sizeof(void*);
  const void* const* par = reinterpret_cast<const void* const*>(&D.param);
  const void* const* gra = reinterpret_cast<const void* const*>(&D.grad);
  for (int i = 0; i < n; ++i) {
    const void* const* const of_v = par + i;
    const bool residual = of_v == &D.param.v0 || of_v == &D.param.v1 || of_v == &D.param.v2;
    ok = ok && par[i] != nullptr && aligned16(par[i]);
    if (backward) ok = ok && (gra[i] != nullptr ? aligned16(gra[i]) : residual && D.L == 1);
  }
  if (backward && D.saved == nullptr) ok = false;
  for (int64_t l = 0; ok && D.saved != nullptr && l < D.L; ++l) ok = D.saved[l] != nullptr && aligned16(D.saved[l]);
  if (!ok) return fail(HIPRWKV_EINVAL, "%s: null or misaligned tensor pointer (16 bytes)", op);
  if (!backward && (D.state == D.new_state || D.s == D.new_s)) return fail(HIPRWKV_EINVAL, "%s: states and new states must be different arrays", op);
  const size_t need = rwkv7_stack_workspace(D, backward);
  if (D.workspace_bytes < need)
    return fail(HIPRWKV_ENOSPACE, "%s: workspace has %llu bytes, %zu needed", op, (unsigned long long)D.workspace_bytes, need);
  return HIPRWKV_OK;
}
}  // namespace

size_t hiprwkv_rwkv7_stack_saved_layer_bytes(const hiprwkv_rwkv7_stack_args* args, int64_t layer) {
  return args == nullptr || !stack_sizes_ok(*args) || layer < 0 || layer >= args->L ? 0 : rwkv7_stack_saved(*args, layer);
}

size_t hiprwkv_rwkv7_stack_saved_bytes(const hiprwkv_rwkv7_stack_args* args) {
  size_t most = 0;
  if (args != nullptr)
    for (int64_t layer : {(int64_t)0, args->L / 2, args->L - 1}) most = std::max(most, hiprwkv_rwkv7_stack_saved_layer_bytes(args, layer));
  return most;
}

size_t hiprwkv_rwkv7_stack_workspace_bytes(const hiprwkv_rwkv7_stack_args* args, int backward) {
  return args == nullptr || !stack_sizes_ok(*args) ? 0 : rwkv7_stack_workspace(*args, backward != 0);
}

int hiprwkv_rwkv7_stack_fwd(hiprwkv_stream stream, const hiprwkv_rwkv7_stack_args* args) {
  if (int rc = check_stack("rwkv7_stack_fwd", args, false)) return rc;
  hipError_t e = hipSuccess;
  if (int rc = launch_rwkv7_stack_fwd(*args, static_cast<hipStream_t>(stream), e)) return rc;
  return gate_done("rwkv7_stack_fwd", e);
}

int hiprwkv_rwkv7_stack_bwd(hiprwkv_stream stream, const hiprwkv_rwkv7_stack_args* args) {
  if (int rc = check_stack("rwkv7_stack_bwd", args, true)) return rc;
  hipError_t e = hipSuccess;
  if (int rc = launch_rwkv7_stack_bwd(*args, static_cast<hipStream_t>(stream), e)) return rc;
  return gate_done("rwkv7_stack_bwd", e);
}

// ---- WKV4 with the receptance applied, sequences cut into parts where the batch leaves the GPU idle
namespace {
size_t wkv4_part_bytes(int64_t B, int64_t T, int64_t C, int floats) {
  int64_t part;
  const int64_t nz = wkv4_parts(B, T, C, &part);
  return align256((size_t)B * (nz - 1) * C * floats * sizeof(float));
}
int check_wkv4(const char* op, int io_dtype, int64_t B, int64_t T, int64_t C, unsigned flags, std::initializer_list<const void*> req,
               std::initializer_list<const void*> opt) {
  if (int rc = check_flags(op, flags)) return rc;
  if (!dtype_ok(io_dtype)) return fail(HIPRWKV_EINVAL, "%s: dtype must be HIPRWKV_F32 or HIPRWKV_BF16", op);
  if (B <= 0 || T <= 0 || C <= 0) return fail(HIPRWKV_EINVAL, "%s: B,T,C must be positive", op);
  if (B * ((C + 63) / 64) > 0x7fffffffLL) return fail(HIPRWKV_EINVAL, "%s: B*C exceeds the grid limit", op);
  if (C > (1LL << 23)) return fail(HIPRWKV_EINVAL, "%s: C exceeds 2^23 channels", op);
  for (const void* p : req)
    if (p == nullptr || !aligned16(p)) return fail(HIPRWKV_EINVAL, "%s: null or misaligned tensor pointer (16 bytes)", op);
  for (const void* p : opt)
    if (p != nullptr && !aligned16(p)) return fail(HIPRWKV_EINVAL, "%s: tensor pointers must be 16-byte aligned", op);
  return HIPRWKV_OK;
}
}  // namespace

size_t hiprwkv_wkv4_mix_workspace_bytes(int64_t B, int64_t T, int64_t C) {
  return B <= 0 || T <= 0 || C <= 0 ? 0 : wkv4_part_bytes(B, T, C, 4);
}

int hiprwkv_wkv4_mix(hiprwkv_stream stream, int io_dtype, int64_t B, int64_t T, int64_t C, const void* w, const void* u,
                     const void* k, const void* v, const void* r, const void* s, const uint32_t* length,
                     const uint8_t* new_starts, void* new_s, void* out, void* ckpt, size_t ckpt_bytes, void* workspace,
                     size_t workspace_bytes, unsigned flags) {
  if (int rc = check_wkv4("wkv4_mix", io_dtype, B, T, C, flags, {w, u, k, v, s, new_s, out}, {r, ckpt, workspace})) return rc;
  const size_t need = hiprwkv_wkv4_mix_workspace_bytes(B, T, C);
  if (workspace_bytes < need || (need != 0 && workspace == nullptr))
    return fail(HIPRWKV_ENOSPACE, "wkv4_mix: workspace has %zu bytes, %zu needed", workspace_bytes, need);
  if (ckpt != nullptr && ckpt_bytes < hiprwkv_wkv4_bwd_workspace_bytes(B, T, C))
    return fail(HIPRWKV_ENOSPACE, "wkv4_mix: checkpoint array has %zu bytes, %zu needed", ckpt_bytes, hiprwkv_wkv4_bwd_workspace_bytes(B, T, C));
  Wkv4Args A;
  memset(&A, 0, sizeof(A));
  A.B = B; A.T = T; A.C = C;
  A.w = w; A.u = u; A.k = k; A.v = v; A.r = r; A.s = s;
  A.length = length; A.ns = new_starts;
  A.new_s = new_s; A.out = out;
  A.ckpt = static_cast<float*>(ckpt);
  A.io_f32 = io_dtype == HIPRWKV_F32;
  A.flags = flags;
  A.nz = wkv4_parts(B, T, C, &A.part);
  A.sums = static_cast<float*>(workspace);
  return gate_done("wkv4_mix", launch_wkv4_fwd(A, static_cast<hipStream_t>(stream)));
}

size_t hiprwkv_wkv4_mix_bwd_workspace_bytes(int64_t B, int64_t T, int64_t C) {
  if (B <= 0 || T <= 0 || C <= 0) return 0;
  int64_t part;
  const int64_t nz = wkv4_parts(B, T, C, &part);
  return wkv4_part_bytes(B, T, C, 8) + align256((size_t)B * nz * 2 * C * sizeof(float));
}

int hiprwkv_wkv4_mix_bwd(hiprwkv_stream stream, int io_dtype, int64_t B, int64_t T, int64_t C, const void* w,
                         const void* u, const void* k, const void* v, const void* r, const void* gout, const void* s,
                         const uint32_t* length, const uint8_t* new_starts, const void* gs_new, void* ckpt,
                         size_t ckpt_bytes, void* gw, void* gu, void* gk, void* gv, void* gr, void* gs, void* workspace,
                         size_t workspace_bytes, unsigned flags) {
  if (int rc = check_wkv4("wkv4_mix_bwd", io_dtype, B, T, C, flags, {w, u, k, v, gout, s, ckpt, gk, gv, gs, workspace}, {r, gr, gs_new}))
    return rc;
  if (gw == nullptr || gu == nullptr || ((r == nullptr) != (gr == nullptr)))
    return fail(HIPRWKV_EINVAL, "wkv4_mix_bwd: null tensor pointer");
  if (ckpt_bytes < hiprwkv_wkv4_bwd_workspace_bytes(B, T, C))
    return fail(HIPRWKV_ENOSPACE, "wkv4_mix_bwd: checkpoint array has %zu bytes, %zu needed", ckpt_bytes, hiprwkv_wkv4_bwd_workspace_bytes(B, T, C));
  const size_t need = hiprwkv_wkv4_mix_bwd_workspace_bytes(B, T, C);
  if (workspace_bytes < need)
    return fail(HIPRWKV_ENOSPACE, "wkv4_mix_bwd: workspace has %zu bytes, %zu needed", workspace_bytes, need);
  Wkv4Args A;
  memset(&A, 0, sizeof(A));
  A.B = B; A.T = T; A.C = C;
  A.w = w; A.u = u; A.k = k; A.v = v; A.r = r; A.s = s;
  A.length = length; A.ns = new_starts;
  A.io_f32 = io_dtype == HIPRWKV_F32;
  A.flags = flags;
  A.gy = gout; A.gs_new = gs_new;
  A.gk = gk; A.gv = gv; A.gr = gr; A.gs = gs;
  A.ckpt = static_cast<float*>(ckpt);
  A.nz = wkv4_parts(B, T, C, &A.part);
  A.maps = static_cast<float*>(workspace);
  A.gw = reinterpret_cast<float*>(static_cast<char*>(workspace) + wkv4_part_bytes(B, T, C, 8));
  A.gu = A.gw + C;
  A.gw_stride = 2 * C;
  hipStream_t st = static_cast<hipStream_t>(stream);
  hipError_t e = launch_wkv4_bwd(A, st);
  if (e == hipSuccess) {
    ReduceArgs R;
    R.part = A.gw; R.rows = B * A.nz; R.nk = 2; R.C = C;
    R.out[0] = gw; R.out[1] = gu;
    e = reduce_parts(A.io_f32, R, nullptr, st);
  }
  return gate_done("wkv4_mix_bwd", e);
}

int hiprwkv_gemm(hiprwkv_stream stream, int n_jobs, const hiprwkv_gemm_job* jobs) {
  if (n_jobs <= 0 || n_jobs > HIPRWKV_GEMM_MAX_JOBS || jobs == nullptr)
    return fail(HIPRWKV_EINVAL, "gemm: 1 to %d jobs", HIPRWKV_GEMM_MAX_JOBS);
  GemmArgs A;
  memset(&A, 0, sizeof(A));
  A.n_jobs = n_jobs;
  int64_t tiles = 0;
  for (int i = 0; i < n_jobs; ++i) {
    const hiprwkv_gemm_job& J = jobs[i];
    if (J.M <= 0 || J.N <= 0 || J.K <= 0 || J.N % 8 || (!J.kn && J.K % 8) || (J.km ? J.M % 8 : J.K % 8))
      return fail(HIPRWKV_EINVAL, "gemm: job %d: sizes must be positive, those contiguous in memory multiples of 8", i);
    if (std::max((int64_t)(J.km ? J.M : 0), (int64_t)(J.kn ? J.N : 0)) * J.K * 2 >= 0x7fffffffLL || (int64_t)J.K * 256 >= 0x7fffffffLL)
      return fail(HIPRWKV_EINVAL, "gemm: job %d: an operand of 2 GiB or more", i);
    if (J.act < 0 || J.act > (J.aux ? 2 : 3)) return fail(HIPRWKV_EINVAL, "gemm: job %d: unknown function", i);
    for (const void* p : {J.x, J.w, static_cast<const void*>(J.out)})
      if (p == nullptr || !aligned16(p)) return fail(HIPRWKV_EINVAL, "gemm: job %d: null or misaligned tensor pointer (16 bytes)", i);
    if (J.aux != nullptr && !aligned16(J.aux)) return fail(HIPRWKV_EINVAL, "gemm: job %d: misaligned tensor pointer (16 bytes)", i);
    tiles += (int64_t)((J.N + 511) / 512 * 8) * ((J.M + 511) / 512 * 8);
    static_cast<hiprwkv_gemm_job&>(A.job[i]) = J;
  }
  if (tiles > 0x7fffffffLL) return fail(HIPRWKV_EINVAL, "gemm: too many tiles for one launch");
  return gate_done("gemm", launch_gemm(A, 1, static_cast<hipStream_t>(stream)));
}

size_t hiprwkv_rwkv7_postmix_bwd2_workspace_bytes(int64_t rows, int64_t H, int64_t N) {
  return rows <= 0 || H <= 0 || N <= 0 ? 0 : (size_t)rwkv7_postmix_bwd_rows(rows, H) * 3 * H * N * sizeof(float);
}

int hiprwkv_rwkv7_postmix_bwd2(hiprwkv_stream stream, int io_dtype, int64_t rows, int64_t H, int64_t N, const void* y,
                               const void* r, const void* k, const void* v, const void* g, const void* ln_w,
                               const void* ln_b, const void* r_k, float eps, const void* gout, void* gy, void* gr,
                               void* gk, void* gv, void* gg, void* const* dparam, void* workspace, size_t workspace_bytes) {
  PreArgs A;      // shape checks as for rwkv7_pre
  memset(&A, 0, sizeof(A));
  A.rows = rows; A.H = H;
  if (int rc = check_pre("rwkv7_postmix_bwd2", io_dtype, N, A, {y, r, k, v, g, ln_w, ln_b, r_k, gout, gy, gr, gk, gv, gg, workspace}, {})) return rc;
  if (dparam == nullptr || dparam[0] == nullptr || dparam[1] == nullptr || dparam[2] == nullptr)
    return fail(HIPRWKV_EINVAL, "rwkv7_postmix_bwd2: null tensor pointer");
  const size_t need = hiprwkv_rwkv7_postmix_bwd2_workspace_bytes(rows, H, N);
  if (workspace_bytes < need)
    return fail(HIPRWKV_ENOSPACE, "rwkv7_postmix_bwd2: workspace has %zu bytes, %zu needed", workspace_bytes, need);
  return gate_done("rwkv7_postmix_bwd2", launch_rwkv7_postmix_bwd(io_dtype == HIPRWKV_F32, rows, H, y, r, k, v, g, ln_w, ln_b, r_k, eps,
                                                                   gout, gy, gr, gk, gv, gg, nullptr, nullptr, nullptr,
                                                                   static_cast<float*>(workspace), dparam, static_cast<hipStream_t>(stream)));
}

}  // extern "C"
