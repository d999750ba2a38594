// Plain argument blocks passed by value to the kernels, and the launcher prototypes the C ABI calls.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <string.h>

#include <atomic>

#include "../../include/hiprwkv.h"

namespace hiprwkv {

struct Wkv7Args {
  int64_t B, T, H;
  const void *w, *r, *k, *v, *a, *b, *s;
  const uint32_t* length;
  const uint8_t* ns;
  void* out;
  void* sa;       // forward residual (may be null): fp32 beside fp32 I/O, IEEE half beside bf16 I/O
  void* new_s;
  int io_f32, st_f32, new_st_f32;      // I/O, s, new_s
  unsigned flags;
  // backward only
  const void* gy;
  const void* sa_in;     // the forward residual, in the forward's type
  const void* gs_out;
  void *gw, *gr, *gk, *gv, *ga, *gb, *gs;
  // workspace, three regions of (B,T,H,64) fp32 each.  The sequential sweeps and the chunked fp32 ones keep dsa in the
  // first as fp32; the chunked bf16 sweeps keep it there as 16-bit fixed point with one scale exponent per chunk and
  // value tile, the exponents in the third region (chunk_common.h dsa_scales).  The chunked sweeps keep e3_t + e2_{t+1}
  // in e2, as records per chunk and wave (chunk_common.h f_record), and do not use e3 otherwise.
  float *dsa, *e2, *e3;
  unsigned* status;      // device word counting workgroups whose hand-shake gave up (may be null)
  // Elements between the states of consecutive sequences in `s` / `new_s`; 0 = dense (H*64*64).  Honoured by the
  // small-T kernel only (states read and written inside a packed model state).
  int64_t s_bstride, new_s_bstride;
  // workspace for the summaries of a sequence in parts (forward: wkv7_fwd_parts, null: whole, the launcher sets the other two;
  // sweep A: wkv7_bwd_parts, n_part < 2: whole)
  void* parts;
  int n_part, part_chunks;
  // The parts of sweeps B and C: n_end of end_chunks chunks.  ends: fp32 I/O the states at their boundaries, (heads, n_end - 1, 64,
  // 64) fp32, left by the forward that keeps sa (null there: none wanted); bf16 I/O records that give them (wkv7_ends.h), made beside
  // sweep A; gends: the cotangents of these states, left by sweep A.
  float *ends, *gends;
  int n_end, end_chunks;
};
int wkv7_fwd_parts(int64_t heads, int64_t T, bool f32, int* chunks);
size_t wkv7_fwd_parts_bytes(int64_t heads, int64_t T, bool f32);
// How the backward splits a sequence: n_end parts for sweeps B and C, and whether sweep A runs in these parts too
struct Wkv7BwdSplit {
  int n_end, end_chunks;
  bool a_parts;
};
Wkv7BwdSplit wkv7_bwd_parts(int64_t heads, int64_t T, bool f32);
size_t wkv7_bwd_sums_bytes(int64_t heads, const Wkv7BwdSplit& S);      // summaries of sweep A
size_t wkv7_ends_bytes(int64_t heads, const Wkv7BwdSplit& S, bool f32);

// Wkv6Args::flags bit: w is (H,64), shared by every token and sequence (HIPRWKV_W_PER_HEAD)
constexpr unsigned FLAG_W_PER_HEAD = 0x10u;

struct Wkv6Args {
  int64_t B, T, H;
  const void *r, *k, *v, *w, *u, *s;
  const uint32_t* length;
  const uint8_t* ns;
  void* out;
  void* new_s;
  int io_f32, st_f32, new_st_f32;      // I/O, s, new_s
  unsigned flags;
  // backward only
  const void* gy;
  const void* gs_out;
  void *gr, *gk, *gv, *gw, *gs;
  float* gu;   // (B,H,64)
  float* er;   // workspace (B,T,H,64): r . (S' dy)
  float* eI;   // workspace (B,H,64): rowsum(dS_out * S_{length-1})
  unsigned* status;   // device word counting workgroups whose hand-shake gave up (may be null)
  // Elements between the states of consecutive sequences in `s` / `new_s`; 0 = dense (H*64*64).  Honoured by the
  // small-T kernel only (states read and written inside a packed model state).
  int64_t s_bstride, new_s_bstride;
  // forward, bf16 I/O: workspace for a sequence in parts (wkv6_fwd_parts), null: whole; the launcher sets the other two
  void* parts;
  int n_part, part_chunks;
};
int wkv6_fwd_parts(int64_t heads, int64_t T, int* chunks);
size_t wkv6_fwd_parts_bytes(int64_t heads, int64_t T);

// Wkv4Args::flags bit: the workspace already holds the checkpoints (HIPRWKV_CKPT_READY)
constexpr unsigned FLAG_CKPT_READY = 0x20u;
// Wkv4Args::flags bit: w is the raw time_decay, the decay is -exp(w) (HIPRWKV_W_RAW)
constexpr unsigned FLAG_W_RAW = 0x80u;

struct Wkv4Args {
  int64_t B, T, C;
  const void *w, *u, *k, *v, *s;
  const uint32_t* length;
  const uint8_t* ns;
  void* new_s;
  void* out;
  int io_f32;
  unsigned flags;
  // backward only
  const void* gy;
  const void* gs_new;
  void *gk, *gv, *gs;
  float *gw, *gu;   // rows of C, gw_stride floats apart: one per sequence and part
  int64_t gw_stride;
  float* ckpt;      // workspace: (B, ceil(T/16), 3, C) states entering every 16th step (forward: optional output)
  // receptance (may be null): out = r wkv, and the backward returns gr
  const void* r;
  void* gr;
  // the sequence in parts of `part` tokens (wkv4_parts); nz = 1: whole, no workspace
  int64_t nz, part;
  float* sums;      // workspace (B, nz-1, C, 4): the parts' summaries
  float* maps;      // workspace (B, nz-1, 2, C, 4): the parts' cotangent maps
};
int64_t wkv4_parts(int64_t B, int64_t T, int64_t C, int64_t* part);

// Residual addition + LayerNorm + token shift and interpolation (rwkv7_block.hip); tensors in the I/O dtype
struct LnMixArgs {
  int64_t B, T, C, run;
  const void *x, *dx;            // (B,T,C); dx may be null (then xs is x itself and is not written)
  const void *ln_w, *ln_b;       // (C,)
  float eps;
  const void* prev;              // (B,C) rows, prev_bstride elements apart: the token before t = 0
  int64_t prev_bstride;
  const uint8_t* ns;
  const int32_t* length;         // (B,) or null: which token's norm goes to `shift`
  const void* mix[6];            // (C,) each
  void* out[6];
  void* xs;                      // forward: x + dx out; backward: the same array in
  void* shift;                   // (B,C) rows, shift_bstride elements apart; may be null
  int64_t shift_bstride;
  float* stats;                  // (B*T, 2) mean and 1/std; forward: may be null
  // backward
  const void* g[6];
  const void *gx, *gshift;       // cotangents of xs and of the shift row (B,C), each may be null
  void *dxs, *dprev;             // dprev (B,C) may be null
  // backward: workspace (workgroups, n_out + 2, C).  Forward: dx as n_part > 1 partial sums (n_part, B*T, C) in place of `dx`
  float* part;
  int n_part;
};
struct ReduceArgs {
  const float* part;             // (rows, nk, C)
  int64_t rows, C;
  int nk;
  void* out[8];                  // nk arrays (C,)
};
// Several of them in one launch: where a launcher below is given one, its sum is added to it instead of launched
struct ReduceJobs {
  int n;
  ReduceArgs job[3];
};
hipError_t launch_reduce_parts(int io_f32, const ReduceJobs& J, hipStream_t stream);
hipError_t reduce_parts(int io_f32, const ReduceArgs& A, ReduceJobs* later, hipStream_t stream);
int64_t ln_shiftmix_bwd_run(int64_t rows);
hipError_t launch_ln_shiftmix(int io_f32, int n_out, LnMixArgs A, hipStream_t stream);
hipError_t launch_ln_shiftmix_bwd(int io_f32, int n_out, LnMixArgs A, void* const* dparam, hipStream_t stream, ReduceJobs* later = nullptr);

// Element-wise work between the projections and the WKV op (rwkv7_pre.hip); token tensors (rows, H, 64), parameters (H, 64)
struct PreArgs {
  int64_t rows, H;
  const void *xw, *k, *xa, *v, *vf, *xv;       // vf null: no value residual (v, vf, xv, v0, v_out and dv, dvf, dxv unused)
  const void *w0, *a0, *v0, *k_k, *k_a;
  void *w, *k_out, *v_out, *a_out, *b_out;
  // backward
  const void *gw, *gk, *gv, *ga, *gb;          // cotangents of w, k_out, v_out, a_out, b_out
  const void *gk2, *gv2;                       // second cotangents of k_out and v_out, added to the first; may be null
  const void *gr, *gr2;                        // two cotangents of r to be added up in dr; may be null
  void* dr;
  void *dxw, *dk, *dv, *dvf, *dxv, *dxa;
  const void* gvf;                             // added to dvf (or to dv_sum); may be null, may be dvf
  void* dv_sum;                                // without the value residual: gv + gv2 + gvf; may be null
  float* part;                                 // workspace (rwkv7_pre_bwd_rows, 4 or 5, H*64)
};
int64_t rwkv7_pre_bwd_rows(int64_t rows, int64_t H);
hipError_t launch_rwkv7_pre(int io_f32, const PreArgs& A, hipStream_t stream);
hipError_t launch_rwkv7_pre_bwd(int io_f32, const PreArgs& A, void* const* dparam, hipStream_t stream, ReduceJobs* later = nullptr);

// Several products per launch (rwkv7_gemm.hip), bf16: out[m][n] = f(sum_k x(m, k) w(n, k)).  The job is the C ABI's
// (hiprwkv_gemm_job) and more; tile0 is the launcher's.
struct GemmJob : ::hiprwkv_gemm_job {
  void* raw;           // without aux: the product itself, beside f of it in out; may be null
};
constexpr int GEMM_ACT_NONE = 0, GEMM_ACT_TANH = 1, GEMM_ACT_SIGMOID = 2, GEMM_ACT_RELUSQ = 3;      // f without aux
constexpr int GEMM_ADD = 0, GEMM_DTANH = 1, GEMM_DSIGMOID = 2, GEMM_DRELUSQ = 3;                    // f with aux
constexpr int GEMM_MAX_JOBS = 14;
constexpr int GEMM_TILE_ROWS = 33;     // rows from which the kernel with LDS tiles takes over
constexpr int GEMM_MAX_SPLIT = 8;
struct GemmArgs {
  int n_jobs;
  int tile0[GEMM_MAX_JOBS];  // the launcher's: a job's first tile; side by side, so that a workgroup finds its job with one load
  GemmJob job[GEMM_MAX_JOBS];
  float* part;         // not null: (split, M, N) fp32 partial sums instead of out; one job, no f
  int log_split;       // the launcher's, few rows
};
int gemm_split(int M, int64_t K, int64_t N);
hipError_t launch_gemm(GemmArgs A, int split, hipStream_t stream);
// The second low-rank products and launch_rwkv7_pre in one pass, bf16: xw, xa, g, xv = hid[i] (rows, d[i]) times w2[i] (d[i], H*64), g to
// out[2], the others, which P's fields of their name do not give, to out[i] where that is not null.  d multiples of 8; without the value
// residual (P.vf null) hid[3], w2[3] and d[3] are not looked at.
struct LoraPreArgs {
  PreArgs P;
  const void *hid[4], *w2[4];
  int d[4];
  void* out[4];
};
hipError_t launch_rwkv7_lora_pre(const LoraPreArgs& A, hipStream_t stream);
// The same products of one or two rows of norm and interpolation (LnMixArgs: bf16, C a multiple of 64, at most 4096; mix and
// out unused): a job's x is that of its aux, the mix vector (C,); K = C, N a multiple of 32, not km.
constexpr int HEAD_GEMM_ROWS = 2;
hipError_t launch_head_gemm(const LnMixArgs& N, GemmArgs A, hipStream_t stream);

using Rwkv7Decode = ::hiprwkv_rwkv7_decode_args;
size_t rwkv7_decode_workspace(const Rwkv7Decode& D);
hipError_t launch_rwkv7_decode(const Rwkv7Decode& D, hipStream_t stream);

using Rwkv7Stack = ::hiprwkv_rwkv7_stack_args;
size_t rwkv7_stack_saved(const Rwkv7Stack& D, int64_t l);
size_t rwkv7_stack_workspace(const Rwkv7Stack& D, bool backward);
int launch_rwkv7_stack_fwd(const Rwkv7Stack& D, hipStream_t stream, hipError_t& e);      // an entry point's error, or e
int launch_rwkv7_stack_bwd(const Rwkv7Stack& D, hipStream_t stream, hipError_t& e);

// Raises a kernel's dynamic-LDS limit once per kernel and device instead of at every enqueue (the attribute call
// goes to the driver; hipGetDevice does not).
struct LdsAttrOnce {
  std::atomic<uint64_t> done{0};   // bit d: set on device d
};
inline hipError_t allow_dynamic_lds(LdsAttrOnce& once, const void* kernel, size_t bytes) {
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  const uint64_t bit = 1ull << (dev & 63);
  if (once.done.load(std::memory_order_acquire) & bit) return hipSuccess;
  e = hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
  if (e == hipSuccess) once.done.fetch_or(bit, std::memory_order_release);
  return e;
}

hipError_t launch_wkv7_seq_fwd(const Wkv7Args& A, hipStream_t stream);
hipError_t launch_wkv7_chunk_fwd(const Wkv7Args& A, hipStream_t stream);
hipError_t launch_wkv7_chunk_fwd_f32(const Wkv7Args& A, hipStream_t stream);
hipError_t launch_wkv7_chunk_bwd_a_f32(const Wkv7Args& A, hipStream_t stream);
hipError_t launch_wkv7_chunk_bwd_b_f32(const Wkv7Args& A, hipStream_t stream);
hipError_t launch_wkv7_chunk_bwd_c_f32(const Wkv7Args& A, hipStream_t stream);
hipError_t launch_wkv7_small_t_fwd(const Wkv7Args& A, hipStream_t stream);
hipError_t launch_wkv6_small_t_fwd(const Wkv6Args& A, hipStream_t stream);
hipError_t launch_wkv7_chunk_bwd_a(const Wkv7Args& A, hipStream_t stream);
hipError_t launch_wkv7_chunk_bwd_b(const Wkv7Args& A, hipStream_t stream);
hipError_t launch_wkv7_chunk_bwd_c(const Wkv7Args& A, hipStream_t stream);
hipError_t launch_wkv7_seq_bwd_a(const Wkv7Args& A, hipStream_t stream);
hipError_t launch_wkv7_seq_bwd_b(const Wkv7Args& A, hipStream_t stream);
hipError_t launch_wkv7_seq_bwd_c(const Wkv7Args& A, hipStream_t stream);
hipError_t launch_wkv6_seq_fwd(const Wkv6Args& A, hipStream_t stream);
hipError_t launch_wkv6_chunk_fwd(const Wkv6Args& A, hipStream_t stream);
hipError_t launch_wkv6_chunk_fwd_f32(const Wkv6Args& A, hipStream_t stream);
hipError_t launch_wkv6_seq_bwd(const Wkv6Args& A, hipStream_t stream);
hipError_t launch_wkv6_chunk_bwd_f(const Wkv6Args& A, hipStream_t stream);
hipError_t launch_wkv6_chunk_bwd_r(const Wkv6Args& A, hipStream_t stream);
hipError_t launch_wkv6_chunk_bwd_f_f32(const Wkv6Args& A, hipStream_t stream);
hipError_t launch_wkv6_chunk_bwd_r_f32(const Wkv6Args& A, hipStream_t stream);
hipError_t launch_wkv4_fwd(const Wkv4Args& A, hipStream_t stream);
hipError_t launch_wkv4_bwd(const Wkv4Args& A, hipStream_t stream);
hipError_t launch_rwkv7_premix(int io_f32, int64_t rows, int64_t H, const void* k, const void* a, const void* k_k,
                               const void* k_a, void* k_out, void* a_out, void* b_out, hipStream_t stream);
hipError_t launch_rwkv7_postmix(int io_f32, int64_t rows, int64_t H, const void* y, const void* r, const void* k,
                                const void* v, const void* g, const void* ln_w, const void* ln_b, const void* r_k,
                                float eps, void* out, hipStream_t stream);
hipError_t launch_rwkv7_decay(int io_f32, int sigmoid, int64_t rows, int64_t C, const void* x, const void* w0, void* w,
                              hipStream_t stream);
hipError_t launch_rwkv7_decay_bwd(int io_f32, int sigmoid, int64_t rows, int64_t C, const void* x, const void* w0,
                                  const void* g, void* dx, float* dw0, hipStream_t stream);
hipError_t launch_rwkv7_relusq(int io_f32, int64_t n, const void* x, const void* g, void* out, hipStream_t stream);
hipError_t launch_rwkv7_vmix(int io_f32, int64_t rows, int64_t C, const void* v, const void* v_first, const void* x,
                             const void* v0, void* out, hipStream_t stream);
hipError_t launch_rwkv7_vmix_bwd(int io_f32, int64_t rows, int64_t C, const void* v, const void* v_first, const void* x,
                                 const void* v0, const void* g, void* dv, void* dv_first, void* dx, float* dv0,
                                 hipStream_t stream);
hipError_t launch_rwkv7_shiftmix(int io_f32, int64_t B, int64_t T, int64_t C, int n_out, const void* x, const void* prev,
                                 int64_t prev_bstride, const uint8_t* ns, const void* const* mix, void* const* out,
                                 hipStream_t stream);
hipError_t launch_rwkv7_shiftmix_bwd(int io_f32, int64_t B, int64_t T, int64_t C, int n_out, const void* x,
                                     const void* prev, int64_t prev_bstride, const uint8_t* ns, const void* const* mix,
                                     const void* const* g, void* dx, void* dprev, int64_t dprev_bstride, float* dmix,
                                     hipStream_t stream);
hipError_t launch_rwkv7_premix_bwd(int io_f32, int64_t rows, int64_t H, const void* k, const void* a, const void* k_k,
                                   const void* k_a, const void* gko, const void* gao, const void* gbo, void* gk,
                                   void* ga, float* gk_k, float* gk_a, hipStream_t stream);
hipError_t launch_rwkv7_postmix_bwd(int io_f32, int64_t rows, int64_t H, const void* y, const void* r, const void* k,
                                    const void* v, const void* g, const void* ln_w, const void* ln_b, const void* r_k,
                                    float eps, const void* go, void* gy, void* gr, void* gk, void* gv, void* gg,
                                    float* gln_w, float* gln_b, float* gr_k, float* part, void* const* dparam,
                                    hipStream_t stream, ReduceJobs* later = nullptr);
int64_t rwkv7_postmix_bwd_rows(int64_t rows, int64_t H);

}  // namespace hiprwkv
