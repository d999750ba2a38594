// An RWKV-7 decode step (at most 8 tokens per sequence, at most 256 tokens in all, bf16) layer by layer from native code:
// eight launches per layer instead of the ~30 operations of the general path, whose host side alone takes 5 ms for 12 layers.
//     1  residual addition, norm, shift and six interpolations               (rwkv7_block.hip)
//     2  r, k, v and the first low-rank factors, tanh / sigmoid applied       skinny_gemm, seven products in one grid
//     3  the second low-rank factors                                          skinny_gemm, four products
//     4  gates, WKV step on the packed state, group norm, bonus, gate         decode_core_kernel
//     5  output projection                                                    skinny_gemm
//     6  residual addition, norm, shift and interpolation                     (rwkv7_block.hip)
//     7  key projection with relu(.)^2                                        skinny_gemm
//     8  value projection                                                     skinny_gemm
// Measured (eager, host included): 12 layers of 768 channels, one user 5.4 ms -> 0.56 ms a step; 24 layers of 2048 channels,
// 256 users 10.9 -> 3.6 ms (7.5 with the weight-streaming product alone: 51 us a launch at 256 rows, 18 tiled).
// References: /root/reference/src/jaxrwkv/rwkv7.py:190-198, :223-267, :269-291.  Products accumulate in fp32 and are rounded
// once; the values between the gates, the recurrence and the group norm are rounded where the general path stores them.
#include "chunk_common.h"
#include "wkv_args.h"

namespace hiprwkv {

namespace {

using chunk::f32x4_t;
using chunk::u32x4_t;
using chunk::mfma;

constexpr int GEMM_WAVES = 8;
enum Act { ACT_NONE = 0, ACT_TANH = 1, ACT_SIGMOID = 2, ACT_RELUSQ = 3 };

// One product out[m][n] = act(sum_k x[m][k] w(n, k)).  NK weights are (N, K) row-major (used as x @ W.T), KN weights (K, N).
struct GemmJob {
  const bf16_t *x, *w;
  bf16_t* out;
  int K, N;
  int kn;          // layout of w
  int act;
  int tile0;       // first column tile of the job in the grid
};
constexpr int MAX_JOBS = 7;
struct GemmArgs {
  GemmJob job[MAX_JOBS];
  int n_jobs;
  int M;
  int tiles;       // column tiles of all jobs
  float* part;     // not null: split partial sums (split, M, N) in fp32 instead of out; one job, no activation
};

__device__ __forceinline__ float activate(float x, int act) {
  switch (act) {
    case ACT_TANH: return 1.f - 2.f / (1.f + __expf(2.f * x));
    case ACT_SIGMOID: return 1.f / (1.f + __expf(-x));
    case ACT_RELUSQ: { const float r = fmaxf(x, 0.f); return r * r; }
    default: return x;
  }
}

// Weight-streaming product for few rows: bound by reading w once.  A workgroup owns 16 columns of one product and 16 MT
// rows; its eight waves split K (every wave of the grid then streams a run of k of sixteen weight rows, so that many
// short streams are in flight however small N is) and add their 16x16 tiles through LDS.  The weights' rows are the
// matrix instruction's A operand straight from memory, 16 bytes per lane, no LDS; x comes from the cache.  KN weights (the
// low-rank factors, a tenth of the bytes) are gathered two bytes at a time.
template <int MT>
__global__ __launch_bounds__(64 * GEMM_WAVES) void skinny_gemm_kernel(GemmArgs A) {
  __shared__ f32x4_t red[GEMM_WAVES][MT][64];
  int ji = 0;
  for (int i = 1; i < A.n_jobs; ++i) ji = (int)blockIdx.x >= A.job[i].tile0 ? i : ji;
  const GemmJob J = A.job[ji];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
  const int n0 = ((int)blockIdx.x - J.tile0) * 16, m0 = (int)blockIdx.y * 16 * MT;
  const int steps = J.K / 32;
  const int s0 = steps * wave / GEMM_WAVES, s1 = steps * (wave + 1) / GEMM_WAVES;
  f32x4_t acc[MT];
  const bf16_t* xp[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t) {
    acc[t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    const int m = m0 + 16 * t + r;
    xp[t] = J.x + (size_t)(m < A.M ? m : A.M - 1) * J.K + 8 * g;
  }
  auto step = [&](const u32x4_t w, int s) {
#pragma unroll
    for (int t = 0; t < MT; ++t) acc[t] = mfma(w, *reinterpret_cast<const u32x4_t*>(xp[t] + 32 * s), acc[t]);
  };
  if (!J.kn) {
    const bf16_t* wp = J.w + (size_t)(n0 + r) * J.K + 8 * g;
    constexpr int UN = MT == 1 ? 8 : 4;
    int s = s0;
    for (; s + UN <= s1; s += UN) {
      u32x4_t w[UN];
#pragma unroll
      for (int u = 0; u < UN; ++u) w[u] = *reinterpret_cast<const u32x4_t*>(wp + 32 * (s + u));
#pragma unroll
      for (int u = 0; u < UN; ++u) step(w[u], s + u);
    }
    for (; s < s1; ++s) step(*reinterpret_cast<const u32x4_t*>(wp + 32 * s), s);
  } else {
    const uint16_t* wp = reinterpret_cast<const uint16_t*>(J.w) + (size_t)(8 * g) * J.N + n0 + r;
    auto gather = [&](int s) {
      u32x4_t w;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const uint16_t* p = wp + (size_t)(32 * s + 2 * i) * J.N;
        w[i] = (uint32_t)p[0] | ((uint32_t)p[J.N] << 16);
      }
      return w;
    };
    int s = s0;
    for (; s + 2 <= s1; s += 2) {
      const u32x4_t w0 = gather(s), w1 = gather(s + 1);
      step(w0, s);
      step(w1, s + 1);
    }
    if (s < s1) step(gather(s), s);
  }
#pragma unroll
  for (int t = 0; t < MT; ++t) red[wave][t][lane] = acc[t];
  __syncthreads();
  if (wave < MT) {
    f32x4_t s = red[0][wave][lane];
#pragma unroll
    for (int q = 1; q < GEMM_WAVES; ++q) s += red[q][wave][lane];
    // lane (column m = lane % 16, g) holds n = 4g .. 4g+3
    const int m = m0 + 16 * wave + r;
    if (m < A.M) {
      const uint2 o = make_uint2(chunk::pack_rn(activate(s[0], J.act), activate(s[1], J.act)),
                                 chunk::pack_rn(activate(s[2], J.act), activate(s[3], J.act)));
      *reinterpret_cast<uint2*>(J.out + (size_t)m * J.N + n0 + 4 * g) = o;
    }
  }
}

// The same for 65 .. 256 rows, where the product is bound by the weights' stream and by LDS about equally (256 rows against
// 6656 columns of 2048: 5.3 us of weights, 6 us of operand reads).  64 x 64 tiles, 64 of k per step through two LDS
// buffers: a thread carries two 16-byte pieces of either operand, requested two steps ahead, and four workgroups share a
// CU, so loads, LDS writes and matrix instructions of different workgroups overlap.  The row tiles of one column tile run
// on one XCD (workgroups go to the eight XCDs round-robin), whose L2 then reads the weights once.  Where one product leaves
// CUs idle (the output and value projections: 128 tiles) K is split over gridDim.y and the parts are added by the norm that
// reads the result.
constexpr int TG = 64, TG_RS = TG + 8;         // tile edge; LDS row stride: 16-byte rows 144 bytes apart
__device__ __forceinline__ uint2 lds_tr4(const uint16_t* p) {      // see wkv7_fwd.hip
  typedef short s16x4_t __attribute__((ext_vector_type(4)));
  typedef __attribute__((address_space(3))) s16x4_t* lds_ptr;
  return __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)(p)));
}
typedef uint16_t TileLds[2][2][TG][TG_RS];     // [buffer][x | w]

template <bool KN>
__device__ __forceinline__ void tile_gemm_body(const GemmArgs& A, const GemmJob& J, int n0, int m0, TileLds& lds) {
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, r = lane & 15, g = lane >> 4;
  const int all = (J.K + TG - 1) / TG;
  const int s0 = all * (int)blockIdx.y / (int)gridDim.y, s1 = all * ((int)blockIdx.y + 1) / (int)gridDim.y;
  const int row = tid >> 3, col = (tid & 7) * 8;
  // Addresses stay inside the operands (rows, columns and k beyond an edge re-read its last piece).  What lies beyond K is
  // zeroed on its way to LDS, in the last step only; what lies beyond M or N reaches results that are not stored.
  const uint4 *xp[2], *wp[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int m = m0 + row + 32 * i < A.M ? m0 + row + 32 * i : A.M - 1;
    xp[i] = reinterpret_cast<const uint4*>(J.x + (size_t)m * J.K);
    if (KN) {
      const int n = n0 + col < J.N ? n0 + col : J.N - 8;
      wp[i] = reinterpret_cast<const uint4*>(J.w + n);
    } else {
      const int n = n0 + row + 32 * i < J.N ? n0 + row + 32 * i : J.N - 1;
      wp[i] = reinterpret_cast<const uint4*>(J.w + (size_t)n * J.K);
    }
  }
  auto load = [&](u32x4_t (&x)[2], u32x4_t (&w)[2], int s) {
    const int k = s * TG + col < J.K ? s * TG + col : J.K - 8;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      x[i] = *reinterpret_cast<const u32x4_t*>(xp[i] + k / 8);
      if (KN) {
        const int kk = s * TG + row + 32 * i < J.K ? s * TG + row + 32 * i : J.K - 1;
        w[i] = *reinterpret_cast<const u32x4_t*>(wp[i] + (size_t)kk * (J.N / 8));
      } else {
        w[i] = *reinterpret_cast<const u32x4_t*>(wp[i] + k / 8);
      }
    }
  };
  auto store = [&](u32x4_t (&x)[2], u32x4_t (&w)[2], int s, int buf) {
    if ((s + 1) * TG > J.K) {
      chunk::rare_path();
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const uint32_t mx = s * TG + col < J.K ? 0xffffffffu : 0u;
        const uint32_t mw = KN ? (s * TG + row + 32 * i < J.K ? 0xffffffffu : 0u) : mx;
#pragma unroll
        for (int c = 0; c < 4; ++c) { x[i][c] &= mx; w[i][c] &= mw; }
      }
    }
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      *reinterpret_cast<u32x4_t*>(&lds[buf][0][row + 32 * i][col]) = x[i];
      *reinterpret_cast<u32x4_t*>(&lds[buf][1][row + 32 * i][col]) = w[i];
    }
  };
  f32x4_t acc[2][2];
#pragma unroll
  for (int i = 0; i < 4; ++i) acc[i >> 1][i & 1] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  const int wn = 32 * (wave & 1), wm = 32 * (wave >> 1);
  auto compute = [&](int buf) {
#pragma unroll
    for (int kh = 0; kh < 2; ++kh) {
      u32x4_t wf[2], xf[2];
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        xf[t] = *reinterpret_cast<const u32x4_t*>(&lds[buf][0][wm + 16 * t + r][32 * kh + 8 * g]);
        if (KN) {
          const uint16_t* p = &lds[buf][1][32 * kh + 8 * g + (r >> 2)][wn + 16 * t + 4 * (r & 3)];
          const uint2 lo = lds_tr4(p), hi = lds_tr4(p + 4 * TG_RS);
          wf[t] = u32x4_t{lo.x, lo.y, hi.x, hi.y};
        } else {
          wf[t] = *reinterpret_cast<const u32x4_t*>(&lds[buf][1][wn + 16 * t + r][32 * kh + 8 * g]);
        }
      }
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int u = 0; u < 2; ++u) acc[t][u] = mfma(wf[t], xf[u], acc[t][u]);
    }
  };
  u32x4_t x0[2], w0[2], x1[2], w1[2];
  load(x0, w0, s0);
  load(x1, w1, s0 + 1);
  int s = s0;
  for (; s + 1 < s1; s += 2) {
    // a buffer is written after the barrier that follows its last readers' step
    store(x0, w0, s, 0);
    load(x0, w0, s + 2);
    __syncthreads();
    compute(0);
    store(x1, w1, s + 1, 1);
    load(x1, w1, s + 3);
    __syncthreads();
    compute(1);
  }
  if (s < s1) {
    store(x0, w0, s, 0);
    __syncthreads();
    compute(0);
  }
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int n = n0 + wn + 16 * t + 4 * g, m = m0 + wm + 16 * u + r;
      if (n >= J.N || m >= A.M) continue;
      const f32x4_t v = acc[t][u];
      if (A.part != nullptr)
        *reinterpret_cast<f32x4_t*>(A.part + ((size_t)blockIdx.y * A.M + m) * J.N + n) = v;
      else
        *reinterpret_cast<uint2*>(J.out + (size_t)m * J.N + n) =
            make_uint2(chunk::pack_rn(activate(v[0], J.act), activate(v[1], J.act)),
                       chunk::pack_rn(activate(v[2], J.act), activate(v[3], J.act)));
    }
}

__global__ __launch_bounds__(256) void tile_gemm_kernel(GemmArgs A) {
  __shared__ __align__(16) TileLds lds;
  const int mt = (A.M + TG - 1) / TG;
  const int grp = (int)blockIdx.x / (8 * mt), in = (int)blockIdx.x % (8 * mt);
  const int tile = grp * 8 + in % 8, m0 = in / 8 * TG;
  if (tile >= A.tiles) return;
  int ji = 0;
  for (int i = 1; i < A.n_jobs; ++i) ji = tile >= A.job[i].tile0 ? i : ji;
  const GemmJob J = A.job[ji];
  const int n0 = (tile - J.tile0) * TG;
  if (J.kn) tile_gemm_body<true>(A, J, n0, m0, lds);
  else tile_gemm_body<false>(A, J, n0, m0, lds);
}

// ---------------------------------------------------------------------------------------------------------------
__device__ __forceinline__ float sigmoidf(float z) { return 1.f / (1.f + __expf(-z)); }
__device__ __forceinline__ float softplusf(float z) { return fmaxf(z, 0.f) + __logf(1.f + __expf(-fabsf(z))); }
__device__ __forceinline__ float rnd(float x) { return bf16_to_f32(f32_to_bf16(x)); }

// sum over the wave, delivered to every lane
__device__ __forceinline__ float wave_sum(float x) {
#pragma unroll
  for (int o = 32; o; o >>= 1) x += __shfl_xor(x, o, 64);
  return x;
}

struct CoreArgs {
  int64_t T, H;
  const bf16_t *r, *k, *v, *vf, *xw, *xa, *xv, *g;          // (B,T,H,64); vf null: the first layer
  const bf16_t *w0, *a0, *v0, *k_k, *k_a, *ln_w, *ln_b, *r_k;   // (H,64)
  float eps;
  const bf16_t* s;             // states: H*64*64 elements per sequence, bstride apart
  bf16_t* new_s;
  int64_t bstride;
  const int32_t* length;
  const uint8_t* ns;
  unsigned flags;              // bit 0: the associative scan's conventions, as in the op
  bf16_t* y;
};

// One workgroup per (sequence, head); thread (row i = tid/4, quarter q = tid%4) holds 16 elements of state row i, as in
// the small-T kernel of the op, whose state traffic (2 x 8 KB per head) is the bound.  The state is requested first; wave 0
// (one lane per channel) meanwhile turns the projections into the op's inputs and hands them over through LDS, and takes
// y back through LDS for the group norm, the bonus and the gate.  B=256 H=32: the state alone is 134 MB each way.
__global__ __launch_bounds__(256) void decode_core_kernel(CoreArgs A) {
  __shared__ float ch[5][64];            // d, k', a_i, b_i, r
  __shared__ float vs[64], ys[64];
  const int64_t b = blockIdx.x / A.H, h = blockIdx.x % A.H;
  const int tid = threadIdx.x, i = tid >> 2, q = tid & 3, c0 = 16 * q;
  const bool lead = tid < 64;
  int64_t L = A.T;
  if (A.length != nullptr) { L = A.length[b]; L = L < 0 ? 0 : L < A.T ? L : A.T; }
  const bool compat = (A.flags & 1u) != 0;
  const uint8_t* ns = A.ns ? A.ns + b * A.T : nullptr;
  const bool q2drop = compat && L < A.T && ns != nullptr && ns[L] != 0;
  const size_t sel = (size_t)b * A.bstride + ((size_t)h * 64 + i) * 64 + c0;
  float S[16];
  ld16<bf16_t>(A.s, sel, S);
  auto put_state = [&]() {
    float lo[8], hi[8];
#pragma unroll
    for (int c = 0; c < 8; ++c) { lo[c] = q2drop ? 0.f : S[c]; hi[c] = q2drop ? 0.f : S[8 + c]; }
    st8(A.new_s + sel, lo);
    st8(A.new_s + sel + 8, hi);
  };
  if (L == 0) put_state();
  const size_t cel = (size_t)h * 64 + tid;
  float w0 = 0.f, a0 = 0.f, v0 = 0.f, k_k = 0.f, k_a = 0.f, ln_w = 0.f, ln_b = 0.f, r_k = 0.f;
  if (lead) {
    w0 = ld_f(A.w0 + cel); a0 = ld_f(A.a0 + cel); k_k = ld_f(A.k_k + cel); k_a = ld_f(A.k_a + cel);
    ln_w = ld_f(A.ln_w + cel); ln_b = ld_f(A.ln_b + cel); r_k = ld_f(A.r_k + cel);
    if (A.vf != nullptr) v0 = ld_f(A.v0 + cel);
  }
  for (int64_t t = 0; t < A.T; ++t) {
    float v = 0.f, gate = 0.f, bonus = 0.f;
    const size_t el = (((size_t)b * A.T + t) * A.H + h) * 64 + tid;
    if (lead) {
      const float k = ld_f(A.k + el), r = ld_f(A.r + el), xw = ld_f(A.xw + el), xa = ld_f(A.xa + el);
      gate = ld_f(A.g + el);
      v = ld_f(A.v + el);
      if (A.vf != nullptr) v = rnd(fmaf(ld_f(A.vf + el) - v, sigmoidf(v0 + ld_f(A.xv + el)), v));
      const float a = rnd(sigmoidf(a0 + xa));
      const float w = rnd(-softplusf(-(w0 + xw)) - 0.5f);
      float kk = k * k_k;
      kk *= 1.f / fmaxf(sqrtf(wave_sum(kk * kk)), 1e-12f);
      const float kp = rnd(k * (1.f + (a - 1.f) * k_a));
      bonus = wave_sum(r * kp * r_k);
      ch[0][tid] = __expf(-__expf(w));
      ch[1][tid] = kp;
      ch[2][tid] = rnd(-kk);
      ch[3][tid] = rnd(kk * a);
      ch[4][tid] = r;
      vs[tid] = v;
    }
    __syncthreads();
    if (ns != nullptr && ns[t]) {
#pragma unroll
      for (int c = 0; c < 16; ++c) S[c] = 0.f;
    }
    float p = 0.f;
#pragma unroll
    for (int c = 0; c < 16; ++c) p = fmaf(S[c], ch[2][c0 + c], p);
    const float sa = quad_sum(p), vi = vs[i];
    float y = 0.f;
#pragma unroll
    for (int c = 0; c < 16; ++c) {
      S[c] = fmaf(S[c], ch[0][c0 + c], fmaf(vi, ch[1][c0 + c], sa * ch[3][c0 + c]));
      y = fmaf(S[c], ch[4][c0 + c], y);
    }
    y = quad_sum(y);
    if (compat && t + 1 < A.T && ns != nullptr && ns[t + 1]) y = 0.f;
    if (q == 0) ys[i] = rnd(y);
    if (t == L - 1) put_state();
    __syncthreads();
    if (lead) {
      const float yv = ys[tid];
      const float d = yv - wave_sum(yv) * (1.f / 64.f);
      const float rstd = rsqrtf(wave_sum(d * d) * (1.f / 64.f) + A.eps);
      st_f(A.y + el, (d * rstd * ln_w + ln_b + bonus * v) * gate);
    }
  }
}

// Up to 64 rows one row tile of the streaming kernel reads the weights once.  Beyond, every further row tile streams them
// again (256 rows, 2048 channels: 51 us a launch on average against 18 us of the tiled kernel).
constexpr int TILE_ROWS = 65;          // rows from which the LDS-tiled kernel takes over
constexpr int MAX_SPLIT = 4;

// Parts that a product's K is split into: enough tiles for about two workgroups per CU
int split_of(int M, int64_t K, int64_t N) {
  if (M < TILE_ROWS) return 1;
  const int64_t tiles = (M + TG - 1) / TG * ((N + TG - 1) / TG);
  const int64_t want = 512 / tiles, most = K / (8 * TG);
  const int64_t n = want < most ? want : most;
  return (int)(n < 1 ? 1 : n > MAX_SPLIT ? MAX_SPLIT : n);
}

hipError_t gemm(const GemmArgs& A0, int split, hipStream_t stream) {
  GemmArgs A = A0;
  const bool tiled = A.M >= TILE_ROWS;
  const int edge = tiled ? TG : 16;
  A.tiles = 0;
  for (int i = 0; i < A.n_jobs; ++i) { A.job[i].tile0 = A.tiles; A.tiles += (A.job[i].N + edge - 1) / edge; }
  const dim3 block(64 * GEMM_WAVES);
  if (tiled) hipLaunchKernelGGL(tile_gemm_kernel, dim3((A.tiles + 7) / 8 * 8 * ((A.M + TG - 1) / TG), split), dim3(256), 0, stream, A);
  else if (A.M <= 16) hipLaunchKernelGGL(skinny_gemm_kernel<1>, dim3(A.tiles, 1), block, 0, stream, A);
  else if (A.M <= 32) hipLaunchKernelGGL(skinny_gemm_kernel<2>, dim3(A.tiles, 1), block, 0, stream, A);
  else hipLaunchKernelGGL(skinny_gemm_kernel<4>, dim3(A.tiles, 1), block, 0, stream, A);
  return hipGetLastError();
}

}  // namespace

size_t rwkv7_decode_workspace(const Rwkv7Decode& D) {
  const size_t rows = (size_t)D.B * D.T;
  const size_t d = D.d_decay + D.d_aaa + D.d_mv + D.d_gate;
  // xs twice, six interpolations, r k v v_first, four low-rank results, y, dx; the low-rank hidden values; the ffn's
  const size_t parts = D.B * D.T < TILE_ROWS ? 0 : rows * D.C * MAX_SPLIT * sizeof(float);
  return rows * (18 * D.C + d + D.F) * 2 + parts + 64 * 256;
}

hipError_t launch_rwkv7_decode(const Rwkv7Decode& D, hipStream_t stream) {
  const size_t rows = (size_t)D.B * D.T, C = D.C;
  char* at = static_cast<char*>(D.workspace);
  auto take = [&](size_t cols) {
    bf16_t* p = reinterpret_cast<bf16_t*>(at);
    at += (rows * cols * 2 + 255) / 256 * 256;
    return p;
  };
  bf16_t* xs[2] = {take(C), take(C)};
  bf16_t* mix[6];
  for (auto& m : mix) m = take(C);
  bf16_t *r = take(C), *k = take(C), *v = take(C), *vf = take(C), *xw = take(C), *xa = take(C), *xv = take(C),
         *g = take(C), *y = take(C), *dx = take(C);
  bf16_t *hw = take(D.d_decay), *ha = take(D.d_aaa), *hv = take(D.d_mv), *hg = take(D.d_gate), *ff = take(D.F);
  // the output and the value projection as sums of parts, which the norm after them adds
  float* parts = rows < TILE_ROWS ? nullptr : reinterpret_cast<float*>(at);
  const int split_out = split_of((int)rows, C, C), split_val = split_of((int)rows, D.F, C);
  int n_part = 1;                              // of the dx that the next norm reads
  auto layer = [&](const void* p, int64_t l, size_t n) { return static_cast<const bf16_t*>(p) + (size_t)l * n; };
  const size_t row_state = (2 + 64) * C, seq_state = (size_t)D.L * row_state;
  const bf16_t* st = static_cast<const bf16_t*>(D.state);
  bf16_t* nst = static_cast<bf16_t*>(D.new_state);

  LnMixArgs N;
  memset(&N, 0, sizeof(N));
  N.B = D.B; N.T = D.T; N.C = D.C; N.eps = 1e-5f;
  N.ns = D.new_starts; N.length = D.length;
  auto head = [&](int n_out, const void* x, const void* add, bf16_t* sum, const void* w, const void* b, int64_t l, int srow,
                  const void* const* mixv, bf16_t* const* outs) {
    LnMixArgs A = N;
    A.x = x; A.dx = add; A.xs = sum;
    if (add != nullptr && n_part > 1) { A.dx = nullptr; A.part = parts; A.n_part = n_part; } A.ln_w = w; A.ln_b = b;
    if (n_out) {
      A.prev = st + (size_t)l * row_state + srow * C; A.prev_bstride = seq_state;
      A.shift = nst + (size_t)l * row_state + srow * C; A.shift_bstride = seq_state;
    }
    for (int i = 0; i < n_out; ++i) A.mix[i] = mixv[i];
    for (int i = 0; i < (n_out ? n_out : 1); ++i) A.out[i] = outs[i];
    return launch_ln_shiftmix(0, n_out, A, stream);
  };
  hipError_t e;
#define HIPRWKV_TRY(x) if ((e = (x)) != hipSuccess) return e
  int cur = 0;
  {
    bf16_t* o[1] = {xs[0]};
    HIPRWKV_TRY(head(0, D.x, nullptr, nullptr, D.ln0_w, D.ln0_b, 0, 0, nullptr, o));
  }
  for (int64_t l = 0; l < D.L; ++l) {
    const void* mv[6];
    const void* stacked[6] = {D.x_r, D.x_w, D.x_k, D.x_v, D.x_a, D.x_g};
    for (int i = 0; i < 6; ++i) mv[i] = layer(stacked[i], l, C);
    HIPRWKV_TRY(head(6, xs[cur], l ? dx : nullptr, xs[cur ^ 1], layer(D.ln1_w, l, C), layer(D.ln1_b, l, C), l, 1, mv, mix));
    if (l) cur ^= 1;
    GemmArgs G;
    memset(&G, 0, sizeof(G));
    G.M = (int)rows;
    auto add = [&](const bf16_t* x, const bf16_t* w, bf16_t* out, int64_t K, int64_t Nn, int kn, int act) {
      GemmJob& J = G.job[G.n_jobs++];
      J.x = x; J.w = w; J.out = out; J.K = (int)K; J.N = (int)Nn; J.kn = kn; J.act = act;
    };
    bf16_t* vl = l == 0 ? vf : v;
    add(mix[0], layer(D.receptance, l, C * C), r, C, C, 0, ACT_NONE);
    add(mix[2], layer(D.key, l, C * C), k, C, C, 0, ACT_NONE);
    add(mix[3], layer(D.value, l, C * C), vl, C, C, 0, ACT_NONE);
    add(mix[1], layer(D.w1, l, C * D.d_decay), hw, C, D.d_decay, 1, ACT_TANH);
    add(mix[4], layer(D.a1, l, C * D.d_aaa), ha, C, D.d_aaa, 1, ACT_NONE);
    add(mix[5], layer(D.g1, l, C * D.d_gate), hg, C, D.d_gate, 1, ACT_SIGMOID);
    if (l) add(mix[3], layer(D.v1, l, C * D.d_mv), hv, C, D.d_mv, 1, ACT_NONE);
    HIPRWKV_TRY(gemm(G, 1, stream));
    G.n_jobs = 0;
    add(hw, layer(D.w2, l, C * D.d_decay), xw, D.d_decay, C, 1, ACT_NONE);
    add(ha, layer(D.a2, l, C * D.d_aaa), xa, D.d_aaa, C, 1, ACT_NONE);
    add(hg, layer(D.g2, l, C * D.d_gate), g, D.d_gate, C, 1, ACT_NONE);
    if (l) add(hv, layer(D.v2, l, C * D.d_mv), xv, D.d_mv, C, 1, ACT_NONE);
    HIPRWKV_TRY(gemm(G, 1, stream));
    CoreArgs A;
    memset(&A, 0, sizeof(A));
    A.T = D.T; A.H = D.H;
    A.r = r; A.k = k; A.v = vl; A.vf = l ? vf : nullptr; A.xw = xw; A.xa = xa; A.xv = xv; A.g = g;
    A.w0 = layer(D.w0, l, C); A.a0 = layer(D.a0, l, C); A.v0 = layer(D.v0, l, C);
    A.k_k = layer(D.k_k, l, C); A.k_a = layer(D.k_a, l, C); A.r_k = layer(D.r_k, l, C);
    A.ln_w = layer(D.lnx_w, l, C); A.ln_b = layer(D.lnx_b, l, C); A.eps = 64e-5f;
    A.s = st + (size_t)l * row_state + 2 * C; A.new_s = nst + (size_t)l * row_state + 2 * C; A.bstride = seq_state;
    A.length = D.length; A.ns = D.new_starts; A.flags = (unsigned)D.flags; A.y = y;
    hipLaunchKernelGGL(decode_core_kernel, dim3((unsigned)(D.B * D.H)), dim3(256), 0, stream, A);
    HIPRWKV_TRY(hipGetLastError());
    G.n_jobs = 0;
    add(y, layer(D.output, l, C * C), dx, C, C, 0, ACT_NONE);
    n_part = split_out;
    G.part = n_part > 1 ? parts : nullptr;
    HIPRWKV_TRY(gemm(G, n_part, stream));
    const void* fm[1] = {layer(D.ffn_x_k, l, C)};
    HIPRWKV_TRY(head(1, xs[cur], dx, xs[cur ^ 1], layer(D.ln2_w, l, C), layer(D.ln2_b, l, C), l, 0, fm, mix));
    cur ^= 1;
    G.n_jobs = 0;
    G.part = nullptr;
    add(mix[0], layer(D.ffn_key, l, C * D.F), ff, C, D.F, 0, ACT_RELUSQ);
    HIPRWKV_TRY(gemm(G, 1, stream));
    G.n_jobs = 0;
    add(ff, layer(D.ffn_value, l, C * D.F), dx, D.F, C, 0, ACT_NONE);
    n_part = split_val;
    G.part = n_part > 1 ? parts : nullptr;
    HIPRWKV_TRY(gemm(G, n_part, stream));
  }
  bf16_t* o[1] = {static_cast<bf16_t*>(D.xn)};
  HIPRWKV_TRY(head(0, xs[cur], dx, xs[cur ^ 1], D.ln_out_w, D.ln_out_b, 0, 0, nullptr, o));
  if (D.logits != nullptr) {
    GemmArgs G;
    memset(&G, 0, sizeof(G));
    G.M = (int)rows; G.n_jobs = 1;
    GemmJob& J = G.job[0];
    J.x = static_cast<const bf16_t*>(D.xn); J.w = static_cast<const bf16_t*>(D.head); J.out = static_cast<bf16_t*>(D.logits);
    J.K = (int)C; J.N = (int)D.vocab;
    HIPRWKV_TRY(gemm(G, 1, stream));
  }
#undef HIPRWKV_TRY
  return hipSuccess;
}

}  // namespace hiprwkv
