// Products beside the RWKV-7 recurrence that a library call serves badly, several of them per launch, bf16 in and out, fp32
// accumulation:
//   * a decode step's projections (few rows: a stream of the weights), skinny_gemm_kernel and, from 65 rows on, tile_gemm_kernel;
//   * the low-rank factors of decay, gate, value residual and output gate in whole-sequence passes, forward and backward
//     (rwkv7.py:237-245): narrow on one side, so that a library call of 10-18 us each is mostly launch and latency.
#include "chunk_common.h"
#include "wkv_args.h"

namespace hiprwkv {

namespace {

using chunk::f32x4_t;
using chunk::u32x4_t;
using chunk::mfma;

constexpr int GEMM_WAVES = 8;

__device__ __forceinline__ float activate(float x, int act) {
  switch (act) {
    case GEMM_ACT_TANH: return 1.f - 2.f / (1.f + __expf(2.f * x));
    case GEMM_ACT_SIGMOID: return 1.f / (1.f + __expf(-x));
    case GEMM_ACT_RELUSQ: { const float r = fmaxf(x, 0.f); return r * r; }
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
  const bf16_t* const jx = static_cast<const bf16_t*>(J.x);
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
  const int n0 = ((int)blockIdx.x - J.tile0) * 16;
  const int steps = J.K / 32;
  const int s0 = steps * wave / GEMM_WAVES, s1 = steps * (wave + 1) / GEMM_WAVES;
  f32x4_t acc[MT];
  const bf16_t* xp[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t) {
    acc[t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    const int m = 16 * t + r;
    xp[t] = jx + (size_t)(m < J.M ? m : J.M - 1) * J.K + 8 * g;
  }
  auto step = [&](const u32x4_t w, int s) {
#pragma unroll
    for (int t = 0; t < MT; ++t) acc[t] = mfma(w, *reinterpret_cast<const u32x4_t*>(xp[t] + 32 * s), acc[t]);
  };
  if (!J.kn) {
    const bf16_t* wp = static_cast<const bf16_t*>(J.w) + (size_t)(n0 + r) * J.K + 8 * g;
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
    const uint16_t* wp = static_cast<const uint16_t*>(J.w) + (size_t)(8 * g) * J.N + n0 + r;
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
    const int m = 16 * wave + r;
    if (m < J.M) {
      const uint2 o = make_uint2(chunk::pack_rn(activate(s[0], J.act), activate(s[1], J.act)),
                                 chunk::pack_rn(activate(s[2], J.act), activate(s[3], J.act)));
      *reinterpret_cast<uint2*>(static_cast<bf16_t*>(J.out) + (size_t)m * J.N + n0 + 4 * g) = o;
    }
  }
}

// 64 x 64 tiles, 64 of k per step through two LDS buffers: a thread carries two 16-byte pieces of either operand, requested two
// steps ahead, and four workgroups share a CU, so loads, LDS writes and matrix instructions of different workgroups
// overlap.  An operand that lies k-major (km, kn) goes to LDS as it lies and is read with the transposing load.  The row tiles
// of one column tile run on one XCD (workgroups go to the eight XCDs round-robin), whose L2 then reads the weights once.
// At 256 rows against 6656 columns of 2048 (a decode step of 256 users) the weights' stream needs 5.3 us and the operand reads
// from LDS 6 us; measured 25.  Where one product leaves CUs idle (the output and value projections there: 128 tiles) K is
// split over gridDim.y and the parts are added by the norm that reads the result.
constexpr int TG = 64, TG_RS = TG + 8;         // tile edge; LDS row stride: 16-byte rows 144 bytes apart
typedef uint16_t TileLds[2][2][TG][TG_RS];     // [buffer][x | w]

__device__ __forceinline__ uint2 lds_tr4(const uint16_t* p) {      // see wkv7_fwd.hip
  typedef short s16x4_t __attribute__((ext_vector_type(4)));
  typedef __attribute__((address_space(3))) s16x4_t* lds_ptr;
  return __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)(p)));
}

// One operand of a tile: R rows (of m or n) by K of k, row-major R x K, or with TR its transpose.
template <bool TR>
struct TileOperand {
  const uint4* p[2];
  int row, col, R, K, r0;
  __device__ __forceinline__ TileOperand(const void* base, int R_, int K_, int r0_) : R(R_), K(K_), r0(r0_) {
    row = threadIdx.x >> 3;
    col = (threadIdx.x & 7) * 8;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int rr = r0 + row + 32 * i < R ? r0 + row + 32 * i : R - 1, cc = r0 + col < R ? r0 + col : R - 8;
      p[i] = reinterpret_cast<const uint4*>(static_cast<const bf16_t*>(base) + (TR ? (size_t)cc : (size_t)rr * K));
    }
  }
  // Addresses stay inside the operand: rows and k beyond an edge re-read its last piece.
  __device__ __forceinline__ void load(u32x4_t (&v)[2], int s) const {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      if (TR) {
        const int kk = s * TG + row + 32 * i < K ? s * TG + row + 32 * i : K - 1;
        v[i] = *reinterpret_cast<const u32x4_t*>(p[i] + (size_t)kk * (R / 8));
      } else {
        const int k = s * TG + col < K ? s * TG + col : K - 8;
        v[i] = *reinterpret_cast<const u32x4_t*>(p[i] + k / 8);
      }
    }
  }
  // What lies beyond K is zeroed on its way to LDS (in the last step only); what lies beyond R reaches results that are not
  // stored.
  __device__ __forceinline__ void store(u32x4_t (&v)[2], int s, uint16_t (&lds)[TG][TG_RS]) const {
    if ((s + 1) * TG > K) {
      chunk::rare_path();
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const uint32_t keep = s * TG + (TR ? row + 32 * i : col) < K ? 0xffffffffu : 0u;
#pragma unroll
        for (int c = 0; c < 4; ++c) v[i][c] &= keep;
      }
    }
#pragma unroll
    for (int i = 0; i < 2; ++i) *reinterpret_cast<u32x4_t*>(&lds[row + 32 * i][col]) = v[i];
  }
  // rows t .. t+15, k 32 kh + 8g .. + 7 of the tile, lane (r, g)
  static __device__ __forceinline__ u32x4_t frag(const uint16_t (&lds)[TG][TG_RS], int t, int kh, int r, int g) {
    if (TR) {
      const uint16_t* q = &lds[32 * kh + 8 * g + (r >> 2)][t + 4 * (r & 3)];
      const uint2 lo = lds_tr4(q), hi = lds_tr4(q + 4 * TG_RS);
      return u32x4_t{lo.x, lo.y, hi.x, hi.y};
    }
    return *reinterpret_cast<const u32x4_t*>(&lds[t + r][32 * kh + 8 * g]);
  }
};

template <bool KM, bool KN>
__device__ __forceinline__ void tile_gemm_body(const GemmArgs& A, const GemmJob& J, int n0, int m0, TileLds& lds) {
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
  const int all = (J.K + TG - 1) / TG;
  const int s0 = all * (int)blockIdx.y / (int)gridDim.y, s1 = all * ((int)blockIdx.y + 1) / (int)gridDim.y;
  const TileOperand<KM> X(J.x, J.M, J.K, m0);
  const TileOperand<KN> W(J.w, J.N, J.K, n0);
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
        xf[t] = TileOperand<KM>::frag(lds[buf][0], wm + 16 * t, kh, r, g);
        wf[t] = TileOperand<KN>::frag(lds[buf][1], wn + 16 * t, kh, r, g);
      }
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int u = 0; u < 2; ++u) acc[t][u] = mfma(wf[t], xf[u], acc[t][u]);
    }
  };
  u32x4_t x0[2], w0[2], x1[2], w1[2];
  X.load(x0, s0); W.load(w0, s0);
  X.load(x1, s0 + 1); W.load(w1, s0 + 1);
  int s = s0;
  for (; s + 1 < s1; s += 2) {
    // a buffer is written after the barrier that follows its last readers' step
    X.store(x0, s, lds[0][0]); W.store(w0, s, lds[0][1]);
    X.load(x0, s + 2); W.load(w0, s + 2);
    __syncthreads();
    compute(0);
    X.store(x1, s + 1, lds[1][0]); W.store(w1, s + 1, lds[1][1]);
    X.load(x1, s + 3); W.load(w1, s + 3);
    __syncthreads();
    compute(1);
  }
  if (s < s1) {
    X.store(x0, s, lds[0][0]); W.store(w0, s, lds[0][1]);
    __syncthreads();
    compute(0);
  }
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int n = n0 + wn + 16 * t + 4 * g, m = m0 + wm + 16 * u + r;
      if (n >= J.N || m >= J.M) continue;
      f32x4_t v = acc[t][u];
      if (A.part != nullptr) {
        *reinterpret_cast<f32x4_t*>(A.part + ((size_t)blockIdx.y * J.M + m) * J.N + n) = v;
        continue;
      }
      const size_t el = (size_t)m * J.N + n;
      if (J.aux != nullptr) {
        const uint2 q = *reinterpret_cast<const uint2*>(static_cast<const bf16_t*>(J.aux) + el);
        const float h[4] = {__uint_as_float(q.x << 16), __uint_as_float(q.x & 0xffff0000u), __uint_as_float(q.y << 16),
                            __uint_as_float(q.y & 0xffff0000u)};
#pragma unroll
        for (int i = 0; i < 4; ++i)
          v[i] = J.act == GEMM_ADD ? v[i] + h[i] : J.act == GEMM_DTANH ? v[i] * (1.f - h[i] * h[i]) : v[i] * (h[i] * (1.f - h[i]));
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = activate(v[i], J.act);
      }
      *reinterpret_cast<uint2*>(static_cast<bf16_t*>(J.out) + el) = make_uint2(chunk::pack_rn(v[0], v[1]), chunk::pack_rn(v[2], v[3]));
    }
}

__global__ __launch_bounds__(256) void tile_gemm_kernel(GemmArgs A) {
  __shared__ __align__(16) TileLds lds;
  int ji = 0;
  for (int i = 1; i < A.n_jobs; ++i) ji = (int)blockIdx.x >= A.job[i].tile0 ? i : ji;
  const GemmJob J = A.job[ji];
  // eight column tiles at a time, all row tiles of each on one XCD
  const int mt = (J.M + TG - 1) / TG, local = (int)blockIdx.x - J.tile0;
  const int grp = local / (8 * mt), in = local % (8 * mt);
  const int n0 = (grp * 8 + in % 8) * TG, m0 = in / 8 * TG;
  if (n0 >= J.N) return;
  if (J.km) {
    if (J.kn) tile_gemm_body<true, true>(A, J, n0, m0, lds);
    else tile_gemm_body<true, false>(A, J, n0, m0, lds);
  } else {
    if (J.kn) tile_gemm_body<false, true>(A, J, n0, m0, lds);
    else tile_gemm_body<false, false>(A, J, n0, m0, lds);
  }
}

}  // namespace

// Parts that a product's K is split into: enough tiles for about two workgroups per CU
int gemm_split(int M, int64_t K, int64_t N) {
  if (M < GEMM_TILE_ROWS) return 1;
  const int64_t tiles = (M + TG - 1) / TG * ((N + TG - 1) / TG);
  const int64_t want = 512 / tiles, most = K / (8 * TG);
  const int64_t n = want < most ? want : most;
  return (int)(n < 1 ? 1 : n > GEMM_MAX_SPLIT ? GEMM_MAX_SPLIT : n);
}

// Up to 64 rows one row tile of the streaming kernel reads the weights once; K is then a multiple of 32, N of 16.  Beyond,
// every further row tile would stream them again (256 rows, 2048 channels: 51 us a launch on average against 18 us tiled).
hipError_t launch_gemm(GemmArgs A, int split, hipStream_t stream) {
  bool skinny = A.part == nullptr;
  int M = 0, tiles = 0;
  for (int i = 0; i < A.n_jobs; ++i) {
    const GemmJob& J = A.job[i];
    M = J.M > M ? J.M : M;
    skinny = skinny && J.M < GEMM_TILE_ROWS && !J.km && J.aux == nullptr && J.K % 32 == 0 && J.N % 16 == 0;
  }
  for (int i = 0; i < A.n_jobs; ++i) {
    GemmJob& J = A.job[i];
    J.tile0 = tiles;
    tiles += skinny ? J.N / 16 : (J.N + 8 * TG - 1) / (8 * TG) * 8 * ((J.M + TG - 1) / TG);
  }
  const dim3 block(64 * GEMM_WAVES);
  if (!skinny) hipLaunchKernelGGL(tile_gemm_kernel, dim3(tiles, split), dim3(256), 0, stream, A);
  else if (M <= 16) hipLaunchKernelGGL(skinny_gemm_kernel<1>, dim3(tiles), block, 0, stream, A);
  else if (M <= 32) hipLaunchKernelGGL(skinny_gemm_kernel<2>, dim3(tiles), block, 0, stream, A);
  else hipLaunchKernelGGL(skinny_gemm_kernel<4>, dim3(tiles), block, 0, stream, A);
  return hipGetLastError();
}

}  // namespace hiprwkv
