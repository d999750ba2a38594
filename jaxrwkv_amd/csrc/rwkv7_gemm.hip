// Products beside the RWKV-7 recurrence that a library call serves badly, several of them per launch, bf16 in and out, fp32
// accumulation:
//   * a decode step's projections (few rows: a stream of the weights), skinny_gemm_kernel and, from 33 rows on, tiles;
//   * the low-rank factors of decay, gate, value residual and output gate in whole-sequence passes, forward and backward
//     (rwkv7.py:237-245): narrow on one side, so that a library call of 10-18 us each is mostly launch and latency.
#include "chunk_common.h"
#include "rwkv7_pre.h"
#include "wkv_args.h"

#include <type_traits>

namespace hiprwkv {

namespace {

using chunk::f32x4_t;
using chunk::u32x4_t;
using chunk::mfma;

constexpr int GEMM_WAVES = 8;

// f of a product, which is rounded to bf16 first, where the separate product would be stored.
// tanh is 1 - 2 / (1 + e^2x) where that keeps its value to 1e-6 (its error is 1e-7 of one whatever x is) and the series below (the
// next term is 62/2835 x^8).  This code is inlined at every store of the kernels of few rows and its length costs them, so tanh
// and sigmoid share the quotient; the tiles apply it in one loop (TileOut::write).
__device__ __forceinline__ float activate(float x, int act) {
  if (act == GEMM_ACT_NONE) return x;
  x = rnd(x);
  if (act == GEMM_ACT_RELUSQ) { const float r = fmaxf(x, 0.f); return r * r; }
  const bool th = act == GEMM_ACT_TANH;
  const float q = 1.f / (1.f + __expf(th ? 2.f * x : -x)), s = x * x;
  const float series = x * fmaf(s, fmaf(s, fmaf(s, -17.f / 315.f, 2.f / 15.f), -1.f / 3.f), 1.f);
  return !th ? q : fabsf(x) < 0.25f ? series : 1.f - 2.f * q;
}

__device__ __forceinline__ float half_of(const u32x4_t v, int e) {        // value e of eight
  return __uint_as_float(e & 1 ? v[e >> 1] & 0xffff0000u : v[e >> 1] << 16);
}

// The job of a tile.  The first tiles are read at once and the job after them: as a loop over the jobs' own first tiles a grid of seven
// began with seven reads that waited for each other.
__device__ __forceinline__ int job_of(const GemmArgs& A, int tile) {
  int ji = 0;
#pragma unroll
  for (int i = 1; i < GEMM_MAX_JOBS; ++i) ji = tile >= A.tile0[i] ? i : ji;      // beyond the last: INT_MAX
  return ji;
}
// columns (or tiles) of a job -> the first tiles; returns their number
template <typename F>
int place_jobs(GemmArgs& A, F&& tiles_of_job) {
  int tiles = 0;
  for (int i = 0; i < GEMM_MAX_JOBS; ++i) {
    A.tile0[i] = i < A.n_jobs ? tiles : INT_MAX;
    if (i < A.n_jobs) tiles += tiles_of_job(A.job[i]);
  }
  return tiles;
}

__device__ __forceinline__ uint2 lds_tr4(const uint16_t* p) {      // see wkv7_fwd.hip
  typedef short s16x4_t __attribute__((ext_vector_type(4)));
  typedef __attribute__((address_space(3))) s16x4_t* lds_ptr;
  return __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)(p)));
}

// Sixteen columns of a KN weight (the low-rank factors) by 32 of k for one wave: two lanes read a row, and the matrix operand (column r, k =
// 8g ..) comes out of a KiB of LDS that only this wave uses, by the transposing read.  As eight reads of two bytes a lane these factors held
// up the launch that they share with r, k and v: 6.9 us a launch (768 channels, one user), 6.0 now.
constexpr int KN_LDS = 512;                    // values a wave
struct KnWeights {
  const uint16_t* at;
  int N, lane;
  __device__ __forceinline__ KnWeights(const void* w, int N_, int n0, int lane_)
      : at(static_cast<const uint16_t*>(w) + (size_t)(lane_ >> 1) * N_ + n0 + 8 * (lane_ & 1)), N(N_), lane(lane_) {}
  __device__ __forceinline__ u32x4_t load(int s, int n = 0) const { return *reinterpret_cast<const u32x4_t*>(at + (size_t)32 * s * N + n); }
  // in the order of the wave's LDS instructions: the next piece may follow at once
  __device__ __forceinline__ u32x4_t operand(u32x4_t v, uint16_t* lds) const {
    *reinterpret_cast<u32x4_t*>(lds + 8 * lane) = v;
    const int r = lane & 15, g = lane >> 4;
    const uint16_t* q = lds + (8 * g + (r >> 2)) * 16 + 4 * (r & 3);
    const uint2 lo = lds_tr4(q), hi = lds_tr4(q + 4 * 16);
    return u32x4_t{lo.x, lo.y, hi.x, hi.y};
  }
};

// Weight-streaming product for few rows: bound by reading w once.  A workgroup owns 16 columns of one product and 16 MT
// rows; its eight waves split K (every wave of the grid then streams a run of k of sixteen weight rows, so that many
// short streams are in flight however small N is) and add their 16x16 tiles through LDS.  The weights' rows are the
// matrix instruction's A operand straight from memory, 16 bytes per lane, no LDS; x comes from the cache.  KN weights: KnWeights.
// ONE: a single product, whose arguments are then one load away.
template <int MT, bool ONE>
__global__ __launch_bounds__(64 * GEMM_WAVES) void skinny_gemm_kernel(GemmArgs A) {
  __shared__ f32x4_t red[GEMM_WAVES][MT][64];
  __shared__ __align__(16) uint16_t kn_lds[GEMM_WAVES][KN_LDS];
  const int ji = ONE ? 0 : job_of(A, blockIdx.x);
  const GemmJob J = A.job[ji];
  const bf16_t* const jx = static_cast<const bf16_t*>(J.x);
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
  const int n0 = ONE ? (int)blockIdx.x * 16 : ((int)blockIdx.x - A.tile0[ji]) * 16;
  const int steps = J.K / 32, part = wave + GEMM_WAVES * (int)blockIdx.y, log_parts = 3 + A.log_split;
  const int s0 = steps * part >> log_parts, s1 = steps * (part + 1) >> log_parts;
  f32x4_t acc[MT];
  const bf16_t* xp[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t) {
    acc[t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    const int m = 16 * t + r;
    xp[t] = jx + (size_t)(m < J.M ? m : J.M - 1) * J.K + 8 * g;
  }
  const bf16_t* const wp = static_cast<const bf16_t*>(J.w) + (size_t)(n0 + r) * J.K + 8 * g;
  const KnWeights wk(J.w, J.N, n0, lane);
  // COUNT steps whose loads are all requested before the first product; four at most, with eight fewer workgroups share a CU (24 layers of 2048
  // channels, 16 users: 1752 us a step with eight, 1664 with four; one step after the other for what is left over: 1684)
  auto steps_of = [&](auto count, int s) {
    constexpr int COUNT = decltype(count)::value;
    u32x4_t w[COUNT], x[COUNT][MT];
#pragma unroll
    for (int u = 0; u < COUNT; ++u) w[u] = J.kn ? wk.load(s + u) : *reinterpret_cast<const u32x4_t*>(wp + 32 * (s + u));
#pragma unroll
    for (int u = 0; u < COUNT; ++u) {
#pragma unroll
      for (int t = 0; t < MT; ++t) x[u][t] = *reinterpret_cast<const u32x4_t*>(xp[t] + 32 * (s + u));
    }
#pragma unroll
    for (int u = 0; u < COUNT; ++u) {
      const u32x4_t wf = J.kn ? wk.operand(w[u], kn_lds[wave]) : w[u];
#pragma unroll
      for (int t = 0; t < MT; ++t) acc[t] = mfma(wf, x[u][t], acc[t]);
    }
  };
  constexpr int UN = 4;
  int s = s0;
  for (; s + UN <= s1; s += UN) steps_of(std::integral_constant<int, UN>(), s);
  switch (s1 - s) {
    case 3: steps_of(std::integral_constant<int, 3>(), s); break;
    case 2: steps_of(std::integral_constant<int, 2>(), s); break;
    case 1: steps_of(std::integral_constant<int, 1>(), s); break;
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
    if (m < J.M && A.part != nullptr) {
      *reinterpret_cast<f32x4_t*>(A.part + ((size_t)blockIdx.y * J.M + m) * J.N + n0 + 4 * g) = s;
    } else if (m < J.M) {
      const uint2 o = make_uint2(chunk::pack_rn(activate(s[0], J.act), activate(s[1], J.act)),
                                 chunk::pack_rn(activate(s[2], J.act), activate(s[3], J.act)));
      *reinterpret_cast<uint2*>(static_cast<bf16_t*>(J.out) + (size_t)m * J.N + n0 + 4 * g) = o;
    }
  }
}

// What ln_shiftmix_kernel and the product above do, in one launch for one or two rows (a decode step of few users).  There a launch of
// its own costs more than doing the norm again in every workgroup while the weights are on their way.  Such a kernel is a chain of
// latencies: 0.4 us until the arguments are there, 0.4 to 0.6 for its rows, 1.4 for weights that no cache holds, 0.2 for a barrier, 2.2 ns an
// instruction of a wave that has its SIMD to itself.  So the rows are requested before the weights (memory answers a wave in order), and a
// wave normalises the channels of its own part of K alone: sixteen lanes a row, eight channels a lane and turn.  One barrier, for the sums:
// mean and squares about it are combined from those of the eight parts, which is as precise as a second pass.  The interpolated values go to
// the matrix instruction's layout through LDS that only this wave uses.  768 channels, one user: 7.4 and 6.2 us a launch (r, k, v; key), now 6.0 and 4.9, of which 1.7 are the launch.
// Workgroup 0 writes the residual stream and the state's shift row.
// G: rows; TURNS: times 128 channels of a wave; NT: times 16 columns of a workgroup.
template <int G, int TURNS, int NT>
__global__ __launch_bounds__(64 * GEMM_WAVES) void head_gemm_kernel(LnMixArgs N, GemmArgs A) {
  __shared__ __align__(16) u32x4_t ops[GEMM_WAVES][G][16 * TURNS];       // 8 channels each
  __shared__ f32x4_t red[GEMM_WAVES][NT][4][G];
  __shared__ __align__(16) uint16_t kn_lds[GEMM_WAVES][KN_LDS];
  __shared__ float2 sums[G][16];                                 // mean and squares about it of a wave's channels
  constexpr int AHEAD_W = TURNS < 2 ? 4 : 8;                     // steps of K whose weights are requested first
  const int ji = job_of(A, blockIdx.x);
  const GemmJob J = A.job[ji];
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, r = lane & 15, g = lane >> 4;
  const int C = (int)N.C, T = (int)N.T;
  const int n0 = ((int)blockIdx.x - A.tile0[ji]) * 16 * NT;
  const int steps = C / 32, s0 = steps * wave / GEMM_WAVES, s1 = steps * (wave + 1) / GEMM_WAVES, count = 32 * (s1 - s0);
  // the norm: row j, channels 32 s0 + 8 (r + 16 i) ..
  const int j = G == 1 ? 0 : g & 1, b = T == 1 ? j : 0, t = T == 1 ? 0 : j;
  const bool reset = N.ns != nullptr && N.ns[j] != 0;
  const int first = 32 * s0 + 8 * r;
  u32x4_t x[TURNS], lnw[TURNS], lnb[TURNS], share[TURNS], before[TURNS];
  f32x4_t d[4][TURNS][2];                        // what the residual stream gains: a product, or its first four partial sums
#pragma unroll
  for (int i = 0; i < TURNS; ++i) {
    x[i] = lnw[i] = lnb[i] = share[i] = before[i] = u32x4_t{0u, 0u, 0u, 0u};
#pragma unroll
    for (int p = 0; p < 4; ++p) d[p][i][0] = d[p][i][1] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  }
  if (g < G) {                                   // only the lanes that a row has: a request costs the CU by its lanes
#pragma unroll
    for (int i = 0; i < TURNS; ++i) {
      const int c = 8 * r + 128 * i < count ? first + 128 * i : 0;       // beyond the part: read, not used
      auto at = [&](const void* p, size_t el) { return *reinterpret_cast<const u32x4_t*>(static_cast<const bf16_t*>(p) + el); };
      x[i] = at(N.x, (size_t)j * C + c);
      if (N.n_part > 1) {
#pragma unroll
        for (int p = 0; p < 4; ++p)
          if (p < 2 || p < N.n_part) {
            const f32x4_t* q = reinterpret_cast<const f32x4_t*>(N.part + (size_t)(p * G + j) * C + c);
            d[p][i][0] = q[0];
            d[p][i][1] = q[1];
          }
      } else if (N.dx != nullptr) {
        d[0][i][0] = __builtin_bit_cast(f32x4_t, at(N.dx, (size_t)j * C + c));
      }
      lnw[i] = at(N.ln_w, c);
      lnb[i] = at(N.ln_b, c);
      share[i] = at(J.aux, c);
      before[i] = at(N.prev, (size_t)b * N.prev_bstride + c);
    }
  }
  const bf16_t* const wp = static_cast<const bf16_t*>(J.w) + (size_t)(n0 + r) * C + 8 * g;
  const KnWeights wk(J.w, J.N, n0, lane);
  auto weights = [&](int s, int q) {
    return J.kn ? wk.load(s, 16 * q) : *reinterpret_cast<const u32x4_t*>(wp + (size_t)16 * q * C + 32 * s);
  };
  auto operand = [&](u32x4_t v) { return J.kn ? wk.operand(v, kn_lds[wave]) : v; };
  u32x4_t w[AHEAD_W][NT];
#pragma unroll
  for (int u = 0; u < AHEAD_W; ++u)
#pragma unroll
    for (int q = 0; q < NT; ++q) w[u][q] = weights(s0 + u < s1 ? s0 + u : steps - 1, q);
  // the residual stream, rounded as it is stored
  float sum = 0.f;
#pragma unroll
  for (int i = 0; i < TURNS; ++i) {
    const bool have = 8 * r + 128 * i < count;
    if (N.n_part > 1) {
      f32x4_t lo = d[0][i][0] + d[1][i][0], hi = d[0][i][1] + d[1][i][1];
      lo = lo + d[2][i][0]; hi = hi + d[2][i][1];
      lo = lo + d[3][i][0]; hi = hi + d[3][i][1];
      for (int p = 4; p < N.n_part; ++p) {
        const f32x4_t* q = reinterpret_cast<const f32x4_t*>(N.part + (size_t)(p * G + j) * C + (have ? first + 128 * i : 0));
        lo += q[0];
        hi += q[1];
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float s0_ = e < 2 ? lo[2 * e] : hi[2 * e - 4], s1_ = e < 2 ? lo[2 * e + 1] : hi[2 * e - 3];
        x[i][e] = chunk::pack_rn(half_of(x[i], 2 * e) + rnd(s0_), half_of(x[i], 2 * e + 1) + rnd(s1_));
      }
    } else if (N.dx != nullptr) {
      const u32x4_t dx = __builtin_bit_cast(u32x4_t, d[0][i][0]);
#pragma unroll
      for (int e = 0; e < 4; ++e)
        x[i][e] = chunk::pack_rn(half_of(x[i], 2 * e) + half_of(dx, 2 * e), half_of(x[i], 2 * e + 1) + half_of(dx, 2 * e + 1));
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) sum += have ? half_of(x[i], e) : 0.f;
  }
  const float mine = row_sum(sum) / (float)(count > 0 ? count : 1);
  float sq = 0.f;
#pragma unroll
  for (int i = 0; i < TURNS; ++i) {
    const bool have = 8 * r + 128 * i < count;
#pragma unroll
    for (int e = 0; e < 8; ++e) { const float v = half_of(x[i], e) - mine; sq = have ? fmaf(v, v, sq) : sq; }
  }
  sq = row_sum(sq);
  if (r == 0 && g < G) sums[g][wave] = make_float2(mine, sq);
  __syncthreads();
  const float invC = 1.f / (float)C;
  const float2 of = sums[j][r & 7];
  const float n = r < 8 ? 32.f * (float)(steps * (r + 1) / GEMM_WAVES - steps * r / GEMM_WAVES) : 0.f;
  const float mean = row_sum(n * of.x) * invC, off = of.x - mean;
  const float rstd = rsqrtf(row_sum(r < 8 ? fmaf(n * off, off, of.y) : 0.f) * invC + N.eps);
  u32x4_t xn[TURNS];
#pragma unroll
  for (int i = 0; i < TURNS; ++i) {
#pragma unroll
    for (int e = 0; e < 4; ++e)
      xn[i][e] = chunk::pack_rn(fmaf((half_of(x[i], 2 * e) - mean) * rstd, half_of(lnw[i], 2 * e), half_of(lnb[i], 2 * e)),
                                fmaf((half_of(x[i], 2 * e + 1) - mean) * rstd, half_of(lnw[i], 2 * e + 1), half_of(lnb[i], 2 * e + 1)));
    u32x4_t p = before[i];
    if (G > 1 && T > 1) {                        // the second token follows the first, sixteen lanes below
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const uint32_t q = (uint32_t)__shfl((int)xn[i][e], lane - 16, 64);
        p[e] = t > 0 ? q : p[e];
      }
    }
    u32x4_t o;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float lo = half_of(xn[i], 2 * e), hi = half_of(xn[i], 2 * e + 1);
      o[e] = chunk::pack_rn(fmaf((reset ? 0.f : half_of(p, 2 * e)) - lo, half_of(share[i], 2 * e), lo),
                            fmaf((reset ? 0.f : half_of(p, 2 * e + 1)) - hi, half_of(share[i], 2 * e + 1), hi));
    }
    if (g < G) ops[wave][j][r + 16 * i] = o;
  }
  // a wave's own writes and reads of LDS are in order
  f32x4_t acc[NT];
#pragma unroll
  for (int q = 0; q < NT; ++q) acc[q] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  const u32x4_t* const op = ops[wave][r < G ? r : G - 1] + g;
#pragma unroll
  for (int u = 0; u < AHEAD_W; ++u)
    if (s0 + u < s1) {
      const u32x4_t o = op[4 * u];
#pragma unroll
      for (int q = 0; q < NT; ++q) acc[q] = mfma(operand(w[u][q]), o, acc[q]);
    }
  for (int s = s0 + AHEAD_W; s < s1; ++s) {
    u32x4_t ws[NT];
#pragma unroll
    for (int q = 0; q < NT; ++q) ws[q] = weights(s, q);
    const u32x4_t o = op[4 * (s - s0)];
#pragma unroll
    for (int q = 0; q < NT; ++q) acc[q] = mfma(operand(ws[q]), o, acc[q]);
  }
  if (r < G) {
#pragma unroll
    for (int q = 0; q < NT; ++q) red[wave][q][g][r] = acc[q];
  }
  __syncthreads();
  if (wave < NT && r < G) {
    f32x4_t v = red[0][wave][g][r];
#pragma unroll
    for (int q = 1; q < GEMM_WAVES; ++q) v += red[q][wave][g][r];
    const uint2 o = make_uint2(chunk::pack_rn(activate(v[0], J.act), activate(v[1], J.act)),
                               chunk::pack_rn(activate(v[2], J.act), activate(v[3], J.act)));
    *reinterpret_cast<uint2*>(static_cast<bf16_t*>(J.out) + (size_t)r * J.N + n0 + 16 * wave + 4 * g) = o;
  }
  if (blockIdx.x == 0 && g < G) {
#pragma unroll
    for (int i = 0; i < TURNS; ++i) {
      if (8 * r + 128 * i >= count) break;
      const int c = first + 128 * i;
      if (N.dx != nullptr || N.n_part > 1) *reinterpret_cast<u32x4_t*>(static_cast<bf16_t*>(N.xs) + (size_t)j * C + c) = x[i];
      if (t == (int)last_token(N.length, b, T))
        *reinterpret_cast<u32x4_t*>(static_cast<bf16_t*>(N.shift) + (size_t)b * N.shift_bstride + c) = xn[i];
    }
  }
}

// 64 x 64 tiles through registers, 64 of K per step through two LDS buffers, for products of a short K alone in their launch (the second
// low-rank factors of a decode step): a thread carries two 16-byte pieces of either operand, requested two steps ahead, and four
// workgroups share a CU, so loads, LDS writes and matrix instructions of different workgroups overlap.  An operand that lies k-major (km, kn) goes to LDS as it lies and is read with the transposing load.  Workgroups go
// to the eight XCDs round-robin; the tiles that share a piece of the longer operand run on one XCD, whose L2 reads it once.
// Its waves wait for 63 % of their time in a decode step of 256 users (profiles/rwkv7_model_bf16.md): a step moves 16 KiB in, 16 KiB to
// LDS and 32 KiB from it for 32 matrix instructions.  Weights straight from memory into the matrix operands were slower (a cache line
// per lane), and so were four steps in flight.  Where one product leaves CUs idle K is split over gridDim.y, in these tiles and those
// below (a decode step's output and value projections: 128 tiles), and the parts are added by the norm that reads the result.
constexpr int TG = 64, TG_RS = TG + 8;         // tile edge; LDS row stride: 16-byte rows 144 bytes apart
constexpr int AHEAD = 2;                       // steps whose operands are in flight (four: 212 registers, 1.6 times slower for short K)
typedef uint16_t TileLds[2][2][TG][TG_RS];     // [buffer][x | w]

using chunk::rsrc_t;
using chunk::make_rsrc;
__device__ __forceinline__ u32x4_t buf_ld16(rsrc_t r, int voff, int soff) {
  return __builtin_bit_cast(u32x4_t, __builtin_amdgcn_raw_buffer_load_b128(r, voff, soff, 0));
}

// One operand of a tile: R rows (of m or n) by K of k, row-major R x K, or with TR its transpose.  Addressed through a buffer
// descriptor: a lane's offset is computed once and a step's is a scalar, so that a request costs one instruction.  Rows
// beyond the edge re-read the last one (what they give is not stored).  EXACT: K is a multiple of the step; otherwise k beyond K
// re-reads the last piece and is zeroed on its way to LDS.  Requests beyond the last step re-read it.
template <bool TR, bool EXACT>
struct TileOperand {
  rsrc_t rs;
  int voff[2], row, col, R, K, last;
  __device__ __forceinline__ TileOperand(const void* base, int R_, int K_, int r0, int tid) : R(R_), K(K_) {
    row = tid >> 3;
    col = (tid & 7) * 8;
    last = (K - 1) / TG;
    // the descriptor starts at the tile, so that offsets stay small whatever the operand's size
    const int64_t first = TR ? (int64_t)(r0 < R ? r0 : R - 8) : (int64_t)(r0 < R ? r0 : R - 1) * K;
    rs = make_rsrc(static_cast<const bf16_t*>(base) + first);
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int rr = r0 + row + 32 * i < R ? row + 32 * i : R - 1 - r0, cc = r0 + col < R ? col : R - 8 - r0;
      voff[i] = TR ? ((row + 32 * i) * R + cc) * 2 : (rr * K + col) * 2;
    }
  }
  __device__ __forceinline__ void load(u32x4_t (&v)[2], int s) const {
    s = s < last ? s : last;
    const int soff = TR ? s * TG * R * 2 : s * TG * 2;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      int o = voff[i];
      if (!EXACT) {
        if (TR) o -= s * TG + row + 32 * i < K ? 0 : (s * TG + row + 32 * i - (K - 1)) * R * 2;
        else o -= s * TG + col < K ? 0 : (s * TG + col - (K - 8)) * 2;
      }
      v[i] = buf_ld16(rs, o, soff);
    }
  }
  __device__ __forceinline__ void store(u32x4_t (&v)[2], int s, uint16_t (&lds)[TG][TG_RS]) const {
    if (!EXACT && (s + 1) * TG > K) {
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

// A tile's results.  Partial sums go to memory as they lie; everything else is rounded first, whatever follows (a separate product would
// be stored there), so the tile goes through LDS as bf16 and out as rows of whole cache lines, eight values a lane, f in a loop whose
// code is short: with f inlined at each of a lane's sixteen stores of 8 bytes, key projections of 2048 rows (768 into 3072, relu^2 beside
// the product) took 31.8 us, 22.4 now, their backward with the weights' cotangents 53.5, 47.8 now; 256 rows of r, k, v and the low-rank inputs
// (2048 channels) 25.4, 22.2 now.
template <int TM, int TN>
struct TileOut {
  static constexpr int STRIDE = TN + 8;
  static constexpr size_t BYTES = (size_t)TM * STRIDE * 2;
  // columns n .. n + 3 of row m of the tile
  static __device__ __forceinline__ void put(const GemmArgs& A, const GemmJob& J, uint16_t* lds, int n0, int m0, int n, int m, f32x4_t v) {
    if (A.part != nullptr) {
      if (n0 + n < J.N && m0 + m < J.M)
        *reinterpret_cast<f32x4_t*>(A.part + ((size_t)blockIdx.y * J.M + m0 + m) * J.N + n0 + n) = v;
      return;
    }
    *reinterpret_cast<uint2*>(lds + m * STRIDE + n) = make_uint2(chunk::pack_rn(v[0], v[1]), chunk::pack_rn(v[2], v[3]));
  }
  // by all threads of a workgroup, after a barrier
  template <int THREADS>
  static __device__ __forceinline__ void write(const GemmArgs& A, const GemmJob& J, const uint16_t* lds, int n0, int m0) {
    if (A.part != nullptr) return;
    constexpr int PIECES = TN / 8;
#pragma unroll 1
    for (int i = threadIdx.x; i < TM * PIECES; i += THREADS) {
      const int m = i / PIECES, n = 8 * (i % PIECES);
      if (m0 + m >= J.M || n0 + n >= J.N) continue;
      const size_t el = (size_t)(m0 + m) * J.N + n0 + n;
      u32x4_t q = *reinterpret_cast<const u32x4_t*>(lds + m * STRIDE + n);
      if (J.aux != nullptr || J.act != GEMM_ACT_NONE) {
        if (J.raw != nullptr) *reinterpret_cast<u32x4_t*>(static_cast<bf16_t*>(J.raw) + el) = q;
        float v[8], h[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = half_of(q, e);
        if (J.aux != nullptr) {
          ld8(static_cast<const bf16_t*>(J.aux) + el, h);
#pragma unroll
          for (int e = 0; e < 8; ++e)
            v[e] = J.act == GEMM_ADD ? v[e] + h[e] : J.act == GEMM_DTANH ? v[e] * (1.f - h[e] * h[e])
                 : J.act == GEMM_DRELUSQ ? 2.f * v[e] * fmaxf(h[e], 0.f) : v[e] * (h[e] * (1.f - h[e]));
        } else if (J.act == GEMM_ACT_RELUSQ) {
#pragma unroll
          for (int e = 0; e < 8; ++e) { const float p = fmaxf(v[e], 0.f); v[e] = p * p; }
        } else {
#pragma unroll
          for (int e = 0; e < 8; ++e) v[e] = activate(v[e], J.act);
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) q[e] = chunk::pack_rn(v[2 * e], v[2 * e + 1]);
      }
      *reinterpret_cast<u32x4_t*>(static_cast<bf16_t*>(J.out) + el) = q;
    }
  }
};

template <bool KM, bool KN, bool EXACT>
__device__ __forceinline__ void tile_gemm_body(const GemmArgs& A, const GemmJob& J, int n0, int m0, TileLds& lds) {
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
  const int all = (J.K + TG - 1) / TG;
  const int s0 = all * (int)blockIdx.y / (int)gridDim.y, s1 = all * ((int)blockIdx.y + 1) / (int)gridDim.y;
  const TileOperand<KM, EXACT> X(J.x, J.M, J.K, m0, threadIdx.x);
  const TileOperand<KN, EXACT> W(J.w, J.N, J.K, n0, threadIdx.x);
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
        xf[t] = TileOperand<KM, EXACT>::frag(lds[buf][0], wm + 16 * t, kh, r, g);
        wf[t] = TileOperand<KN, EXACT>::frag(lds[buf][1], wn + 16 * t, kh, r, g);
      }
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int u = 0; u < 2; ++u) acc[t][u] = mfma(wf[t], xf[u], acc[t][u]);
    }
  };
  u32x4_t x[AHEAD][2], w[AHEAD][2];
#pragma unroll
  for (int j = 0; j < AHEAD; ++j) { X.load(x[j], s0 + j); W.load(w[j], s0 + j); }
  int s = s0;
  // no branches in the loop: the waits for memory then name exactly the loads that a step needs
  for (; s + AHEAD <= s1; s += AHEAD) {
#pragma unroll
    for (int j = 0; j < AHEAD; ++j) {
      // a buffer is written after the barrier that follows its last readers' step
      X.store(x[j], s + j, lds[j & 1][0]); W.store(w[j], s + j, lds[j & 1][1]);
      X.load(x[j], s + j + AHEAD); W.load(w[j], s + j + AHEAD);
      __syncthreads();
      compute(j & 1);
    }
  }
#pragma unroll
  for (int j = 0; j < AHEAD - 1; ++j) {
    if (s + j < s1) {
      X.store(x[j], s + j, lds[j & 1][0]); W.store(w[j], s + j, lds[j & 1][1]);
      __syncthreads();
      compute(j & 1);
    }
  }
  typedef TileOut<TG, TG> Out;
  uint16_t* const out = &lds[0][0][0][0];
  __syncthreads();                               // every wave has read the last step
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int u = 0; u < 2; ++u) Out::put(A, J, out, n0, m0, wn + 16 * t + 4 * g, wm + 16 * u + r, acc[t][u]);
  __syncthreads();
  Out::write<256>(A, J, out, n0, m0);
}

// job and tile of a workgroup: along the longer side of the tile grid eight tiles at a time, one per XCD; all tiles across from
// each on the same XCD
__device__ __forceinline__ bool tile_of(const GemmArgs& A, int tm, int tn, int& ji, int& n0, int& m0) {
  ji = job_of(A, blockIdx.x);
  const int M = A.job[ji].M, N = A.job[ji].N;
  const int mt = (M + tm - 1) / tm, nt = (N + tn - 1) / tn, local = (int)blockIdx.x - A.tile0[ji];
  const int across = mt < nt ? mt : nt;
  const int p = local / (8 * across) * 8 + local % 8, q = local % (8 * across) / 8;
  n0 = (mt < nt ? p : q) * tn;
  m0 = (mt < nt ? q : p) * tm;
  return n0 < N && m0 < M;
}
// workgroups of a job: the longer side comes in eights, what is beyond it returns at once
int tiles_of(const GemmJob& J, int tm, int tn) {
  const int mt = (J.M + tm - 1) / tm, nt = (J.N + tn - 1) / tn;
  return ((mt < nt ? nt : mt) + 7) / 8 * 8 * (mt < nt ? mt : nt);
}
// those of them that work
int64_t real_tiles(const GemmJob& J, int tm, int tn) { return (int64_t)((J.M + tm - 1) / tm) * ((J.N + tn - 1) / tn); }

// Tiles of 64 to 256 rows and 64 or 128 columns with the operands requested straight into LDS, BUFS - 1 steps ahead: no registers are held by what
// is in flight.  Any K (launch_gemm: from 256 on, multiples of the step, or beside a product of 1024): the last step of one that is no
// multiple is masked where it is read.  A wave's request fills 1 KiB as it lies, eight rows of 128 bytes or, of a 128-wide k-major
// operand, four of 256, so rows cannot be padded: 16-byte piece p of row q lies at p ^ swizzle(q) instead (no bank conflicts counted in
// the loop).  Weights that no cache holds, 64 x 64 tiles against those through registers: 64 rows of 2048 channels into 8192 columns 19.0 -> 15.3 us, K = 8192 into 2048 unsplit 57.9 -> 37.8;
// 128 rows 19.3 -> 15.4; r, k, v and the low-rank inputs at 128 rows 20.5 -> 16.6; 256 rows into 8192 columns 23.5 -> 22.8 with
// 64-row tiles, 19.9 with 128, 19.2 with eight waves.  Bound by a step's way through LDS (see launch_gemm): in a step of 256 users (128 x 64, 17.8 us for 43.7 MB
// read) the waves wait for half of their time, for arriving operands and each other, an LDS read is why in 1 %, and the matrix units work
// a fifth of it (profiles/rwkv7_model_bf16.md); five and seven steps in flight took as long, and so did a first step that differs from tile
// to tile.
constexpr int stream_step(int tm, int tn) { return (tm + tn) * TG; }     // bf16 values of a step in LDS: TM rows of x, TN of w
typedef __attribute__((address_space(3))) uint16_t* lds_u16_ptr;

// 16 bytes per lane to 1 KiB of LDS at `lds` (a wave-uniform address).  In assembly because the compiler waits for every request
// under way before any LDS read; it has no result registers, the waits are the reader's.
__device__ __forceinline__ void request_lds(u32x4_t rs, int voff, int soff, uint32_t lds) {
  asm volatile("s_nop 0\n\tbuffer_load_dwordx4 %0, %1, %2 offen lds" ::"v"(voff), "s"(rs), "s"(soff), "{m0}"(lds) : "memory");
}

// ROWS (64, 128 or 256) rows of m or n by 64 of k; with TR the operand lies k-major and so does its piece of LDS.  The last step of a K
// that is no multiple of 64 asks for the last k again where there are no more; what it gives is masked (`keep`).
template <bool TR, int ROWS, int WAVES>
struct StreamOperand {
  static constexpr int PIECES = ROWS / 8 / WAVES;                           // requests of a wave per step
  static constexpr int PER_ROW = TR ? ROWS / 8 : TG / 8;             // 16-byte pieces of an LDS row
  static constexpr int LINES = 64 / PER_ROW;                         // LDS rows that a request fills
  u32x4_t rs;
  int voff[PIECES], stride, last, at, lane, R, over;
  static __device__ __forceinline__ int swizzle(int q) {
    return TR ? 2 * ((q ^ (q >> 3)) & 3) : (q & 3) | ((q >> 1) & 4);
  }
  __device__ __forceinline__ StreamOperand(const void* base, int R_, int K, int r0, int wave, int lane_) : lane(lane_), R(R_) {
    last = (K - 1) / TG;
    over = (last + 1) * TG - K;                                      // of the last step
    stride = TR ? TG * R * 2 : TG * 2;
    const uint64_t first = reinterpret_cast<uint64_t>(static_cast<const bf16_t*>(base) + (TR ? (int64_t)r0 : (int64_t)r0 * K));
    rs = u32x4_t{(uint32_t)first, (uint32_t)(first >> 32) & 0xffffu, 0x7fffffffu, 0x00020000u};      // as make_rsrc
    at = wave * PIECES * 1024;
#pragma unroll
    for (int i = 0; i < PIECES; ++i) {
      const int q = line(i), c = column(i);
      voff[i] = TR ? (q * R + (r0 + c < R ? c : R - 8 - r0)) * 2 : ((r0 + q < R ? q : R - 1 - r0) * K + c) * 2;
    }
  }
  __device__ __forceinline__ int line(int i) const { return LINES * (at / 1024 + i) + lane / PER_ROW; }
  __device__ __forceinline__ int column(int i) const { return 8 * ((lane % PER_ROW) ^ swizzle(line(i))); }
  __device__ __forceinline__ void request(int s, uint16_t* lds) const {
    const int soff = (s < last ? s : last) * stride;
    const uint32_t to = (uint32_t)(uintptr_t)(lds_u16_ptr)(lds) + at;
    if (s >= last && over != 0) {
#pragma unroll
      for (int i = 0; i < PIECES; ++i) {
        const int k = TR ? line(i) : column(i), past = k - (TG - over - (TR ? 1 : 8));      // beyond the last that there is
        request_lds(rs, voff[i] - (past > 0 ? past * (TR ? 2 * R : 2) : 0), soff, to + 1024 * i);
      }
      return;
    }
#pragma unroll
    for (int i = 0; i < PIECES; ++i) request_lds(rs, voff[i], soff, to + 1024 * i);
  }
  // eight of k (32 kh + 8g ..) of row n; with TR the lane's own row comes out of the transposing read, n is that of its request
  static __device__ __forceinline__ u32x4_t frag(const uint16_t* lds, int n, int kh, int r, int g) {
    if (TR) {
      const int k = 32 * kh + 8 * g + (r >> 2);
      const uint2 lo = lds_tr4(lds + k * ROWS + 8 * ((n >> 3) ^ swizzle(k)) + (n & 7));
      const uint2 hi = lds_tr4(lds + (k + 4) * ROWS + 8 * ((n >> 3) ^ swizzle(k + 4)) + (n & 7));
      return u32x4_t{lo.x, lo.y, hi.x, hi.y};
    }
    return *reinterpret_cast<const u32x4_t*>(lds + n * TG + 8 * ((4 * kh + g) ^ swizzle(n)));
  }
};
// v with its eight k (from k0 on) cleared from `end` on
__device__ __forceinline__ u32x4_t keep_k(u32x4_t v, int k0, int end) {
#pragma unroll
  for (int c = 0; c < 4; ++c) v[c] = k0 + 2 * c + 1 < end ? v[c] : k0 + 2 * c < end ? v[c] & 0xffffu : 0u;
  return v;
}

// TM x TN tiles, WM x WN waves
template <int TM, int TN, int BUFS, int WM, int WN, bool KM, bool KN>
__device__ __forceinline__ void stream_gemm_body(const GemmArgs& A, const GemmJob& J, int n0, int m0, uint16_t* lds) {
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
  constexpr int WAVES = WM * WN, MT = TM / WM / 16, NT = TN / WN / 16, STEP = stream_step(TM, TN), IN_STEP = (TM + TN) / 8 / WAVES;
  const int all = (J.K + TG - 1) / TG;
  const int s0 = all * (int)blockIdx.y / (int)gridDim.y, s1 = all * ((int)blockIdx.y + 1) / (int)gridDim.y;
  typedef StreamOperand<KM, TM, WAVES> OpX;
  typedef StreamOperand<KN, TN, WAVES> OpW;
  const OpX X(J.x, J.M, J.K, m0, wave, lane);
  const OpW W(J.w, J.N, J.K, n0, wave, lane);
  f32x4_t acc[NT][MT];
#pragma unroll
  for (int i = 0; i < NT * MT; ++i) acc[i / MT][i % MT] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  const int wn = TN / WN * (wave % WN), wm = TM / WM * (wave / WN);
  auto request = [&](int s, int buf) {
    X.request(s, lds + buf * STEP);
    W.request(s, lds + buf * STEP + TM * TG);
  };
#pragma unroll
  for (int j = 0; j < BUFS - 1; ++j) request(s0 + j, j);
  // `end`: k of this step that there are (64 but for the last step of a K that is no multiple of it)
  auto compute = [&](int buf, bool whole, int end) {
    const uint16_t* const xs = lds + buf * STEP;
    const uint16_t* const ws = xs + TM * TG;
#pragma unroll
    for (int kh = 0; kh < 2; ++kh) {
      u32x4_t wf[NT], xf[MT];
#pragma unroll
      for (int t = 0; t < NT; ++t) wf[t] = OpW::frag(ws, wn + 16 * t + (KN ? 4 * (r & 3) : r), kh, r, g);
#pragma unroll
      for (int u = 0; u < MT; ++u) xf[u] = OpX::frag(xs, wm + 16 * u + (KM ? 4 * (r & 3) : r), kh, r, g);
      if (!whole) {
#pragma unroll
        for (int t = 0; t < NT; ++t) wf[t] = keep_k(wf[t], 32 * kh + 8 * g, end);
#pragma unroll
        for (int u = 0; u < MT; ++u) xf[u] = keep_k(xf[u], 32 * kh + 8 * g, end);
      }
#pragma unroll
      for (int u = 0; u < MT; ++u)
#pragma unroll
        for (int t = 0; t < NT; ++t) acc[t][u] = mfma(wf[t], xf[u], acc[t][u]);
    }
  };
  auto arrive = [&](int s, int buf) {
    // this wave's part of step s has arrived; after the barrier all parts, and nobody reads the buffer of step s - 1 any more
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(IN_STEP * (BUFS - 2)) : "memory");
    request(s + BUFS - 1, (buf + BUFS - 1) % BUFS);
  };
  const int tail = s1 == all && J.K % TG != 0 ? 1 : 0, sw = s1 - tail;          // whole steps
  int s = s0;
  for (; s + BUFS <= sw; s += BUFS)
#pragma unroll
    for (int j = 0; j < BUFS; ++j) {
      arrive(s + j, j);
      compute(j, true, TG);
    }
  int buf = 0;
#pragma unroll
  for (int j = 0; j < BUFS - 1; ++j)
    if (s + j < sw) {
      arrive(s + j, j);
      compute(j, true, TG);
      buf = j + 1;
    }
  if (tail) {
    arrive(s1 - 1, buf);
    compute(buf, false, J.K % TG);
  }
  // the requests beyond the last step write to LDS as well: none may be under way when the tile goes there, nor may a wave read the last
  // step
  typedef TileOut<TM, TN> Out;
  static_assert(Out::BYTES <= (size_t)BUFS * STEP * 2, "the tile fits in the buffers");
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int u = 0; u < MT; ++u) Out::put(A, J, lds, n0, m0, wn + 16 * t + 4 * g, wm + 16 * u + r, acc[t][u]);
  __syncthreads();
  Out::template write<64 * WM * WN>(A, J, lds, n0, m0);
}

template <int TM, int TN, int BUFS, int WM, int WN>
__global__ __launch_bounds__(64 * WM * WN) void stream_gemm_kernel(GemmArgs A) {
  extern __shared__ __align__(1024) uint16_t stream_lds[];
  int ji, n0, m0;
  if (!tile_of(A, TM, TN, ji, n0, m0)) return;
  const GemmJob J = A.job[ji];
  if constexpr (TM > 2 * TG) {                   // launch_gemm gives these tiles no transposed operands
    stream_gemm_body<TM, TN, BUFS, WM, WN, false, false>(A, J, n0, m0, stream_lds);
  } else {
    switch ((J.km ? 2 : 0) + (J.kn ? 1 : 0)) {
      case 0: stream_gemm_body<TM, TN, BUFS, WM, WN, false, false>(A, J, n0, m0, stream_lds); break;
      case 1: stream_gemm_body<TM, TN, BUFS, WM, WN, false, true>(A, J, n0, m0, stream_lds); break;
      case 2: stream_gemm_body<TM, TN, BUFS, WM, WN, true, false>(A, J, n0, m0, stream_lds); break;
      default: stream_gemm_body<TM, TN, BUFS, WM, WN, true, true>(A, J, n0, m0, stream_lds); break;
    }
  }
}
template <int TM, int TN, int BUFS, int WM, int WN>
hipError_t launch_stream(const GemmArgs& A, int tiles, int split, hipStream_t stream) {
  static LdsAttrOnce attr;
  constexpr size_t bytes = (size_t)BUFS * stream_step(TM, TN) * 2;
  const auto kernel = stream_gemm_kernel<TM, TN, BUFS, WM, WN>;
  hipError_t e = allow_dynamic_lds(attr, reinterpret_cast<const void*>(kernel), bytes);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(kernel, dim3(tiles, split), dim3(64 * WM * WN), bytes, stream, A);
  return hipGetLastError();
}

__global__ __launch_bounds__(256) void tile_gemm_kernel(GemmArgs A) {
  __shared__ __align__(16) TileLds lds;
  int ji, n0, m0;
  if (!tile_of(A, TG, TG, ji, n0, m0)) return;
  const GemmJob J = A.job[ji];
  switch ((J.km ? 4 : 0) + (J.kn ? 2 : 0) + (J.K % TG == 0 ? 1 : 0)) {
    case 0: tile_gemm_body<false, false, false>(A, J, n0, m0, lds); break;
    case 1: tile_gemm_body<false, false, true>(A, J, n0, m0, lds); break;
    case 2: tile_gemm_body<false, true, false>(A, J, n0, m0, lds); break;
    case 3: tile_gemm_body<false, true, true>(A, J, n0, m0, lds); break;
    case 4: tile_gemm_body<true, false, false>(A, J, n0, m0, lds); break;
    case 5: tile_gemm_body<true, false, true>(A, J, n0, m0, lds); break;
    case 6: tile_gemm_body<true, true, false>(A, J, n0, m0, lds); break;
    default: tile_gemm_body<true, true, true>(A, J, n0, m0, lds); break;
  }
}

// The second low-rank products of 64 tokens and one head, and everything element-wise behind them.  In separate launches the products'
// results made a trip through memory each way: 4084 tokens, 32 heads (inner sizes 96, 96, 64, 288) 44 + 36 us, here 68; 2048 tokens, 12
// heads 11.3 + 9.6, here 16.3.  The vector units take 27 of the 68 (the element-wise part), the barrier of each of ten steps most of the
// rest; four waves of twice the tile took as long.  The factors' steps of 64 of k follow each other without a stop, two in flight; their
// products wait in LDS, rounded, for the last one.  Heads run fastest through the grid: an XCD reads the rows of hidden values that its
// eight neighbours read as well, and of the weights only its own heads'.
constexpr int LORA_THREADS = 512;
template <bool VMIX>
__global__ __launch_bounds__(LORA_THREADS) void lora_pre_kernel(LoraPreArgs A) {
  constexpr int NF = VMIX ? 4 : 3;
  __shared__ __align__(16) TileLds lds;
  __shared__ __align__(16) uint16_t low[NF][TG][TG_RS];
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, r = lane & 15, g = lane >> 4;
  const int H = (int)A.P.H, C = 64 * H, h = (int)blockIdx.x % H, m0 = (int)blockIdx.x / H * TG, M = (int)A.P.rows;
  const int row = tid >> 3, col = 8 * (tid & 7);                 // of the tiles: a token or a k, and eight k or channels
  const bool live = m0 + row < M;
  const int mc = live ? m0 + row : M - 1;
  const size_t el = (size_t)mc * C + 64 * h + col;
  int first[NF + 1];                              // a factor's first step
  first[0] = 0;
#pragma unroll
  for (int f = 0; f < NF; ++f) first[f + 1] = first[f] + (A.d[f] + TG - 1) / TG;
  const int all = first[NF];
  auto factor = [&](int s) {
    int f = 0;
#pragma unroll
    for (int i = 1; i < NF; ++i) f = s >= first[i] ? i : f;
    return f;
  };
  auto load = [&](u32x4_t& x, u32x4_t& w, int s_) {
    const int s = s_ < all ? s_ : all - 1, f = factor(s);
    int at = first[0], d = A.d[0];
    const bf16_t *hid = static_cast<const bf16_t*>(A.hid[0]), *w2 = static_cast<const bf16_t*>(A.w2[0]);
#pragma unroll
    for (int i = 1; i < NF; ++i) {
      at = f == i ? first[i] : at;
      d = f == i ? A.d[i] : d;
      hid = f == i ? static_cast<const bf16_t*>(A.hid[i]) : hid;
      w2 = f == i ? static_cast<const bf16_t*>(A.w2[i]) : w2;
    }
    const int k0 = (s - at) * TG;
    const int kx = k0 + col, kw = k0 + row;
    auto at16 = [](const bf16_t* p, uint32_t el) { return *reinterpret_cast<const u32x4_t*>(reinterpret_cast<const char*>(p) + 2u * el); };
    if (k0 + TG <= d) {
      x = at16(hid, (uint32_t)mc * (uint32_t)d + (uint32_t)kx);
      w = at16(w2, (uint32_t)kw * (uint32_t)C + (uint32_t)(64 * h + col));
    } else {
      x = at16(hid, (uint32_t)mc * (uint32_t)d + (uint32_t)(kx < d ? kx : d - 8));
      w = at16(w2, (uint32_t)(kw < d ? kw : d - 1) * (uint32_t)C + (uint32_t)(64 * h + col));
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        x[c] = kx < d ? x[c] : 0u;
        w[c] = kw < d ? w[c] : 0u;
      }
    }
  };
  u32x4_t x[2], w[2], kq, vq, vfq;
  load(x[0], w[0], 0);
  load(x[1], w[1], 1);
  kq = *reinterpret_cast<const u32x4_t*>(static_cast<const bf16_t*>(A.P.k) + el);
  if (VMIX) {
    vq = *reinterpret_cast<const u32x4_t*>(static_cast<const bf16_t*>(A.P.v) + el);
    vfq = *reinterpret_cast<const u32x4_t*>(static_cast<const bf16_t*>(A.P.vf) + el);
  }
  f32x4_t acc[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
  const int wn = 16 * (wave & 3), wm = 32 * (wave >> 2);
  auto step = [&](int s, int buf) {
    *reinterpret_cast<u32x4_t*>(&lds[buf][0][row][col]) = x[buf];
    *reinterpret_cast<u32x4_t*>(&lds[buf][1][row][col]) = w[buf];
    load(x[buf], w[buf], s + 2);
    __syncthreads();
#pragma unroll
    for (int kh = 0; kh < 2; ++kh) {
      const u32x4_t wf = TileOperand<true, true>::frag(lds[buf][1], wn, kh, r, g);
#pragma unroll
      for (int u = 0; u < 2; ++u) acc[u] = mfma(wf, TileOperand<false, true>::frag(lds[buf][0], wm + 16 * u, kh, r, g), acc[u]);
    }
    const int f = factor(s);
    if (s + 1 == all || factor(s + 1) != f) {
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        *reinterpret_cast<uint2*>(&low[f][wm + 16 * u + r][wn + 4 * g]) = make_uint2(chunk::pack_rn(acc[u][0], acc[u][1]), chunk::pack_rn(acc[u][2], acc[u][3]));
        acc[u] = f32x4_t{0.f, 0.f, 0.f, 0.f};
      }
    }
  };
  int s = 0;
  for (; s + 2 <= all; s += 2) { step(s, 0); step(s + 1, 1); }
  if (s < all) step(s, 0);
  __syncthreads();
  u32x4_t q[4];
#pragma unroll
  for (int f = 0; f < 4; ++f) {
    q[f] = f < NF ? *reinterpret_cast<const u32x4_t*>(&low[f < NF ? f : 0][row][col]) : u32x4_t{0u, 0u, 0u, 0u};
    if (f < NF && live && A.out[f] != nullptr) *reinterpret_cast<u32x4_t*>(static_cast<bf16_t*>(A.out[f]) + el) = q[f];
  }
  float xw[8], k[8], xa[8], v[8], vf[8], xv[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    xw[e] = half_of(q[0], e); xa[e] = half_of(q[1], e); xv[e] = half_of(q[3], e);
    k[e] = half_of(kq, e);
    v[e] = VMIX ? half_of(vq, e) : 0.f;
    vf[e] = VMIX ? half_of(vfq, e) : 0.f;
  }
  pre_unit<bf16_t, VMIX>(A.P, el, (size_t)64 * h + col, live, xw, k, xa, v, vf, xv);
}

}  // namespace

// Parts that a product's K is split into: enough tiles for about two workgroups per CU, at least 256 of k each (few rows: three
// steps of a wave.  One user's value projection of 3072 into 768 had 48 workgroups)
int gemm_split(int M, int64_t K, int64_t N) {
  const bool skinny = M < GEMM_TILE_ROWS;
  const int64_t tiles = skinny ? (N + 15) / 16 : (M + TG - 1) / TG * ((N + TG - 1) / TG);
  const int64_t want = 512 / tiles, most = skinny ? K / (32 * GEMM_WAVES * 3) : K / 256;
  int64_t n = want < most ? want : most;
  n = n < 1 ? 1 : n > GEMM_MAX_SPLIT ? GEMM_MAX_SPLIT : n;
  while (skinny && (n & (n - 1)) != 0) n &= n - 1;               // a power of two: a wave finds its part by a shift
  return (int)n;
}

// Up to 32 rows the streaming kernel (K a multiple of 32, N of 16, no aux): its operand loads touch a cache line per lane,
// 64 cycles a KiB, which a stream of weights can afford but repeated reads of x cannot (8192 columns of 2048: 14 us at 32
// rows, 16 at 33, 21 at 64; tiled 15 us up to 128 rows, 22 at 256).
// From 33 rows tiles, straight to LDS (through registers where an operand of a narrow K is no multiple of a step: the second low-rank
// factors, which the other kernel would mostly mask).  Which: a step takes in proportion to what passes through a CU's LDS (its operands
// are written at 64 bytes a cycle and read twice at 128: 4 (TM + TN) cycles; measured 0.29 us for 64 x 64, 0.40 for 128 x 64, 0.54 for 128
// x 128, 0.79 for 256 x 128 with one workgroup a CU; by the counters the waves wait for what arrives, not for what they read), so the tile
// that takes the fewest steps a CU times TM + TN.  Products of one K run in rounds over the CUs; of several, the longest or the mean counts.
// Eight waves from 128 rows on: one reads LDS while the other of its SIMD multiplies.  us with four waves and with eight, weights that no
// cache holds: three 768x768 of 2048 rows in 128 x 128 tiles 14.4 / 13.3, one in 128 x 64 7.7 / 6.8, its K = 3072 22.2 / 21.0; the same in
// a training step, 768 into 3072 forward 128 x 128 24.9 / 22.2 and, without transposed operands, 256 x 128 20.6; its two backward products
// in one launch 128 x 64 47.4 / 41.3, 128 x 128 43.6 / 37.8, 64 x 64 52.8; K = 3072 backward 128 x 64 33.4 / 34.5, 128 x 128 with three
// buffers 31.3; six of 768 x 768 and the low-rank ones 41.2 / 38.2 and 37.8; r, k, v and the low-rank inputs 26.6 / 25.0, 24.9 / 22.8,
// 256 x 128 26.1 (transposed ones among them).  4084 rows, three 2048 x 2048: 128 x 128 102 / 99, 256 x 128 95.  Large tiles of several K
// leave less to balance: they have to be a tenth better by that count.  Products split over K keep four waves (256 rows of 8192 columns
// 14.7 / 15.0).  512 rows: 2048 into 8192 64 x 64 36, 128 x 64 29, 128 x 128 25, 8192 into 2048 37 / 52 / 75.
// Empty workgroups of the tiles of 128 columns do not count: with
// them, and as edges, 24 layers of 2048 channels fell back to 128 x 64 at 2200 rows, 12.9 ms forward, now 12.0, at 2600 14.6, now 12.8, at
// 3200 18.7, now 14.8.  Those of the smaller tiles do: 12 layers of 768 channels were 1 % slower without them (700 and 1500 rows).  More
// requests in flight change nothing: four steps took as long as three (one workgroup per CU), and so did two groups of waves half a step apart
// and tiles handed out in blocks of several rows and columns an XCD.
constexpr int CUS = 256, WIDE_TILES = 192;
hipError_t launch_gemm(GemmArgs A, int split, hipStream_t stream) {
  bool skinny = true, stream_k = true, same_k = true, plain = true;
  int M = 0, longest = 0, tiles = 0;
  // the longest first: what is left at the end is short
  for (int i = 1; i < A.n_jobs; ++i)
    for (int j = i; j > 0 && A.job[j].K > A.job[j - 1].K; --j) { const GemmJob t = A.job[j]; A.job[j] = A.job[j - 1]; A.job[j - 1] = t; }
  for (int i = 0; i < A.n_jobs; ++i) {
    const GemmJob& J = A.job[i];
    M = J.M > M ? J.M : M;
    longest = J.K > longest ? J.K : longest;
    same_k = same_k && J.K == A.job[0].K;
    plain = plain && !J.km && !J.kn;
    stream_k = stream_k && (J.K % TG == 0 || J.K >= 4 * TG);
    skinny = skinny && J.M < GEMM_TILE_ROWS && !J.km && J.aux == nullptr && J.raw == nullptr && J.K % 32 == 0 && J.N % 16 == 0;
  }
  stream_k = stream_k || longest >= 16 * TG;       // beside a long one the short ones' masked steps do not count
  auto place = [&](int tm, int tn) { tiles = place_jobs(A, [&](const GemmJob& J) { return skinny ? J.N / 16 : tiles_of(J, tm, tn); }); };
  const dim3 block(64 * GEMM_WAVES);
  if (!skinny && stream_k && (split > 1 || A.part != nullptr)) {
    place(2 * TG, TG);
    if (M > TG && tiles * split >= WIDE_TILES && tiles * split <= CUS) return launch_stream<2 * TG, TG, 4, 2, 2>(A, tiles, split, stream);
    place(TG, TG);
    return launch_stream<TG, TG, 4, 2, 2>(A, tiles, split, stream);
  }
  if (!skinny && stream_k) {
    auto cost = [&](int tm, int tn) {
      int64_t n = 0, steps = 0, area = 0;
      for (int i = 0; i < A.n_jobs; ++i) {
        const int64_t t = tn > TG ? real_tiles(A.job[i], tm, tn) : tiles_of(A.job[i], tm, tn);
        n += t;
        area += (int64_t)A.job[i].M * A.job[i].N;
        steps += t * ((A.job[i].K + TG - 1) / TG);
      }
      const int64_t one = (longest + TG - 1) / TG, mean = (steps + CUS - 1) / CUS;
      if (tn > TG && 100 * area < 85 * n * tm * tn) return INT64_MAX;         // mostly edges (the low-rank inputs alone: 38 us and 34)
      return (same_k ? (n + CUS - 1) / CUS * one : mean > one ? mean : one) * (tm + tn);
    };
    const int64_t small = cost(TG, TG), wide = M > TG ? cost(2 * TG, TG) : small, large = M > TG ? cost(2 * TG, 2 * TG) : wide;
    const int64_t huge = M > 2 * TG && same_k && plain ? cost(4 * TG, 2 * TG) : large;
    if (huge < large && huge < wide && huge < small) {
      place(4 * TG, 2 * TG);
      return launch_stream<4 * TG, 2 * TG, 3, 4, 2>(A, tiles, split, stream);
    }
    if (large < (same_k ? wide : wide - wide / 11) && large < small) {
      place(2 * TG, 2 * TG);
      return tiles > CUS ? launch_stream<2 * TG, 2 * TG, 2, 2, 4>(A, tiles, split, stream) : launch_stream<2 * TG, 2 * TG, 3, 2, 4>(A, tiles, split, stream);
    }
    if (wide < small) {
      place(2 * TG, TG);
      return tiles > CUS ? launch_stream<2 * TG, TG, 3, 4, 2>(A, tiles, split, stream) : launch_stream<2 * TG, TG, 4, 4, 2>(A, tiles, split, stream);
    }
    place(TG, TG);
    return launch_stream<TG, TG, 4, 2, 2>(A, tiles, split, stream);
  }
  place(TG, TG);
  if (!skinny) hipLaunchKernelGGL(tile_gemm_kernel, dim3(tiles, split), dim3(256), 0, stream, A);
  else {
    while (2 << A.log_split <= split) ++A.log_split;             // gemm_split: a power of two
    auto kernel = A.n_jobs == 1 ? (M <= 16 ? skinny_gemm_kernel<1, true> : skinny_gemm_kernel<2, true>)
                                : (M <= 16 ? skinny_gemm_kernel<1, false> : skinny_gemm_kernel<2, false>);
    hipLaunchKernelGGL(kernel, dim3(tiles, split), block, 0, stream, A);
  }
  return hipGetLastError();
}

template <int G, int TURNS, int NT>
static hipError_t launch_head(const LnMixArgs& N, GemmArgs& A, hipStream_t stream) {
  const int tiles = place_jobs(A, [](const GemmJob& J) { return J.N / (16 * NT); });
  hipLaunchKernelGGL((head_gemm_kernel<G, TURNS, NT>), dim3(tiles), dim3(64 * GEMM_WAVES), 0, stream, N, A);
  return hipGetLastError();
}
// 32 columns a workgroup from 1025 channels on: with 16 there are two turns of workgroups, each with its norm (24 layers of 2048
// channels, one user, before requests were bundled: 1536 us with 16, 1360 with 32, 1439 with norms of their own; 1213 now)
hipError_t launch_head_gemm(const LnMixArgs& N, GemmArgs A, hipStream_t stream) {
  const bool one = A.job[0].M == 1;
  if (N.C <= 1024) return one ? launch_head<1, 1, 1>(N, A, stream) : launch_head<2, 1, 1>(N, A, stream);
  if (N.C <= 2048) return one ? launch_head<1, 2, 2>(N, A, stream) : launch_head<2, 2, 2>(N, A, stream);
  return one ? launch_head<1, 4, 2>(N, A, stream) : launch_head<2, 4, 2>(N, A, stream);
}

hipError_t launch_rwkv7_lora_pre(const LoraPreArgs& A, hipStream_t stream) {
  const dim3 grid((unsigned)((A.P.rows + TG - 1) / TG * A.P.H)), block(LORA_THREADS);
  if (A.P.vf != nullptr) hipLaunchKernelGGL(lora_pre_kernel<true>, grid, block, 0, stream, A);
  else hipLaunchKernelGGL(lora_pre_kernel<false>, grid, block, 0, stream, A);
  return hipGetLastError();
}

}  // namespace hiprwkv
