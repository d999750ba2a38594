// Everything element-wise between RWKV-7's projections and the WKV op in one pass (reference:
// /root/reference/src/jaxrwkv/rwkv7.py:237, :241-242, :244, :248-252, :257):
//     w  = -softplus(-(w0 + xw)) - 0.5              xw, xv, xa: the low-rank terms of decay, value residual and gate
//     v' = v + (v_first - v) sigmoid(v0 + xv)       layers after the first; the first layer has v' = v
//     a  = sigmoid(a0 + xa)
//     kk = normalize_head(k k_k) ;  k' = k (1 + (a - 1) k_a) ;  a_i = -kk ;  b_i = kk a
// Memory bound: six token tensors in, five out (the separate kernels move seventeen, and `a` makes a trip through memory
// in between).  Measured in bf16 at 4084 tokens and 32 heads: 37 us, 5.0 TB/s, against 49 us for the four kernels.  Eight lanes per (token, head), eight channels per lane: one 16-byte access per lane and array in bf16, the
// norm's sum over a head is three DPP steps.  fp32 arithmetic, one rounding per output; `a` is rounded to the I/O dtype
// where the reference stores it.
//
// Backward: from the cotangents of w, k', v', a_i, b_i to those of xw, k, v, v_first, xv, xa and of the five parameters.
// A workgroup works on one head and steps over the tokens with the parameter sums in registers; they meet in LDS and leave
// as one row per workgroup, which launch_reduce_parts adds up.
#include "common.h"
#include "rwkv7_pre.h"
#include "wkv_args.h"

namespace hiprwkv {

namespace {

constexpr int PRE_THREADS = 256;            // 32 units
constexpr int PRE_UNITS = PRE_THREADS / 8;

template <typename T, bool VMIX>
__global__ __launch_bounds__(PRE_THREADS) void rwkv7_pre_kernel(PreArgs A) {
  // units beyond the end redo the last one: whole rows stay active for the reductions
  int64_t unit = (int64_t)blockIdx.x * PRE_UNITS + (threadIdx.x >> 3);
  unit = unit < A.rows * A.H ? unit : A.rows * A.H - 1;
  const int c8 = 8 * (threadIdx.x & 7);
  const size_t el = (size_t)unit * 64 + c8, ch = (size_t)(unit % A.H) * 64 + c8;
  auto in = [&](const void* p, float (&o)[8]) { ld8(reinterpret_cast<const T*>(p) + el, o); };
  float xw[8], k[8], xa[8], v[8], vf[8], xv[8];
  in(A.xw, xw); in(A.k, k); in(A.xa, xa);
  if (VMIX) { in(A.v, v); in(A.vf, vf); in(A.xv, xv); }
  pre_unit<T, VMIX>(A, el, ch, true, xw, k, xa, v, vf, xv);
}

constexpr int BWD_THREADS = 16 * PRE_UNITS;

// Four channels a lane: with eight the requests of a token took so many registers (228) that a SIMD held two waves of the three it had been given.
// B=4 T=512 H=12, bf16: 22 us a launch when the arrays were requested as they were needed (four to five waits for memory in series), 20.4 requested
// at once by lanes of eight channels, 17.8 by lanes of four (72 MB, 4.0 TB/s).
// Workgroup b: head b % H, tokens (b / H) * PRE_UNITS + unit, stepping by PRE_UNITS * (gridDim.x / H)
template <typename T, bool VMIX>
__global__ __launch_bounds__(BWD_THREADS) void rwkv7_pre_bwd_kernel(PreArgs A) {
  constexpr int NP = VMIX ? 5 : 4;
  __shared__ float red[NP][PRE_UNITS / 4][64];
  const int64_t h = blockIdx.x % A.H, rb = blockIdx.x / A.H, nrb = gridDim.x / A.H;
  const int unit = threadIdx.x >> 4, c4 = 4 * (threadIdx.x & 15);
  Held4<T> w0, a0, kkw, kaw, v0;
  auto param = [&](const void* p, Held4<T>& x) { x.load(reinterpret_cast<const T*>(p) + h * 64 + c4); };
  param(A.w0, w0); param(A.a0, a0); param(A.k_k, kkw); param(A.k_a, kaw);
  if (VMIX) param(A.v0, v0);
  float part[NP][4];
#pragma unroll
  for (int p = 0; p < NP; ++p)
#pragma unroll
    for (int c = 0; c < 4; ++c) part[p][c] = 0.f;
  // every unit runs the same number of rounds; tokens beyond the end redo the last one without storing
  for (int64_t base = rb * PRE_UNITS; base < A.rows; base += nrb * PRE_UNITS) {
    const int64_t row = base + unit;
    const bool live = row < A.rows;
    const float lv = live ? 1.f : 0.f;
    const size_t el = (size_t)((live ? row : A.rows - 1) * A.H + h) * 64 + c4;
    auto put = [&](void* p, const float (&o)[4]) { if (live) st_n(reinterpret_cast<T*>(p) + el, o); };
    // everything is requested before anything is looked at
    Held4<T> hxw, hk, hxa, hgw, hgk, hgk2, hga, hgb, hgr, hgr2, hv, hvf, hxv, hgv, hgv2, hgvf;
    auto request = [&](const void* p, Held4<T>& h) { if (p != nullptr) h.load(reinterpret_cast<const T*>(p) + el); };
    request(A.gk, hgk); request(A.gk2, hgk2);
    if (A.dr != nullptr) { request(A.gr, hgr); request(A.gr2, hgr2); }
    if (VMIX) { request(A.v, hv); request(A.vf, hvf); request(A.xv, hxv); }
    if (VMIX || A.dv_sum != nullptr) { request(A.gv, hgv); request(A.gv2, hgv2); request(A.gvf, hgvf); }
    request(A.gw, hgw); request(A.xw, hxw); request(A.k, hk); request(A.xa, hxa); request(A.ga, hga); request(A.gb, hgb);
    w0.pin(); a0.pin(); kkw.pin(); kaw.pin();
    if (VMIX) v0.pin();
    float k[4], gk[4], gbi[4], o[4];
    auto sum = [&](const Held4<T>& x, const Held4<T>& y, float (&z)[4]) {
#pragma unroll
      for (int c = 0; c < 4; ++c) z[c] = round_io<T>(x[c] + y[c]);      // as their separate sum would be
    };
    auto take = [&](const Held4<T>& x, float (&z)[4]) {
#pragma unroll
      for (int c = 0; c < 4; ++c) z[c] = x[c];
    };
    if (A.gk2 != nullptr) sum(hgk, hgk2, gk);
    else take(hgk, gk);
    if (A.dr != nullptr) {
      sum(hgr, hgr2, o);
      put(A.dr, o);
    }
    if (VMIX) {
      float gv[4], o1[4], o2[4];
      if (A.gv2 != nullptr) sum(hgv, hgv2, gv);
      else take(hgv, gv);
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const float s = sigmoidf(v0[c] + hxv[c]);
        o1[c] = gv[c] * (1.f - s);
        o2[c] = gv[c] * s;
        o[c] = gv[c] * (hvf[c] - hv[c]) * s * (1.f - s);
        part[NP - 1][c] = fmaf(lv, o[c], part[NP - 1][c]);
      }
      if (A.gvf != nullptr) {
#pragma unroll
        for (int c = 0; c < 4; ++c) o2[c] += hgvf[c];
      }
      put(A.dv, o1); put(A.dvf, o2); put(A.dxv, o);
    } else if (A.dv_sum != nullptr) {
#pragma unroll
      for (int c = 0; c < 4; ++c) o[c] = hgv[c] + hgv2[c];
      if (A.gvf != nullptr) {
#pragma unroll
        for (int c = 0; c < 4; ++c) o[c] += hgvf[c];
      }
      put(A.dv_sum, o);
    }
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      o[c] = hgw[c] * (1.f - sigmoidf(w0[c] + hxw[c]));
      part[0][c] = fmaf(lv, o[c], part[0][c]);
    }
    put(A.dxw, o);
    float kk[4], ss = 0.f;
    take(hk, k);
    take(hgb, gbi);
#pragma unroll
    for (int c = 0; c < 4; ++c) { kk[c] = k[c] * kkw[c]; ss = fmaf(kk[c], kk[c], ss); }
    const float nrm = sqrtf(row_sum(ss));
    const float inv = 1.f / fmaxf(nrm, 1e-12f);
    float a[4], gkk[4], dot = 0.f;
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      a[c] = round_io<T>(sigmoidf(a0[c] + hxa[c]));
      kk[c] *= inv;
      gkk[c] = gbi[c] * a[c] - hga[c];              // a_i = -kk, b_i = kk a
      dot = fmaf(kk[c], gkk[c], dot);
    }
    dot = nrm >= 1e-12f ? row_sum(dot) : 0.f;       // below the clamp the norm is a constant
    float ok[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const float graw = (gkk[c] - kk[c] * dot) * inv;              // cotangent of k . k_k
      ok[c] = gk[c] * (1.f + (a[c] - 1.f) * kaw[c]) + graw * kkw[c];
      const float gav = gbi[c] * kk[c] + gk[c] * k[c] * kaw[c];     // cotangent of a
      o[c] = gav * a[c] * (1.f - a[c]);
      part[1][c] = fmaf(lv, o[c], part[1][c]);
      part[2][c] = fmaf(lv * graw, k[c], part[2][c]);
      part[3][c] = fmaf(lv * gk[c] * k[c], a[c] - 1.f, part[3][c]);
    }
    put(A.dk, ok); put(A.dxa, o);
  }
  // the four units of a wave by permutes, the waves through LDS
#pragma unroll
  for (int p = 0; p < NP; ++p) {
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      part[p][c] += __shfl_xor(part[p][c], 16, 64);
      part[p][c] += __shfl_xor(part[p][c], 32, 64);
    }
    if ((unit & 3) == 0) st_n(&red[p][unit >> 2][c4], part[p]);
  }
  __syncthreads();
  for (int i = threadIdx.x; i < NP * 64; i += BWD_THREADS) {
    float s = 0.f;
#pragma unroll
    for (int u = 0; u < PRE_UNITS / 4; ++u) s += red[i >> 6][u][i & 63];
    A.part[((size_t)rb * NP + (i >> 6)) * (A.H * 64) + h * 64 + (i & 63)] = s;
  }
}

}  // namespace

// workgroups per head of the backward: about four per CU, never more than there are groups of PRE_UNITS tokens
int64_t rwkv7_pre_bwd_rows(int64_t rows, int64_t H) {
  const int64_t want = (1024 + H - 1) / H, have = (rows + PRE_UNITS - 1) / PRE_UNITS;
  return want < have ? want : have;
}

hipError_t launch_rwkv7_pre(int io_f32, const PreArgs& A, hipStream_t stream) {
  const dim3 grid((unsigned)((A.rows * A.H + PRE_UNITS - 1) / PRE_UNITS)), block(PRE_THREADS);
  const bool vmix = A.vf != nullptr;
  if (io_f32) {
    if (vmix) hipLaunchKernelGGL((rwkv7_pre_kernel<float, true>), grid, block, 0, stream, A);
    else hipLaunchKernelGGL((rwkv7_pre_kernel<float, false>), grid, block, 0, stream, A);
  } else {
    if (vmix) hipLaunchKernelGGL((rwkv7_pre_kernel<bf16_t, true>), grid, block, 0, stream, A);
    else hipLaunchKernelGGL((rwkv7_pre_kernel<bf16_t, false>), grid, block, 0, stream, A);
  }
  return hipGetLastError();
}

// dparam: w0, a0, k_k, k_a and, with the value residual, v0
hipError_t launch_rwkv7_pre_bwd(int io_f32, const PreArgs& A, void* const* dparam, hipStream_t stream, ReduceJobs* later) {
  const int64_t nrb = rwkv7_pre_bwd_rows(A.rows, A.H);
  const dim3 grid((unsigned)(nrb * A.H)), block(BWD_THREADS);
  const bool vmix = A.vf != nullptr;
  if (io_f32) {
    if (vmix) hipLaunchKernelGGL((rwkv7_pre_bwd_kernel<float, true>), grid, block, 0, stream, A);
    else hipLaunchKernelGGL((rwkv7_pre_bwd_kernel<float, false>), grid, block, 0, stream, A);
  } else {
    if (vmix) hipLaunchKernelGGL((rwkv7_pre_bwd_kernel<bf16_t, true>), grid, block, 0, stream, A);
    else hipLaunchKernelGGL((rwkv7_pre_bwd_kernel<bf16_t, false>), grid, block, 0, stream, A);
  }
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  ReduceArgs R;
  R.part = A.part; R.rows = nrb; R.nk = vmix ? 5 : 4; R.C = A.H * 64;
  for (int i = 0; i < R.nk; ++i) R.out[i] = dparam[i];
  return reduce_parts(io_f32, R, later, stream);
}

}  // namespace hiprwkv
