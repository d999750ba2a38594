// What rwkv7_pre.hip and the kernel that makes the second low-rank products (rwkv7_gemm.hip) do with eight channels of one token and
// head; the eight lanes of a head lie side by side.
#pragma once
#include "common.h"
#include "wkv_args.h"

namespace hiprwkv {

namespace {

// sum over the 8 lanes of half a DPP row, delivered to all of them
__device__ __forceinline__ float oct_sum(float x) {
  x = quad_sum(x);
  x += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), 0x141, 0xf, 0xf, true));   // row_half_mirror
  return x;
}

// el: the element of the token tensors, ch: of the parameters.  All eight lanes come here; only `live` ones store.
template <typename T, bool VMIX>
__device__ __forceinline__ void pre_unit(const PreArgs& A, size_t el, size_t ch, bool live, const float (&xw)[8], const float (&k)[8],
                                         const float (&xa)[8], const float (&v)[8], const float (&vf)[8], const float (&xv)[8]) {
  auto in = [&](const void* p, float (&o)[8]) { ld8(reinterpret_cast<const T*>(p) + ch, o); };
  auto put = [&](void* p, const float (&o)[8]) { if (live) st8(reinterpret_cast<T*>(p) + el, o); };
  float p0[8], p1[8], p2[8], o[8];
  in(A.w0, p0); in(A.k_k, p1); in(A.k_a, p2);
#pragma unroll
  for (int c = 0; c < 8; ++c) o[c] = -softplusf(-(p0[c] + xw[c])) - 0.5f;
  put(A.w, o);
  if (VMIX) {
    float pv[8];
    in(A.v0, pv);
#pragma unroll
    for (int c = 0; c < 8; ++c) o[c] = fmaf(vf[c] - v[c], sigmoidf(pv[c] + xv[c]), v[c]);
    put(A.v_out, o);
  }
  in(A.a0, p0);
  float kk[8], ss = 0.f;
#pragma unroll
  for (int c = 0; c < 8; ++c) { kk[c] = k[c] * p1[c]; ss = fmaf(kk[c], kk[c], ss); }
  const float inv = 1.f / fmaxf(sqrtf(oct_sum(ss)), 1e-12f);
  float ko[8], bo[8];
#pragma unroll
  for (int c = 0; c < 8; ++c) {
    const float a = round_io<T>(sigmoidf(p0[c] + xa[c]));
    kk[c] *= inv;
    ko[c] = k[c] * (1.f + (a - 1.f) * p2[c]);
    o[c] = -kk[c];
    bo[c] = kk[c] * a;
  }
  put(A.k_out, ko); put(A.a_out, o); put(A.b_out, bo);
}

}  // namespace

}  // namespace hiprwkv
