// Shared device helpers for the gfx950 WKV kernels.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <type_traits>

namespace hiprwkv {

struct bf16_t { uint16_t bits; };

__device__ __forceinline__ float bf16_to_f32(uint16_t h) { return __uint_as_float(((uint32_t)h) << 16); }

// round-to-nearest-even, NaN stays NaN: the hardware conversion (v_cvt_pk_bf16_f32), one instruction
__device__ __forceinline__ uint16_t f32_to_bf16(float f) { return __builtin_bit_cast(uint16_t, (__bf16)f); }

__device__ __forceinline__ float ld_f(const float* p) { return *p; }
__device__ __forceinline__ float ld_f(const bf16_t* p) { return bf16_to_f32(p->bits); }
__device__ __forceinline__ void st_f(float* p, float x) { *p = x; }
__device__ __forceinline__ void st_f(bf16_t* p, float x) { p->bits = f32_to_bf16(x); }

// x as it is stored in bf16, or in the type T
__device__ __forceinline__ float rnd(float x) { return bf16_to_f32(f32_to_bf16(x)); }
template <typename T>
__device__ __forceinline__ float round_io(float x);
template <>
__device__ __forceinline__ float round_io<float>(float x) { return x; }
template <>
__device__ __forceinline__ float round_io<bf16_t>(float x) { return rnd(x); }

__device__ __forceinline__ float sigmoidf(float z) { return 1.f / (1.f + __expf(-z)); }
// softplus(z) = log(1 + e^z) = max(z, 0) + log(1 + e^-|z|): the argument of the logarithm lies in (1, 2], where the
// hardware logarithm is accurate to a few 1e-7 absolute (log1pf, a software routine, made the kernel of the decay three times slower)
__device__ __forceinline__ float softplusf(float z) { return fmaxf(z, 0.f) + __logf(1.f + __expf(-fabsf(z))); }

// sum over the 16 lanes of a DPP row, delivered to all of them
__device__ __forceinline__ float row_sum(float x) {
  x += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x128, 0xf, 0xf, false));   // row_ror:8
  x += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x124, 0xf, 0xf, false));   // row_ror:4
  x += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x122, 0xf, 0xf, false));   // row_ror:2
  x += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x121, 0xf, 0xf, false));   // row_ror:1
  return x;
}

// Tokens of sequence b that count: at most T.  FLAG_LENGTH_I32 (HIPRWKV_LENGTH_I32): the array is int32, negative = 0.
constexpr unsigned FLAG_LENGTH_I32 = 0x40u;
__device__ __forceinline__ int64_t seq_length(const uint32_t* length, int64_t b, int64_t T, unsigned flags) {
  if (length == nullptr) return T;
  const uint32_t L = length[b];
  return (flags & FLAG_LENGTH_I32) && (int32_t)L < 0 ? 0 : (int64_t)L;
}

// in-sequence index of the token whose xn a token-shift state keeps: x[length - 1] with the wrap-around of negative indices
__device__ __forceinline__ int64_t last_token(const int32_t* length, int64_t b, int64_t T) {
  if (length == nullptr) return T - 1;
  const int64_t t = ((int64_t)length[b] - 1) % T;
  return t < 0 ? t + T : t;
}

// 8 consecutive elements <-> 8 floats (pointer must be 16-byte aligned for bf16, 32 for fp32)
__device__ __forceinline__ void ld8(const float* p, float (&o)[8]) {
  float4 a = *reinterpret_cast<const float4*>(p);
  float4 b = *reinterpret_cast<const float4*>(p + 4);
  o[0] = a.x; o[1] = a.y; o[2] = a.z; o[3] = a.w; o[4] = b.x; o[5] = b.y; o[6] = b.z; o[7] = b.w;
}
__device__ __forceinline__ void ld8(const bf16_t* p, float (&o)[8]) {
  uint4 a = *reinterpret_cast<const uint4*>(p);
  uint32_t w[4] = {a.x, a.y, a.z, a.w};
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    o[2 * i] = __uint_as_float(w[i] << 16);
    o[2 * i + 1] = __uint_as_float(w[i] & 0xffff0000u);
  }
}
__device__ __forceinline__ void st8(float* p, const float (&o)[8]) {
  *reinterpret_cast<float4*>(p) = make_float4(o[0], o[1], o[2], o[3]);
  *reinterpret_cast<float4*>(p + 4) = make_float4(o[4], o[5], o[6], o[7]);
}
__device__ __forceinline__ void st8(bf16_t* p, const float (&o)[8]) {
  uint32_t w[4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
    w[i] = (uint32_t)f32_to_bf16(o[2 * i]) | ((uint32_t)f32_to_bf16(o[2 * i + 1]) << 16);
  *reinterpret_cast<uint4*>(p) = make_uint4(w[0], w[1], w[2], w[3]);
}

// Eight values kept as they lie in memory: in bf16 half the registers of eight floats
template <typename T>
struct Held;
template <>
struct Held<float> {
  float v[8];
  __device__ __forceinline__ void load(const float* p) { ld8(p, v); }
  __device__ __forceinline__ void pin() {}
  __device__ __forceinline__ float operator[](int c) const { return v[c]; }
};
template <>
struct Held<bf16_t> {
  uint32_t v[4];
  __device__ __forceinline__ void load(const bf16_t* p) {
    const uint4 a = *reinterpret_cast<const uint4*>(p);
    v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
  }
  // in a loop: keeps the compiler from unpacking once in front of it
  __device__ __forceinline__ void pin() { asm volatile("" : "+v"(v[0]), "+v"(v[1]), "+v"(v[2]), "+v"(v[3])); }
  __device__ __forceinline__ float operator[](int c) const {
    return __uint_as_float((c & 1) ? (v[c >> 1] & 0xffff0000u) : (v[c >> 1] << 16));
  }
};

// Four consecutive values kept as they lie in memory
template <typename T>
struct Held4;
template <>
struct Held4<float> {
  float4 v;
  __device__ __forceinline__ void load(const float* p) { v = *reinterpret_cast<const float4*>(p); }
  __device__ __forceinline__ void pin() {}
  __device__ __forceinline__ float operator[](int c) const { return c == 0 ? v.x : c == 1 ? v.y : c == 2 ? v.z : v.w; }
};
template <>
struct Held4<bf16_t> {
  uint32_t v[2];
  __device__ __forceinline__ void load(const bf16_t* p) {
    const uint2 a = *reinterpret_cast<const uint2*>(p);
    v[0] = a.x; v[1] = a.y;
  }
  __device__ __forceinline__ void pin() { asm volatile("" : "+v"(v[0]), "+v"(v[1])); }
  __device__ __forceinline__ float operator[](int c) const {
    return __uint_as_float((c & 1) ? (v[c >> 1] & 0xffff0000u) : (v[c >> 1] << 16));
  }
};
template <typename T, int E>
using HeldOf = std::conditional_t<E == 8, Held<T>, Held4<T>>;
template <typename T, int E>
__device__ __forceinline__ void ld_n(const T* p, float (&o)[E]) {
  HeldOf<T, E> h;
  h.load(p);
#pragma unroll
  for (int c = 0; c < E; ++c) o[c] = h[c];
}
template <typename T>
__device__ __forceinline__ void st_n(T* p, const float (&o)[8]) { st8(p, o); }
__device__ __forceinline__ void st_n(float* p, const float (&o)[4]) { *reinterpret_cast<float4*>(p) = make_float4(o[0], o[1], o[2], o[3]); }
__device__ __forceinline__ void st_n(bf16_t* p, const float (&o)[4]) {
  *reinterpret_cast<uint2*>(p) = make_uint2((uint32_t)f32_to_bf16(o[0]) | ((uint32_t)f32_to_bf16(o[1]) << 16),
                                            (uint32_t)f32_to_bf16(o[2]) | ((uint32_t)f32_to_bf16(o[3]) << 16));
}

// IEEE half: the forward residual sa of the bf16 paths (11 significant bits where bf16 has 8)
__device__ __forceinline__ void ld8(const _Float16* p, float (&o)[8]) {
  typedef _Float16 h8_t __attribute__((ext_vector_type(8)));
  const h8_t a = *reinterpret_cast<const h8_t*>(p);
#pragma unroll
  for (int i = 0; i < 8; ++i) o[i] = (float)a[i];
}
__device__ __forceinline__ void st8(_Float16* p, const float (&o)[8]) {
  typedef _Float16 h8_t __attribute__((ext_vector_type(8)));
  h8_t a;
#pragma unroll
  for (int i = 0; i < 8; ++i) a[i] = (_Float16)o[i];
  *reinterpret_cast<h8_t*>(p) = a;
}

// 16 consecutive elements starting at element `el` of a typed array -> 16 floats
template <typename T>
__device__ __forceinline__ void ld16(const void* base, size_t el, float (&o)[16]) {
  const T* p = reinterpret_cast<const T*>(base) + el;
  float lo[8], hi[8];
  ld8(p, lo);
  ld8(p + 8, hi);
#pragma unroll
  for (int c = 0; c < 8; ++c) { o[c] = lo[c]; o[8 + c] = hi[c]; }
}

// sum over the 4 lanes of a quad (lanes 4m..4m+3); every lane gets the total
__device__ __forceinline__ float quad_sum(float x) {
  x += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), 0xB1, 0xf, 0xf, true));  // quad_perm [1,0,3,2]
  x += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), 0x4E, 0xf, 0xf, true));  // quad_perm [2,3,0,1]
  return x;
}

}  // namespace hiprwkv
