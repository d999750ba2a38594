// WKV7 sequences in parts, shared by the chunked kernels (wkv7_fwd.hip, wkv7_bwd_a.hip and their fp32 counterparts).
//
// Two things cross the boundary between two parts of a sequence:
//   * summaries.  The state (in the reverse sweep the cotangent of the state) that leaves a part is an affine map of the one that
//     enters it, S_end = S_start M + B.  Workgroups of a first launch make M and B of every part, those of a second one fold the
//     summaries before theirs into their entering state.
//   * ends.  Sweeps B and C need nothing from other parts but the state at a boundary and its cotangent.  The cotangents are left in
//     memory by sweep A, which carries them past the boundaries, the states in fp32 by the forward (when it keeps `sa`).  The
//     bf16 forward carries its state with fp16 operands, five bits fewer than sweep B's pairs (gw came out up to 1.1 % further from
//     64 bits from there), so in bf16 workgroups beside sweep A (wkv7_ends.h) leave a record per part, EndSum, and the sweeps
//     fold those before their part.
#pragma once
#include "chunk_common.h"
#include "wkv_args.h"

namespace hiprwkv {
namespace chunk {

// eight fp16 values (11 significant bits) as bf16 hi and lo parts; the pair is exact
__device__ __forceinline__ void split8h(const uint4 raw, u32x4_t& h, u32x4_t& l) {
  typedef _Float16 h8_t __attribute__((ext_vector_type(8)));
  const h8_t x = __builtin_bit_cast(h8_t, raw);
  uint32_t a, b;
  split2((float)x[0], (float)x[1], a, b); h[0] = a; l[0] = b;
  split2((float)x[2], (float)x[3], a, b); h[1] = a; l[1] = b;
  split2((float)x[4], (float)x[5], a, b); h[2] = a; l[2] = b;
  split2((float)x[6], (float)x[7], a, b); h[3] = a; l[3] = b;
}

// What a workgroup does with its sequence: all of it, a part's summary, or a part.
enum { WHOLE = 0, SUMMARY = 1, PART = 2 };

// One record per (sequence, head, part) in fp32, laid out as the operands that the fold takes (rows of 256 bytes instead: 64
// cycles a KiB, 2.3 us a predecessor), and eight words (one per consumer wave of the two workgroups that make it) that are not
// zero where the summary must not be used.  Parts count in the direction of the sweep.
struct PartSum {
  f32x4_t M[4][4][64];     // [tile][jt], lane (x, g): M[key 16 tile + 4g + i][key 16 jt + x]; for the fp64 fold key 16 tile + 4i + g
  f32x4_t B[4][4][64];     // [q][tile]: consumer q's state tiles, their keys in the same order
};
constexpr float PART_MAX_GAIN = 4.f;
__device__ __forceinline__ PartSum* part_sum(const Wkv7Args& A, int64_t head, int part) {
  return reinterpret_cast<PartSum*>(A.parts) + head * (A.n_part - 1) + part;
}
__device__ __forceinline__ int* part_flags(const Wkv7Args& A, int64_t head, int part) {
  return reinterpret_cast<int*>(reinterpret_cast<PartSum*>(A.parts) + A.B * A.H * (A.n_part - 1)) +
         (head * (A.n_part - 1) + part) * 8;
}
// the first part before `part` whose summary is not usable, else `part`; a lane looks at four of its eight words
__device__ __forceinline__ int first_unusable(const Wkv7Args& A, int64_t head, int part, int lane) {
  const int4 f = lane < 2 * part ? *reinterpret_cast<const int4*>(part_flags(A, head, 0) + 4 * lane) : make_int4(0, 0, 0, 0);
  const uint64_t bad = __ballot((f.x | f.y | f.z | f.w) != 0);
  return bad != 0 ? __builtin_ctzll(bad) >> 1 : part;
}

// The state entering part `part` > 0, S <- S M + B over the summaries before it, in fp32.  The state tiles are the B operand
// of the products M^T S^T as they are (k-slot g of step i of a tile is key 16 tile + 4g + i); a predecessor costs a consumer 64
// instructions of 32 cycles and 20 KiB from the cache.
__device__ __forceinline__ void fold_parts(f32x4_t (&S)[4], int q, int lane, const Wkv7Args& A, int64_t head, int part) {
#pragma unroll
  for (int tile = 0; tile < 4; ++tile) S[tile] = part_sum(A, head, 0)->B[q][tile][lane];
  if (part < 2) return;
  // a predecessor's 20 KiB are requested while the one before it is multiplied
  f32x4_t acc[4], m[4][4];
  auto load_m = [&](int p, int tile) {
#pragma unroll
    for (int jt = 0; jt < 4; ++jt)
      m[tile][jt] = part_sum(A, head, p)->M[tile][jt][lane];
  };
#pragma unroll
  for (int jt = 0; jt < 4; ++jt) acc[jt] = part_sum(A, head, 1)->B[q][jt][lane];
#pragma unroll
  for (int tile = 0; tile < 4; ++tile) load_m(1, tile);
  for (int p = 1; p < part; ++p) {
    const int next = p + 1 < part ? p + 1 : p;
    f32x4_t b[4];
#pragma unroll
    for (int jt = 0; jt < 4; ++jt) b[jt] = part_sum(A, head, next)->B[q][jt][lane];
#pragma unroll
    for (int tile = 0; tile < 4; ++tile) {
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int jt = 0; jt < 4; ++jt) acc[jt] = __builtin_amdgcn_mfma_f32_16x16x4f32(m[tile][jt][i], S[tile][i], acc[jt], 0, 0, 0);
      load_m(next, tile);
    }
#pragma unroll
    for (int jt = 0; jt < 4; ++jt) {
      S[jt] = acc[jt];
      acc[jt] = b[jt];
    }
  }
}
// The same on the fp64 matrix instruction, for the fp32 kernels, at 64 cycles an instruction: with sums of 64 terms in fp32 the state
// at a boundary was 1.4 times as far from 64 bits as the whole sequence's (B=1 T=1024 H=2, decay exp(-exp(-2.5))).  Its register i
// holds row 4i + g of a tile where the fp32 one holds 4g + i; the summaries lie in that order, so that a lane's operands are 16 bytes
// (gathered from the fp32 order they were 80 requests of four bytes a predecessor, waited for tile by tile), and the last step turns the
// tiles back.  B=3 T=777 H=12: forward in five parts 46.5 -> 41.2 us, sweep A in seven 51.6 -> 39.8.
__device__ __forceinline__ void fold_parts_f64(f32x4_t (&S)[4], int q, int lane, const Wkv7Args& A, int64_t head, int part) {
  typedef double f64x4_t __attribute__((ext_vector_type(4)));
  const int x = lane & 15, g = lane >> 4;
  f64x4_t s[4], acc[4];
  f32x4_t m[4][4], b[4];
  auto load_b = [&](int p) {
#pragma unroll
    for (int jt = 0; jt < 4; ++jt) b[jt] = part_sum(A, head, p)->B[q][jt][lane];
  };
  auto load_m = [&](int p, int tile) {
#pragma unroll
    for (int jt = 0; jt < 4; ++jt) m[tile][jt] = part_sum(A, head, p)->M[tile][jt][lane];
  };
  auto widen = [&](f64x4_t (&o)[4]) {
#pragma unroll
    for (int jt = 0; jt < 4; ++jt)
#pragma unroll
      for (int i = 0; i < 4; ++i) o[jt][i] = (double)b[jt][i];
  };
  load_b(0);
  widen(s);
  if (part > 1) {
    load_b(1);
#pragma unroll
    for (int tile = 0; tile < 4; ++tile) load_m(1, tile);
  }
  // a predecessor's 20 KiB are requested while the one before it is multiplied
  for (int p = 1; p < part; ++p) {
    const int next = p + 1 < part ? p + 1 : p;
    widen(acc);
    load_b(next);
#pragma unroll
    for (int tile = 0; tile < 4; ++tile) {
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int jt = 0; jt < 4; ++jt) acc[jt] = __builtin_amdgcn_mfma_f64_16x16x4f64((double)m[tile][jt][i], s[tile][i], acc[jt], 0, 0, 0);
      load_m(next, tile);
    }
#pragma unroll
    for (int jt = 0; jt < 4; ++jt) s[jt] = acc[jt];
  }
#pragma unroll
  for (int tile = 0; tile < 4; ++tile)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      // row 4g + i lies in register g of lane (x, i)
      float r = 0.f;
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const float v = __shfl((float)s[tile][k], x + 16 * i, 64);
        r = g == k ? v : r;
      }
      S[tile][i] = r;
    }
}
// writes a consumer's rows of one half of a summary, in the order of the fold that reads it; not zero if it must not be used
template <bool F64>
__device__ __forceinline__ int store_summary(const f32x4_t (&S)[4], int q, int lane, PartSum& ps, bool map) {
  const int x = lane & 15, g = lane >> 4;
  const float limit = map ? PART_MAX_GAIN : 3.0e38f;
  bool bad = false;
#pragma unroll
  for (int tile = 0; tile < 4; ++tile) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      bad |= !(fabsf(S[tile][i]) <= limit);
      // key x of the tile is (x >> 2, x & 3) as (lane, register) of the fp32 instruction's operand and the other way round of the fp64 one's
      if (map) reinterpret_cast<float*>(&ps.M[q][tile][16 * (F64 ? x & 3 : x >> 2) + 4 * g + i])[F64 ? x >> 2 : x & 3] = S[tile][i];
      else if (F64) reinterpret_cast<float*>(&ps.B[q][tile][16 * i + x])[g] = S[tile][i];
    }
    if (!map && !F64) ps.B[q][tile][lane] = S[tile];
  }
  return __ballot(bad) != 0 ? 1 : 0;
}

// The matrix (64 values x 64 keys, fp32) at the boundary in front of part `part` >= 1 of the backward's parts
__device__ __forceinline__ float* end_of(float* ends, const Wkv7Args& A, int64_t head, int part) {
  return ends + (head * (A.n_end - 1) + part - 1) * 4096;
}
// consumer q's rows of it (tiles of a value-row split, as in the forward and in sweep A), bits cleared where `kept` is 0
__device__ __forceinline__ void store_end(const f32x4_t (&S)[4], int q, int lane, float* ends, const Wkv7Args& A, int64_t head, int part,
                                          uint32_t kept = 0xffffffffu) {
  float* const p = end_of(ends, A, head, part) + (16 * q + (lane & 15)) * 64 + 4 * (lane >> 4);
#pragma unroll
  for (int tile = 0; tile < 4; ++tile)
    *reinterpret_cast<u32x4_t*>(p + 16 * tile) = u32x4_t{__float_as_uint(S[tile][0]) & kept, __float_as_uint(S[tile][1]) & kept,
                                                         __float_as_uint(S[tile][2]) & kept, __float_as_uint(S[tile][3]) & kept};
}
// For a cotangent in front of chunk c: exactly zero where the chunk starts a sequence (in sweep A what is not finite comes through
// a reset as 0 times it, in sweep C it does not).  A mask and not a branch: with one, hipcc 7.2 left the first of the sixteen
// registers unset on the path without a reset.
__device__ __forceinline__ uint32_t end_kept(const Wkv7Args& A, int64_t b, int c) {
  return A.ns != nullptr && A.ns[b * A.T + (int64_t)c * CK] != 0 ? 0u : 0xffffffffu;
}
// a workgroup whose hand-shake failed: NaN at the boundaries in front of chunks c0 .. c1
__device__ __forceinline__ void poison_ends(float* ends, const Wkv7Args& A, int64_t head, int c0, int c1) {
  for (int part = 1; part < A.n_end; ++part) {
    if (part * A.end_chunks < c0 || part * A.end_chunks > c1) continue;
    float* const p = end_of(ends, A, head, part);
    for (int i = threadIdx.x; i < 4096; i += blockDim.x) p[i] = __uint_as_float(0x7fc00000u);
  }
}
// bf16: what a part does to the state.  With sa_t known (the residual) the state is linear key by key, so the map is a decay per key.
struct EndSum {
  f32x4_t S[4][4][64];     // [consumer q][value tile]: the part's own contribution, tiles of a key-column split
  float decay[64];         // per key; negative where the part holds a reset: nothing that entered is left
};
__device__ __forceinline__ EndSum* end_sum(const Wkv7Args& A, int64_t head, int part) {
  return reinterpret_cast<EndSum*>(A.ends) + head * (A.n_end - 1) + part;
}
// The state in front of part `part` >= 0, key columns 16q ..: S[vt][i] = value 16 vt + 4g + i, key 16q + n
__device__ __forceinline__ void fold_ends(f32x4_t (&S)[4], int q, int lane, const Wkv7Args& A, int64_t head, int part) {
  const size_t el = ((size_t)head * 64 + 4 * (lane >> 4)) * 64 + 16 * q + (lane & 15);
#pragma unroll
  for (int vt = 0; vt < 4; ++vt)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const size_t e = el + (size_t)(16 * vt + i) * 64;
      S[vt][i] = A.st_f32 ? static_cast<const float*>(A.s)[e] : bf16_to_f32(static_cast<const uint16_t*>(A.s)[e]);
    }
#pragma unroll 4
  for (int p = 0; p < part; ++p) {
    const EndSum* const e = end_sum(A, head, p);
    const float d = e->decay[16 * q + (lane & 15)];
#pragma unroll
    for (int vt = 0; vt < 4; ++vt) {
      const f32x4_t add = e->S[q][vt][lane];
#pragma unroll
      for (int i = 0; i < 4; ++i) S[vt][i] = d < 0.f ? add[i] : fmaf(S[vt][i], d, add[i]);
    }
  }
  // the loads are waited for here and not, as far as the compiler can tell, in the chunk loop that follows
#pragma unroll
  for (int vt = 0; vt < 4; ++vt) asm volatile("" : "+v"(S[vt]));
}
// key columns 16q .. of it (tiles of a key-column split, as in sweeps B and C): S[vt][i] = value 16 vt + 4g + i, key 16q + n
__device__ __forceinline__ void load_end_cols(f32x4_t (&S)[4], int q, int lane, const float* p) {
#pragma unroll
  for (int vt = 0; vt < 4; ++vt)
#pragma unroll
    for (int i = 0; i < 4; ++i) S[vt][i] = p[(16 * vt + 4 * (lane >> 4) + i) * 64 + 16 * q + (lane & 15)];
}

// The running sum of the decay gradient that enters a part of sweep C from the tokens after it (see wkv7_chunk_bwd_c.hip): with G
// the cotangent of the state S between the parts, sum over the values of G S, one key per lane (all four lanes of a key).
// Where the next token starts a sequence G is zero, whatever S holds.
__device__ __forceinline__ float end_carry(const f32x4_t (&G)[4], const f32x4_t (&S)[4]) {
  float p = 0.f;
#pragma unroll
  for (int vt = 0; vt < 4; ++vt)
#pragma unroll
    for (int i = 0; i < 4; ++i) p += G[vt][i] == 0.f ? 0.f : G[vt][i] * S[vt][i];
  p += __shfl_xor(p, 16, 64);
  p += __shfl_xor(p, 32, 64);
  return p;
}

}  // namespace chunk
}  // namespace hiprwkv
