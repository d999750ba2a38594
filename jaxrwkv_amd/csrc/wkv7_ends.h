// What each part of a sequence does to the state, for the sweeps of the WKV7 backward that start inside it (bf16 I/O, gfx950;
// reference of the recurrence: /root/reference/src/jaxrwkv/rwkv7.py:200-220).
//
// With sa_t known (the forward's residual) the state obeys a recurrence that is linear key by key,
//     S_t = S_{t-1} diag(d_t) + sa_t b_t^T + v_t k_t^T
// so a part that does not reset leaves S_in diag(decay) + S_own, S_own what it makes from zero: one EndSum per part but the last.
// The operands of a chunk are those of sweep B (wkv7_chunk_bwd_b.hip: bf16 pairs, the same decay floor), so the state at a
// boundary is as near to 64 bits as the one that sweep B would carry there.
//
// Sweep A does not need the records and B and C come after it, so they are made by workgroups of their own behind those of sweep A's
// first launch, on CUs that it leaves idle or in its last round.  As a launch of their own beside the forward they cost 5 to 19 us
// (B=1 T=256 H=12 70 us forward and backward, now 65; B=4 T=1024 H=32 271, now 255).
// Nothing of a chunk depends on another one before the sums meet, so there is no hand-shake: sweep A's twelve waves are six groups with a
// sixth of the part's chunks each, one wave per 32 keys, operands straight from memory to registers (the transposing products leave
// them as the update wants them), the next chunk requested ahead; the groups' results are joined in LDS.
#pragma once
#include "wkv7_parts.h"

namespace hiprwkv {
namespace chunk {

constexpr int END_GROUPS = 6;              // of two waves
struct EndHalf {                           // what a wave's chunks add up to: half of an EndSum
  f32x4_t S[2][4][64];
  float decay[32];
};
constexpr size_t END_LDS = 2 * END_GROUPS * sizeof(EndHalf);

// a decay behind another one; negative: nothing is left
__device__ __forceinline__ float join_decay(float first, float second) {
  // not below the smallest normal number: what is infinite stays so, as it does chunk by chunk
  return first < 0.f || second < 0.f ? -1.f : fmaxf(first * second, 1.17549435e-38f);
}

// unit: (head, part before the last); by 128 END_GROUPS threads
__device__ __forceinline__ void make_ends(const Wkv7Args& A, int64_t unit, unsigned char* smem) {
  struct Raw {
    uint4 w, k, b, v[2], sa[2];
  };
  EndHalf* const sums = reinterpret_cast<EndHalf*>(smem);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, t = lane & 15, g = lane >> 4;
  const int group = wave >> 1, hf = wave & 1;
  const int64_t head = unit / (A.n_end - 1);
  const int part = (int)(unit % (A.n_end - 1));
  const int64_t b = head / A.H, h = head % A.H;
  const int c_in = part * A.end_chunks, first = c_in + A.end_chunks * group / END_GROUPS, last = c_in + A.end_chunks * (group + 1) / END_GROUPS;
  const f32x4_t zero4 = {0.f, 0.f, 0.f, 0.f};
  auto pack4 = [](const f32x4_t d) { return make_uint2(pack_exact(d[0], d[1]), pack_exact(d[2], d[3])); };      // of a transposing product
  EndHalf& own = sums[wave];
  u32x4_t sel[2];
  make_sel(sel, lane);
  f32x4_t S[2][4];         // [key tile of the half][value tile]
  float decay[2];          // of the wave's chunks so far, keys 32 hf + 16 x2 + t
#pragma unroll
  for (int x2 = 0; x2 < 2; ++x2) {
    decay[x2] = 1.f;
#pragma unroll
    for (int vt = 0; vt < 4; ++vt) S[x2][vt] = zero4;
  }
  Raw next;
  uint32_t ns_next = 0u;
  auto request = [&](int c) {              // a part before the last is whole chunks
    ns_next = chunk_flag_prefetch(A.ns, A.T, b, (int64_t)c * CK, lane);
    const size_t el = (((size_t)b * A.T + (size_t)c * CK + t) * A.H + h) * 64 + 8 * g;
    auto ld = [&](const void* p, int half) { return *reinterpret_cast<const uint4*>(static_cast<const uint16_t*>(p) + el + 32 * half); };
    next.w = ld(A.w, hf); next.k = ld(A.k, hf); next.b = ld(A.b, hf);
#pragma unroll
    for (int i = 0; i < 2; ++i) { next.v[i] = ld(A.v, i); next.sa[i] = ld(A.sa_in, i); }
  };
  if (first < last) request(first);
  for (int c = first; c < last; ++c) {
    const Raw x = next;
    const uint32_t resets = chunk_flags_of(A.ns, ns_next, A.flags, A.T, (int64_t)c * CK, 0).ns & 0xffffu;
    if (c + 1 < last) request(c + 1);
    bool restart = false;
    int seg_src = 0;
    if (resets) {
      rare_path();
      const uint32_t upto = resets & ((2u << t) - 1u);
      const int pr = upto ? 31 - __builtin_clz(upto) : 0;
      restart = pr > 0;
      seg_src = (lane & 48) | (pr > 0 ? pr - 1 : 0);
#pragma unroll
      for (int i = 0; i < 8; ++i) S[i >> 2][i & 3] = zero4;
    }
    u32x4_t A1[4], A3[4];                            // rows: values, k-slots (sa | v) of tokens 4g ..
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      const u32x4_t vop = {x.v[half].x, x.v[half].y, x.v[half].z, x.v[half].w};
      u32x4_t sa_h, sa_l;
      split8h(x.sa[half], sa_h, sa_l);
#pragma unroll
      for (int x2 = 0; x2 < 2; ++x2) {
        const uint2 vv = pack4(mfma(vop, sel[x2], zero4));
        const uint2 hi = pack4(mfma(sa_h, sel[x2], zero4)), lo = pack4(mfma(sa_l, sel[x2], zero4));
        A1[2 * half + x2] = u32x4_t{hi.x, hi.y, vv.x, vv.y};
        A3[2 * half + x2] = u32x4_t{lo.x, lo.y, 0u, 0u};
      }
    }
    if (resets) {                                    // tokens from the last reset on
      rare_path();
      const uint32_t keep = ~((1u << (31 - __builtin_clz(resets))) - 1u) >> (4 * g);
      const uint32_t m0 = (keep & 1u ? 0xffffu : 0u) | (keep & 2u ? 0xffff0000u : 0u), m1 = (keep & 4u ? 0xffffu : 0u) | (keep & 8u ? 0xffff0000u : 0u);
#pragma unroll
      for (int vt = 0; vt < 4; ++vt) {
        A1[vt][0] &= m0; A1[vt][2] &= m0; A3[vt][0] &= m0;
        A1[vt][1] &= m1; A1[vt][3] &= m1; A3[vt][1] &= m1;
      }
    }
    float E[8];
    unpack8(x.w, E);
#pragma unroll
    for (int e = 0; e < 8; ++e) E[e] = row_scan(fmaxf(-exp2_fast(E[e] * LOG2E) * LOG2E, MIN_STEP_L2));
    cap_chunk_decay(E, lane, nullptr);               // the sweeps count it
    if (resets) {
      rare_path();
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float base = __shfl(E[e], seg_src, 64);
        if (restart) E[e] -= base;
      }
    }
    u32x4_t kh, kl, bh, bl;
    {
      float fk[8], fb[8];
      unpack8(x.k, fk); unpack8(x.b, fb);
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float l2 = fmaxf(E[e], MIN_CUM_L2), einv = exp2_fast(-l2);
        E[e] = exp2_fast(l2);
        fk[e] *= einv; fb[e] *= einv;
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        uint32_t hi, lo;
        split2(fk[2 * j], fk[2 * j + 1], hi, lo); kh[j] = hi; kl[j] = lo;
        split2(fb[2 * j], fb[2 * j + 1], hi, lo); bh[j] = hi; bl[j] = lo;
      }
    }
    // the chunk's decay from the lanes of its last token to those of the update, through this wave's own LDS
    if (t == 15) {
      float* const gp = own.decay + 8 * g;
      *reinterpret_cast<float4*>(gp) = make_float4(E[0], E[1], E[2], E[3]);
      *reinterpret_cast<float4*>(gp + 4) = make_float4(E[4], E[5], E[6], E[7]);
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
    for (int x2 = 0; x2 < 2; ++x2) {
      const uint2 b_h = pack4(mfma(bh, sel[x2], zero4)), b_l = pack4(mfma(bl, sel[x2], zero4));
      const uint2 k_h = pack4(mfma(kh, sel[x2], zero4)), k_l = pack4(mfma(kl, sel[x2], zero4));
      const u32x4_t Bh = {b_h.x, b_h.y, k_h.x, k_h.y}, Bl = {b_l.x, b_l.y, k_l.x, k_l.y};
      const float gm = own.decay[16 * x2 + t];
#pragma unroll
      for (int vt = 0; vt < 4; ++vt) {
        f32x4_t acc = S[x2][vt];
        acc = mfma(A1[vt], Bh, acc);
        acc = mfma(A1[vt], Bl, acc);
        acc = mfma(A3[vt], Bh, acc);
        acc[0] *= gm; acc[1] *= gm; acc[2] *= gm; acc[3] *= gm;
        S[x2][vt] = acc;
      }
      decay[x2] = join_decay(decay[x2], resets ? -1.f : gm);
    }
  }
#pragma unroll
  for (int x2 = 0; x2 < 2; ++x2) {
#pragma unroll
    for (int vt = 0; vt < 4; ++vt) own.S[x2][vt][lane] = S[x2][vt];
    if (g == 0) own.decay[16 * x2 + t] = decay[x2];
  }
  __syncthreads();
  EndSum* const rec = end_sum(A, head, part);
  for (int i = threadIdx.x; i < 16 * 64; i += 128 * END_GROUPS) {
    const int q = i >> 8, vt = (i >> 6) & 3, l = i & 63;
    f32x4_t acc = sums[q >> 1].S[q & 1][vt][l];
#pragma unroll
    for (int w = 1; w < END_GROUPS; ++w) {
      const EndHalf& s = sums[2 * w + (q >> 1)];
      const f32x4_t add = s.S[q & 1][vt][l];
      const float d = s.decay[16 * (q & 1) + (l & 15)];
#pragma unroll
      for (int e = 0; e < 4; ++e) acc[e] = d < 0.f ? add[e] : fmaf(acc[e], d, add[e]);
    }
    rec->S[q][vt][l] = acc;
  }
  if (threadIdx.x < 64) {
    float d = 1.f;
#pragma unroll
    for (int w = 0; w < END_GROUPS; ++w) d = join_decay(d, sums[2 * w + (threadIdx.x >> 5)].decay[threadIdx.x & 31]);
    rec->decay[threadIdx.x] = d;
  }
}

}  // namespace chunk
}  // namespace hiprwkv
