// What each part of a sequence does to the state, for the sweeps of the WKV7 backward that start inside it (bf16 I/O, gfx950;
// reference of the recurrence: /root/reference/src/jaxrwkv/rwkv7.py:200-220).
//
// With sa_t known (the forward's residual) the state obeys a recurrence that is linear key by key,
//     S_t = S_{t-1} diag(d_t) + sa_t b_t^T + v_t k_t^T
// so a part that does not reset leaves S_in diag(decay) + S_own, S_own what it makes from zero: one EndSum per part but the last.
// The operands of a chunk are those of sweep B (wkv7_chunk_bwd_b.hip: bf16 pairs, the same decay floor), so the state at a
// boundary is as near to 64 bits as the one that sweep B would carry there.
//
// Nothing of a chunk depends on another one before the sums meet, so there is no hand-shake: each of eight waves takes an eighth of
// the part's chunks, its operands straight from memory to registers (the transposing products leave them as the update wants them),
// the next chunk requested ahead, and the eight results are joined in LDS.  Bound by the vector units, two waves of a SIMD in turn
// (one chunk a part 5 us, of which the launch and the joining are 4; as a variant of sweep B, with its ring, the same).  What a call that
// keeps the records takes longer for, forward alone: B=1 T=256 H=12 19.4 -> 25.0 us, B=1 T=2048 H=32 56.8 -> 69.6, B=4 T=1024 H=32, where
// 128 workgroups have four chunks a wave, 57 -> 76.
#include "chunk_common.h"
#include "wkv_args.h"
#include "wkv7_parts.h"

namespace hiprwkv {

namespace {

using namespace chunk;

constexpr int WAVES = 8;

struct Raw {
  uint4 w[2], k[2], b[2], v[2], sa[2];
};
// a part before the last is whole chunks
__device__ __forceinline__ void load_raw(Raw& x, const Wkv7Args& A, int64_t b, int64_t h, int64_t c0, int lane) {
  const size_t el = (((size_t)b * A.T + c0 + (lane & 15)) * A.H + h) * 64 + 8 * (lane >> 4);
  auto ld = [&](const void* p, uint4 (&o)[2]) {
    o[0] = *reinterpret_cast<const uint4*>(reinterpret_cast<const char*>(p) + el * 2);
    o[1] = *reinterpret_cast<const uint4*>(reinterpret_cast<const char*>(p) + el * 2 + 64);
  };
  ld(A.w, x.w); ld(A.k, x.k); ld(A.b, x.b); ld(A.v, x.v); ld(A.sa_in, x.sa);
}
// four consecutive tokens of a transposing product
__device__ __forceinline__ uint2 pack4(const f32x4_t d) { return make_uint2(pack_exact(d[0], d[1]), pack_exact(d[2], d[3])); }
// a decay behind another one; negative: nothing is left
__device__ __forceinline__ float join_decay(float first, float second) {
  // not below the smallest normal number: what is infinite stays so, as it does chunk by chunk
  return first < 0.f || second < 0.f ? -1.f : fmaxf(first * second, 1.17549435e-38f);
}

}  // namespace

__global__ __launch_bounds__(64 * WAVES) void wkv7_ends_kernel(Wkv7Args A) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  EndSum* const sums = reinterpret_cast<EndSum*>(smem_raw);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, t = lane & 15, g = lane >> 4;
  const int64_t head = blockIdx.x / (A.n_end - 1);
  const int part = (int)(blockIdx.x % (A.n_end - 1));
  const int64_t b = head / A.H, h = head % A.H;
  const int first = part * A.end_chunks + A.end_chunks * wave / WAVES, last = part * A.end_chunks + A.end_chunks * (wave + 1) / WAVES;
  const f32x4_t zero4 = {0.f, 0.f, 0.f, 0.f};
  EndSum& own = sums[wave];
  u32x4_t sel[2];
  make_sel(sel, lane);
  f32x4_t S[4][4];         // [key tile][value tile]
  float decay[4];          // of the wave's chunks so far, keys 16q + t
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    decay[q] = 1.f;
#pragma unroll
    for (int vt = 0; vt < 4; ++vt) S[q][vt] = zero4;
  }
  Raw next;
  uint32_t ns_next = 0u;
  auto request = [&](int c) {
    ns_next = chunk_flag_prefetch(A.ns, A.T, b, (int64_t)c * CK, lane);
    load_raw(next, A, b, h, (int64_t)c * CK, lane);
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
      for (int i = 0; i < 16; ++i) S[i >> 2][i & 3] = zero4;
    }
    u32x4_t A1[4], A3[4];                            // rows: values, k-slots (sa | v) of tokens 4g ..
#pragma unroll
    for (int hf = 0; hf < 2; ++hf) {
      const u32x4_t vop = {x.v[hf].x, x.v[hf].y, x.v[hf].z, x.v[hf].w};
      u32x4_t sa_h, sa_l;
      split8h(x.sa[hf], sa_h, sa_l);
#pragma unroll
      for (int x2 = 0; x2 < 2; ++x2) {
        const uint2 vv = pack4(mfma(vop, sel[x2], zero4));
        const uint2 hi = pack4(mfma(sa_h, sel[x2], zero4)), lo = pack4(mfma(sa_l, sel[x2], zero4));
        A1[2 * hf + x2] = u32x4_t{hi.x, hi.y, vv.x, vv.y};
        A3[2 * hf + x2] = u32x4_t{lo.x, lo.y, 0u, 0u};
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
#pragma unroll
    for (int hf = 0; hf < 2; ++hf) {
      float E[8];
      unpack8(x.w[hf], E);
#pragma unroll
      for (int e = 0; e < 8; ++e) E[e] = row_scan(fmaxf(-exp2_fast(E[e] * LOG2E) * LOG2E, MIN_STEP_L2));
      cap_chunk_decay(E, lane, nullptr);             // the forward counts it
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
        unpack8(x.k[hf], fk); unpack8(x.b[hf], fb);
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
        float* const gp = own.decay + 32 * hf + 8 * g;
        *reinterpret_cast<float4*>(gp) = make_float4(E[0], E[1], E[2], E[3]);
        *reinterpret_cast<float4*>(gp + 4) = make_float4(E[4], E[5], E[6], E[7]);
      }
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
      for (int x2 = 0; x2 < 2; ++x2) {
        const int q = 2 * hf + x2;
        const uint2 b_h = pack4(mfma(bh, sel[x2], zero4)), b_l = pack4(mfma(bl, sel[x2], zero4));
        const uint2 k_h = pack4(mfma(kh, sel[x2], zero4)), k_l = pack4(mfma(kl, sel[x2], zero4));
        const u32x4_t Bh = {b_h.x, b_h.y, k_h.x, k_h.y}, Bl = {b_l.x, b_l.y, k_l.x, k_l.y};
        const float gm = own.decay[16 * q + t];
#pragma unroll
        for (int vt = 0; vt < 4; ++vt) {
          f32x4_t acc = S[q][vt];
          acc = mfma(A1[vt], Bh, acc);
          acc = mfma(A1[vt], Bl, acc);
          acc = mfma(A3[vt], Bh, acc);
          acc[0] *= gm; acc[1] *= gm; acc[2] *= gm; acc[3] *= gm;
          S[q][vt] = acc;
        }
        decay[q] = join_decay(decay[q], resets ? -1.f : gm);
      }
    }
  }
#pragma unroll
  for (int q = 0; q < 4; ++q) {
#pragma unroll
    for (int vt = 0; vt < 4; ++vt) own.S[q][vt][lane] = S[q][vt];
    if (g == 0) own.decay[16 * q + t] = decay[q];
  }
  __syncthreads();
  EndSum* const rec = end_sum(A, head, part);
  for (int i = threadIdx.x; i < 16 * 64; i += 64 * WAVES) {
    const int q = i >> 8, vt = (i >> 6) & 3, l = i & 63;
    f32x4_t acc = sums[0].S[q][vt][l];
#pragma unroll
    for (int w = 1; w < WAVES; ++w) {
      const f32x4_t add = sums[w].S[q][vt][l];
      const float d = sums[w].decay[16 * q + (l & 15)];
#pragma unroll
      for (int e = 0; e < 4; ++e) acc[e] = d < 0.f ? add[e] : fmaf(acc[e], d, add[e]);
    }
    rec->S[q][vt][l] = acc;
  }
  if (threadIdx.x < 64) {
    float d = sums[0].decay[threadIdx.x];
#pragma unroll
    for (int w = 1; w < WAVES; ++w) d = join_decay(d, sums[w].decay[threadIdx.x]);
    rec->decay[threadIdx.x] = d;
  }
}

// A.sa_in, A.ns, the inputs, A.n_end >= 2 parts of A.end_chunks chunks -> A.ends
hipError_t launch_wkv7_ends(const Wkv7Args& A, hipStream_t stream) {
  constexpr size_t smem = WAVES * sizeof(EndSum);
  static LdsAttrOnce once;
  const hipError_t attr = allow_dynamic_lds(once, reinterpret_cast<const void*>(wkv7_ends_kernel), smem);
  if (attr != hipSuccess) return attr;
  hipLaunchKernelGGL(wkv7_ends_kernel, dim3((unsigned)(A.B * A.H * (A.n_end - 1))), dim3(64 * WAVES), smem, stream, A);
  return hipGetLastError();
}

}  // namespace hiprwkv
