// An RWKV-7 decode step (at most 8 tokens per sequence, at most 256 tokens in all, bf16) layer by layer from native code:
// eight launches per layer instead of the ~30 operations of the general path, whose host side alone takes 5 ms for 12 layers.  With one
// or two tokens 1 and 2, 3 and 4, and 6 and 7 are one launch each.
//     1  residual addition, norm, shift and six interpolations               (rwkv7_block.hip)
//     2  r, k, v and the first low-rank factors, tanh / sigmoid applied       rwkv7_gemm.hip, seven products in one grid
//     3  the second low-rank factors                                          rwkv7_gemm.hip, four products
//     4  gates, WKV step on the packed state, group norm, bonus, gate         decode_core_kernel
//     5  output projection                                                    rwkv7_gemm.hip
//     6  residual addition, norm, shift and interpolation                     (rwkv7_block.hip)
//     7  key projection with relu(.)^2                                        rwkv7_gemm.hip
//     8  value projection                                                     rwkv7_gemm.hip
// Measured (eager, host included), with the general path's operations, with a launch for each line above, and now: 12 layers of 768 channels, one
// user 5.4 ms, 0.57, 0.32 a step, 16 users -, 0.61, 0.50; 24 layers of 2048 channels, one user -, 1.61, 1.21, 16 -, 1.89, 1.66, 256 10.9, 3.6, 3.1.
// Norms inside the products: three users as long as with norms of their own, two 0.50 -> 0.42 ms (12 x 768; 0.32 now).
// References: /root/reference/src/jaxrwkv/rwkv7.py:190-198, :223-267, :269-291.  Products accumulate in fp32 and are rounded
// once; the values between the gates, the recurrence and the group norm are rounded where the general path stores them.
#include "chunk_common.h"
#include "wkv_args.h"

namespace hiprwkv {

namespace {

// ---------------------------------------------------------------------------------------------------------------
// Sum over the wave, delivered to every lane: rows of 16 lanes by DPP, the four rows through scalar registers.  Every lane of the wave takes
// part.  (Six __shfl_xor are six trips through LDS in series, about 100 cycles each; a step's four sums were a sixth of the kernel below.)
__device__ __forceinline__ float wave_sum(float x) {
  const int v = __float_as_int(row_sum(x));
  const float a = __int_as_float(__builtin_amdgcn_readlane(v, 0)) + __int_as_float(__builtin_amdgcn_readlane(v, 16));
  const float b = __int_as_float(__builtin_amdgcn_readlane(v, 32)) + __int_as_float(__builtin_amdgcn_readlane(v, 48));
  return a + b;
}

struct CoreArgs {
  int64_t B, T, H;
  int per;                     // sequences of a workgroup
  const bf16_t* par[2][6];     // (H,64) parameters of waves 0 and 1: a0 k_k k_a r_k ln_w ln_b | w0 v0
  const bf16_t* tok[2][4];     // (B,T,H,64): k r xa g | v xw v_first xv
  int vmix;                    // there is a value residual
  float eps;
  const bf16_t* s;             // states: H*64*64 elements per sequence, bstride apart
  bf16_t* new_s;
  int64_t bstride;
  const int32_t* length;
  const uint8_t* ns;
  unsigned flags;              // bit 0: the associative scan's conventions, as in the op
  bf16_t* y;
};

// A workgroup has one head of `per` consecutive sequences, one after the other; thread (row i = tid/4, quarter q = tid%4) holds 16 elements
// of state row i, as in the small-T kernel of the op, whose state traffic (2 x 8 KB per head) is the bound.  Waves 0 and 1 (one lane per
// channel) turn the projections into the op's inputs and hand them over through LDS, wave 0 takes y back through LDS for the group norm,
// the bonus and the gate.  A sequence is a chain of waits; the state and the operands of the next one are requested before this one's are
// used, so that memory works through it.  B=256 H=32: the state alone is 67 MB each way; 38.5 us a launch with one wave for the op's inputs
// and sums by way of LDS, 34.6 with a workgroup a sequence (six of them a CU), 31.3 now with four a CU (4.6 TB/s; five 32.1, and for six the
// registers spill: 51).
constexpr int CORE_PER_CU = 4;
__global__ __launch_bounds__(256, CORE_PER_CU) void decode_core_kernel(CoreArgs A) {
  __shared__ __align__(16) float ch[5][64];            // d, k', a_i, b_i, r
  __shared__ float vs[64], ys[64];
  const int h = blockIdx.x;
  const int64_t b0 = (int64_t)blockIdx.y * A.per, b1 = b0 + A.per < A.B ? b0 + A.per : A.B;
  const int tid = threadIdx.x, i = tid >> 2, q = tid & 3, c0 = 16 * q;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, role = wave & 1;
  const bool maker = wave < 2;                         // wave 0: what comes of k, r, a and the end; wave 1: decay and values
  const size_t in_state = ((size_t)h * 64 + i) * 64 + c0;
  uint4 s0, s1;                                        // the next sequence's state and first token, as they lie
  uint32_t tk[4];
  auto request_token = [&](int64_t row) {
#pragma unroll
    for (int z = 0; z < 4; ++z) tk[z] = A.tok[role][z][(row * A.H + h) * 64 + lane].bits;
  };
  auto request = [&](int64_t b) {
    const uint4* p = reinterpret_cast<const uint4*>(A.s + (size_t)b * A.bstride + in_state);
    s0 = p[0];
    s1 = p[1];
    if (maker) request_token(b * A.T);
  };
  uint32_t pv[6] = {0u, 0u, 0u, 0u, 0u, 0u};
  if (maker) {
#pragma unroll
    for (int z = 0; z < 6; ++z) pv[z] = A.par[role][z][h * 64 + lane].bits;
  }
  request(b0);
  const bool compat = (A.flags & 1u) != 0;
  for (int64_t b = b0; b < b1; ++b) {
    int64_t L = A.T;
    if (A.length != nullptr) { L = A.length[b]; L = L < 0 ? 0 : L < A.T ? L : A.T; }
    const uint8_t* ns = A.ns ? A.ns + b * A.T : nullptr;
    const bool q2drop = compat && L < A.T && ns != nullptr && ns[L] != 0;
    bf16_t* const out = A.new_s + (size_t)b * A.bstride + in_state;
    asm volatile("" : "+v"(s0.x), "+v"(s0.y), "+v"(s0.z), "+v"(s0.w), "+v"(s1.x), "+v"(s1.y), "+v"(s1.z), "+v"(s1.w));
    float S[16];
    {
      const uint32_t w[8] = {s0.x, s0.y, s0.z, s0.w, s1.x, s1.y, s1.z, s1.w};
#pragma unroll
      for (int c = 0; c < 8; ++c) {
        S[2 * c] = __uint_as_float(w[c] << 16);
        S[2 * c + 1] = __uint_as_float(w[c] & 0xffff0000u);
      }
    }
    auto put_state = [&]() {
      float lo[8], hi[8];
#pragma unroll
      for (int c = 0; c < 8; ++c) { lo[c] = q2drop ? 0.f : S[c]; hi[c] = q2drop ? 0.f : S[8 + c]; }
      st8(out, lo);
      st8(out + 8, hi);
    };
    if (L == 0) put_state();
    for (int64_t t = 0; t < A.T; ++t) {
      asm volatile("" : "+v"(tk[0]), "+v"(tk[1]), "+v"(tk[2]), "+v"(tk[3]));
      const float t0 = __uint_as_float(tk[0] << 16), t1 = __uint_as_float(tk[1] << 16), t2 = __uint_as_float(tk[2] << 16),
                  t3 = __uint_as_float(tk[3] << 16);
      if (t + 1 < A.T) {
        if (maker) request_token(b * A.T + t + 1);
      } else if (b + 1 < b1) {
        request(b + 1);
      }
      asm volatile("" : "+v"(pv[0]), "+v"(pv[1]), "+v"(pv[2]), "+v"(pv[3]), "+v"(pv[4]), "+v"(pv[5]));
      auto param = [&](int z) { return __uint_as_float(pv[z] << 16); };
      float bonus = 0.f, v = 0.f;
      if (wave == 0) {
        const float a = rnd(sigmoidf(param(0) + t2));
        float kk = t0 * param(1);
        kk *= 1.f / fmaxf(sqrtf(wave_sum(kk * kk)), 1e-12f);
        const float kp = rnd(t0 * (1.f + (a - 1.f) * param(2)));
        bonus = wave_sum(t1 * kp * param(3));
        ch[1][lane] = kp;
        ch[2][lane] = rnd(-kk);
        ch[3][lane] = rnd(kk * a);
        ch[4][lane] = t1;
      } else if (wave == 1) {
        const float w = rnd(-softplusf(-(param(0) + t1)) - 0.5f);
        ch[0][lane] = __expf(-__expf(w));
        vs[lane] = A.vmix ? rnd(fmaf(t2 - t0, sigmoidf(param(1) + t3), t0)) : t0;
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
      if (wave == 0) v = vs[lane];                       // before wave 1 writes the next token's
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
      if (wave == 0) {
        const float yv = ys[lane];
        const float d = yv - wave_sum(yv) * (1.f / 64.f);
        const float rstd = rsqrtf(wave_sum(d * d) * (1.f / 64.f) + A.eps);
        st_f(A.y + ((b * A.T + t) * A.H + h) * 64 + lane, (d * rstd * param(4) + param(5) + bonus * v) * t3);
      }
    }
  }
}

// The same for one or two tokens in all (a decode step of few users), where a workgroup's time is a chain of instructions and latencies
// and CUs stand idle: sixteen waves, four elements of the state a lane, the op's inputs made by four waves, and the second low-rank
// products here as well (one launch less; their weights are read once per sequence).  Eight lanes read a row of a factor; four waves take a
// factor, and the wave that needs a product adds their parts.  What a wave reads is named by a table in the arguments: as conditions in the
// code every choice became a branch that waited for its own loads.  768 channels, one user: 8.1 us a launch with four waves, 5.8 now.
struct FewArgs {
  int64_t T, H;
  const bf16_t* par[4][4];     // (H,64) parameters of waves 0 to 3: a0 k_k ln_w ln_b | a0 k_a r_k | w0 | v0
  const bf16_t* tok[4][2];     // (B,T,H,64): k | k r | | v v_first
  const bf16_t *hid[4], *w2[4];   // the factors of xw, xa, g, xv: (B,T,d) and (d,H,64), d a multiple of 32 or 0 (none)
  int d[4];
  const bf16_t* s;
  bf16_t* new_s;
  int64_t bstride;
  const int32_t* length;
  const uint8_t* ns;
  bf16_t* y;
  float eps;
  unsigned flags;
  int vmix;                    // there is a value residual
};
__global__ __launch_bounds__(1024) void decode_few_kernel(FewArgs A) {
  __shared__ __align__(16) float lora[16][4][64];                 // [wave][16 of its lanes][channel]
  __shared__ __align__(16) float ch[5][64];                       // d, k', a_i, b_i, r
  __shared__ float vs[64], ys[64], gs[64], bonus_s;
  const int64_t b = blockIdx.y, h = blockIdx.x;
  const int tid = threadIdx.x, i = tid >> 4, c0 = 4 * (tid & 15);
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, q = wave & 3, f = wave >> 2;
  const int d = A.d[f];
  const size_t sel = (size_t)b * A.bstride + ((size_t)h * 64 + i) * 64 + c0, cel = (size_t)h * 64 + lane;
  uint2 s4 = *reinterpret_cast<const uint2*>(A.s + sel);
  uint32_t pv[4];                                                 // as they lie: a conversion would wait for them
#pragma unroll
  for (int z = 0; z < 4; ++z) pv[z] = A.par[q][z][cel].bits;
  int64_t L = A.T;
  if (A.length != nullptr) { L = A.length[b]; L = L < 0 ? 0 : L < A.T ? L : A.T; }
  const bool compat = (A.flags & 1u) != 0;
  const uint8_t* ns = A.ns ? A.ns + b * A.T : nullptr;
  const bool q2drop = compat && L < A.T && ns != nullptr && ns[L] != 0;
  float S[4] = {0.f, 0.f, 0.f, 0.f};
  for (int64_t t = 0; t < A.T; ++t) {
    const size_t row = (size_t)b * A.T + t, el = (row * A.H + h) * 64 + lane;
    uint32_t u0v = A.tok[q][0][el].bits, u1v = A.tok[q][1][el].bits;
    {
      const int first = 8 * q + (lane >> 3), c8 = 8 * (lane & 7);
      const bf16_t *hid = A.hid[f] + row * d + first, *w2 = A.w2[f] + ((size_t)first * A.H + h) * 64 + c8;
      const size_t stride = (size_t)32 * 64 * A.H;
      float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
      for (int j0 = 0; j0 < d; j0 += 128) {
        uint4 w[4];
        uint32_t x[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const int uu = j0 + 32 * u < d ? u : 0;                // beyond the factor: read again, not used
          w[u] = *reinterpret_cast<const uint4*>(w2 + uu * stride);
          x[u] = hid[32 * uu].bits;
        }
#pragma unroll
        for (int u = 0; u < 4; ++u)
          if (j0 + 32 * u < d) {
            const uint32_t q4[4] = {w[u].x, w[u].y, w[u].z, w[u].w};
            const float xu = __uint_as_float(x[u] << 16);
#pragma unroll
            for (int c = 0; c < 4; ++c) {
              acc[2 * c] = fmaf(xu, __uint_as_float(q4[c] << 16), acc[2 * c]);
              acc[2 * c + 1] = fmaf(xu, __uint_as_float(q4[c] & 0xffff0000u), acc[2 * c + 1]);
            }
          }
        hid += 128;
        w2 += 4 * stride;
      }
#pragma unroll
      for (int c = 0; c < 8; ++c)
        acc[c] += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(acc[c]), 0x128, 0xf, 0xf, false));   // row_ror:8
      if ((lane & 8) == 0) st8(&lora[wave][lane >> 4][c8], acc);
    }
    __syncthreads();
    asm volatile("" : "+v"(u0v), "+v"(u1v), "+v"(pv[0]), "+v"(pv[1]), "+v"(pv[2]), "+v"(pv[3]));      // conversions stay behind the barrier
    const float p0 = __uint_as_float(pv[0] << 16), p1 = __uint_as_float(pv[1] << 16), p2 = __uint_as_float(pv[2] << 16), p3 = __uint_as_float(pv[3] << 16);
    const float u0 = __uint_as_float(u0v << 16), u1 = __uint_as_float(u1v << 16);
    auto low = [&](int of) {
      float s = 0.f;
#pragma unroll
      for (int u = 0; u < 16; ++u) s += lora[4 * of + (u >> 2)][u & 3][lane];
      return rnd(s);
    };
    if (wave == 0) {
      float kk = u0 * p1;
      kk *= 1.f / fmaxf(sqrtf(wave_sum(kk * kk)), 1e-12f);
      const float a = rnd(sigmoidf(p0 + low(1)));
      ch[2][lane] = rnd(-kk);
      ch[3][lane] = rnd(kk * a);
    } else if (wave == 1) {
      const float a = rnd(sigmoidf(p0 + low(1)));
      const float kp = rnd(u0 * (1.f + (a - 1.f) * p1));
      ch[1][lane] = kp;
      ch[4][lane] = u1;
      bonus_s = wave_sum(u1 * kp * p2);                           // every lane the same
    } else if (wave == 2) {
      const float w = rnd(-softplusf(-(p0 + low(0))) - 0.5f);
      ch[0][lane] = __expf(-__expf(w));
    } else if (wave == 3) {
      vs[lane] = A.vmix ? rnd(fmaf(u1 - u0, sigmoidf(p0 + low(3)), u0)) : u0;
    } else if (wave == 4) {
      gs[lane] = low(2);
    }
    __syncthreads();
    if (t == 0) {
      asm volatile("" : "+v"(s4.x), "+v"(s4.y));
      S[0] = __uint_as_float(s4.x << 16); S[1] = __uint_as_float(s4.x & 0xffff0000u);
      S[2] = __uint_as_float(s4.y << 16); S[3] = __uint_as_float(s4.y & 0xffff0000u);
    }
    if (ns != nullptr && ns[t]) {
#pragma unroll
      for (int c = 0; c < 4; ++c) S[c] = 0.f;
    }
    float p = 0.f;
#pragma unroll
    for (int c = 0; c < 4; ++c) p = fmaf(S[c], ch[2][c0 + c], p);
    const float sa = row_sum(p), vi = vs[i];
    float y = 0.f;
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      S[c] = fmaf(S[c], ch[0][c0 + c], fmaf(vi, ch[1][c0 + c], sa * ch[3][c0 + c]));
      y = fmaf(S[c], ch[4][c0 + c], y);
    }
    y = row_sum(y);
    if (compat && t + 1 < A.T && ns != nullptr && ns[t + 1]) y = 0.f;
    if ((tid & 15) == 0) ys[i] = rnd(y);
    if (t == L - 1) s4 = make_uint2(chunk::pack_rn(S[0], S[1]), chunk::pack_rn(S[2], S[3]));
    __syncthreads();
    if (wave == 0) {                                              // the others wait at the next token's first barrier
      const float yv = ys[lane];
      const float dv = yv - wave_sum(yv) * (1.f / 64.f);
      const float rstd = rsqrtf(wave_sum(dv * dv) * (1.f / 64.f) + A.eps);
      st_f(A.y + el, (dv * rstd * p2 + p3 + bonus_s * vs[lane]) * gs[lane]);
    }
  }
  *reinterpret_cast<uint2*>(A.new_s + sel) = q2drop ? make_uint2(0u, 0u) : s4;      // L = 0: the state itself
}

}  // namespace

size_t rwkv7_decode_workspace(const Rwkv7Decode& D) {
  const size_t rows = (size_t)D.B * D.T;
  const size_t d = D.d_decay + D.d_aaa + D.d_mv + D.d_gate;
  // xs twice, six interpolations, r k v v_first, four low-rank results, y, dx; the low-rank hidden values; the ffn's
  const size_t parts = rows * D.C * GEMM_MAX_SPLIT * sizeof(float);
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
  float* parts = reinterpret_cast<float*>(at);
  const int split_out = gemm_split((int)rows, C, C), split_val = gemm_split((int)rows, D.F, C);
  int n_part = 1;                              // of the dx that the next norm reads
  auto layer = [&](const void* p, int64_t l, size_t n) { return static_cast<const bf16_t*>(p) + (size_t)l * n; };
  const bool few = rows <= HEAD_GEMM_ROWS;     // norms inside the products, second low-rank products inside the recurrence
  const size_t row_state = (2 + 64) * C, seq_state = (size_t)D.L * row_state;
  const bf16_t* st = static_cast<const bf16_t*>(D.state);
  bf16_t* nst = static_cast<bf16_t*>(D.new_state);

  LnMixArgs N;
  memset(&N, 0, sizeof(N));
  N.B = D.B; N.T = D.T; N.C = D.C; N.eps = 1e-5f;
  N.ns = D.new_starts; N.length = D.length;
  auto head_args = [&](int n_out, const void* x, const void* add, bf16_t* sum, const void* w, const void* b, int64_t l, int srow) {
    LnMixArgs A = N;
    A.x = x; A.dx = add; A.xs = sum;
    if (add != nullptr && n_part > 1) { A.dx = nullptr; A.part = parts; A.n_part = n_part; }
    A.ln_w = w; A.ln_b = b;
    if (n_out) {
      A.prev = st + (size_t)l * row_state + srow * C; A.prev_bstride = seq_state;
      A.shift = nst + (size_t)l * row_state + srow * C; A.shift_bstride = seq_state;
    }
    return A;
  };
  auto head = [&](int n_out, const LnMixArgs& of, const void* const* mixv, bf16_t* const* outs) {
    LnMixArgs A = of;
    for (int i = 0; i < n_out; ++i) A.mix[i] = mixv[i];
    for (int i = 0; i < (n_out ? n_out : 1); ++i) A.out[i] = outs[i];
    return launch_ln_shiftmix(0, n_out, A, stream);
  };
  hipError_t e;
#define HIPRWKV_TRY(x) if ((e = (x)) != hipSuccess) return e
  int cur = 0;
  {
    bf16_t* o[1] = {xs[0]};
    HIPRWKV_TRY(head(0, head_args(0, D.x, nullptr, nullptr, D.ln0_w, D.ln0_b, 0, 0), nullptr, o));
  }
  for (int64_t l = 0; l < D.L; ++l) {
    const void* mv[6];
    const void* stacked[6] = {D.x_r, D.x_w, D.x_k, D.x_v, D.x_a, D.x_g};
    for (int i = 0; i < 6; ++i) mv[i] = layer(stacked[i], l, C);
    const LnMixArgs ln1 = head_args(6, xs[cur], l ? dx : nullptr, xs[cur ^ 1], layer(D.ln1_w, l, C), layer(D.ln1_b, l, C), l, 1);
    if (!few) HIPRWKV_TRY(head(6, ln1, mv, mix));
    if (l) cur ^= 1;
    GemmArgs G;
    memset(&G, 0, sizeof(G));
    auto add = [&](const bf16_t* x, const bf16_t* w, bf16_t* out, int64_t K, int64_t Nn, int kn, int act) {
      GemmJob& J = G.job[G.n_jobs++];
      memset(&J, 0, sizeof(J));
      J.x = x; J.w = w; J.out = out; J.M = (int)rows; J.K = (int)K; J.N = (int)Nn; J.kn = kn; J.act = act;
    };
    bf16_t* vl = l == 0 ? vf : v;
    add(mix[0], layer(D.receptance, l, C * C), r, C, C, 0, GEMM_ACT_NONE);
    add(mix[2], layer(D.key, l, C * C), k, C, C, 0, GEMM_ACT_NONE);
    add(mix[3], layer(D.value, l, C * C), vl, C, C, 0, GEMM_ACT_NONE);
    add(mix[1], layer(D.w1, l, C * D.d_decay), hw, C, D.d_decay, 1, GEMM_ACT_TANH);
    add(mix[4], layer(D.a1, l, C * D.d_aaa), ha, C, D.d_aaa, 1, GEMM_ACT_NONE);
    add(mix[5], layer(D.g1, l, C * D.d_gate), hg, C, D.d_gate, 1, GEMM_ACT_SIGMOID);
    if (l) add(mix[3], layer(D.v1, l, C * D.d_mv), hv, C, D.d_mv, 1, GEMM_ACT_NONE);
    const dim3 heads((unsigned)D.H, (unsigned)D.B);
    const bf16_t *const w0 = layer(D.w0, l, C), *const a0 = layer(D.a0, l, C), *const v0 = layer(D.v0, l, C), *const k_k = layer(D.k_k, l, C),
                 *const k_a = layer(D.k_a, l, C), *const r_k = layer(D.r_k, l, C), *const ln_w = layer(D.lnx_w, l, C), *const ln_b = layer(D.lnx_b, l, C);
    const bf16_t* const s = st + (size_t)l * row_state + 2 * C;
    bf16_t* const new_s = nst + (size_t)l * row_state + 2 * C;
    if (few) {
      const int of_mix[7] = {0, 2, 3, 1, 4, 5, 3};
      for (int i = 0; i < G.n_jobs; ++i) G.job[i].aux = mv[of_mix[i]];
      HIPRWKV_TRY(launch_head_gemm(ln1, G, stream));
      FewArgs A = {};
      const bf16_t* const second[4] = {layer(D.w2, l, C * D.d_decay), layer(D.a2, l, C * D.d_aaa), layer(D.g2, l, C * D.d_gate),
                                       layer(l ? D.v2 : D.w2, l, C * D.d_mv)};
      const bf16_t* const first[4] = {hw, ha, hg, l ? hv : hw};
      const int64_t d[4] = {D.d_decay, D.d_aaa, D.d_gate, l ? D.d_mv : 0};
      const bf16_t* const par[4][4] = {{a0, k_k, ln_w, ln_b}, {a0, k_a, r_k, r_k}, {w0, w0, w0, w0}, {l ? v0 : w0, w0, w0, w0}};
      const bf16_t* const tok[4][2] = {{k, k}, {k, r}, {k, k}, {vl, l ? vf : vl}};
      for (int i = 0; i < 4; ++i) {
        A.hid[i] = first[i]; A.w2[i] = second[i]; A.d[i] = (int)d[i];
        for (int z = 0; z < 4; ++z) A.par[i][z] = par[i][z];
        for (int z = 0; z < 2; ++z) A.tok[i][z] = tok[i][z];
      }
      A.T = D.T; A.H = D.H; A.eps = 64e-5f; A.vmix = l > 0;
      A.s = s; A.new_s = new_s; A.bstride = seq_state;
      A.length = D.length; A.ns = D.new_starts; A.flags = (unsigned)D.flags; A.y = y;
      hipLaunchKernelGGL(decode_few_kernel, heads, dim3(1024), 0, stream, A);
      HIPRWKV_TRY(hipGetLastError());
    } else {
      HIPRWKV_TRY(launch_gemm(G, 1, stream));
      G.n_jobs = 0;
      add(hw, layer(D.w2, l, C * D.d_decay), xw, D.d_decay, C, 1, GEMM_ACT_NONE);
      add(ha, layer(D.a2, l, C * D.d_aaa), xa, D.d_aaa, C, 1, GEMM_ACT_NONE);
      add(hg, layer(D.g2, l, C * D.d_gate), g, D.d_gate, C, 1, GEMM_ACT_NONE);
      if (l) add(hv, layer(D.v2, l, C * D.d_mv), xv, D.d_mv, C, 1, GEMM_ACT_NONE);
      HIPRWKV_TRY(launch_gemm(G, 1, stream));
      CoreArgs A = {};
      const bf16_t* const par[2][6] = {{a0, k_k, k_a, r_k, ln_w, ln_b}, {w0, l ? v0 : w0, w0, w0, w0, w0}};
      const bf16_t* const tok[2][4] = {{k, r, xa, g}, {vl, xw, l ? vf : vl, l ? xv : vl}};
      memcpy(A.par, par, sizeof(par));
      memcpy(A.tok, tok, sizeof(tok));
      A.B = D.B; A.T = D.T; A.H = D.H; A.eps = 64e-5f; A.vmix = l > 0;
      // as many workgroups as the GPU holds at once
      A.per = (int)((D.B * D.H + 256 * CORE_PER_CU - 1) / (256 * CORE_PER_CU));
      A.s = s; A.new_s = new_s; A.bstride = seq_state;
      A.length = D.length; A.ns = D.new_starts; A.flags = (unsigned)D.flags; A.y = y;
      hipLaunchKernelGGL(decode_core_kernel, dim3((unsigned)D.H, (unsigned)((D.B + A.per - 1) / A.per)), dim3(256), 0, stream, A);
      HIPRWKV_TRY(hipGetLastError());
    }
    G.n_jobs = 0;
    add(y, layer(D.output, l, C * C), dx, C, C, 0, GEMM_ACT_NONE);
    n_part = split_out;
    G.part = n_part > 1 ? parts : nullptr;
    HIPRWKV_TRY(launch_gemm(G, n_part, stream));
    const void* fm[1] = {layer(D.ffn_x_k, l, C)};
    const LnMixArgs ln2 = head_args(1, xs[cur], dx, xs[cur ^ 1], layer(D.ln2_w, l, C), layer(D.ln2_b, l, C), l, 0);
    if (!few) HIPRWKV_TRY(head(1, ln2, fm, mix));
    cur ^= 1;
    G.n_jobs = 0;
    G.part = nullptr;
    add(mix[0], layer(D.ffn_key, l, C * D.F), ff, C, D.F, 0, GEMM_ACT_RELUSQ);
    G.job[0].aux = few ? fm[0] : nullptr;
    HIPRWKV_TRY(few ? launch_head_gemm(ln2, G, stream) : launch_gemm(G, 1, stream));
    G.n_jobs = 0;
    add(ff, layer(D.ffn_value, l, C * D.F), dx, D.F, C, 0, GEMM_ACT_NONE);
    n_part = split_val;
    G.part = n_part > 1 ? parts : nullptr;
    HIPRWKV_TRY(launch_gemm(G, n_part, stream));
  }
  bf16_t* o[1] = {static_cast<bf16_t*>(D.xn)};
  HIPRWKV_TRY(head(0, head_args(0, xs[cur], dx, xs[cur ^ 1], D.ln_out_w, D.ln_out_b, 0, 0), nullptr, o));
  if (D.logits != nullptr) {
    GemmArgs G;
    memset(&G, 0, sizeof(G));
    G.n_jobs = 1;
    GemmJob& J = G.job[0];
    J.x = D.xn; J.w = D.head; J.out = D.logits;
    J.M = (int)rows; J.K = (int)C; J.N = (int)D.vocab;
    HIPRWKV_TRY(launch_gemm(G, 1, stream));
  }
#undef HIPRWKV_TRY
  return hipSuccess;
}

}  // namespace hiprwkv
