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
// Measured (eager, host included), general path -> separate launches -> now: 12 layers of 768 channels, one user 5.4 ms -> 0.57 -> 0.41
// a step, two 0.43, 16 0.61 -> 0.54; 24 layers of 2048 channels, one user 1.61 -> 1.36, 16 1.89 -> 1.69, 256 10.9 -> 3.6 -> 3.2 (7.5
// with the weight-streaming product alone: 51 us a launch at 256 rows, 18 tiled).  Norms inside the products: one user 0.50 -> 0.42 (12 x
// 768), three as long as before; second low-rank products inside the recurrence 0.42 -> 0.41.
// References: /root/reference/src/jaxrwkv/rwkv7.py:190-198, :223-267, :269-291.  Products accumulate in fp32 and are rounded
// once; the values between the gates, the recurrence and the group norm are rounded where the general path stores them.
#include "chunk_common.h"
#include "wkv_args.h"

namespace hiprwkv {

namespace {

// ---------------------------------------------------------------------------------------------------------------
// sum over the wave, delivered to every lane
__device__ __forceinline__ float wave_sum(float x) {
#pragma unroll
  for (int o = 32; o; o >>= 1) x += __shfl_xor(x, o, 64);
  return x;
}

struct CoreArgs {
  int64_t T, H;
  const bf16_t *r, *k, *v, *vf, *xw, *xa, *xv, *g;          // (B,T,H,64); vf null: the first layer
  const bf16_t *hid[4], *w2[4];   // or the factors of xw, xa, g, xv: (B,T,d) and (d,H,64), d a multiple of 32
  int d[4];
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
// LORA: the second low-rank products are made here, each workgroup its head's 64 columns (one launch less, but their weights are read
// once per sequence).  Eight lanes read a row of a factor, a wave eight rows, the requests of 128 rows of all four together.
template <bool LORA>
__global__ __launch_bounds__(256, LORA ? 1 : 6) void decode_core_kernel(CoreArgs A) {
  __shared__ __align__(16) float lora[LORA ? 16 : 1][4][64];      // [wave, 16 of its lanes][factor][channel]; then lora[0] the results
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
    float v = 0.f, gate = 0.f, bonus = 0.f, k = 0.f, r = 0.f, vf = 0.f, xw = 0.f, xa = 0.f, xv = 0.f;
    const size_t el = (((size_t)b * A.T + t) * A.H + h) * 64 + tid;
    if (lead) {
      k = ld_f(A.k + el); r = ld_f(A.r + el); v = ld_f(A.v + el);
      if (A.vf != nullptr) vf = ld_f(A.vf + el);
      if (!LORA) {
        xw = ld_f(A.xw + el); xa = ld_f(A.xa + el); gate = ld_f(A.g + el);
        if (A.vf != nullptr) xv = ld_f(A.xv + el);
      }
    }
    if (LORA) {
      const int wave = tid >> 6, lane = tid & 63, first = 8 * wave + (lane >> 3), c8 = 8 * (lane & 7);
      const size_t row = (size_t)b * A.T + t;
      float acc[4][8];
#pragma unroll
      for (int f = 0; f < 4; ++f)
#pragma unroll
        for (int c = 0; c < 8; ++c) acc[f][c] = 0.f;
      for (int j0 = 0; j0 < A.d[0] || j0 < A.d[1] || j0 < A.d[2] || j0 < A.d[3]; j0 += 128) {
        uint4 w[4][4];
        float x[4][4];
#pragma unroll
        for (int f = 0; f < 4; ++f)
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            const int j = j0 + 32 * u + first, jj = j < A.d[f] ? j : A.d[f] - 1;      // no factor (d = 0): that of the decay, unused
            w[f][u] = *reinterpret_cast<const uint4*>(A.w2[f] + ((size_t)(jj < 0 ? 0 : jj) * A.H + h) * 64 + c8);
            x[f][u] = ld_f(A.hid[f] + row * A.d[f] + (jj < 0 ? 0 : jj));
          }
#pragma unroll
        for (int f = 0; f < 4; ++f)
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            // beyond the factor the last row is read again: both are cleared, either may not be finite
            const uint32_t have = j0 + 32 * u < A.d[f] ? 0xffffffffu : 0u;
            const float xs = __uint_as_float(__float_as_uint(x[f][u]) & have);
            const uint32_t q[4] = {w[f][u].x & have, w[f][u].y & have, w[f][u].z & have, w[f][u].w & have};
#pragma unroll
            for (int c = 0; c < 4; ++c) {
              acc[f][2 * c] = fmaf(xs, __uint_as_float(q[c] << 16), acc[f][2 * c]);
              acc[f][2 * c + 1] = fmaf(xs, __uint_as_float(q[c] & 0xffff0000u), acc[f][2 * c + 1]);
            }
          }
      }
#pragma unroll
      for (int f = 0; f < 4; ++f) {
#pragma unroll
        for (int c = 0; c < 8; ++c)
          acc[f][c] += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(acc[f][c]), 0x128, 0xf, 0xf, false));   // row_ror:8
        if ((lane & 8) == 0) st8(&lora[tid >> 4][f][c8], acc[f]);
      }
      __syncthreads();
      float s = 0.f;
#pragma unroll
      for (int u = 0; u < 16; ++u) s += lora[u][wave][lane];
      __syncthreads();
      lora[0][wave][lane] = rnd(s);
      __syncthreads();
      if (lead) { xw = lora[0][0][tid]; xa = lora[0][1][tid]; gate = lora[0][2][tid]; xv = lora[0][3][tid]; }
    }
    if (lead) {
      if (A.vf != nullptr) v = rnd(fmaf(vf - v, sigmoidf(v0 + xv), v));
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
    CoreArgs A;
    memset(&A, 0, sizeof(A));
    if (few) {
      const int of_mix[7] = {0, 2, 3, 1, 4, 5, 3};
      for (int i = 0; i < G.n_jobs; ++i) G.job[i].aux = mv[of_mix[i]];
      HIPRWKV_TRY(launch_head_gemm(ln1, G, stream));
      const bf16_t* const second[4] = {layer(D.w2, l, C * D.d_decay), layer(D.a2, l, C * D.d_aaa), layer(D.g2, l, C * D.d_gate),
                                       layer(l ? D.v2 : D.w2, l, C * D.d_mv)};
      const bf16_t* const first[4] = {hw, ha, hg, l ? hv : hw};
      const int64_t d[4] = {D.d_decay, D.d_aaa, D.d_gate, l ? D.d_mv : 0};
      for (int i = 0; i < 4; ++i) { A.hid[i] = first[i]; A.w2[i] = second[i]; A.d[i] = (int)d[i]; }
    } else {
      HIPRWKV_TRY(launch_gemm(G, 1, stream));
      G.n_jobs = 0;
      add(hw, layer(D.w2, l, C * D.d_decay), xw, D.d_decay, C, 1, GEMM_ACT_NONE);
      add(ha, layer(D.a2, l, C * D.d_aaa), xa, D.d_aaa, C, 1, GEMM_ACT_NONE);
      add(hg, layer(D.g2, l, C * D.d_gate), g, D.d_gate, C, 1, GEMM_ACT_NONE);
      if (l) add(hv, layer(D.v2, l, C * D.d_mv), xv, D.d_mv, C, 1, GEMM_ACT_NONE);
      HIPRWKV_TRY(launch_gemm(G, 1, stream));
    }
    A.T = D.T; A.H = D.H;
    A.r = r; A.k = k; A.v = vl; A.vf = l ? vf : nullptr; A.xw = xw; A.xa = xa; A.xv = xv; A.g = g;
    A.w0 = layer(D.w0, l, C); A.a0 = layer(D.a0, l, C); A.v0 = layer(D.v0, l, C);
    A.k_k = layer(D.k_k, l, C); A.k_a = layer(D.k_a, l, C); A.r_k = layer(D.r_k, l, C);
    A.ln_w = layer(D.lnx_w, l, C); A.ln_b = layer(D.lnx_b, l, C); A.eps = 64e-5f;
    A.s = st + (size_t)l * row_state + 2 * C; A.new_s = nst + (size_t)l * row_state + 2 * C; A.bstride = seq_state;
    A.length = D.length; A.ns = D.new_starts; A.flags = (unsigned)D.flags; A.y = y;
    if (few) hipLaunchKernelGGL(decode_core_kernel<true>, dim3((unsigned)(D.B * D.H)), dim3(256), 0, stream, A);
    else hipLaunchKernelGGL(decode_core_kernel<false>, dim3((unsigned)(D.B * D.H)), dim3(256), 0, stream, A);
    HIPRWKV_TRY(hipGetLastError());
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
