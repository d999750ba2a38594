// The head of an RWKV-7 sub-block in one pass: residual addition, LayerNorm, token shift and interpolation
// (reference: /root/reference/src/jaxrwkv/rwkv7.py:8-12, :226-235 / :192-195 and :269-291):
//     xs  = x (+ dx)                                   the residual stream, rounded to the I/O dtype as stored
//     xn  = (xs - mean) rstd ln_w + ln_b               rounded to the I/O dtype, as the reference's layer_norm returns it
//     out_i = xn + (xn_prev - xn) mix_i                xn_prev: the token before, the state row at t = 0, 0 at new_starts
// NOUT = 6 (time mixing), 1 (channel mixing) or 0 (the norm alone: out_0 = xn).  The xn of token (length - 1) mod T of
// every sequence goes to the shift row of the new model state.
//
// Memory bound.  As separate operations (addition, cast to fp32, norm, cast back, gather of the state row, shift and
// interpolation) the six-output head of a layer moved 21 token tensors in bf16 units, this moves 9.  Measured in bf16 at
// B=4 T=1021 C=2048: 37 us (4.1 TB/s) and 24 us with one output, against 72 and 55 us for the separate kernels; backward
// with six cotangents at B=4 T=512 C=768: 13 + 5 us with its reduction, against 66 us for the shift kernel alone.
// A workgroup spans all channels (eight per thread, one 16-byte access in bf16) and walks a run of consecutive tokens,
// GROUP at a time so that the loads of a group are in flight together and a pair of barriers serves all of them; the
// xn of the token before stays in registers.  The first token of a run needs the xn of the one before it, which is
// computed again: with runs of 8 tokens an eighth of the reads of x, which come from L2.
//
// Backward, for cotangents g_i of the outputs, gx of xs and gshift of the shift row:
//     dxn_t = sum_i g_i,t (1 - mix_i) + (t+1 < T and not new_starts[t+1]) sum_i g_i,t+1 mix_i (+ gshift_t)
//     dxs   = rstd (dxn w - mean(dxn w) - xhat mean(dxn w xhat)) + gx         (the cotangent of x and of dx)
//     dmix_i = sum g_i (xn_prev - xn), dln_w = sum dxn xhat, dln_b = sum dxn,  dprev = not new_starts[0] ? sum_i g_i,0 mix_i : 0
// The runs are walked downwards, sums over tokens stay in registers and every workgroup writes them once to a workspace;
// a second small kernel adds the workgroups' rows and rounds to the parameters' type.  (One fp32 atomic per channel and
// workgroup instead, with the zero fills and casts around it, is what the separate shift kernel does: its time is set by
// the atomics from 512 workgroups on.)
#include "common.h"
#include "wkv_args.h"

namespace hiprwkv {

namespace {

constexpr int MAX_WAVES = 8;           // 512 threads: C <= 4096, and 256 registers per thread (with 16 waves the kernels spill)

// G sums over the workgroup at once.  `buf` is not read by anyone when a thread gets here (callers alternate two).
template <int G>
__device__ __forceinline__ void block_sum(float (&x)[G], float* buf) {
  const int row = threadIdx.x >> 4, nrow = blockDim.x >> 4;
#pragma unroll
  for (int j = 0; j < G; ++j) x[j] = row_sum(x[j]);
  if ((threadIdx.x & 15) == 0) {
#pragma unroll
    for (int j = 0; j < G; ++j) buf[row * G + j] = x[j];
  }
  __syncthreads();
#pragma unroll
  for (int j = 0; j < G; ++j) x[j] = 0.f;
  for (int r = 0; r < nrow; r += 4)            // blockDim.x is a multiple of 64
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
      for (int j = 0; j < G; ++j) x[j] += buf[(r + q) * G + j];
}

template <typename T>
__device__ __forceinline__ void zero_or_ld8(const T* p, bool take, float (&o)[8]) {
  if (take) {
    ld8(p, o);
  } else {
#pragma unroll
    for (int c = 0; c < 8; ++c) o[c] = 0.f;
  }
}

// GROUP: tokens whose loads are in flight together, chosen by the launcher so that runs are whole groups (a decode step's token has
// none before it; with groups of four its loads were asked for four times, partial sums of a product among them: 256 rows of 2048
// channels, six outputs 10.7 -> 8.1 us, one 10.4 -> 7.2)
template <typename T, int NOUT, int GROUP>
__global__ __launch_bounds__(64 * MAX_WAVES) void ln_shiftmix_kernel(LnMixArgs A) {
  __shared__ float buf[2][GROUP * MAX_WAVES * 4];
  const int64_t C = A.C, Tn = A.T, total = A.B * A.T;
  const int c8 = threadIdx.x * 8;
  const bool on = c8 < C;
  const int cc = on ? c8 : 0;
  const float invC = 1.f / (float)C;
  Held<T> w, bias, m[NOUT ? NOUT : 1];
  w.load(reinterpret_cast<const T*>(A.ln_w) + cc);
  bias.load(reinterpret_cast<const T*>(A.ln_b) + cc);
#pragma unroll
  for (int i = 0; i < NOUT; ++i) m[i].load(reinterpret_cast<const T*>(A.mix[i]) + cc);
  const int64_t n0 = (int64_t)blockIdx.x * A.run;
  const int64_t n1 = n0 + A.run < total ? n0 + A.run : total;
  // the token before the run, unless the run starts a sequence
  const int64_t first = (NOUT != 0 && n0 % Tn != 0) ? n0 - 1 : n0;
  float before[8];                             // xn of the last token handled
#pragma unroll
  for (int c = 0; c < 8; ++c) before[c] = 0.f;
  for (int64_t g0 = first; g0 < n1; g0 += GROUP) {
    w.pin(); bias.pin();
#pragma unroll
    for (int i = 0; i < NOUT; ++i) m[i].pin();
    float x[GROUP][8], s[GROUP];
#pragma unroll
    for (int j = 0; j < GROUP; ++j) {
      const int64_t n = g0 + j < n1 ? g0 + j : n1 - 1;
      zero_or_ld8(reinterpret_cast<const T*>(A.x) + n * C + cc, on, x[j]);
    }
    if (A.dx != nullptr || A.n_part > 1) {
#pragma unroll
      for (int j = 0; j < GROUP; ++j) {
        const int64_t n = g0 + j < n1 ? g0 + j : n1 - 1;
        float d[8];
        if (A.n_part > 1) {                    // a product's partial sums: dx is their sum, rounded as the product's result
          zero_or_ld8(A.part + n * C + cc, on, d);
#pragma unroll 4
          for (int p = 1; p < A.n_part; ++p) {
            float e[8];
            zero_or_ld8(A.part + (p * total + n) * C + cc, on, e);
#pragma unroll
            for (int c = 0; c < 8; ++c) d[c] += e[c];
          }
#pragma unroll
          for (int c = 0; c < 8; ++c) d[c] = round_io<T>(d[c]);
        } else {
          zero_or_ld8(reinterpret_cast<const T*>(A.dx) + n * C + cc, on, d);
        }
#pragma unroll
        for (int c = 0; c < 8; ++c) x[j][c] = round_io<T>(x[j][c] + d[c]);
        if (on && g0 + j >= n0 && g0 + j < n1) st8(reinterpret_cast<T*>(A.xs) + n * C + cc, x[j]);
      }
    }
#pragma unroll
    for (int j = 0; j < GROUP; ++j) {
      s[j] = 0.f;
#pragma unroll
      for (int c = 0; c < 8; ++c) s[j] += x[j][c];
    }
    block_sum(s, buf[0]);
    float q[GROUP];
#pragma unroll
    for (int j = 0; j < GROUP; ++j) {
      s[j] *= invC;
      q[j] = 0.f;
#pragma unroll
      for (int c = 0; c < 8; ++c) { const float d = x[j][c] - s[j]; q[j] = fmaf(d, d, q[j]); }
      if (!on) q[j] = 0.f;
    }
    block_sum(q, buf[1]);
#pragma unroll
    for (int j = 0; j < GROUP; ++j) {
      const int64_t n = g0 + j;
      if (n >= n1) break;
      const float rstd = rsqrtf(q[j] * invC + A.eps);
      float xn[8];
#pragma unroll
      for (int c = 0; c < 8; ++c) xn[c] = round_io<T>(fmaf((x[j][c] - s[j]) * rstd, w[c], bias[c]));
      if (n >= n0) {
        if (A.stats != nullptr && threadIdx.x == 0) *reinterpret_cast<float2*>(A.stats + 2 * n) = make_float2(s[j], rstd);
        if (on) {
          if (NOUT == 0) {
            st8(reinterpret_cast<T*>(A.out[0]) + n * C + c8, xn);
          } else {
            const int64_t b = n / Tn, t = n - b * Tn;
            if (A.shift != nullptr && t == last_token(A.length, b, Tn)) st8(reinterpret_cast<T*>(A.shift) + b * A.shift_bstride + c8, xn);
            const bool reset = A.ns != nullptr && A.ns[n] != 0;
            float pv[8];
            if (t == 0) ld8(reinterpret_cast<const T*>(A.prev) + b * A.prev_bstride + c8, pv);
#pragma unroll
            for (int c = 0; c < 8; ++c) pv[c] = reset ? 0.f : (t == 0 ? pv[c] : before[c]);
#pragma unroll
            for (int i = 0; i < NOUT; ++i) {
              float o[8];
#pragma unroll
              for (int c = 0; c < 8; ++c) o[c] = fmaf(pv[c] - xn[c], m[i][c], xn[c]);
              st8(reinterpret_cast<T*>(A.out[i]) + n * C + c8, o);
            }
          }
        }
      }
#pragma unroll
      for (int c = 0; c < 8; ++c) before[c] = xn[c];
    }
  }
}

// The loads of a token are requested a token ahead: with the few waves that a SIMD has (512 workgroups at 2048 tokens of 768 channels) a token
// took 6.5 us when its loads were waited for, most of it latency.  E channels a thread: four up to 2048 channels (eight make a token's chain
// of instructions twice as long, spill with six cotangents and leave a quarter of the lanes idle at 768), eight beyond, where four need more
// threads than registers allow.  B=4 T=512 C=768, six cotangents: 26.2 us waiting, two tokens' loads at a time with one (14.7 us); requested ahead
// 22.1 and 10.6 with eight channels, 13.0 and 9.0 with four.
template <typename T, int NOUT, int E>
__global__ __launch_bounds__(64 * MAX_WAVES) void ln_shiftmix_bwd_kernel(LnMixArgs A) {
  constexpr int NG = NOUT ? NOUT : 1;          // cotangent tensors
  constexpr int NP = NOUT + 2;                 // parameter cotangents: mix_0.., ln_w, ln_b
  constexpr bool AHEAD = NOUT != 6 || E != 8;  // there the registers do not hold them
  __shared__ float buf[2][2 * MAX_WAVES * 4];
  const int64_t C = A.C, Tn = A.T, total = A.B * A.T;
  const int ce = threadIdx.x * E;
  const bool on = ce < C;
  const int cc = on ? ce : 0;
  const float invC = 1.f / (float)C;
  float acc[NP][E];
  HeldOf<T, E> w, bias, m[NG];
  w.load(reinterpret_cast<const T*>(A.ln_w) + cc);
  bias.load(reinterpret_cast<const T*>(A.ln_b) + cc);
#pragma unroll
  for (int i = 0; i < NOUT; ++i) m[i].load(reinterpret_cast<const T*>(A.mix[i]) + cc);
#pragma unroll
  for (int i = 0; i < NP; ++i)
#pragma unroll
    for (int c = 0; c < E; ++c) acc[i][c] = 0.f;
  const int64_t n0 = (int64_t)blockIdx.x * A.run;
  const int64_t n1 = (n0 + A.run < total ? n0 + A.run : total) - 1;      // last token of the run
  // a token's cotangents and the one of xs, xs and its statistics of the token before; threads beyond C read channels that others have
  HeldOf<T, E> g[NG], gx, x0, x1;
  float2 st0, st1;
  auto request = [&](int64_t n) {
#pragma unroll
    for (int i = 0; i < NG; ++i) g[i].load(reinterpret_cast<const T*>(A.g[i]) + n * C + cc);
    if (A.gx != nullptr) gx.load(reinterpret_cast<const T*>(A.gx) + n * C + cc);
  };
  auto request_x = [&](int64_t n) {
    n = n < 0 ? 0 : n;
    x1.load(reinterpret_cast<const T*>(A.xs) + n * C + cc);
    st1 = *reinterpret_cast<const float2*>(A.stats + 2 * n);
  };
  request_x(n1);
  x0 = x1; st0 = st1;
  // sum_i g_i mix_i of the token after, if that token takes its shifted value from the one before it
  float gm_next[E];
#pragma unroll
  for (int c = 0; c < E; ++c) gm_next[c] = 0.f;
  if (NOUT != 0 && n1 + 1 < total && (n1 + 1) % Tn != 0 && !(A.ns != nullptr && A.ns[n1 + 1] != 0)) {
    request(n1 + 1);
#pragma unroll
    for (int i = 0; i < NOUT; ++i)
#pragma unroll
      for (int c = 0; c < E; ++c) gm_next[c] = fmaf(g[i][c], m[i][c], gm_next[c]);
  }
  if (AHEAD) request(n1);
  request_x(n1 - 1);
  int ph = 0;
  int64_t b = n1 / Tn, t = n1 - b * Tn;
  for (int64_t n = n1; n >= n0; --n, ph ^= 1) {
    if (!AHEAD) request(n);
    w.pin(); bias.pin();
#pragma unroll
    for (int i = 0; i < NOUT; ++i) m[i].pin();
    const float rstd = st0.y;
    const bool reset = NOUT != 0 && A.ns != nullptr && A.ns[n] != 0;
    float xh[E], dxn[E], red[2];
    x0.pin();
#pragma unroll
    for (int c = 0; c < E; ++c) xh[c] = (x0[c] - st0.x) * rstd;
    if (NOUT == 0) {
#pragma unroll
      for (int c = 0; c < E; ++c) dxn[c] = g[0][c];
    } else {
      float pv[E], d[E], gm[E];
      if (t == 0) ld_n(reinterpret_cast<const T*>(A.prev) + b * A.prev_bstride + cc, pv);
#pragma unroll
      for (int c = 0; c < E; ++c) {
        const float xn = round_io<T>(fmaf(xh[c], w[c], bias[c]));
        const float xb = round_io<T>(fmaf((x1[c] - st1.x) * st1.y, w[c], bias[c]));
        d[c] = (reset ? 0.f : (t == 0 ? pv[c] : xb)) - xn;
        gm[c] = 0.f;
        dxn[c] = 0.f;
      }
#pragma unroll
      for (int i = 0; i < NOUT; ++i) {
        g[i].pin();
#pragma unroll
        for (int c = 0; c < E; ++c) {
          const float gi = g[i][c];
          dxn[c] += gi;
          gm[c] = fmaf(gi, m[i][c], gm[c]);
          acc[i][c] = fmaf(gi, d[c], acc[i][c]);
        }
      }
      const bool last_of_seq = t == Tn - 1;
#pragma unroll
      for (int c = 0; c < E; ++c) dxn[c] += (last_of_seq ? 0.f : gm_next[c]) - gm[c];
      if (A.gshift != nullptr && t == last_token(A.length, b, Tn)) {
        float gs[E];
        ld_n(reinterpret_cast<const T*>(A.gshift) + b * C + cc, gs);
#pragma unroll
        for (int c = 0; c < E; ++c) dxn[c] += gs[c];
      }
#pragma unroll
      for (int c = 0; c < E; ++c) gm_next[c] = reset ? 0.f : gm[c];
      if (t == 0 && on && A.dprev != nullptr) st_n(reinterpret_cast<T*>(A.dprev) + b * C + ce, gm_next);
    }
    // what the token before needs, while the sums below wait for each other
    const HeldOf<T, E> gx_now = gx;
    if (AHEAD && n > n0) request(n - 1);
    x0 = x1; st0 = st1;
    if (NOUT != 0 || n > n0) request_x(n - 2);
    red[0] = red[1] = 0.f;
#pragma unroll
    for (int c = 0; c < E; ++c) {
      acc[NOUT][c] = fmaf(dxn[c], xh[c], acc[NOUT][c]);
      acc[NOUT + 1][c] += dxn[c];
      const float gw = dxn[c] * w[c];
      red[0] += gw;
      red[1] = fmaf(gw, xh[c], red[1]);
    }
    if (!on) red[0] = red[1] = 0.f;
    block_sum(red, buf[ph]);
    if (on) {
      const float s1 = red[0] * invC, s2 = red[1] * invC;
      float o[E];
#pragma unroll
      for (int c = 0; c < E; ++c) o[c] = (A.gx != nullptr ? gx_now[c] : 0.f) + rstd * (dxn[c] * w[c] - s1 - xh[c] * s2);
      st_n(reinterpret_cast<T*>(A.dxs) + n * C + ce, o);
    }
    if (--t < 0) { t = Tn - 1; --b; }
  }
  if (on) {
#pragma unroll
    for (int i = 0; i < NP; ++i) st_n(A.part + ((size_t)blockIdx.x * NP + i) * C + ce, acc[i]);
  }
}

// out_k[c] = sum over p of part[p][k][c]; a workgroup owns 64 consecutive of the nk*C columns, its sixteen waves every sixteenth row.
// Bound by the wait for the rows, eight of a wave's in flight; with four waves and four rows a training step of
// 12 layers of 768 channels and 2048 tokens (its 50 sums, up to 512 rows of 6144 columns) took 8.6 us each on average, then 4.8, about 2 of
// them the launch.  Three of a layer's four go into one now (26 launches: the step 6341 -> 6237 us).
constexpr int REDUCE_WAVES = 16;
template <typename T>
__global__ __launch_bounds__(64 * REDUCE_WAVES) void reduce_parts_kernel(ReduceJobs J) {
  __shared__ float red[REDUCE_WAVES][64];
  int64_t block = blockIdx.x;
  int ji = 0;
  for (; ji + 1 < J.n; ++ji) {
    const int64_t blocks = ((int64_t)J.job[ji].nk * J.job[ji].C + 63) / 64;
    if (block < blocks) break;
    block -= blocks;
  }
  const ReduceArgs& A = J.job[ji];
  const int64_t cols = (int64_t)A.nk * A.C;
  const int64_t col = block * 64 + (threadIdx.x & 63);
  const int wv = threadIdx.x >> 6;
  float s[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  if (col < cols) {
    const float* p = A.part + col;
    int64_t r = wv;
    for (; r + 7 * REDUCE_WAVES < A.rows; r += 8 * REDUCE_WAVES)
#pragma unroll
      for (int i = 0; i < 8; ++i) s[i] += p[(r + i * REDUCE_WAVES) * cols];
#pragma unroll
    for (int i = 0; i < 7; ++i)
      if (r + i * REDUCE_WAVES < A.rows) s[i] += p[(r + i * REDUCE_WAVES) * cols];
  }
  red[wv][threadIdx.x & 63] = ((s[0] + s[1]) + (s[2] + s[3])) + ((s[4] + s[5]) + (s[6] + s[7]));
  __syncthreads();
  if (wv == 0 && col < cols) {
    float t[4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
      t[i] = (red[4 * i][threadIdx.x] + red[4 * i + 1][threadIdx.x]) + (red[4 * i + 2][threadIdx.x] + red[4 * i + 3][threadIdx.x]);
    st_f(reinterpret_cast<T*>(A.out[col / A.C]) + col % A.C, (t[0] + t[1]) + (t[2] + t[3]));
  }
}

}  // namespace

hipError_t launch_reduce_parts(int io_f32, const ReduceJobs& J, hipStream_t stream) {
  int64_t blocks = 0;
  for (int i = 0; i < J.n; ++i) blocks += ((int64_t)J.job[i].nk * J.job[i].C + 63) / 64;
  const dim3 grid((unsigned)blocks), block(64 * REDUCE_WAVES);
  if (io_f32) hipLaunchKernelGGL(reduce_parts_kernel<float>, grid, block, 0, stream, J);
  else hipLaunchKernelGGL(reduce_parts_kernel<bf16_t>, grid, block, 0, stream, J);
  return hipGetLastError();
}
hipError_t reduce_parts(int io_f32, const ReduceArgs& A, ReduceJobs* later, hipStream_t stream) {
  if (later != nullptr) {
    later->job[later->n++] = A;
    return hipSuccess;
  }
  ReduceJobs J;
  memset(&J, 0, sizeof(J));
  J.n = 1;
  J.job[0] = A;
  return launch_reduce_parts(io_f32, J, stream);
}

// Tokens per workgroup.  Forward: 8 keep the re-reading of the token before a run at an eighth; shorter runs while that
// leaves fewer than 1024 workgroups.
int64_t ln_shiftmix_run(int64_t rows) {
  const int64_t run = rows / 1024;
  return run < 1 ? 1 : run > 8 ? 8 : run;
}
// Backward: a workgroup writes NP rows of C sums, so runs grow with the token count (at most about 1024 workgroups).
int64_t ln_shiftmix_bwd_run(int64_t rows) {
  const int64_t run = (rows + 1023) / 1024;
  return run < 4 ? 4 : (run + 1) / 2 * 2;
}

#define HIPRWKV_BLOCK_DISPATCH(KERNEL, ...)                                                                          \
  if (io_f32) {                                                                                                     \
    if (n_out == 6) hipLaunchKernelGGL((KERNEL<float, 6 __VA_ARGS__>), grid, block, 0, stream, A);                  \
    else if (n_out == 1) hipLaunchKernelGGL((KERNEL<float, 1 __VA_ARGS__>), grid, block, 0, stream, A);             \
    else hipLaunchKernelGGL((KERNEL<float, 0 __VA_ARGS__>), grid, block, 0, stream, A);                             \
  } else {                                                                                                          \
    if (n_out == 6) hipLaunchKernelGGL((KERNEL<bf16_t, 6 __VA_ARGS__>), grid, block, 0, stream, A);                 \
    else if (n_out == 1) hipLaunchKernelGGL((KERNEL<bf16_t, 1 __VA_ARGS__>), grid, block, 0, stream, A);            \
    else hipLaunchKernelGGL((KERNEL<bf16_t, 0 __VA_ARGS__>), grid, block, 0, stream, A);                            \
  }
#define HIPRWKV_COMMA ,

hipError_t launch_ln_shiftmix(int io_f32, int n_out, LnMixArgs A, hipStream_t stream) {
  A.run = ln_shiftmix_run(A.B * A.T);
  const dim3 grid((unsigned)((A.B * A.T + A.run - 1) / A.run)), block((unsigned)((A.C / 8 + 63) / 64 * 64));
  // a run and, where tokens are shifted, the one before it; runs of 3 and 8 leave a rest (9 tokens: three groups of three)
  const int64_t tokens = A.run + (n_out != 0 && A.T > 1 ? 1 : 0);
  if (tokens == 1) { HIPRWKV_BLOCK_DISPATCH(ln_shiftmix_kernel, HIPRWKV_COMMA 1) }
  else if (tokens == 2) { HIPRWKV_BLOCK_DISPATCH(ln_shiftmix_kernel, HIPRWKV_COMMA 2) }
  else if (tokens % 3 == 0) { HIPRWKV_BLOCK_DISPATCH(ln_shiftmix_kernel, HIPRWKV_COMMA 3) }
  else { HIPRWKV_BLOCK_DISPATCH(ln_shiftmix_kernel, HIPRWKV_COMMA 4) }
  return hipGetLastError();
}

hipError_t launch_ln_shiftmix_bwd(int io_f32, int n_out, LnMixArgs A, void* const* dparam, hipStream_t stream, ReduceJobs* later) {
  A.run = ln_shiftmix_bwd_run(A.B * A.T);
  const bool four = A.C <= 4 * 64 * MAX_WAVES;
  const dim3 grid((unsigned)((A.B * A.T + A.run - 1) / A.run)), block((unsigned)((A.C / (four ? 4 : 8) + 63) / 64 * 64));
  if (four) { HIPRWKV_BLOCK_DISPATCH(ln_shiftmix_bwd_kernel, HIPRWKV_COMMA 4) }
  else { HIPRWKV_BLOCK_DISPATCH(ln_shiftmix_bwd_kernel, HIPRWKV_COMMA 8) }
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  ReduceArgs R;
  R.part = A.part; R.rows = grid.x; R.nk = n_out + 2; R.C = A.C;
  for (int i = 0; i < n_out + 2; ++i) R.out[i] = dparam[i];
  return reduce_parts(io_f32, R, later, stream);
}

}  // namespace hiprwkv
