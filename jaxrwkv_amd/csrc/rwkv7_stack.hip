// The stack of RWKV-7 blocks over whole sequences, forward and backward, launched layer by layer from native code (bf16; references:
// /root/reference/src/jaxrwkv/rwkv7.py:190-198, :223-291).
// What bounds it: launched from Python a layer costs the host 0.3 ms forward and 0.8 ms backward, whatever the rows (12 layers of 768
// channels, 4 x 512 tokens, forward and backward: 12.9 ms, of which the GPU worked 9.9; 4 x 64 tokens as long).  From here a launch
// costs 2 to 3 us and there are fewer of them: products that do not wait for each other share one (rwkv7_gemm.hip), relu^2 and its
// derivative are applied where a product is stored, and the cotangents that several layers or kernels give are added where one is made.
// Forward and backward now: 4 x 512 tokens 12.7 -> 6.8 ms (the GPU's time), 1 x 23 tokens 11.0 -> 3.0; 8 layers of 1024 channels,
// 4 x 19 tokens 8.2 -> 2.5; forward alone of 24 layers of 2048 channels, 4 x 250 tokens 7.7 -> 5.7, 3 x 39 7.8 -> 2.4.
//   forward:  norm, shift, six interpolations | r, k, v, first low-rank factors | second ones, gates | recurrence | group norm, bonus,
//             gate | output | norm, shift, interpolation | key | value
//   backward: value | key | norm | output | group norm | recurrence | gates | r, k, v, low-rank factors (two launches) | norm, each
//             product's two cotangents in one launch
// Values are rounded where the separate operations store them, and a cotangent that is a sum of several once instead of after each.
#include "common.h"
#include "wkv_args.h"

namespace hiprwkv {

namespace {

constexpr float EPS = 1e-5f, EPS_X = 64e-5f;

// Pieces of one allocation.  The large ones start 128 bytes further apart each, modulo 1 KiB: rows of several arrays at one address
// modulo 1 KiB compete for the same part of the memory system (ops._PHASES).
struct Arena {
  char* base;
  size_t used = 0;
  int n = 0;
  template <typename T = bf16_t>
  T* take(size_t elements) {
    used = (used + 1023) / 1024 * 1024 + 128 * (size_t)(n++ % 8);
    char* const p = base + used;
    used += elements * sizeof(T);
    return reinterpret_cast<T*>(p);
  }
};

// What the backward reads of a layer's forward, without what at_layer puts in its place.  Without a backward to come all layers use the
// same memory (`l` then is any layer between the first and the last).
struct Layer {
  bf16_t *x, *mix[6], *r, *k, *v, *hid[4], *lora[4], *w, *k2, *v2, *a, *b, *yw, *y, *x2, *xk2, *ff, *fr;      // hid, lora: w, a, g, v
  float *stats1, *stats2;
  void* sa;
};
constexpr int MIX_R = 0, MIX_W = 1, MIX_K = 2, MIX_V = 3, MIX_A = 4, MIX_G = 5;
constexpr int LORA_MIX[4] = {MIX_W, MIX_A, MIX_G, MIX_V};

struct Stack {
  const Rwkv7Stack& D;
  size_t rows, C, F, d[4];
  explicit Stack(const Rwkv7Stack& D_) : D(D_), rows((size_t)D_.B * D_.T), C(D_.C), F(D_.F) {
    d[0] = D.d_decay; d[1] = D.d_aaa; d[2] = D.d_gate; d[3] = D.d_mv;
  }
  size_t ends_bytes() const { return hiprwkv_wkv7_ends_bytes(HIPRWKV_BF16, D.B, D.T, D.H, 64); }
  Layer layer(Arena& A, bool keep, int64_t l) const {
    Layer S;
    memset(&S, 0, sizeof(S));
    const size_t n = rows * C;
    const bool first = keep && l == 0, last = keep && l == D.L - 1;
    if (!first) S.x = A.take(n);
    for (auto& m : S.mix) m = A.take(n);
    S.r = A.take(n); S.k = A.take(n); S.v = A.take(n);
    for (int i = 0; i < (first ? 3 : 4); ++i) {
      S.hid[i] = A.take(rows * d[i]);
      if (keep || i == 2) S.lora[i] = A.take(n);           // the gate's alone is read again in the forward
    }
    S.w = A.take(n); S.k2 = A.take(n); S.a = A.take(n); S.b = A.take(n);
    if (!first) S.v2 = A.take(n);
    S.yw = A.take(n); S.y = A.take(n); S.xk2 = A.take(n); S.fr = A.take(rows * F);
    if (!last) S.x2 = A.take(n);
    if (keep) {
      S.ff = A.take(rows * F);
      S.stats1 = A.take<float>(2 * rows); S.stats2 = A.take<float>(2 * rows);
      S.sa = A.take(n);
    }
    return S;
  }
};
// layer l as the forward and the backward see it: the first has no value residual and reads the call's x, the last returns its x2
Layer at_layer(const Stack& K, Layer S, int64_t l, const bf16_t* v_first) {
  if (l == 0) { S.x = static_cast<bf16_t*>(const_cast<void*>(K.D.x)); S.v = const_cast<bf16_t*>(v_first); S.v2 = S.v; }
  if (l == K.D.L - 1) S.x2 = static_cast<bf16_t*>(K.D.xs);
  return S;
}

struct Products {
  GemmArgs G;
  Products() { memset(&G, 0, sizeof(G)); }
  // out (M, N) = f(x w): x (M, K), or with km (K, M); w (N, K), or with kn (K, N)
  GemmJob& add(void* out, const void* x, const void* w, size_t M, size_t N, size_t K, int km, int kn, int act = 0, const void* aux = nullptr) {
    GemmJob& J = G.job[G.n_jobs++];
    J.out = out; J.x = x; J.w = w; J.M = (int)M; J.N = (int)N; J.K = (int)K; J.km = km; J.kn = kn; J.act = act; J.aux = aux;
    return J;
  }
  hipError_t launch(hipStream_t stream) { return G.n_jobs ? launch_gemm(G, 1, stream) : hipSuccess; }
};

struct Forward {
  Layer one;                 // without a backward to come
  bf16_t *v_first, *dx;
  float* parts;              // a product's partial sums
  void* wkv;
  size_t wkv_bytes;
  Forward(const Stack& K, Arena& A) {
    const size_t n = K.rows * K.C;
    one = K.D.saved == nullptr ? K.layer(A, false, 0) : Layer();
    v_first = K.D.saved == nullptr ? A.take(n) : nullptr;
    dx = A.take(n);
    const int out = gemm_split((int)K.rows, K.C, K.C), val = gemm_split((int)K.rows, K.F, K.C), most = out > val ? out : val;
    parts = A.take<float>(most > 1 ? n * most : 0);
    wkv_bytes = hiprwkv_wkv7_fwd_workspace_bytes(HIPRWKV_BF16, K.D.B, K.D.T, K.D.H, 64);
    wkv = wkv_bytes ? A.take<char>(wkv_bytes) : nullptr;
  }
};

struct Backward {
  bf16_t *gff, *gxk2, *dx2, *dx, *gy, *gyw, *gr1, *gk1, *gv1, *gg, *gr2, *gw, *gk2, *gv2, *ga, *gb, *gs, *gr, *dl[4], *dk, *dv, *dvf,
      *dmix[6], *dh[4];
  float *part, *parts[3];      // the first head's; channel mixing's head, group norm, gates
  void *wkv, *ends;
  size_t wkv_bytes;
  Backward(const Stack& K, Arena& A) {
    const auto& D = K.D;
    const size_t n = K.rows * K.C;
    // gy and gyw come when gff has been read for the last time, the six of dmix when the recurrence's cotangents have
    gff = A.take(K.rows * K.F > 2 * n + 1024 ? K.rows * K.F : 2 * n + 1024);
    gy = gff; gyw = gff + (n + 511) / 512 * 512 + 64;
    for (bf16_t** p : {&gxk2, &dx2, &dx, &gr1, &gk1, &gv1, &gg, &gr2, &gw, &gk2, &gv2, &ga, &gb, &gr, &dk, &dv, &dvf}) *p = A.take(n);
    bf16_t* const over[6] = {gr2, gw, gk2, gv2, ga, gb};
    for (int i = 0; i < 6; ++i) dmix[i] = over[i];
    gs = A.take((size_t)D.B * D.H * 4096);
    for (int i = 0; i < 4; ++i) { dl[i] = i == 2 ? gg : A.take(n); dh[i] = A.take(K.rows * K.d[i]); }
    // workgroups' rows of sums: three kernels' side by side, which one launch adds up, then the first head's in the same memory (more of them
    // than of the three together, but for models of a head or two)
    const size_t bytes = hiprwkv_rwkv7_ln_shiftmix_bwd_workspace_bytes(D.B, D.T, D.C, 6);
    const size_t each[3] = {hiprwkv_rwkv7_ln_shiftmix_bwd_workspace_bytes(D.B, D.T, D.C, 1),
                            hiprwkv_rwkv7_postmix_bwd2_workspace_bytes(D.B * D.T, D.H, 64),
                            hiprwkv_rwkv7_pre_bwd_workspace_bytes(D.B * D.T, D.H, 64)};
    size_t at[4] = {0, 0, 0, 0};
    for (int i = 0; i < 3; ++i) at[i + 1] = at[i] + (each[i] + 255) / 256 * 256;
    char* const rows = A.take<char>(bytes > at[3] ? bytes : at[3]);
    part = reinterpret_cast<float*>(rows);
    for (int i = 0; i < 3; ++i) parts[i] = reinterpret_cast<float*>(rows + at[i]);
    wkv_bytes = K.ends_bytes() ? hiprwkv_wkv7_bwd_ends_workspace_bytes(HIPRWKV_BF16, D.B, D.T, D.H, 64)
                               : hiprwkv_wkv7_bwd_workspace_bytes(D.B, D.T, D.H, 64);
    wkv = A.take<char>(wkv_bytes);
    ends = K.ends_bytes() ? A.take<char>(K.ends_bytes()) : nullptr;      // in bf16 the recurrence's backward fills it itself
  }
};

const bf16_t* of(const void* p, int64_t l, size_t n) { return static_cast<const bf16_t*>(p) + (size_t)l * n; }
void* to(const void* p, int64_t l, size_t n) { return const_cast<bf16_t*>(of(p, l, n)); }      // of a parameter's cotangent

}  // namespace

size_t rwkv7_stack_saved(const Rwkv7Stack& D, int64_t l) {
  Arena A{nullptr};
  Stack(D).layer(A, true, l);
  return A.used;
}
size_t rwkv7_stack_workspace(const Rwkv7Stack& D, bool backward) {
  Arena A{nullptr};
  const Stack K(D);
  if (backward) Backward(K, A);
  else Forward(K, A);
  return A.used;
}

#define HIPRWKV_TRY(x) if ((e = (x)) != hipSuccess) return HIPRWKV_OK
#define HIPRWKV_TRY_RC(x) if (const int rc = (x)) return rc

int launch_rwkv7_stack_fwd(const Rwkv7Stack& D, hipStream_t stream, hipError_t& e) {
  const Stack K(D);
  const size_t C = K.C, F = K.F, M = K.rows, row_state = 66 * C;
  const bool keep = D.saved != nullptr;
  Arena A{static_cast<char*>(D.workspace)};
  const Forward W(K, A);
  const auto& P = D.param;
  const bf16_t* const st = static_cast<const bf16_t*>(D.state);
  bf16_t* const nst = static_cast<bf16_t*>(D.new_state);
  const bf16_t *x = static_cast<const bf16_t*>(D.x), *v_first = W.v_first;
  const int split_out = gemm_split((int)M, C, C), split_val = gemm_split((int)M, F, C);
  int n_part = 0;                                // of the dx to come: none, itself, or its partial sums
  auto head = [&](int n_out, const void* in, bf16_t* sum, const void* w, const void* b, int64_t l, int srow, const void* const* mix,
                  bf16_t* const* out, float* stats) {
    LnMixArgs N;
    memset(&N, 0, sizeof(N));
    N.B = D.B; N.T = D.T; N.C = D.C; N.eps = EPS; N.ns = D.new_starts; N.length = D.length;
    N.x = in; N.xs = sum; N.ln_w = w; N.ln_b = b; N.stats = stats;
    if (n_part == 1) N.dx = W.dx;
    if (n_part > 1) { N.part = W.parts; N.n_part = n_part; }
    N.prev = st + l * row_state + srow * C; N.prev_bstride = D.L * row_state;
    N.shift = nst + l * row_state + srow * C; N.shift_bstride = D.L * row_state;
    for (int i = 0; i < n_out; ++i) { N.mix[i] = mix[i]; N.out[i] = out[i]; }
    return launch_ln_shiftmix(0, n_out, N, stream);
  };
  for (int64_t l = 0; l < D.L; ++l) {
    Arena own{keep ? static_cast<char*>(D.saved[l]) : nullptr};
    Layer S = keep ? K.layer(own, true, l) : W.one;
    if (l == 0 && keep) v_first = S.v;
    S = at_layer(K, S, l, v_first);
    const void* const mixv[6] = {of(P.x_r, l, C), of(P.x_w, l, C), of(P.x_k, l, C), of(P.x_v, l, C), of(P.x_a, l, C), of(P.x_g, l, C)};
    HIPRWKV_TRY(head(6, x, S.x, of(P.ln1_w, l, C), of(P.ln1_b, l, C), l, 1, mixv, S.mix, S.stats1));
    const int n_lora = l ? 4 : 3;
    const void* const f1[4] = {of(P.w1, l, C * K.d[0]), of(P.a1, l, C * K.d[1]), of(P.g1, l, C * K.d[2]), of(P.v1, l, C * K.d[3])};
    const void* const f2[4] = {of(P.w2, l, C * K.d[0]), of(P.a2, l, C * K.d[1]), of(P.g2, l, C * K.d[2]), of(P.v2, l, C * K.d[3])};
    const int act[4] = {GEMM_ACT_TANH, GEMM_ACT_NONE, GEMM_ACT_SIGMOID, GEMM_ACT_NONE};
    {
      Products G;
      G.add(S.r, S.mix[MIX_R], of(P.receptance, l, C * C), M, C, C, 0, 0);
      G.add(S.k, S.mix[MIX_K], of(P.key, l, C * C), M, C, C, 0, 0);
      G.add(S.v, S.mix[MIX_V], of(P.value, l, C * C), M, C, C, 0, 0);
      for (int i = 0; i < n_lora; ++i) G.add(S.hid[i], S.mix[LORA_MIX[i]], f1[i], M, K.d[i], C, 0, 1, act[i]);
      HIPRWKV_TRY(G.launch(stream));
    }
    LoraPreArgs X;
    memset(&X, 0, sizeof(X));
    for (int i = 0; i < n_lora; ++i) {
      X.hid[i] = S.hid[i]; X.w2[i] = f2[i]; X.d[i] = (int)K.d[i];
      X.out[i] = keep || i == 2 ? S.lora[i] : nullptr;
    }
    PreArgs& R = X.P;
    R.rows = M; R.H = D.H;
    R.k = S.k;
    if (l) { R.v = S.v; R.vf = v_first; R.v0 = of(P.v0, l, C); R.v_out = S.v2; }
    R.w0 = of(P.w0, l, C); R.a0 = of(P.a0, l, C); R.k_k = of(P.k_k, l, C); R.k_a = of(P.k_a, l, C);
    R.w = S.w; R.k_out = S.k2; R.a_out = S.a; R.b_out = S.b;
    HIPRWKV_TRY(launch_rwkv7_lora_pre(X, stream));
    const size_t states = (size_t)D.B * 64 * C;
    HIPRWKV_TRY_RC(hiprwkv_wkv7_fwd_parts(stream, HIPRWKV_BF16, HIPRWKV_BF16, D.B, D.T, D.H, 64, S.w, S.r, S.k2, S.v2, S.a, S.b,
                                         of(D.s, l, states), reinterpret_cast<const uint32_t*>(D.length), D.new_starts, S.yw, S.sa,
                                         to(D.new_s, l, states), W.wkv, W.wkv_bytes, (unsigned)D.flags | HIPRWKV_LENGTH_I32));
    HIPRWKV_TRY(launch_rwkv7_postmix(0, M, D.H, S.yw, S.r, S.k2, S.v2, S.lora[2], of(P.lnx_w, l, C), of(P.lnx_b, l, C), of(P.r_k, l, C),
                                     EPS_X, S.y, stream));
    Products O;
    O.add(W.dx, S.y, of(P.output, l, C * C), M, C, C, 0, 0);
    n_part = split_out;
    O.G.part = n_part > 1 ? W.parts : nullptr;
    HIPRWKV_TRY(launch_gemm(O.G, n_part, stream));
    const void* const fmix[1] = {of(P.ffn_x_k, l, C)};
    HIPRWKV_TRY(head(1, S.x, S.x2, of(P.ln2_w, l, C), of(P.ln2_b, l, C), l, 0, fmix, &S.xk2, S.stats2));
    Products E;
    E.add(S.fr, S.xk2, of(P.ffn_key, l, C * F), M, F, C, 0, 0, GEMM_ACT_RELUSQ).raw = S.ff;
    HIPRWKV_TRY(E.launch(stream));
    Products V;
    const bool last = l == D.L - 1;
    V.add(last ? D.dx : W.dx, S.fr, of(P.ffn_value, l, C * F), M, C, F, 0, 0);
    n_part = last ? 1 : split_val;
    V.G.part = n_part > 1 ? W.parts : nullptr;
    HIPRWKV_TRY(launch_gemm(V.G, n_part, stream));
    x = S.x2;
  }
  return HIPRWKV_OK;
}

int launch_rwkv7_stack_bwd(const Rwkv7Stack& D, hipStream_t stream, hipError_t& e) {
  const Stack K(D);
  const size_t C = K.C, F = K.F, M = K.rows, row_state = 66 * C, states = (size_t)D.B * 64 * C;
  Arena A{static_cast<char*>(D.workspace)};
  const Backward W(K, A);
  const auto &P = D.param, &G = D.grad;
  const bf16_t* const st = static_cast<const bf16_t*>(D.state);
  const bf16_t* v_first;
  {
    Arena first{static_cast<char*>(D.saved[0])};
    v_first = K.layer(first, true, 0).v;
  }
  auto head = [&](int n_out, const bf16_t* x, float* stats, const void* w, const void* b, int64_t l, int srow, const void* const* mix,
                  bf16_t* const* g, const void* gx, void* out, void* const* dparam, float* part, ReduceJobs* later) {
    LnMixArgs N;
    memset(&N, 0, sizeof(N));
    N.B = D.B; N.T = D.T; N.C = D.C; N.eps = EPS; N.ns = D.new_starts; N.length = D.length;
    N.xs = const_cast<bf16_t*>(x); N.stats = stats; N.ln_w = w; N.ln_b = b;
    N.prev = st + l * row_state + srow * C; N.prev_bstride = D.L * row_state;
    N.gx = gx; N.dxs = out; N.part = part;
    if (D.g_shift != nullptr) N.gshift = static_cast<const bf16_t*>(D.g_shift) + ((size_t)srow * D.L + l) * D.B * C;
    for (int i = 0; i < n_out; ++i) { N.mix[i] = mix[i]; N.g[i] = g[i]; }
    return launch_ln_shiftmix_bwd(0, n_out, N, dparam, stream, later);
  };
  const void *g_x = D.g_xs, *g_dx = D.g_dx;
  for (int64_t l = D.L - 1; l >= 0; --l) {
    Arena own{static_cast<char*>(D.saved[l])};
    const Layer S = at_layer(K, K.layer(own, true, l), l, v_first);
    // channel mixing
    {
      Products Q;
      Q.add(W.gff, g_dx, of(P.ffn_value, l, C * F), M, F, C, 0, 1, GEMM_DRELUSQ, S.ff);
      Q.add(to(G.ffn_value, l, C * F), g_dx, S.fr, C, F, M, 1, 1);
      HIPRWKV_TRY(Q.launch(stream));
    }
    {
      Products Q;
      Q.add(W.gxk2, W.gff, of(P.ffn_key, l, C * F), M, C, F, 0, 1);
      Q.add(to(G.ffn_key, l, C * F), W.gff, S.xk2, F, C, M, 1, 1);
      HIPRWKV_TRY(Q.launch(stream));
    }
    const void* const fmix[1] = {of(P.ffn_x_k, l, C)};
    ReduceJobs sums;
    memset(&sums, 0, sizeof(sums));
    void* const dhead2[3] = {to(G.ffn_x_k, l, C), to(G.ln2_w, l, C), to(G.ln2_b, l, C)};
    HIPRWKV_TRY(head(1, S.x2, S.stats2, of(P.ln2_w, l, C), of(P.ln2_b, l, C), l, 0, fmix, &W.gxk2, g_x, W.dx2, dhead2, W.parts[0],
                     &sums));
    // time mixing: output projection, group norm and gate
    {
      Products Q;
      Q.add(W.gy, W.dx2, of(P.output, l, C * C), M, C, C, 0, 1);
      Q.add(to(G.output, l, C * C), W.dx2, S.y, C, C, M, 1, 1);
      HIPRWKV_TRY(Q.launch(stream));
    }
    void* const dpost[3] = {to(G.lnx_w, l, C), to(G.lnx_b, l, C), to(G.r_k, l, C)};
    HIPRWKV_TRY(launch_rwkv7_postmix_bwd(0, M, D.H, S.yw, S.r, S.k2, S.v2, S.lora[2], of(P.lnx_w, l, C), of(P.lnx_b, l, C),
                                         of(P.r_k, l, C), EPS_X, W.gy, W.gyw, W.gr1, W.gk1, W.gv1, W.gg, nullptr, nullptr, nullptr,
                                         W.parts[1], dpost, stream, &sums));
    // the recurrence
    HIPRWKV_TRY_RC(hiprwkv_wkv7_bwd_ends(stream, HIPRWKV_BF16, HIPRWKV_BF16, D.B, D.T, D.H, 64, S.w, S.r, S.k2, S.v2, S.a, S.b,
                                         of(D.s, l, states), reinterpret_cast<const uint32_t*>(D.length), D.new_starts, W.gyw, S.sa,
                                         D.g_s == nullptr ? nullptr : of(D.g_s, l, states), W.ends, W.gw, W.gr2, W.gk2, W.gv2, W.ga,
                                         W.gb, W.gs, W.wkv, W.wkv_bytes, (unsigned)D.flags | HIPRWKV_LENGTH_I32));
    // gates; the value residual's cotangents of all layers meet in W.dvf and in the first layer's values
    PreArgs R;
    memset(&R, 0, sizeof(R));
    R.rows = M; R.H = D.H;
    R.xw = S.lora[0]; R.k = S.k; R.xa = S.lora[1];
    R.w0 = of(P.w0, l, C); R.a0 = of(P.a0, l, C); R.k_k = of(P.k_k, l, C); R.k_a = of(P.k_a, l, C);
    R.gw = W.gw; R.gk = W.gk1; R.gk2 = W.gk2; R.gv = W.gv1; R.gv2 = W.gv2; R.ga = W.ga; R.gb = W.gb;
    R.gr = W.gr1; R.gr2 = W.gr2; R.dr = W.gr;
    R.dxw = W.dl[0]; R.dk = W.dk; (l ? R.dv : R.dv_sum) = W.dv; R.dxa = W.dl[1];
    R.gvf = l == D.L - 1 ? nullptr : W.dvf;
    if (l) { R.v = S.v; R.vf = v_first; R.xv = S.lora[3]; R.v0 = of(P.v0, l, C); R.dvf = W.dvf; R.dxv = W.dl[3]; }
    R.part = W.parts[2];
    void* const dpre[5] = {to(G.w0, l, C), to(G.a0, l, C), to(G.k_k, l, C), to(G.k_a, l, C), l ? to(G.v0, l, C) : nullptr};
    HIPRWKV_TRY(launch_rwkv7_pre_bwd(0, R, dpre, stream, &sums));
    HIPRWKV_TRY(launch_reduce_parts(0, sums, stream));
    // projections
    const int n_lora = l ? 4 : 3;
    const void* const f1[4] = {of(P.w1, l, C * K.d[0]), of(P.a1, l, C * K.d[1]), of(P.g1, l, C * K.d[2]), of(P.v1, l, C * K.d[3])};
    const void* const f2[4] = {of(P.w2, l, C * K.d[0]), of(P.a2, l, C * K.d[1]), of(P.g2, l, C * K.d[2]), of(P.v2, l, C * K.d[3])};
    const void* const d1[4] = {G.w1, G.a1, G.g1, G.v1};
    const void* const d2[4] = {G.w2, G.a2, G.g2, G.v2};
    const int act[4] = {GEMM_DTANH, GEMM_ADD, GEMM_DSIGMOID, GEMM_ADD};
    {
      Products Q;
      Q.add(W.dmix[MIX_R], W.gr, of(P.receptance, l, C * C), M, C, C, 0, 1);
      Q.add(W.dmix[MIX_K], W.dk, of(P.key, l, C * C), M, C, C, 0, 1);
      Q.add(W.dmix[MIX_V], W.dv, of(P.value, l, C * C), M, C, C, 0, 1);
      Q.add(to(G.receptance, l, C * C), W.gr, S.mix[MIX_R], C, C, M, 1, 1);
      Q.add(to(G.key, l, C * C), W.dk, S.mix[MIX_K], C, C, M, 1, 1);
      Q.add(to(G.value, l, C * C), W.dv, S.mix[MIX_V], C, C, M, 1, 1);
      for (int i = 0; i < n_lora; ++i) {
        Q.add(W.dh[i], W.dl[i], f2[i], M, K.d[i], C, 0, 0, act[i], act[i] == GEMM_ADD ? nullptr : S.hid[i]);
        Q.add(to(d2[i], l, C * K.d[i]), S.hid[i], W.dl[i], K.d[i], C, M, 1, 1);
      }
      HIPRWKV_TRY(Q.launch(stream));
    }
    Products Q;
    for (int i = 0; i < n_lora; ++i) {
      bf16_t* const out = W.dmix[LORA_MIX[i]];
      Q.add(out, W.dh[i], f1[i], M, C, K.d[i], 0, 0, GEMM_ADD, i == 3 ? out : nullptr);      // the value residual's on top of v's
      Q.add(to(d1[i], l, C * K.d[i]), S.mix[LORA_MIX[i]], W.dh[i], C, K.d[i], M, 1, 1);
    }
    HIPRWKV_TRY(Q.launch(stream));
    const void* const mixv[6] = {of(P.x_r, l, C), of(P.x_w, l, C), of(P.x_k, l, C), of(P.x_v, l, C), of(P.x_a, l, C), of(P.x_g, l, C)};
    void* const dhead1[8] = {to(G.x_r, l, C), to(G.x_w, l, C), to(G.x_k, l, C), to(G.x_v, l, C), to(G.x_a, l, C), to(G.x_g, l, C),
                             to(G.ln1_w, l, C), to(G.ln1_b, l, C)};
    void* const out = l ? W.dx : D.g_x;
    HIPRWKV_TRY(head(6, S.x, S.stats1, of(P.ln1_w, l, C), of(P.ln1_b, l, C), l, 1, mixv, W.dmix, W.dx2, out, dhead1, W.part, nullptr));
    g_x = g_dx = out;
  }
  return HIPRWKV_OK;
}

#undef HIPRWKV_TRY
#undef HIPRWKV_TRY_RC

}  // namespace hiprwkv
