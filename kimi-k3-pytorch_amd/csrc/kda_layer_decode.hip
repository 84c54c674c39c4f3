// One decode step of a whole KDA layer in three launches: every projection of
// the token (multi_linear_kernel), everything between the projections and the
// output projection per (sequence, head) (layer_core_kernel), and the output
// projection (multi_linear_kernel again).
//
// Reference: KimiDeltaAttention.forward in decode (src/kda/kda.py:98-183) over
// KDAProjections.forward (src/kda/projections.py:144-225).  The composition of
// the single stages takes fifteen launches: eight skinny GEMMs, the large ones
// bound by the reading of their weights (9 us each for 8 MB at 32 sequences,
// 1 TB/s), and kernels of a few microseconds over tensors of a few kilobytes.
// Rounding happens where the stages' tensors round: every projection, q, k, v,
// beta, z, g, the operator's output and its gated norm are values of the
// activation type; arithmetic between them is f32, the state f32.
#include "kda_launch.h"

namespace kda {

typedef __bf16 dec_bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 dec_f16x8 __attribute__((ext_vector_type(8)));
typedef float dec_f32x4 __attribute__((ext_vector_type(4)));

template <class IT>
struct Vec8;
template <>
struct Vec8<bf16> {
  using type = dec_bf16x8;
};
template <>
struct Vec8<f16> {
  using type = dec_f16x8;
};

__device__ __forceinline__ dec_f32x4 mfma8(dec_bf16x8 a, dec_bf16x8 b, dec_f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ dec_f32x4 mfma8(dec_f16x8 a, dec_f16x8 b, dec_f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
}

// ---- y_j = x W_j^T (+ bias_j) for several weights of one activation ------------
// x [M, K], W_j [N_j, K] row-major, y_j [M, N_j]; K a multiple of 64.  Bound: the
// weights' bytes, read once.  A workgroup of eight waves owns 16 NT weight rows
// and the whole reduction, wave w the 64-wide slices w, w + 8, ..: each lane's
// two 16-byte loads per row and slice read 64 consecutive bytes a row each, the
// loads of four slices in flight; x comes from L2.  The waves' partial tiles meet
// in LDS.  With one 32-row tile per workgroup the six projections of a d_model
// 2048 layer (261 workgroups) fill the CUs in one round.  Measured there at 32
// sequences: 18.8 us for 34 MB of weights (1.8 TB/s; non-temporal loads 21.9, two
// slices in flight 20.1), against 53 us in six library GEMMs; the output
// projection 7.8 us for 8.4 MB (1.1 TB/s), against 9.1.
constexpr int kLinThreads = 512;
constexpr int kLinWaves = kLinThreads / 64;
constexpr int kMaxLinear = 6;
constexpr int kSlice = 64;  // reduction columns per step

template <class IT>
struct MultiLinear {
  const IT* x;
  const IT* w[kMaxLinear];
  const IT* bias[kMaxLinear];  // entries may be null
  IT* y[kMaxLinear];
  int n[kMaxLinear];        // rows of W_j
  int first[kMaxLinear + 1];  // first workgroup of weight j
  int count;
  int M, K;
};

template <class IT, int MT, int NT>
__global__ __launch_bounds__(kLinThreads) void multi_linear_kernel(const MultiLinear<IT> a) {
  using v8 = typename Vec8<IT>::type;
  __shared__ __attribute__((aligned(16))) float red[kLinWaves][NT * MT][256];
  const int tid = threadIdx.x, lane = tid & 63, li = lane & 15, g = lane >> 4;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  int j = 0;
  while (j + 1 < a.count && static_cast<int>(blockIdx.x) >= a.first[j + 1]) ++j;
  const int n0 = (static_cast<int>(blockIdx.x) - a.first[j]) * 16 * NT, N = a.n[j];
  const int64_t m0 = static_cast<int64_t>(blockIdx.y) * 16 * MT;
  const IT *wp[NT], *xp[MT];
#pragma unroll
  for (int t = 0; t < NT; ++t) {  // rows past the weight repeat its last one; their results are dropped
    const int row = n0 + 16 * t + li;
    wp[t] = a.w[j] + static_cast<int64_t>(row < N ? row : N - 1) * a.K + 8 * g;
  }
#pragma unroll
  for (int t = 0; t < MT; ++t) {
    const int64_t row = m0 + 16 * t + li;
    xp[t] = a.x + (row < a.M ? row : a.M - 1) * a.K + 8 * g;
  }
  dec_f32x4 acc[NT][MT];
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int m = 0; m < MT; ++m) acc[t][m] = dec_f32x4{0.f, 0.f, 0.f, 0.f};
  const int slices = a.K / kSlice;
  // slices in flight: the weights of U, and of them the activation's too (as
  // many as the registers of two waves per SIMD hold)
  constexpr int U = 4;
  for (int s0 = w; s0 < slices; s0 += kLinWaves * U) {
    v8 wv[U][NT][2], xv[U][MT][2];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int s = s0 + u * kLinWaves;
      const int k = (s < slices ? s : s0) * kSlice;  // past the end: a slice already read, not used
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int e = 0; e < 2; ++e)
          wv[u][t][e] = *reinterpret_cast<const v8*>(wp[t] + k + 32 * e);
#pragma unroll
      for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int e = 0; e < 2; ++e) xv[u][m][e] = *reinterpret_cast<const v8*>(xp[m] + k + 32 * e);
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (s0 + u * kLinWaves < slices) {  // uniform
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
          for (int m = 0; m < MT; ++m)
#pragma unroll
            for (int e = 0; e < 2; ++e) acc[t][m] = mfma8(wv[u][t][e], xv[u][m][e], acc[t][m]);
      }
    }
  }
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int m = 0; m < MT; ++m) *reinterpret_cast<dec_f32x4*>(&red[w][t * MT + m][4 * lane]) = acc[t][m];
  __syncthreads();
  // sum the waves' tiles: element (n, m) of tile (t, mt) lies at lane m + 16 (n / 4), register n % 4
  for (int idx = tid; idx < NT * MT * 256; idx += kLinThreads) {
    const int nl = idx % (16 * NT), ml = idx / (16 * NT);
    const int t = nl >> 4, n = nl & 15, mt = ml >> 4, m = ml & 15;
    const int at = 4 * (m + 16 * (n >> 2)) + (n & 3);
    float s = 0.f;
#pragma unroll
    for (int v = 0; v < kLinWaves; ++v) s += red[v][t * MT + mt][at];
    const int row = n0 + nl;
    const int64_t mm = m0 + ml;
    if (row < N && mm < a.M) {
      if (a.bias[j] != nullptr) s += to_float(a.bias[j][row]);
      a.y[j][mm * N + row] = from_compute<IT>(s);
    }
  }
}

// ---- the layer between its projections, one token ------------------------------
// One workgroup of 256 threads per (head, sequence): ShortConv + SiLU (+ L2 norm)
// of the head's q, k, v and their next histories, the decay logits z = d
// alpha_up^T of the head, decay and beta gates, the recurrence step on the
// [K][V] state tile (held in registers as in recurrent_kernel, its loads issued
// first), and RMSNorm x output gate.  Bound: the state, read and written once
// (67 MB, 11 us at 32 sequences of 16 heads, K = V = 128), and the latency of the
// stages before it: 19 us, against 45 us in eight launches (three ShortConvs,
// alpha_up, the gates, the recurrence, the norm and the offsets).
template <class IT>
struct LayerCore {
  const IT *ql, *kl, *vl, *gl, *bl, *dl;  // projections [B, *]: q, k, v, gate logits, beta logits, alpha_down
  const IT* alpha_up;                     // [H K, rank]
  const IT *qw, *kw, *vw;                 // ShortConv weights [C, taps], lag order
  const IT *qb, *kb, *vb;                 // ShortConv biases or null
  const IT *qh, *kh, *vh;                 // histories [B, taps - 1, C], oldest first, or null (zeros)
  IT *qho, *kho, *vho;
  const IT* b_alpha;                      // [H, K]
  const float* a_log;                     // [H]
  const IT* norm_w;                       // [H, V], [V] or null
  int norm_per_head;
  const float* s_in;                      // [B, H, K, V] or null (zeros)
  float* s_out;
  const int64_t* off_in;                  // [B] or null (zeros)
  int64_t* off_out;
  IT* gated;                              // [B, H V]
  int H, taps, rank;
  float g_min, eps, lo, hi;
};

constexpr int kCoreThreads = 256;
constexpr int kMaxRank = 256;
constexpr int kMaxTaps = 8;

template <class IT, int K, int V>
__global__ __launch_bounds__(kCoreThreads) void layer_core_kernel(const LayerCore<IT> a) {
  using v8 = typename Vec8<IT>::type;
  constexpr int TV = V / 4, TK = kCoreThreads / TV, KPT = K / TK;  // thread (tk, tv): KPT rows, 4 columns
  static_assert(TK * TV == kCoreThreads && KPT * TK == K, "the state tile must split over the threads");
  __shared__ float conv[2 * K + V];     // SiLU outputs, then q, k, v as the operator reads them
  __shared__ float dS[kMaxRank];
  __shared__ float alphaS[K];
  __shared__ float norms[2];
  __shared__ __attribute__((aligned(16))) float red_r[TK][V];
  __shared__ __attribute__((aligned(16))) float red_o[TK][V];
  __shared__ float red_kq[TK];
  const int tid = threadIdx.x, lane = tid & 63, tv = tid % TV, tk = tid / TV;
  const int h = blockIdx.x, H = a.H;
  const int64_t b = blockIdx.y;
  const int64_t tile = (b * H + h) * K * V;
  // the head's alpha_up rows, sixteen lanes a row and eight columns each (the
  // first 128 columns; the few past them in the reduction below), ahead of all
  const int part = tid & 15, row0 = tid >> 4;
  auto up_row = [&](int u, int col) {
    return *reinterpret_cast<const v8*>(a.alpha_up + static_cast<int64_t>(h * K + row0 + 16 * u) * a.rank + col);
  };
  v8 wv[K / 16];
#pragma unroll
  for (int u = 0; u < K / 16; ++u) wv[u] = up_row(u, 8 * part < a.rank ? 8 * part : 0);
  float st[KPT][4];
#pragma unroll
  for (int i = 0; i < KPT; ++i) {
    dec_f32x4 x{0.f, 0.f, 0.f, 0.f};
    if (a.s_in != nullptr)
      x = __builtin_nontemporal_load(reinterpret_cast<const dec_f32x4*>(a.s_in + tile + (tk * KPT + i) * V + 4 * tv));
#pragma unroll
    for (int e = 0; e < 4; ++e) st[i][e] = x[e];
  }
  if (tid < a.rank) dS[tid] = to_float(a.dl[b * a.rank + tid]);
  // ShortConv + SiLU of the head's channels; the next history drops the oldest input
  const int H1 = a.taps - 1;
  for (int idx = tid; idx < 2 * K + V; idx += kCoreThreads) {
    const int kind = idx < K ? 0 : (idx < 2 * K ? 1 : 2);
    const int D = kind < 2 ? K : V, c = h * D + (idx - kind * K), W = H * D;
    const IT* xl = kind == 0 ? a.ql : kind == 1 ? a.kl : a.vl;
    const IT* w = (kind == 0 ? a.qw : kind == 1 ? a.kw : a.vw) + static_cast<int64_t>(c) * a.taps;
    const IT* bias = kind == 0 ? a.qb : kind == 1 ? a.kb : a.vb;
    const IT* hi = kind == 0 ? a.qh : kind == 1 ? a.kh : a.vh;
    IT* ho = kind == 0 ? a.qho : kind == 1 ? a.kho : a.vho;
    const IT x = xl[b * W + c];
    IT old[kMaxTaps], wt[kMaxTaps];
#pragma unroll
    for (int j = 1; j < kMaxTaps; ++j) {  // every load before the first use
      wt[j] = j <= H1 ? w[j] : from_compute<IT>(0.f);
      old[j] = j <= H1 && hi != nullptr ? hi[(b * H1 + H1 - j) * W + c] : from_compute<IT>(0.f);
    }
    float acc = (bias != nullptr ? to_float(bias[c]) : 0.f) + to_float(w[0]) * to_float(x);
#pragma unroll
    for (int j = 1; j < kMaxTaps; ++j) {
      if (j <= H1) acc += to_float(wt[j]) * to_float(old[j]);
      if (j < H1) ho[(b * H1 + H1 - 1 - j) * W + c] = old[j];
    }
    if (H1 > 0) ho[(b * H1 + H1 - 1) * W + c] = x;
    conv[idx] = acc * sigmoid(acc);
  }
  __syncthreads();
  // z of the head (rank a multiple of 8), then its decay factors
  {
    const float scale = fexp(a.a_log[h]);
    float z[K / 16];
#pragma unroll
    for (int u = 0; u < K / 16; ++u) z[u] = 0.f;
    for (int col = 8 * part; col < a.rank; col += 128) {
#pragma unroll
      for (int u = 0; u < K / 16; ++u) {
        const v8 x = col < 128 ? wv[u] : up_row(u, col);
#pragma unroll
        for (int e = 0; e < 8; ++e) z[u] += to_float(static_cast<IT>(x[e])) * dS[col + e];
      }
    }
#pragma unroll
    for (int u = 0; u < K / 16; ++u) {
      const float sum = group_sum<16>(z[u]);
      const int c = row0 + 16 * u;
      if (part == 0) {
        const float gg = lower_bounded_decay(to_float(from_compute<IT>(sum)), to_float(a.b_alpha[h * K + c]), scale,
                                             a.g_min, a.lo, a.hi);
        alphaS[c] = fast_exp(to_float(from_compute<IT>(gg)));
      }
    }
  }
  // L2 norms of q (wave 0) and k (wave 1)
  if (tid < 128) {
    const float* p = conv + (tid >> 6) * K;
    float ss = 0.f;
#pragma unroll
    for (int c = 0; c < K; c += 64) ss += p[c + lane] * p[c + lane];
    ss = group_sum<64>(ss);
    if (lane == 0) norms[tid >> 6] = ss > a.eps * a.eps ? frsqrt(ss) : 1.f / a.eps;
  }
  __syncthreads();
  for (int idx = tid; idx < 2 * K + V; idx += kCoreThreads) {
    const float x = conv[idx] * (idx < K ? norms[0] : idx < 2 * K ? norms[1] : 1.f);
    conv[idx] = to_float(from_compute<IT>(x));
  }
  __syncthreads();
  float p = sigmoid(to_float(a.bl[b * H + h]));
  p = p < a.lo ? a.lo : (p > a.hi ? a.hi : p);
  const float bt = to_float(from_compute<IT>(p));
  const float *qs = conv, *ks = conv + K, *vs = conv + 2 * K;
  float pr[4] = {0.f, 0.f, 0.f, 0.f}, po[4] = {0.f, 0.f, 0.f, 0.f}, kq = 0.f;
#pragma unroll
  for (int i = 0; i < KPT; ++i) {
    const float kk = ks[tk * KPT + i], qq = qs[tk * KPT + i], al = alphaS[tk * KPT + i];
    kq += kk * qq;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      st[i][e] *= al;
      pr[e] += st[i][e] * kk;
      po[e] += st[i][e] * qq;
    }
  }
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    red_r[tk][4 * tv + e] = pr[e];
    red_o[tk][4 * tv + e] = po[e];
  }
  if (tv == 0) red_kq[tk] = kq;
  __syncthreads();
  float r[4] = {0.f, 0.f, 0.f, 0.f}, o[4] = {0.f, 0.f, 0.f, 0.f}, kqs = 0.f;
#pragma unroll
  for (int u = 0; u < TK; ++u) {
    kqs += red_kq[u];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      r[e] += red_r[u][4 * tv + e];
      o[e] += red_o[u][4 * tv + e];
    }
  }
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const float err = vs[4 * tv + e] - r[e];
    o[e] = to_float(from_compute<IT>(o[e] + bt * kqs * err));
    r[e] = err;
  }
#pragma unroll
  for (int i = 0; i < KPT; ++i) {
    const float bk = bt * ks[tk * KPT + i];
    dec_f32x4 x;
#pragma unroll
    for (int e = 0; e < 4; ++e) x[e] = st[i][e] + bk * r[e];
    __builtin_nontemporal_store(x, reinterpret_cast<dec_f32x4*>(a.s_out + tile + (tk * KPT + i) * V + 4 * tv));
  }
  // RMSNorm x output gate: every row group holds the whole output; the first TV threads write it
  float ss = tid < TV ? o[0] * o[0] + o[1] * o[1] + o[2] * o[2] + o[3] * o[3] : 0.f;
  ss = group_sum<64>(ss);  // TV <= 32: wave 0 alone holds terms
  if (tid < TV) {
    const float inv = frsqrt(ss / static_cast<float>(V) + a.eps);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int c = 4 * tv + e;
      float y = o[e] * inv;
      if (a.norm_w != nullptr) y *= to_float(a.norm_w[(a.norm_per_head ? h * V : 0) + c]);
      y *= sigmoid(to_float(a.gl[(b * H + h) * V + c]));
      a.gated[(b * H + h) * V + c] = from_compute<IT>(y);
    }
  }
  if (h == 0 && tid == 0) a.off_out[b] = (a.off_in != nullptr ? a.off_in[b] : 0) + 1;
}

}  // namespace kda

namespace kda_host {

using namespace kda;

template <class IT, int NT>
static void launch_linear(const MultiLinear<IT>& a, hipStream_t s) {
  const int mt = a.M <= 16 ? 1 : (a.M <= 32 ? 2 : 4);
  const dim3 grid(static_cast<unsigned>(a.first[a.count]), static_cast<unsigned>((a.M + 16 * mt - 1) / (16 * mt)));
  if (mt == 1)
    hipLaunchKernelGGL((multi_linear_kernel<IT, 1, NT>), grid, dim3(kLinThreads), 0, s, a);
  else if (mt == 2)
    hipLaunchKernelGGL((multi_linear_kernel<IT, 2, NT>), grid, dim3(kLinThreads), 0, s, a);
  else
    hipLaunchKernelGGL((multi_linear_kernel<IT, 4, NT>), grid, dim3(kLinThreads), 0, s, a);
}

template <class IT, int K, int V>
static void launch_core(const LayerCore<IT>& c, int64_t B, hipStream_t s) {
  hipLaunchKernelGGL((layer_core_kernel<IT, K, V>), dim3(static_cast<unsigned>(c.H), static_cast<unsigned>(B)),
                     dim3(kCoreThreads), 0, s, c);
}

// Elements of the workspace: the six projections, then the gated norm.
static int64_t decode_elems(const kda_layer_decode_args& d) {
  const int64_t kw = d.heads * d.key_dim, vw = d.heads * d.value_dim;
  return d.batch * (2 * kw + 3 * vw + d.heads + d.rank) + 7 * 8;
}

size_t layer_decode_workspace_bytes(const kda_layer_decode_args& d) { return static_cast<size_t>(decode_elems(d)) * 2; }

template <class IT>
static int run_layer_decode(const kda_layer_decode_args& d, hipStream_t s) {
  const int64_t B = d.batch, H = d.heads, kw = H * d.key_dim, vw = H * d.value_dim;
  IT* p = static_cast<IT*>(d.workspace);
  auto take = [&](int64_t n) {  // 16-byte aligned pieces
    IT* r = p;
    p += (n + 7) / 8 * 8;
    return r;
  };
  IT *ql = take(B * kw), *kl = take(B * kw), *vl = take(B * vw), *gl = take(B * vw), *bl = take(B * H),
     *dl = take(B * d.rank), *gated = take(B * vw);
  auto in = [](const void* q) { return static_cast<const IT*>(q); };
  MultiLinear<IT> a{};
  a.x = in(d.x);
  a.M = static_cast<int>(B);
  a.K = static_cast<int>(d.d_model);
  const void* w[kMaxLinear] = {d.beta_proj, d.alpha_down, d.q_proj, d.k_proj, d.v_proj, d.gate_proj};
  const void* bias[kMaxLinear] = {d.beta_bias, nullptr, d.q_bias, d.k_bias, d.v_bias, d.gate_bias};
  IT* y[kMaxLinear] = {bl, dl, ql, kl, vl, gl};
  const int64_t n[kMaxLinear] = {H, d.rank, kw, kw, vw, vw};
  a.count = kMaxLinear;
  for (int j = 0; j < kMaxLinear; ++j) {
    a.w[j] = in(w[j]), a.bias[j] = in(bias[j]), a.y[j] = y[j], a.n[j] = static_cast<int>(n[j]);
    a.first[j + 1] = a.first[j] + static_cast<int>((n[j] + 31) / 32);
  }
  launch_linear<IT, 2>(a, s);
  LayerCore<IT> c{};
  c.ql = ql, c.kl = kl, c.vl = vl, c.gl = gl, c.bl = bl, c.dl = dl;
  c.alpha_up = in(d.alpha_up);
  c.qw = in(d.q_conv), c.kw = in(d.k_conv), c.vw = in(d.v_conv);
  c.qb = in(d.q_conv_bias), c.kb = in(d.k_conv_bias), c.vb = in(d.v_conv_bias);
  c.qh = in(d.q_hist), c.kh = in(d.k_hist), c.vh = in(d.v_hist);
  c.qho = static_cast<IT*>(d.q_hist_out), c.kho = static_cast<IT*>(d.k_hist_out), c.vho = static_cast<IT*>(d.v_hist_out);
  c.b_alpha = in(d.b_alpha), c.a_log = d.a_log, c.norm_w = in(d.norm_weight), c.norm_per_head = d.norm_per_head;
  c.s_in = d.state_in, c.s_out = d.state_out, c.off_in = d.offset_in, c.off_out = d.offset_out;
  c.gated = gated;
  c.H = static_cast<int>(H), c.taps = static_cast<int>(d.taps), c.rank = static_cast<int>(d.rank);
  const float eps = __is_same(IT, bf16) ? 0.0078125f : 0.0009765625f;  // the type's machine epsilon
  c.g_min = static_cast<float>(d.g_min), c.eps = static_cast<float>(d.eps), c.lo = eps, c.hi = 1.f - eps;
  if (d.key_dim == 128 && d.value_dim == 128)
    launch_core<IT, 128, 128>(c, B, s);
  else if (d.key_dim == 128)
    launch_core<IT, 128, 64>(c, B, s);
  else if (d.value_dim == 128)
    launch_core<IT, 64, 128>(c, B, s);
  else
    launch_core<IT, 64, 64>(c, B, s);
  MultiLinear<IT> o{};
  o.x = gated, o.M = static_cast<int>(B), o.K = static_cast<int>(vw), o.count = 1;
  o.w[0] = in(d.output_proj), o.bias[0] = in(d.output_bias), o.y[0] = static_cast<IT*>(d.out);
  o.n[0] = static_cast<int>(d.out_dim);
  // one weight alone: 16-row tiles spread it over twice as many CUs
  o.first[1] = static_cast<int>((d.out_dim + 15) / 16);
  launch_linear<IT, 1>(o, s);
  return check_launch("layer_decode");
}

int launch_layer_decode(const kda_layer_decode_args& d, hipStream_t stream) {
  if (d.dtype != KDA_DTYPE_BF16 && d.dtype != KDA_DTYPE_F16) {
    set_detail("layer_decode: bf16 or f16 tensors (dtype %d)", d.dtype);
    return KDA_ERR_UNSUPPORTED;
  }
  const bool dims = (d.key_dim == 64 || d.key_dim == 128) && (d.value_dim == 64 || d.value_dim == 128);
  if (!dims || d.d_model % kSlice != 0 || d.rank % 8 != 0 || d.rank > kMaxRank || d.taps > kMaxTaps ||
      d.heads > 65535 || d.batch > 65535 || d.d_model > 0x7fffff || d.out_dim > 0x7fffff) {
    set_detail("layer_decode: key and value dims 64 or 128, d_model a multiple of 64, rank a multiple of 8 up to 256, "
               "up to 8 ShortConv taps");
    return KDA_ERR_UNSUPPORTED;
  }
  if (d.workspace_bytes < layer_decode_workspace_bytes(d)) {
    set_detail("layer_decode: workspace of %zu bytes needed", layer_decode_workspace_bytes(d));
    return KDA_ERR_WORKSPACE;
  }
  return d.dtype == KDA_DTYPE_BF16 ? run_layer_decode<bf16>(d, stream) : run_layer_decode<f16>(d, stream);
}

}  // namespace kda_host
