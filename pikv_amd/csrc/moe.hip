// Float32 pieces of the mixture-of-experts layer around its library products: small linear layers that share one input
// (key projection, router hidden layers) in one launch, the rest of the adaptive router, the means of the cached values,
// and everything behind the experts' products.
//
// Bound: launches and latency.  A [128 x 256] x [256 x 256] product is 17 MFLOP; as a library call it runs on a
// single compute unit (one 256 x 128 tile, 33 us).  Here a tile is 32 x 32 and the contraction is split over the
// wavefronts of its block, so that one launch of all layers covers the chip and no chain is longer than a quarter of
// the contraction.  Everything is float32 (v_mfma_f32_32x32x2_f32): products, sums and results; error against
// float64 2.1e-7 where the library's is 4.1e-7.  The experts' own products keep the library's order of sums - one launch
// of linear_tiled at the sizes where that order was measured to be the same, library calls elsewhere: their outputs are quantised into the
// caches and come back as means in the next call, where another order - 2e-7, a code in 10^4 - grew to 1e-4 of a cached row's
// scale.  The second factor of their LoRA is taken in expert_combine.  Evaluation pass of 128 tokens x 256, 4 experts: 644 -> 513 us.
// Measured: linear_group, three layers of 2048 x 2048 over 8 rows 23 us a call and 19 in a replayed graph (61 and 26 as
// three library calls), over 128 rows 55 a call (59); adaptive router with 128 tokens of 256, 4 experts 7.7 + 5.2 + 7.0 +
// 3.0 us of kernels for 35 launches.  The kernels are made for that scale: no LDS tile in linear_group, one block a sequence
// for the blend, one block for the balance loss.  dense.py holds the sizes where the library takes over, with both sides.
#include "common.hpp"

namespace pikv {

typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int kMaxGroups = 20;   // layers of one launch
constexpr int kMaxRank = 8;      // LoRA rank
constexpr int kTileMN = 32;
constexpr int kTilePitch = 33;

// ---- linear layers over one input ---------------------------------------------------------
struct LinearLayer {
  const float* w;        // [N][K]
  const float* bias;     // [N]
  const float* lora_a;   // [K][rank] or null
  const float* lora_b;   // [rank][N]
  float* out;            // [T][N]
  float scaling;
  int N, relu;
};
struct LinearArgs {
  LinearLayer l[kMaxGroups];
  const float* x;        // [T][K]
  float* t;              // [n_layers][T][rank]: x lora_a
  int64_t T;
  int K, n_layers, rank;
};

// x lora_a: a wavefront per token and layer.
__global__ __launch_bounds__(256) void lora_in_kernel(LinearArgs a) {
  const int lane = threadIdx.x & 63;
  const int64_t tok = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (tok >= a.T) return;
  const float* x = a.x + tok * a.K;
  const int g = blockIdx.y;
  const float* A = a.l[g].lora_a;
  if (A == nullptr) return;
  float acc[kMaxRank];
#pragma unroll
  for (int j = 0; j < kMaxRank; ++j) acc[j] = 0.f;
  for (int k = lane; k < a.K; k += 64) {
    const float xv = x[k];
#pragma unroll
    for (int j = 0; j < kMaxRank; ++j)
      if (j < a.rank) acc[j] = fmaf(xv, A[(int64_t)k * a.rank + j], acc[j]);
  }
#pragma unroll
  for (int j = 0; j < kMaxRank; ++j) {
    if (j >= a.rank) break;
    const float s = group_sum_dpp(acc[j], 64);
    if (lane == 0) a.t[((int64_t)g * a.T + tok) * a.rank + j] = s;
  }
}

// One 32 x 32 tile of one layer's output per block; each of the four wavefronts contracts a quarter of K.
__global__ __launch_bounds__(256) void linear_group_kernel(LinearArgs a) {
  __shared__ float part[4][kTileMN * kTilePitch];
  const LinearLayer& L = a.l[blockIdx.z];
  const int n0 = blockIdx.x * kTileMN;
  if (n0 >= L.N) return;                 // layers of one launch may differ in width
  const int64_t m0 = (int64_t)blockIdx.y * kTileMN;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int half = lane >> 5, ln = lane & 31;
  const int kw = a.K / 4;
  const int64_t row = m0 + ln < a.T ? m0 + ln : a.T - 1;
  const float* xp = a.x + row * a.K + wave * kw + half * 16;
  const float* wp = L.w + (int64_t)(n0 + ln) * a.K + wave * kw + half * 16;
  f32x16 acc;
#pragma unroll
  for (int i = 0; i < 16; ++i) acc[i] = 0.f;
  float4 xv[4], wv[4], xn[4], wn[4];
  auto load = [&](int k, float4 (&xd)[4], float4 (&wd)[4]) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      xd[i] = *reinterpret_cast<const float4*>(xp + k + 4 * i);
      wd[i] = *reinterpret_cast<const float4*>(wp + k + 4 * i);
    }
  };
  load(0, xv, wv);
  for (int k = 0; k < kw; k += 32) {
    load(k + 32 < kw ? k + 32 : k, xn, wn);   // in flight during the products of this step
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      acc = __builtin_amdgcn_mfma_f32_32x32x2f32(xv[i].x, wv[i].x, acc, 0, 0, 0);
      acc = __builtin_amdgcn_mfma_f32_32x32x2f32(xv[i].y, wv[i].y, acc, 0, 0, 0);
      acc = __builtin_amdgcn_mfma_f32_32x32x2f32(xv[i].z, wv[i].z, acc, 0, 0, 0);
      acc = __builtin_amdgcn_mfma_f32_32x32x2f32(xv[i].w, wv[i].w, acc, 0, 0, 0);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) { xv[i] = xn[i]; wv[i] = wn[i]; }
  }
#pragma unroll
  for (int i = 0; i < 16; ++i) part[wave][(8 * (i >> 2) + 4 * half + (i & 3)) * kTilePitch + ln] = acc[i];
  __syncthreads();
  for (int i = threadIdx.x; i < kTileMN * kTileMN; i += 256) {
    const int m = i >> 5, n = i & 31;
    if (m0 + m >= a.T) break;
    float y = (part[0][m * kTilePitch + n] + part[1][m * kTilePitch + n]) +
              (part[2][m * kTilePitch + n] + part[3][m * kTilePitch + n]) + L.bias[n0 + n];
    if (L.lora_a != nullptr) {
      const float* t = a.t + ((int64_t)blockIdx.z * a.T + m0 + m) * a.rank;
      float s = 0.f;
      for (int j = 0; j < a.rank; ++j) s = fmaf(t[j], L.lora_b[(int64_t)j * L.N + n0 + n], s);
      y = y + s * L.scaling;
    }
    if (L.relu) y = y < 0.f ? 0.f : y;   // a NaN stays
    L.out[(m0 + m) * L.N + n0 + n] = y;
  }
}

// ---- means of the cached rows ---------------------------------------------------------------
struct MeanArgs {
  const void* codes;
  const void* scale;
  const void* zero;
  const int64_t* row_base;
  const int32_t* fill;
  float* part;           // [chunk][cache][D]
  float* out;            // [cache][D]
  int64_t rows_per_chunk;
  int D, group, n_caches, n_chunks;
};

// Sums of one chunk of a cache's rows: 64 lanes x 4 columns, four wavefronts a row apart.
template <int SCHEME>
__global__ __launch_bounds__(256) void cache_sum_kernel(MeanArgs a) {
  using Q = QScheme<SCHEME>;
  __shared__ float4 sums[4][64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int c = blockIdx.y;
  const int d0 = (blockIdx.x * 64 + lane) * 4;
  const int64_t first = blockIdx.z * a.rows_per_chunk;
  int64_t end = first + a.rows_per_chunk;
  if (end > a.fill[c]) end = a.fill[c];
  float4 s = make_float4(0.f, 0.f, 0.f, 0.f);
  if (d0 < a.D) {
    const int64_t base = a.row_base[c];
#pragma unroll 4
    for (int64_t r = first + wave; r < end; r += 4) {
      const int64_t row = base + r;
      const char* p = reinterpret_cast<const char*>(a.codes) + (row * a.D + d0) * Q::bits / 8;
      uint32_t w;
      if constexpr (Q::bits == 8) w = *reinterpret_cast<const uint32_t*>(p);
      else w = *reinterpret_cast<const uint16_t*>(p);
      const int64_t mi = row * (a.D / a.group) + d0 / a.group;
      const float sc = load_meta<SCHEME>(a.scale, mi);
      float z = 0.f;
      if constexpr (!Q::sym) z = load_meta<SCHEME>(a.zero, mi);
      float f[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int b = (int)((w >> (Q::bits * j)) & ((1u << Q::bits) - 1u));
        f[j] = ((float)(Q::sym ? (b ^ (1 << (Q::bits - 1))) - (1 << (Q::bits - 1)) : b) - z) * sc;
      }
      s.x += f[0]; s.y += f[1]; s.z += f[2]; s.w += f[3];
    }
  }
  sums[wave][lane] = s;
  __syncthreads();
  if (wave == 0 && d0 < a.D) {
    const float4 p = sums[0][lane], q = sums[1][lane], r = sums[2][lane], t = sums[3][lane];
    *reinterpret_cast<float4*>(a.part + ((int64_t)blockIdx.z * a.n_caches + c) * a.D + d0) =
        make_float4((p.x + q.x) + (r.x + t.x), (p.y + q.y) + (r.y + t.y), (p.z + q.z) + (r.z + t.z),
                    (p.w + q.w) + (r.w + t.w));
  }
}

__global__ __launch_bounds__(256) void cache_mean_kernel(MeanArgs a) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int64_t n = (int64_t)a.n_caches * a.D;
  if (i >= n) return;
  float s = 0.f;
  for (int k = 0; k < a.n_chunks; ++k) s += a.part[k * n + i];
  const int f = a.fill[i / a.D];
  a.out[i] = s / (float)(f > 1 ? f : 1);
}

// Chunks of a cache: 64 rows, or as many more as keep them at 64.
static int64_t mean_rows_per_chunk(int64_t max_len) {
  const int64_t r = (max_len + 63) / 64;
  return r < 64 ? 64 : r;
}

// ---- value LoRA of the means ------------------------------------------------------------------
struct ValueLoraArgs {
  const float* a[kMaxGroups];   // [H][rank]
  const float* b[kMaxGroups];   // [rank][H]
  float scaling[kMaxGroups];
  const float* mean;            // [E][H]
  float* out;
  int H, rank;
};

__global__ __launch_bounds__(256) void value_lora_kernel(ValueLoraArgs a) {
  __shared__ float sums[4][kMaxRank];
  const int e = blockIdx.x, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const float* m = a.mean + (int64_t)e * a.H;
  float acc[kMaxRank];
#pragma unroll
  for (int j = 0; j < kMaxRank; ++j) acc[j] = 0.f;
  for (int k = threadIdx.x; k < a.H; k += 256) {
#pragma unroll
    for (int j = 0; j < kMaxRank; ++j)
      if (j < a.rank) acc[j] = fmaf(m[k], a.a[e][(int64_t)k * a.rank + j], acc[j]);
  }
#pragma unroll
  for (int j = 0; j < kMaxRank; ++j) {
    const float s = group_sum_dpp(acc[j], 64);
    if (lane == 0) sums[wave][j] = s;
  }
  __syncthreads();
  for (int k = threadIdx.x; k < a.H; k += 256) {
    float s = 0.f;
    for (int j = 0; j < a.rank; ++j)
      s = fmaf((sums[0][j] + sums[1][j]) + (sums[2][j] + sums[3][j]), a.b[e][(int64_t)j * a.H + k], s);
    a.out[(int64_t)e * a.H + k] = m[k] + s * a.scaling[e];
  }
}

// ---- experts behind their products ----------------------------------------------------------------
struct ExpertArgs {
  const float* dense[kMaxGroups];   // [T][H]
  const float* lora[kMaxGroups];    // [T][H]; with factors [T][rank]
  const float* lora_b[kMaxGroups];  // with factors [rank][H]
  float scaling[kMaxGroups];
  const float* add;                 // [E][H]
  const float* w;                   // [T][E]
  float* outs;                      // [E][T][H]
  float* mix;                       // [T][H]
  int64_t T;
  int E, H4, rank;
};

// outs[e] = relu(dense[e] + lora[e] * scaling[e]) + add[e]; mix[t] = sum over e, in order, of outs[e][t] * w[t][e].
// FACTORS: lora[e] is the product of two factors of a small rank, added up here by fused multiply-adds in ascending order, without a
// launch of its own (8 us each for 128 tokens of 256).  The library's product gave the same bits for ranks 1 to 8, 128 to 1024
// columns and 1 to 2048 tokens.
template <bool FACTORS>
__global__ __launch_bounds__(256) void expert_combine_kernel(ExpertArgs a) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= a.T * a.H4) return;
  const int64_t t = i / a.H4;
  const int h = (int)(i - t * a.H4);
  float s[4] = {0.f, 0.f, 0.f, 0.f};
  for (int e = 0; e < a.E; ++e) {
    const float4 d = reinterpret_cast<const float4*>(a.dense[e])[i];
    float4 l = make_float4(0.f, 0.f, 0.f, 0.f);
    if constexpr (FACTORS) {
      for (int j = 0; j < a.rank; ++j) {
        const float u = a.lora[e][t * a.rank + j];
        const float4 b = reinterpret_cast<const float4*>(a.lora_b[e])[j * a.H4 + h];
        l = make_float4(fmaf(u, b.x, l.x), fmaf(u, b.y, l.y), fmaf(u, b.z, l.z), fmaf(u, b.w, l.w));
      }
    } else {
      l = reinterpret_cast<const float4*>(a.lora[e])[i];
    }
    const float4 c = reinterpret_cast<const float4*>(a.add)[(int64_t)e * a.H4 + h];
    const float dv[4] = {d.x, d.y, d.z, d.w}, lv[4] = {l.x, l.y, l.z, l.w}, cv[4] = {c.x, c.y, c.z, c.w};
    const float we = a.w[t * a.E + e];
    float o[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      float y = dv[j] + lv[j] * a.scaling[e];
      y = y < 0.f ? 0.f : y;             // a NaN stays
      o[j] = y + cv[j];
      s[j] = s[j] + o[j] * we;
    }
    reinterpret_cast<float4*>(a.outs)[e * a.T * a.H4 + i] = make_float4(o[0], o[1], o[2], o[3]);
  }
  reinterpret_cast<float4*>(a.mix)[i] = make_float4(s[0], s[1], s[2], s[3]);
}

// ---- adaptive router behind its hidden layers -------------------------------------------------------
struct AdaptiveArgs {
  const float* x_mean;                   // [B][H]
  const float *sel_w1, *sel_b1;          // [H2][H], [H2]
  const float *sel_w2, *sel_b2;          // [2][H2], [2]
  float* blend;                          // [B][2]
  const float *h_lb, *h_imp, *h_pred;    // [T][H], [T][H], [T][H2]
  const float *w_lb, *b_lb, *w_imp, *b_imp, *w_pred, *b_pred;
  const float* mask;                     // [E] or null
  float *lb_probs, *weights, *importance, *topk_w;
  int64_t* topk_idx;
  int64_t T;
  int S, H, H2, E, k;
  float temp_lb, temp_imp;
};

// Blend of one sequence: softmax of the selector's two outputs.
__global__ __launch_bounds__(1024) void router_blend_kernel(AdaptiveArgs a) {
  __shared__ float lg[2][16];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const float* x = a.x_mean + (int64_t)blockIdx.x * a.H;
  float s0 = 0.f, s1 = 0.f;
  for (int n0 = wave * 8; n0 < a.H2; n0 += 128) {      // eight rows in flight together
    float d[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) d[j] = 0.f;
    for (int k = lane; k < a.H; k += 64) {
      const float xv = x[k];
#pragma unroll
      for (int j = 0; j < 8; ++j)
        d[j] = fmaf(xv, a.sel_w1[(int64_t)(n0 + j < a.H2 ? n0 + j : a.H2 - 1) * a.H + k], d[j]);
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const float s = group_sum_dpp(d[j], 64);
      if (n0 + j >= a.H2) continue;
      float h = s + a.sel_b1[n0 + j];
      h = h < 0.f ? 0.f : h;
      s0 = fmaf(h, a.sel_w2[n0 + j], s0);
      s1 = fmaf(h, a.sel_w2[a.H2 + n0 + j], s1);
    }
  }
  if (lane == 0) { lg[0][wave] = s0; lg[1][wave] = s1; }
  __syncthreads();
  if (threadIdx.x == 0) {
    float l0 = 0.f, l1 = 0.f;
    for (int w = 0; w < 16; ++w) { l0 += lg[0][w]; l1 += lg[1][w]; }
    l0 += a.sel_b2[0];
    l1 += a.sel_b2[1];
    const float m = fmaxf(l0, l1);
    const float e0 = expf(l0 - m), e1 = expf(l1 - m);
    a.blend[2 * blockIdx.x] = e0 / (e0 + e1);
    a.blend[2 * blockIdx.x + 1] = e1 / (e0 + e1);
  }
}

__device__ __forceinline__ float dot_lanes(const float* x, const float* w, int n, int lane) {
  float d = 0.f;
  for (int k = lane; k < n; k += 64) d = fmaf(x[k], w[k], d);
  return group_sum_dpp(d, 64);
}

__device__ __forceinline__ float softmax_lanes(float lg, bool in, int lane) {
  const float m = group_max_dpp(in ? lg : -__builtin_inff(), 64);
  const float ex = in ? expf(lg - m) : 0.f;
  return ex / group_sum_dpp(ex, 64);
}

// A wavefront per token, lane e holds expert e: second layers, both softmaxes, the importance factor, the blend,
// top-k (value descending, lower expert first, NaN last) and its renormalisation.
__global__ __launch_bounds__(256) void adaptive_tail_kernel(AdaptiveArgs a) {
  const int lane = threadIdx.x & 63;
  const int64_t t = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (t >= a.T) return;
  const bool in = lane < a.E;
  float l1 = 0.f, l2 = 0.f;
  const float *h1 = a.h_lb + t * a.H, *h2 = a.h_imp + t * a.H;
  for (int e0 = 0; e0 < a.E; e0 += 8) {                // eight experts' rows in flight together
    const int n = a.E - e0 < 8 ? a.E - e0 : 8;
    float d1[8], d2[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) d1[j] = d2[j] = 0.f;
    for (int k = lane; k < a.H; k += 64) {
      const float x1 = h1[k], x2 = h2[k];
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const int64_t w = (int64_t)(e0 + (j < n ? j : n - 1)) * a.H + k;
        d1[j] = fmaf(x1, a.w_lb[w], d1[j]);
        d2[j] = fmaf(x2, a.w_imp[w], d2[j]);
      }
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const float s1 = group_sum_dpp(d1[j], 64), s2 = group_sum_dpp(d2[j], 64);
      if (j < n && lane == e0 + j) { l1 = s1; l2 = s2; }
    }
  }
  const float z = dot_lanes(a.h_pred + t * a.H2, a.w_pred, a.H2, lane) + a.b_pred[0];
  const float imp = 1.f / (1.f + expf(-z));
  if (in) {
    l1 = (l1 + a.b_lb[lane]) / a.temp_lb;
    l2 = (l2 + a.b_imp[lane]) / a.temp_imp;
    if (a.mask != nullptr) { l1 = l1 + a.mask[lane]; l2 = l2 + a.mask[lane]; }
  }
  const float p1 = softmax_lanes(l1, in, lane);
  float p2 = softmax_lanes(l2, in, lane) * imp;
  p2 = p2 / group_sum_dpp(in ? p2 : 0.f, 64);
  const float* bl = a.blend + t / a.S * 2;
  const float w = bl[0] * p1 + bl[1] * p2;
  if (in) {
    a.lb_probs[t * a.E + lane] = p1;
    a.weights[t * a.E + lane] = w;
  }
  if (lane == 0) a.importance[t] = imp;
  bool left = in;
  float sum = 0.f, mine = 0.f;
  int my_idx = 0;
  for (int j = 0; j < a.k; ++j) {
    const float key = left ? w : -__builtin_inff();
    const float mx = group_max_dpp(key, 64);
    uint64_t cand = __ballot(left && key == mx);
    if (cand == 0) cand = __ballot(left);              // only NaNs left
    const int win = (int)__builtin_ctzll(cand);        // k <= E: a lane is left
    const float wv = __shfl(w, win, PIKV_WAVE);
    sum = sum + wv;
    if (lane == j) { mine = wv; my_idx = win; }
    if (lane == win) left = false;
  }
  if (lane < a.k) {
    a.topk_idx[t * a.k + lane] = my_idx;
    a.topk_w[t * a.k + lane] = mine / sum;
  }
}

// balance_weight * std / mean of the experts' mean probabilities (std with n - 1).
__global__ __launch_bounds__(1024) void balance_loss_kernel(const float* probs, int64_t T, int E, float weight, float* loss) {
  __shared__ float sums[16];
  __shared__ float usage[64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  for (int e = 0; e < E; ++e) {
    float s = 0.f;
    for (int64_t t = threadIdx.x; t < T; t += 1024) s += probs[t * E + e];
    s = group_sum_dpp(s, 64);
    if (lane == 0) sums[wave] = s;
    __syncthreads();
    if (threadIdx.x == 0) {
      float u = 0.f;
      for (int i = 0; i < 16; ++i) u += sums[i];
      usage[e] = u / (float)T;
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    float m = 0.f, v = 0.f;
    for (int e = 0; e < E; ++e) m += usage[e];
    m /= (float)E;
    for (int e = 0; e < E; ++e) v += (usage[e] - m) * (usage[e] - m);
    *loss = weight * (sqrtf(v / (float)(E - 1)) / m);   // E = 1: 0 / 0, as the reference's std of one value
  }
}

}  // namespace pikv

using namespace pikv;

extern "C" int64_t pikv_linear_group_workspace_bytes(int64_t T, int n_layers, int rank) {
  if (T < 0 || n_layers < 1 || rank < 0) return 0;
  return (int64_t)n_layers * T * rank * (int64_t)sizeof(float);
}

extern "C" int pikv_linear_group(const float* x, int64_t T, int K, int n_layers, const float* const* w,
                                 const float* const* bias, const int32_t* n_out, const int32_t* relu, int rank,
                                 const float* const* lora_a, const float* const* lora_b, const float* scaling,
                                 float* const* out, void* workspace, int64_t workspace_bytes, void* stream) {
  if (!x || !w || !bias || !n_out || !relu || !out) return PIKV_ERR_NULL;
  if (T < 1 || K < 1 || n_layers < 1 || rank < 0) return PIKV_ERR_SHAPE;
  if (K % 128 != 0 || n_layers > kMaxGroups || rank > kMaxRank || (T + kTileMN - 1) / kTileMN > 65535)
    return PIKV_ERR_UNSUPPORTED;
  LinearArgs a{};
  a.x = x; a.T = T; a.K = K; a.n_layers = n_layers; a.rank = rank;
  int max_n = 0;
  bool lora = false;
  for (int g = 0; g < n_layers; ++g) {
    LinearLayer& l = a.l[g];
    l.w = w[g]; l.bias = bias[g]; l.out = out[g]; l.N = n_out[g]; l.relu = relu[g];
    if (!l.w || !l.bias || !l.out) return PIKV_ERR_NULL;
    if (l.N < 1) return PIKV_ERR_SHAPE;
    if (l.N % kTileMN != 0) return PIKV_ERR_UNSUPPORTED;
    if (rank > 0 && lora_a && lora_a[g]) {
      if (!lora_b || !lora_b[g] || !scaling) return PIKV_ERR_NULL;
      l.lora_a = lora_a[g]; l.lora_b = lora_b[g]; l.scaling = scaling[g];
      lora = true;
    }
    if (l.N > max_n) max_n = l.N;
  }
  hipStream_t st = (hipStream_t)stream;
  if (lora) {
    if (!workspace || workspace_bytes < pikv_linear_group_workspace_bytes(T, n_layers, rank)) return PIKV_ERR_WORKSPACE;
    a.t = reinterpret_cast<float*>(workspace);
    hipLaunchKernelGGL(lora_in_kernel, dim3((unsigned)((T + 3) / 4), (unsigned)n_layers), dim3(256), 0, st, a);
    PIKV_CHECK_LAUNCH();
  }
  hipLaunchKernelGGL(linear_group_kernel,
                     dim3((unsigned)(max_n / kTileMN), (unsigned)((T + kTileMN - 1) / kTileMN), (unsigned)n_layers),
                     dim3(256), 0, st, a);
  PIKV_CHECK_LAUNCH();
  return PIKV_OK;
}

extern "C" int64_t pikv_cache_mean_workspace_bytes(int n_caches, int D, int64_t max_len) {
  if (n_caches < 1 || D < 1 || max_len < 0) return 0;
  const int64_t r = mean_rows_per_chunk(max_len);
  const int64_t chunks = max_len > 0 ? (max_len + r - 1) / r : 1;
  return chunks * n_caches * D * (int64_t)sizeof(float);
}

extern "C" int pikv_cache_mean(const void* codes, const void* scale, const void* zero, int scheme, int group, int D,
                               const int64_t* cache_row_base, const int32_t* cache_fill, int n_caches, int64_t max_len,
                               float* out, void* workspace, int64_t workspace_bytes, void* stream) {
  if (!codes || !scale || !cache_row_base || !cache_fill || !out || !workspace) return PIKV_ERR_NULL;
  if (scheme < 0 || scheme > 3) return PIKV_ERR_UNSUPPORTED;
  if ((scheme == PIKV_Q_I8_ASYM || scheme == PIKV_Q_I4_ASYM) && !zero) return PIKV_ERR_NULL;
  if (n_caches < 1 || n_caches > 65535 || max_len < 0 || D < 1 || group < 16 || D % group != 0) return PIKV_ERR_SHAPE;
  if (workspace_bytes < pikv_cache_mean_workspace_bytes(n_caches, D, max_len)) return PIKV_ERR_WORKSPACE;
  MeanArgs a{};
  a.codes = codes; a.scale = scale; a.zero = zero; a.row_base = cache_row_base; a.fill = cache_fill;
  a.part = reinterpret_cast<float*>(workspace); a.out = out;
  a.rows_per_chunk = mean_rows_per_chunk(max_len);
  a.n_chunks = max_len > 0 ? (int)((max_len + a.rows_per_chunk - 1) / a.rows_per_chunk) : 1;
  a.D = D; a.group = group; a.n_caches = n_caches;
  hipStream_t st = (hipStream_t)stream;
  const dim3 grid((unsigned)((D + 255) / 256), (unsigned)n_caches, (unsigned)a.n_chunks);
  switch (scheme) {
    case PIKV_Q_I8_SYM: hipLaunchKernelGGL((cache_sum_kernel<PIKV_Q_I8_SYM>), grid, dim3(256), 0, st, a); break;
    case PIKV_Q_I8_ASYM: hipLaunchKernelGGL((cache_sum_kernel<PIKV_Q_I8_ASYM>), grid, dim3(256), 0, st, a); break;
    case PIKV_Q_I4_ASYM: hipLaunchKernelGGL((cache_sum_kernel<PIKV_Q_I4_ASYM>), grid, dim3(256), 0, st, a); break;
    default: hipLaunchKernelGGL((cache_sum_kernel<PIKV_Q_I4_SYM>), grid, dim3(256), 0, st, a); break;
  }
  PIKV_CHECK_LAUNCH();
  const int64_t n = (int64_t)n_caches * D;
  hipLaunchKernelGGL(cache_mean_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, a);
  PIKV_CHECK_LAUNCH();
  return PIKV_OK;
}

extern "C" int pikv_value_lora(const float* mean, int n_experts, int H, int rank, const float* const* lora_a,
                               const float* const* lora_b, const float* scaling, float* out, void* stream) {
  if (!mean || !lora_a || !lora_b || !scaling || !out) return PIKV_ERR_NULL;
  if (n_experts < 1 || H < 1 || rank < 1) return PIKV_ERR_SHAPE;
  if (n_experts > kMaxGroups || rank > kMaxRank) return PIKV_ERR_UNSUPPORTED;
  ValueLoraArgs a{};
  for (int e = 0; e < n_experts; ++e) {
    if (!lora_a[e] || !lora_b[e]) return PIKV_ERR_NULL;
    a.a[e] = lora_a[e]; a.b[e] = lora_b[e]; a.scaling[e] = scaling[e];
  }
  a.mean = mean; a.out = out; a.H = H; a.rank = rank;
  hipLaunchKernelGGL(value_lora_kernel, dim3((unsigned)n_experts), dim3(256), 0, (hipStream_t)stream, a);
  PIKV_CHECK_LAUNCH();
  return PIKV_OK;
}

static int expert_combine(const float* const* dense, const float* const* lora, const float* const* lora_b, int rank,
                          const float* scaling, const float* add, const float* weights, int64_t T, int E, int H, float* outs,
                          float* mix, void* stream) {
  if (!dense || !lora || !scaling || !add || !weights || !outs || !mix) return PIKV_ERR_NULL;
  if (T < 1 || E < 1 || H < 4 || H % 4 != 0 || (T * (H / 4) + 255) / 256 > 0x7fffffffLL) return PIKV_ERR_SHAPE;
  if (E > kMaxGroups) return PIKV_ERR_UNSUPPORTED;
  ExpertArgs a{};
  for (int e = 0; e < E; ++e) {
    if (!dense[e] || !lora[e] || (lora_b && !lora_b[e])) return PIKV_ERR_NULL;
    a.dense[e] = dense[e]; a.lora[e] = lora[e]; a.scaling[e] = scaling[e];
    if (lora_b) a.lora_b[e] = lora_b[e];
  }
  a.add = add; a.w = weights; a.outs = outs; a.mix = mix; a.T = T; a.E = E; a.H4 = H / 4; a.rank = rank;
  const dim3 grid((unsigned)((T * (H / 4) + 255) / 256));
  if (lora_b) hipLaunchKernelGGL(expert_combine_kernel<true>, grid, dim3(256), 0, (hipStream_t)stream, a);
  else hipLaunchKernelGGL(expert_combine_kernel<false>, grid, dim3(256), 0, (hipStream_t)stream, a);
  PIKV_CHECK_LAUNCH();
  return PIKV_OK;
}

extern "C" int pikv_expert_combine(const float* const* dense, const float* const* lora, const float* scaling,
                                   const float* add, const float* weights, int64_t T, int E, int H, float* outs,
                                   float* mix, void* stream) {
  return expert_combine(dense, lora, nullptr, 0, scaling, add, weights, T, E, H, outs, mix, stream);
}

extern "C" int pikv_expert_combine_factors(const float* const* dense, const float* const* lora_t, const float* const* lora_b,
                                           int rank, const float* scaling, const float* add, const float* weights, int64_t T,
                                           int E, int H, float* outs, float* mix, void* stream) {
  if (!lora_b) return PIKV_ERR_NULL;
  if (rank < 1) return PIKV_ERR_SHAPE;
  return expert_combine(dense, lora_t, lora_b, rank, scaling, add, weights, T, E, H, outs, mix, stream);
}

extern "C" int pikv_adaptive_router(const float* x_mean, int n_seqs, int S, int H, int H2, int E, int top_k,
                                    const float* sel_w1, const float* sel_b1, const float* sel_w2, const float* sel_b2,
                                    const float* h_lb, const float* w_lb, const float* b_lb, float temp_lb,
                                    const float* h_imp, const float* w_imp, const float* b_imp, float temp_imp,
                                    const float* h_pred, const float* w_pred, const float* b_pred, const float* mask,
                                    float balance_weight, float* blend, float* lb_probs, float* weights,
                                    int64_t* topk_idx, float* topk_w, float* importance, float* balance_loss,
                                    void* stream) {
  if (!x_mean || !sel_w1 || !sel_b1 || !sel_w2 || !sel_b2 || !h_lb || !w_lb || !b_lb || !h_imp || !w_imp || !b_imp ||
      !h_pred || !w_pred || !b_pred || !blend || !lb_probs || !weights || !topk_idx || !topk_w || !importance || !balance_loss)
    return PIKV_ERR_NULL;
  if (n_seqs < 1 || S < 1 || H < 1 || H2 < 1 || E < 1 || E > 64 || top_k < 1 || top_k > E) return PIKV_ERR_SHAPE;
  const int64_t T = (int64_t)n_seqs * S;
  if ((T + 3) / 4 > 0x7fffffffLL) return PIKV_ERR_SHAPE;
  AdaptiveArgs a{x_mean, sel_w1, sel_b1, sel_w2, sel_b2, blend, h_lb, h_imp, h_pred, w_lb, b_lb, w_imp, b_imp, w_pred,
                 b_pred, mask, lb_probs, weights, importance, topk_w, topk_idx, T, S, H, H2, E, top_k, temp_lb, temp_imp};
  hipStream_t st = (hipStream_t)stream;
  hipLaunchKernelGGL(router_blend_kernel, dim3((unsigned)n_seqs), dim3(1024), 0, st, a);
  PIKV_CHECK_LAUNCH();
  hipLaunchKernelGGL(adaptive_tail_kernel, dim3((unsigned)((T + 3) / 4)), dim3(256), 0, st, a);
  PIKV_CHECK_LAUNCH();
  hipLaunchKernelGGL(balance_loss_kernel, dim3(1), dim3(1024), 0, st, lb_probs, T, E, balance_weight, balance_loss);
  PIKV_CHECK_LAUNCH();
  return PIKV_OK;
}
