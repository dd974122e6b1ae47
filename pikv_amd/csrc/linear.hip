// Float32 linear layers over one input with many tokens (q, k and v of a prompt chunk): tiles through LDS, one launch for all layers.
//
// Bound: the float32 matrix cores (v_mfma_f32_16x16x4_f32, 157 TFLOP/s for the chip).  Eight wavefronts share a 128 x 128 tile
// (64 x 32 each, 32 products to six 16-byte LDS reads for 16 k-values), the operands of the next 16 k-values are read
// while these are multiplied, the next stage but one is on its way from memory.  A wavefront issues in order, and with its
// LDS reads, LDS writes and loads each in a row the matrix core ran dry behind every row of them: one such operation
// between products took 8192^3 from 137 to 147 TFLOP/s with stages of 32 k-values (143 with 64, which are the faster ones where a
// compute unit has one block: 125 against 137 us for 1000 tokens x 2048 -> 4096, a barrier every 256 products).  Where
// 128 x 128 tiles would leave compute units idle the tile is 64 x 128, 64 x 64 or 32 x 64 (tile_variant).
// The lane with k-values 16 c + 4 quad .. + 3 feeds one of them to each of four instructions, so sums run over k in steps of 16.
//
// Measured, one launch against one library call a layer (us, back to back): 1000 tokens x 2048 -> 2048 + 1024 + 1024 (128 x 128,
// 256 blocks = the chip) 125 / 130; 1280 x 2048 -> 3072 125 / 144; 1000 x 512 -> 2048 21 / 56; 500 x 1536 -> 4096 52 / 66; 250 x 3072 -> 3072 56 / 57; 66 x 1536 -> 4096
// 20 / 57 (three library calls take the host 56 us).  Against: 1000 x 3072 -> 3072 150 / 146, 4000 x 3072 -> 3072 537 / 528, and rounds
// that stay half empty: 330 x 3072 -> 3072 97 / 73.  A single layer is
// no faster than the library's (1000 x 2048 -> 2048 67 / 62).  dense.py says which calls come here.
#include "common.hpp"

namespace pikv {

typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kMaxTiledLayers = 20;   // of one launch

struct TiledLayer {
  const float* w;        // [N][K]
  const float* bias;     // [N]
  float* out;            // [T][N]
  int N, tile0;          // outputs; column tiles of the layers before
};
struct TiledArgs {
  TiledLayer l[kMaxTiledLayers];
  const float* x;        // [T][K]
  int64_t T;
  int K, n_layers, m_tiles, n_tiles;
};

// A block computes BM tokens x BN outputs, a wavefront WM x WN of them.
template <int BM, int BN, int WM, int WN, int BK>
__global__ __launch_bounds__(64 * (BM / WM) * (BN / WN)) void linear_tiled_kernel(TiledArgs a) {
  constexpr int THREADS = 64 * (BM / WM) * (BN / WN);
  constexpr int P = BK + 4;                          // row pitch in LDS: 16-byte reads of 16 rows touch every bank once
  constexpr int LPR = BK / 4, RPP = THREADS / LPR;   // lanes of a row, rows of one pass of the block
  constexpr int NX = BM / RPP, NW = BN / RPP, MT = WM / 16, NT = WN / 16;
  __shared__ float sx[2][BM * P], sw[2][BN * P];
  // Consecutive blocks go round the eight XCDs: each gets a run of tiles of its own, eight row tiles by its columns,
  // so that what its blocks read together is in its L2.
  const int total = a.m_tiles * a.n_tiles;
  const int q = total / 8, r = total % 8, xcd = blockIdx.x % 8;
  const int pos = xcd * q + (xcd < r ? xcd : r) + (int)blockIdx.x / 8;
  const int span = 8 * a.n_tiles, first = pos / span * 8;
  const int rows = a.m_tiles - first < 8 ? a.m_tiles - first : 8;
  const int64_t m0 = (int64_t)(first + pos % span % rows) * BM;
  const int nt = pos % span / rows;
  int g = 0;
  while (g + 1 < a.n_layers && nt >= a.l[g + 1].tile0) ++g;
  const TiledLayer& L = a.l[g];
  const int n0 = (nt - L.tile0) * BN;

  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int quad = lane >> 4, ln = lane & 15;
  const int wm = wave / (BN / WN) * WM, wn = wave % (BN / WN) * WN;
  const int lr = threadIdx.x / LPR, lc = threadIdx.x % LPR * 4;
  const float *px[NX], *pw[NW];
#pragma unroll
  for (int i = 0; i < NX; ++i) {
    const int64_t m = m0 + i * RPP + lr;
    px[i] = a.x + (m < a.T ? m : a.T - 1) * a.K + lc;
  }
#pragma unroll
  for (int i = 0; i < NW; ++i) {
    const int n = n0 + i * RPP + lr;
    pw[i] = L.w + (int64_t)(n < L.N ? n : L.N - 1) * a.K + lc;
  }
  f32x4 vx[NX], vw[NW];
  auto load = [&](int i, int k) {
    if (i < NX) vx[i] = *reinterpret_cast<const f32x4*>(px[i] + k);
    else vw[i - NX] = *reinterpret_cast<const f32x4*>(pw[i - NX] + k);
  };
  auto stage = [&](int i, int b) {
    if (i < NX) *reinterpret_cast<f32x4*>(&sx[b][(i * RPP + lr) * P + lc]) = vx[i];
    else *reinterpret_cast<f32x4*>(&sw[b][((i - NX) * RPP + lr) * P + lc]) = vw[i - NX];
  };
  f32x4 acc[NT][MT];
#pragma unroll
  for (int i = 0; i < NT; ++i)
#pragma unroll
    for (int j = 0; j < MT; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

  f32x4 fx[2][MT], fw[2][NT];
  auto fetch = [&](int i, int b, int c, int p) {
    if (i < NT) fw[p][i] = *reinterpret_cast<const f32x4*>(&sw[b][(wn + 16 * i + ln) * P + 16 * c + 4 * quad]);
    else fx[p][i - NT] = *reinterpret_cast<const f32x4*>(&sx[b][(wm + 16 * (i - NT) + ln) * P + 16 * c + 4 * quad]);
  };
  constexpr int C = BK / 16, M = 4 * NT * MT, F = NT + MT, W = NX + NW;   // C is even
#pragma unroll
  for (int i = 0; i < W; ++i) load(i, 0);
#pragma unroll
  for (int i = 0; i < W; ++i) stage(i, 0);
#pragma unroll
  for (int i = 0; i < W; ++i) load(i, BK < a.K ? BK : 0);
  __syncthreads();
#pragma unroll
  for (int i = 0; i < F; ++i) fetch(i, 0, 0, 0);
  for (int k = 0, b = 0; k < a.K; k += BK, b ^= 1) {
    const int k2 = k + 2 * BK < a.K ? k + 2 * BK : k;
#pragma unroll
    for (int c = 0; c < C; ++c) {
      // Memory operations go between the products one by one: a wavefront issues in order, and several in a row leave
      // the matrix core idle.
      const int ops = c == 0 ? F + 2 * W : F;
#pragma unroll
      for (int m = 0; m < M; ++m) {
        const int e = m / (NT * MT), i = m / MT % NT, j = m % MT;
        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(fw[c & 1][i][e], fx[c & 1][j][e], acc[i][j], 0, 0, 0);
        if (c + 1 == C && m == 0) __syncthreads();
        const int from = m * ops / M, to = (m + 1) * ops / M;
        if (from < to) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int o = 0; o < F + 2 * W; ++o) {
          if (o < from || o >= to) continue;
          if (o < F) { if (c + 1 < C) fetch(o, b, c + 1, (c + 1) & 1); else fetch(o, b ^ 1, 0, 0); }
          else if (o < F + W) stage(o - F, b ^ 1);     // the next stage; its buffer was last read before the barrier
          else load(o - F - W, k2);                    // the one after it, in flight for a whole stage
        }
        if (from < to) __builtin_amdgcn_sched_barrier(0);
      }
    }
  }

  // a lane holds outputs 4 quad + (0..3) of token ln of every 16 x 16 tile
  const bool whole = L.N % 4 == 0;
#pragma unroll
  for (int i = 0; i < NT; ++i) {
    const int n = n0 + wn + 16 * i + 4 * quad;
    if (n >= L.N) continue;
    float bias[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) bias[e] = L.bias[n + e < L.N ? n + e : L.N - 1];
#pragma unroll
    for (int j = 0; j < MT; ++j) {
      const int64_t m = m0 + wm + 16 * j + ln;
      if (m >= a.T) continue;
      float* o = L.out + m * L.N + n;
      if (whole) {
        *reinterpret_cast<f32x4*>(o) = acc[i][j] + f32x4{bias[0], bias[1], bias[2], bias[3]};
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (n + e < L.N) o[e] = acc[i][j][e] + bias[e];
      }
    }
  }
}

// Which tile: the fewest rounds of blocks over the 256 compute units, each round at what it measured for a k-value, in percent
// of a 128 x 128 round (57 ns): 64 x 128 30, 64 x 64 16.6, 32 x 64 11 ns.
static int tile_variant(const TiledArgs& a) {
  static const int kTile[4][3] = {{128, 128, 100}, {64, 128, 53}, {64, 64, 29}, {32, 64, 19}};
  int best = 0;
  int64_t least = INT64_MAX;
  for (int v = 0; v < 4; ++v) {
    int64_t tiles = 0;
    for (int g = 0; g < a.n_layers; ++g) tiles += ((int64_t)a.l[g].N + kTile[v][1] - 1) / kTile[v][1];
    const int64_t cost = ((a.T + kTile[v][0] - 1) / kTile[v][0] * tiles + 255) / 256 * kTile[v][2];
    if (cost < least) { least = cost; best = v; }
  }
  return best;
}

template <int BM, int BN, int WM, int WN, int BK>
static int launch_tiled(TiledArgs& a, hipStream_t st) {
  int64_t tiles = 0;
  for (int g = 0; g < a.n_layers; ++g) {
    a.l[g].tile0 = (int)tiles;
    tiles += ((int64_t)a.l[g].N + BN - 1) / BN;
  }
  const int64_t m_tiles = (a.T + BM - 1) / BM;
  if (tiles > 0x7fffff || m_tiles > 0x7fffff || tiles * m_tiles > 0x0fffffff) return PIKV_ERR_SHAPE;
  a.m_tiles = (int)m_tiles; a.n_tiles = (int)tiles;
  hipLaunchKernelGGL((linear_tiled_kernel<BM, BN, WM, WN, BK>), dim3((unsigned)(tiles * m_tiles)),
                     dim3(64 * (BM / WM) * (BN / WN)), 0, st, a);
  PIKV_CHECK_LAUNCH();
  return PIKV_OK;
}

}  // namespace pikv

using namespace pikv;

extern "C" int pikv_linear_tiled(const float* x, int64_t T, int K, int n_layers, const float* const* w,
                                 const float* const* bias, const int32_t* n_out, float* const* out, void* stream) {
  if (!x || !w || !bias || !n_out || !out) return PIKV_ERR_NULL;
  if (T < 1 || K < 1 || n_layers < 1) return PIKV_ERR_SHAPE;
  if (K % 64 != 0 || n_layers > kMaxTiledLayers || (uintptr_t)x % 16 != 0) return PIKV_ERR_UNSUPPORTED;
  TiledArgs a{};
  a.x = x; a.T = T; a.K = K; a.n_layers = n_layers;
  for (int g = 0; g < n_layers; ++g) {
    if (!w[g] || !bias[g] || !out[g]) return PIKV_ERR_NULL;
    if (n_out[g] < 1) return PIKV_ERR_SHAPE;
    if ((uintptr_t)w[g] % 16 != 0 || (n_out[g] % 4 == 0 && (uintptr_t)out[g] % 16 != 0)) return PIKV_ERR_UNSUPPORTED;
    a.l[g].w = w[g]; a.l[g].bias = bias[g]; a.l[g].out = out[g]; a.l[g].N = n_out[g];
  }
  hipStream_t st = (hipStream_t)stream;
  switch (tile_variant(a)) {
    case 0: return launch_tiled<128, 128, 64, 32, 64>(a, st);
    case 1: return launch_tiled<64, 128, 32, 32, 64>(a, st);
    case 2: return launch_tiled<64, 64, 32, 16, 32>(a, st);
    default: return launch_tiled<32, 64, 32, 16, 64>(a, st);
  }
}
