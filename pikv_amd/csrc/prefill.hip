// Attention of a prompt chunk in float32: the chunk's queries over [cached rows ; the chunk's own rows],
// softmax(q.k / sqrt(d)) V without a score matrix in memory.
//
// Bound: the float32 matrix cores (v_mfma_f32_32x32x2_f32, 157 TFLOP/s for the chip); scores, probabilities and
// output stay float32 throughout.  Both products are computed transposed, S^T = K Q^T and O^T = V^T P^T: the
// 32 x 32 result of the first holds, lane by lane, exactly the operand the second one reads, so probabilities
// never leave the registers, and a query's running maximum and sum are one value per lane.  The contraction
// index of either product is laid out so that a lane reads 16 contiguous bytes of a K or V row; codes of cached rows
// are expanded on the way in.
//
// A block owns 32 (query, head) rows of one kv head - the heads that share a kv head side by side, so that their
// causal ends meet - and its four wavefronts take every fourth tile of 32 keys, merging once at the end: a prompt
// of 2 x 500 tokens x 16 heads has only 512 such blocks, and rows split over wavefronts instead would leave half
// of the chip idle.  K and V rows are read along the rows and reach the operand layout through the wavefront's LDS tile: V of a
// tile is on its way during the scores, K of the next one during the values, and takes the place of K in LDS in between.  Cached and
// own rows have a loop each: in one loop the rows in flight are copied where its branches meet, and every copy waits for them.
//
// On this chip a float32 product and float32 vector instructions run in turn (exp_nonpositive): what is not a product adds to
// the time, so the instructions around the products were counted - addresses from one exclusive or, masks only at an end, output
// rescaled only where a maximum moved, a short exponential: 1530 -> about 600 a tile of cached rows.
//
// Measured (us, back to back, before -> now; before: K of a tile loaded and waited for, queries and V in registers, 26 spilled
// registers): 2 x 500 tokens, 16 heads of 128 over 8 kv heads 43.8 -> 35.3, over 500 cached rows of 8 bits 97 -> 81; 4 x 1000 over 1000, 32
// heads 1216 -> 978 (101 TFLOP/s, 64 % of the products' rate); 700 over 700 rows of 4 bits 234 -> 147; 4 x 333, 32 heads of 64 50 -> 34;
// 40 tokens 16.8 -> 10.6.  Heads of 128 take 246 registers, none spilled.  Error against float64 and that of the float32 torch path,
// 2-norms, 2 x 500 tokens and the same over 500 cached rows of 8 bits: heads of 128 3.1e-7 / 3.4e-7 and 4.7e-7 / 6.2e-7, of 64 2.4e-7 / 2.8e-7
// and 3.9e-7 / 5.7e-7; with scores eight times as large 1.2e-6 / 1.2e-6 and 1.5e-6 / 1.5e-6.
//
// A NaN or infinity in a V row that a query does not see reaches that query only from the query's own last tile (a
// zero probability times it); a product over the whole score matrix spreads it to every row.
#include "common.hpp"

namespace pikv {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int kPfRows = 32;    // (query, head) rows of a block
constexpr int kPfKeys = 32;    // keys of a tile
constexpr int kPfWaves = 4;

struct PrefillArgs {
  const float* q;        // [B][S][Hq][DH]
  const float* k;        // [B][S][Hkv][DH]
  const float* v;
  const void* codes[2];  // cached K / V rows, or null: no context
  const void* scale[2];
  const void* zero[2];
  const int64_t* row_base;
  const int32_t* fill;
  float* out;            // [B][S][Hq][DH]
  float* part;           // n_split > 1: [split][B * Hkv * n_rows] rows of DH sums, max, sum
  int64_t max_cached;    // fill is cut to it
  int S, n_kv, rep, group, causal, n_split, out16;   // out16: out begins at 16 bytes
  int64_t n_rows;        // S * rep
  float scale_qk;
};

// Orders the LDS accesses of a wavefront's lanes before it against those after it.
__device__ __forceinline__ void wave_lds_exchange() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// An LDS tile holds rows of DH floats without padding (two blocks fill the 160 KB of a compute unit): 16-byte piece `piece` of row
// `row` lies at piece ^ (row & 15), so that 16 rows read at one piece touch every bank once.  Offsets in bytes; those of several
// rows or pieces are one of them, a constant added to its bits by exclusive or, and a multiple of the row's bytes.
template <int DH>
__device__ __forceinline__ int lds_at(int row, int piece) { return row * DH * 4 + ((piece ^ (row & 15)) << 4); }

// A copy the compiler knows nothing about: what is computed from it stays inside the tile loop, where a hundred addresses kept
// in registers across it would spill.  (Emits nothing.)
__device__ __forceinline__ int in_loop(int x) {
  asm volatile("" : "+v"(x));
  return x;
}

// exp(x) for x <= 0, NaN for NaN: 2^t with t = x log2(e) in two parts; what is below 2^-126 is 0.  Ten instructions; expf of
// any argument takes twenty, and the matrix core and the vector unit of a SIMD do float32 in turn, not side by side (a slot of one
// 32 x 32 x 2 product and 16 multiply-adds from two wavefronts takes 145 cycles: 66 + 80).
__device__ __forceinline__ float exp_nonpositive(float x) {
  constexpr float kLog2eHi = 0x1.715476p+0f, kLog2eLo = 0x1.4ae0cp-26f, kLn2 = 0x1.62e430p-1f;
  x = x < -120.f ? -120.f : x;           // 0 as a float32 probability
  const float t = x * kLog2eHi;
  const float e = __builtin_amdgcn_exp2f(t);
  const float r = fmaf(x, kLog2eLo, fmaf(x, kLog2eHi, -t));      // what t lost
  return fmaf(e, r * kLn2, e);
}

// 32 rows of K (WHICH 0) or V (1) on their way from memory to an LDS tile, 16 bytes a lane along the rows: the chunk's own
// rows, or (CACHED) rows of a cache, expanded on the way into LDS.  Rows past `last` are read from it; row addresses are uniform.
template <int SCHEME, int DH, int WHICH, bool CACHED>
struct RowsInFlight {
  using Q = QScheme<SCHEME>;
  static constexpr int kPieces = DH / (CACHED ? Q::epl : 4);     // lanes of a row
  static constexpr int kPass = 64 / kPieces, N = kPfKeys / kPass;
  f32x4 x[N];
  float sc[CACHED ? N : 1], zr[CACHED ? N : 1];

  __device__ __forceinline__ void load(const PrefillArgs& a, int64_t row0, int kvh, int last, int lane) {
    const uint32_t D = a.n_kv * DH, piece = lane % kPieces;
    if constexpr (!CACHED) {
      const char* p = reinterpret_cast<const char*>((WHICH == 0 ? a.k : a.v) + row0 * D + kvh * DH);
#pragma unroll
      for (int i = 0; i < N; ++i) {
        const int r = i * kPass + lane / kPieces;
        x[i] = *reinterpret_cast<const f32x4*>(p + ((uint32_t)(r < last ? r : last) * D + piece * 4) * 4u);
      }
    } else {
      const uint32_t metas = D / a.group, e0 = kvh * DH + piece * Q::epl, m0 = e0 / a.group;
      const char* codes = reinterpret_cast<const char*>(a.codes[WHICH]) + row0 * D * Q::bits / 8;
      const char* scale = reinterpret_cast<const char*>(a.scale[WHICH]) + row0 * metas * Q::meta_bytes;
      const char* zero = reinterpret_cast<const char*>(a.zero[WHICH]) + row0 * metas * Q::meta_bytes;
#pragma unroll
      for (int i = 0; i < N; ++i) {
        const int ri = i * kPass + lane / kPieces;
        const uint32_t r = ri < last ? ri : last;
        x[i] = *reinterpret_cast<const f32x4*>(codes + (r * D + e0) * Q::bits / 8);
        sc[i] = load_meta<SCHEME>(scale + (r * metas + m0) * Q::meta_bytes, 0);
        zr[i] = 0.f;
        if constexpr (!Q::sym) zr[i] = load_meta<SCHEME>(zero + (r * metas + m0) * Q::meta_bytes, 0);
      }
    }
  }
  // (the registers are another's from here on: kept, the last tile's rows would be spilled across every tile)
  __device__ __forceinline__ void drop() {
#pragma unroll
    for (int i = 0; i < N; ++i) x[i] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < (CACHED ? N : 1); ++i) sc[i] = zr[i] = 0.f;
  }
  __device__ __forceinline__ void stage(int lane, char* tile) const {
    const int o = lds_at<DH>(lane / kPieces, lane % kPieces * (CACHED ? Q::epl / 4 : 1));
#pragma unroll
    for (int i = 0; i < N; ++i) {
      if constexpr (!CACHED) {
        *reinterpret_cast<f32x4*>(tile + ((o ^ ((i * kPass & 15) << 4)) + i * kPass * DH * 4)) = x[i];
      } else {
        int c[Q::epl];
        unpack_codes<SCHEME>(__builtin_bit_cast(uint4, x[i]), c);
#pragma unroll
        for (int j = 0; j < Q::epl / 4; ++j) {
          f32x4 y;
#pragma unroll
          for (int e = 0; e < 4; ++e) y[e] = ((float)c[4 * j + e] - zr[i]) * sc[i];
          *reinterpret_cast<f32x4*>(tile + ((o ^ (((i * kPass & 15) ^ j) << 4)) + i * kPass * DH * 4)) = y;
        }
      }
    }
  }
};

template <int SCHEME, int DH>
__global__ __launch_bounds__(64 * kPfWaves, 2) void prefill_attend_kernel(PrefillArgs a) {
  constexpr int NC = DH / 32;            // dimensions of a lane in the second product
  constexpr int kTile = kPfKeys * DH * 4;
  typedef float vec __attribute__((ext_vector_type(NC)));
  // the queries, and a tile of every wavefront (K, then V of the same keys, at the end its output)
  __shared__ __align__(16) char buf[(1 + kPfWaves) * kTile];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);   // uniform: so are its tiles
  const int half = lane >> 5, ln = lane & 31;
  const int b = blockIdx.x / a.n_kv, kvh = blockIdx.x % a.n_kv;
  // With a causal end the last rows see the most keys.  They start first; where all blocks are on the chip at
  // once, two to a compute unit, the second half of them starts with the shortest.
  const int late = ((int)gridDim.y + 1) / 2;
  const bool paired = gridDim.x * gridDim.y * gridDim.z <= 512u;
  const int row_tile = paired && (int)blockIdx.y >= late ? (int)blockIdx.y - late : (int)(gridDim.y - 1 - blockIdx.y);
  const uint32_t r0 = (uint32_t)row_tile * kPfRows, n_rows = (uint32_t)a.n_rows, rep = a.rep;   // rows: below 2^30
  const int Hq = a.n_kv * a.rep;
  char* const tile = buf + (1 + wave) * kTile;

  int64_t cached = 0, base = 0;
  if (a.codes[0] != nullptr) {
    cached = a.fill[b] < a.max_cached ? a.fill[b] : a.max_cached;
    base = a.row_base[b];
  }
  const int64_t own0 = (int64_t)b * a.S;
  const int my_query = r0 + ln < n_rows ? (int)((r0 + ln) / rep) : a.S - 1;
  const uint32_t r_last = r0 + kPfRows < n_rows ? r0 + kPfRows - 1 : n_rows - 1;
  const int own = a.causal ? (int)(r_last / rep) + 1 : a.S;       // own keys some row of the block sees
  const int64_t tiles_cached = (cached + kPfKeys - 1) / kPfKeys;
  const int64_t n_tiles = tiles_cached + (own + kPfKeys - 1) / kPfKeys;
  const int64_t per = (n_tiles + a.n_split - 1) / a.n_split;
  const int64_t t_begin = per * blockIdx.z, t_end = t_begin + per < n_tiles ? t_begin + per : n_tiles;
  // this wavefront's tiles, every fourth: cached ones, then own ones (counted from the first own key)
  const int64_t t_first = t_begin + wave, c_end = t_end < tiles_cached ? t_end : tiles_cached;
  const int64_t c_mine = t_first < c_end ? (c_end - t_first + kPfWaves - 1) / kPfWaves : 0;
  const int64_t o_first = t_first + c_mine * kPfWaves - tiles_cached, o_end = t_end - tiles_cached;

  auto last_row = [](int64_t left) { return left < kPfKeys ? (int)left - 1 : kPfKeys - 1; };
  RowsInFlight<SCHEME, DH, 0, true> kc;
  RowsInFlight<SCHEME, DH, 0, false> ko;
  if (c_mine > 0) kc.load(a, base + t_first * kPfKeys, kvh, last_row(cached - t_first * kPfKeys), lane);
  else if (o_first < o_end) ko.load(a, own0 + o_first * kPfKeys, kvh, last_row(own - o_first * kPfKeys), lane);
  for (int i = threadIdx.x; i < kPfRows * DH / 4; i += 64 * kPfWaves) {
    const uint32_t r = i / (DH / 4), c = i % (DH / 4);
    const uint32_t row = r0 + r < n_rows ? r0 + r : n_rows - 1, t = row / rep;
    *reinterpret_cast<f32x4*>(buf + lds_at<DH>(r, c)) = *reinterpret_cast<const f32x4*>(
        a.q + ((own0 + t) * Hq + kvh * rep + (row - t * rep)) * DH + 4 * c);
  }
  __syncthreads();

  float m = -__builtin_inff(), l = 0.f;
  f32x16 acc[NC];
#pragma unroll
  for (int c = 0; c < NC; ++c)
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[c][i] = 0.f;

  // One tile: its K rows are in `kin`, those of the next tile (at row0 + next, if any) are asked for.
  auto step = [&](auto& kin, auto vin, int64_t row0, int64_t key0, int64_t n_keys, bool more, bool causal) {
    const int lane_t = in_loop(lane), ln_t = lane_t & 31, half_t = lane_t >> 5;
    wave_lds_exchange();                 // the reads of the tile before come first
    kin.stage(lane_t, tile);
    wave_lds_exchange();
    vin.load(a, row0 + key0, kvh, last_row(n_keys - key0), lane_t);   // in flight during the scores
    __builtin_amdgcn_sched_barrier(0);
    f32x16 s;
#pragma unroll
    for (int i = 0; i < 16; ++i) s[i] = 0.f;
    const int row_at = lds_at<DH>(ln_t, half_t * (DH / 8));
    // Operands of the next eight products are read while these eight run.
    f32x4 kf[2][2], qf[2][2];
    auto operands = [&](int g) {
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        kf[g & 1][e] = *reinterpret_cast<const f32x4*>(tile + (row_at ^ ((2 * g + e) << 4)));
        qf[g & 1][e] = *reinterpret_cast<const f32x4*>(buf + (row_at ^ ((2 * g + e) << 4)));
      }
      __builtin_amdgcn_sched_barrier(0);
    };
    operands(0);
#pragma unroll
    for (int g = 0; g < DH / 16; ++g) {
      if (g + 1 < DH / 16) operands(g + 1);
#pragma unroll
      for (int j = 0; j < 8; ++j)
        s = __builtin_amdgcn_mfma_f32_32x32x2f32(kf[g & 1][j >> 2][j & 3], qf[g & 1][j >> 2][j & 3], s, 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
    }
    wave_lds_exchange();
    vin.stage(lane_t, tile);
    wave_lds_exchange();
    if (more) {                          // in flight during the softmax and the values
      const int64_t next = key0 + kPfWaves * kPfKeys;
      kin.load(a, row0 + next, kvh, last_row(n_keys - next), lane_t);
    } else {
      kin.drop();
    }
    __builtin_amdgcn_sched_barrier(0);
    // s[i]: key key0 + 8 (i / 4) + 4 half + i % 4 of row ln, seen by the row if below `seen`
    const int64_t end = !causal || my_query + 1 > n_keys ? n_keys : my_query + 1;
    if (__ballot(end - key0 < kPfKeys) != 0) {
      const int seen = end - key0 < kPfKeys ? (int)(end - key0) : kPfKeys;
#pragma unroll
      for (int i = 0; i < 16; ++i)
        s[i] = 8 * (i >> 2) + 4 * half + (i & 3) < seen ? s[i] * a.scale_qk : -__builtin_inff();
    } else {
#pragma unroll
      for (int i = 0; i < 16; ++i) s[i] *= a.scale_qk;
    }
    float tm = -__builtin_inff();
#pragma unroll
    for (int i = 0; i < 16; ++i) tm = fmaxf(tm, s[i]);
    tm = fmaxf(tm, __shfl_xor(tm, 32, PIKV_WAVE));
    const float mn = fmaxf(m, tm);
    const float ref = mn == -__builtin_inff() ? 0.f : mn;         // nothing seen yet
    const float f = exp_nonpositive(m - ref);
    m = mn;
    l *= f;
    if (__ballot(!(f == 1.f)) != 0) {    // some row's maximum moved
#pragma unroll
      for (int c = 0; c < NC; ++c)
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[c][i] *= f;
    }
    const int key_at = lds_at<DH>(4 * half_t, NC * ln_t / 4) + NC * ln_t % 4 * 4;
    vec vf[2][2];
    auto values = [&](int g) {
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        const int key = 8 * ((2 * g + e) >> 2) + ((2 * g + e) & 3);   // + 4 half
        vf[g & 1][e] = *reinterpret_cast<const vec*>(tile + ((key_at ^ ((key & 15) << 4)) + key * DH * 4));
      }
      __builtin_amdgcn_sched_barrier(0);
    };
    values(0);
#pragma unroll
    for (int g = 0; g < 8; ++g) {
      if (g + 1 < 8) values(g + 1);
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        const float p = exp_nonpositive(s[2 * g + e] - ref);
        l += p;
#pragma unroll
        for (int c = 0; c < NC; ++c) acc[c] = __builtin_amdgcn_mfma_f32_32x32x2f32(vf[g & 1][e][c], p, acc[c], 0, 0, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  if (c_mine > 0) {
    for (int64_t i = 0, t = t_first; i < c_mine; ++i, t += kPfWaves)
      step(kc, RowsInFlight<SCHEME, DH, 1, true>(), base, t * kPfKeys, cached, i + 1 < c_mine, false);
    if (o_first < o_end) ko.load(a, own0 + o_first * kPfKeys, kvh, last_row(own - o_first * kPfKeys), lane);
  }
  for (int64_t t = o_first; t < o_end; t += kPfWaves)
    step(ko, RowsInFlight<SCHEME, DH, 1, false>(), own0, t * kPfKeys, own, t + kPfWaves < o_end, a.causal != 0);
  l += __shfl_xor(l, 32, PIKV_WAVE);

  // merge of the four wavefronts
  __syncthreads();                       // every wavefront is done with its tile and the queries
  float (*const stat)[kPfWaves][kPfRows] = reinterpret_cast<float (*)[kPfWaves][kPfRows]>(buf);
  if (half == 0) { stat[0][wave][ln] = m; stat[1][wave][ln] = l; }
  __syncthreads();
  float mx = -__builtin_inff(), lr = 0.f;
#pragma unroll
  for (int w = 0; w < kPfWaves; ++w) mx = fmaxf(mx, stat[0][w][ln]);
  const float ref = mx == -__builtin_inff() ? 0.f : mx;
  const float f = exp_nonpositive(m - ref);
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const int d0 = NC * (8 * (i >> 2) + 4 * half + (i & 3));
    vec x;
#pragma unroll
    for (int c = 0; c < NC; ++c) x[c] = acc[c][i] * f;
    *reinterpret_cast<vec*>(tile + lds_at<DH>(ln, d0 / 4) + d0 % 4 * 4) = x;
  }
  if (wave == 0) {
#pragma unroll
    for (int w = 0; w < kPfWaves; ++w) lr += stat[1][w][ln] * exp_nonpositive(stat[0][w][ln] - ref);
    if (half == 0) { stat[2][0][ln] = mx; stat[2][1][ln] = lr; }
  }
  __syncthreads();
#pragma unroll
  for (int i = threadIdx.x; i < kPfRows * DH / 4; i += 64 * kPfWaves) {
    const uint32_t r = i / (DH / 4), c = i % (DH / 4);
    if (r0 + r >= n_rows) break;
    f32x4 o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < kPfWaves; ++w) o += *reinterpret_cast<const f32x4*>(buf + (1 + w) * kTile + lds_at<DH>(r, c));
    const float lr = stat[2][1][r];
    if (a.n_split == 1) {
      const uint32_t t = (r0 + r) / rep;
      float* p = a.out + ((own0 + t) * Hq + kvh * rep + (r0 + r - t * rep)) * DH + 4 * c;
      const f32x4 y = {o[0] / lr, o[1] / lr, o[2] / lr, o[3] / lr};
      if (a.out16) {
        *reinterpret_cast<f32x4*>(p) = y;
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) p[e] = y[e];
      }
    } else {
      float* p = a.part + (((int64_t)blockIdx.z * gridDim.x + blockIdx.x) * a.n_rows + r0 + r) * (DH + 2);
#pragma unroll
      for (int e = 0; e < 4; ++e) p[4 * c + e] = o[e];
      if (c == 0) { p[DH] = stat[2][0][r]; p[DH + 1] = lr; }
    }
  }
}

// Key ranges of the blocks that share a row: one wavefront per (sequence, query, head).
__global__ __launch_bounds__(256) void prefill_merge_kernel(PrefillArgs a, int DH, int64_t rows_total) {
  const int lane = threadIdx.x & 63;
  const int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);   // (b * n_kv + kvh) * n_rows + r
  if (row >= rows_total) return;
  const int P = DH + 2;
  float mx = -__builtin_inff();
  for (int s = 0; s < a.n_split; ++s) mx = fmaxf(mx, a.part[(s * rows_total + row) * P + DH]);
  const float ref = mx == -__builtin_inff() ? 0.f : mx;
  float o[2] = {0.f, 0.f}, l = 0.f;
  for (int s = 0; s < a.n_split; ++s) {
    const float* p = a.part + (s * rows_total + row) * P;
    const float f = expf(p[DH] - ref);
    l += p[DH + 1] * f;
    o[0] += p[lane] * f;
    if (DH > 64) o[1] += p[64 + lane] * f;
  }
  const int64_t r = row % a.n_rows, bk = row / a.n_rows;
  const int64_t b = bk / a.n_kv;
  const int h = (int)(bk % a.n_kv) * a.rep + (int)(r % a.rep);
  float* out = a.out + ((b * a.S + r / a.rep) * (a.n_kv * a.rep) + h) * DH;
  out[lane] = o[0] / l;
  if (DH > 64) out[64 + lane] = o[1] / l;
}

// Blocks that share a row's keys.  The chip holds two blocks per compute unit; with fewer rows than that a row's
// keys go to several blocks, but none gets less than eight tiles (two per wavefront) of the longest context.
static int prefill_splits(int64_t blocks, int64_t max_cached, int S) {
  const int64_t tiles = (max_cached + S + kPfKeys - 1) / kPfKeys;
  int64_t n = blocks > 0 ? 512 / blocks : 1;
  if (n > tiles / 8) n = tiles / 8;
  return (int)(n < 1 ? 1 : n > 16 ? 16 : n);
}

template <int SCHEME>
static void launch_prefill(const PrefillArgs& a, int head_dim, int n_seqs, hipStream_t st) {
  const dim3 grid((unsigned)(n_seqs * a.n_kv), (unsigned)((a.n_rows + kPfRows - 1) / kPfRows), (unsigned)a.n_split);
  if (head_dim == 128) hipLaunchKernelGGL((prefill_attend_kernel<SCHEME, 128>), grid, dim3(64 * kPfWaves), 0, st, a);
  else hipLaunchKernelGGL((prefill_attend_kernel<SCHEME, 64>), grid, dim3(64 * kPfWaves), 0, st, a);
}

}  // namespace pikv

using namespace pikv;

extern "C" int64_t pikv_prefill_attend_workspace_bytes(int n_seqs, int S, int n_kv_heads, int n_q_heads, int head_dim,
                                                       int64_t max_cached) {
  if (n_seqs < 1 || S < 1 || n_kv_heads < 1 || n_q_heads < n_kv_heads || max_cached < 0) return 0;
  const int64_t rows = (int64_t)S * (n_q_heads / n_kv_heads);
  const int64_t blocks = (rows + kPfRows - 1) / kPfRows * n_seqs * n_kv_heads;
  const int n = prefill_splits(blocks, max_cached, S);
  return n == 1 ? 0 : (int64_t)n * n_seqs * n_kv_heads * rows * (head_dim + 2) * (int64_t)sizeof(float);
}

extern "C" int pikv_prefill_attend(const float* q, const float* k, const float* v, int n_seqs, int S, int n_kv_heads,
                                   int n_q_heads, int head_dim, int causal, float scale_qk, const void* k_codes,
                                   const void* k_scale, const void* k_zero, const void* v_codes, const void* v_scale,
                                   const void* v_zero, int scheme, int group, const int64_t* cache_row_base,
                                   const int32_t* cache_fill, int64_t max_cached, float* out, void* workspace,
                                   int64_t workspace_bytes, void* stream) {
  if (!q || !k || !v || !out) return PIKV_ERR_NULL;
  if (n_seqs < 1 || S < 1 || n_kv_heads < 1 || n_q_heads < 1 || n_q_heads % n_kv_heads != 0 || max_cached < 0)
    return PIKV_ERR_SHAPE;
  if (head_dim != 64 && head_dim != 128) return PIKV_ERR_UNSUPPORTED;
  if (((uintptr_t)q | (uintptr_t)k | (uintptr_t)v) % 16 != 0) return PIKV_ERR_UNSUPPORTED;   // read as float4
  if (scheme < 0 || scheme > 3) return PIKV_ERR_UNSUPPORTED;
  const bool asym = (scheme == PIKV_Q_I8_ASYM || scheme == PIKV_Q_I4_ASYM);
  const int epl = (scheme == PIKV_Q_I8_SYM || scheme == PIKV_Q_I8_ASYM) ? 16 : 32;
  if (k_codes) {
    if (!k_scale || !v_codes || !v_scale || !cache_row_base || !cache_fill || (asym && (!k_zero || !v_zero)))
      return PIKV_ERR_NULL;
    if (group < epl || !is_pow2(group) || (n_kv_heads * head_dim) % group != 0) return PIKV_ERR_SHAPE;
  }
  PrefillArgs a{};
  a.q = q; a.k = k; a.v = v;
  a.codes[0] = k_codes; a.codes[1] = v_codes;
  a.scale[0] = k_scale; a.scale[1] = v_scale;
  a.zero[0] = k_zero; a.zero[1] = v_zero;
  a.row_base = cache_row_base; a.fill = cache_fill; a.out = out;
  a.max_cached = k_codes ? max_cached : 0;
  a.S = S; a.n_kv = n_kv_heads; a.rep = n_q_heads / n_kv_heads; a.group = k_codes ? group : 1;
  a.causal = causal; a.scale_qk = scale_qk; a.out16 = (uintptr_t)out % 16 == 0;
  a.n_rows = (int64_t)S * a.rep;
  const int64_t need = pikv_prefill_attend_workspace_bytes(n_seqs, S, n_kv_heads, n_q_heads, head_dim, a.max_cached);
  if (need > 0 && (!workspace || workspace_bytes < need)) return PIKV_ERR_WORKSPACE;
  a.part = reinterpret_cast<float*>(workspace);
  const int64_t blocks = (a.n_rows + kPfRows - 1) / kPfRows * n_seqs * n_kv_heads;
  if ((a.n_rows + kPfRows - 1) / kPfRows > 65535 || (int64_t)n_seqs * n_kv_heads > 0x7fffffLL || a.n_rows > 0x3fffffffLL)
    return PIKV_ERR_SHAPE;
  a.n_split = need > 0 ? prefill_splits(blocks, a.max_cached, S) : 1;
  hipStream_t st = (hipStream_t)stream;
  switch (scheme) {
    case PIKV_Q_I8_SYM: launch_prefill<PIKV_Q_I8_SYM>(a, head_dim, n_seqs, st); break;
    case PIKV_Q_I8_ASYM: launch_prefill<PIKV_Q_I8_ASYM>(a, head_dim, n_seqs, st); break;
    case PIKV_Q_I4_ASYM: launch_prefill<PIKV_Q_I4_ASYM>(a, head_dim, n_seqs, st); break;
    default: launch_prefill<PIKV_Q_I4_SYM>(a, head_dim, n_seqs, st); break;
  }
  PIKV_CHECK_LAUNCH();
  if (a.n_split > 1) {
    const int64_t rows_total = (int64_t)n_seqs * a.n_kv * a.n_rows;
    hipLaunchKernelGGL(prefill_merge_kernel, dim3((unsigned)((rows_total + 3) / 4)), dim3(256), 0, st, a, head_dim,
                       rows_total);
    PIKV_CHECK_LAUNCH();
  }
  return PIKV_OK;
}
