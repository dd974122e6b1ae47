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
// of the chip idle.  A wavefront stages its K tile in LDS along the rows - read straight into the operand layout, a
// lane to a row, a load touched 64 lines and every line came from L2 up to eight times - and reads V along the rows.
//
// Measured, 2 x 500 tokens, 16 heads of 128 over 8 kv heads, kernel time: 45 us for the first chunk and 107 us for
// the second (over 500 cached rows of 8 bits), 59 and 129 us with K read into the operand layout and the longest
// blocks side by side; the two layer calls 1104 us with the score matrix in torch, 541 us now, of which 410 us are
// their projections.  Heads of 128 use all 256 registers and spill: 10 values with 8-bit rows, 26 with 4-bit asymmetric,
// 11 with 4-bit symmetric ones (44, 108 and 48 bytes of scratch a lane); heads of 64 use 200 and spill none.
// Against float64 the error is that of the torch path or below (4.7e-7 and 6.2e-7).
//
// A NaN or infinity in a V row that a query does not see reaches that query only from the query's own last tile (a
// zero probability times it); a product over the whole score matrix spreads it to every row.
#include "common.hpp"

namespace pikv {

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
  int S, n_kv, rep, group, causal, n_split;
  int64_t n_rows;        // S * rep
  float scale_qk;
};

// Orders the LDS accesses of a wavefront's lanes before it against those after it.
__device__ __forceinline__ void wave_lds_exchange() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// The tile's K rows, 16 bytes a lane along the rows, into the wavefront's LDS rows of QP floats.
template <int DH, int QP>
__device__ __forceinline__ void stage_own_k(const float* k, int D, int last, int lane, float* rows) {
  constexpr int LPR = DH / 4, N = kPfKeys * LPR / 64 / 2;   // lanes of a row, rounds of one of two batches
#pragma unroll
  for (int g = 0; g < 2; ++g) {
    float4 x[N];
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const int r = (g * N + i) * (64 / LPR) + lane / LPR;
      x[i] = *reinterpret_cast<const float4*>(k + ((r < last ? r : last) * D + lane % LPR * 4));
    }
#pragma unroll
    for (int i = 0; i < N; ++i)
      *reinterpret_cast<float4*>(rows + ((g * N + i) * (64 / LPR) + lane / LPR) * QP + lane % LPR * 4) = x[i];
    __builtin_amdgcn_sched_barrier(0);   // with all rounds in flight at once more registers spill
  }
}

template <int SCHEME, int DH, int QP>
__device__ __forceinline__ void stage_cached_k(const PrefillArgs& a, int64_t row0, int kvh, int last, int lane, float* rows) {
  using Q = QScheme<SCHEME>;
  constexpr int LPR = DH / Q::epl, N = kPfKeys * LPR / 64 > 0 ? kPfKeys * LPR / 64 : 1;
  const int D = a.n_kv * DH;
  const int e0 = kvh * DH + lane % LPR * Q::epl;
  uint4 w[N];
  float sc[N], zr[N];
#pragma unroll
  for (int i = 0; i < N; ++i) {
    const int r = i * (64 / LPR) + lane / LPR;
    const int64_t row = row0 + (r < last ? r : last);
    w[i] = ld16(reinterpret_cast<const char*>(a.codes[0]) + (row * D + e0) * Q::bits / 8);
    const int64_t mi = row * (D / a.group) + e0 / a.group;
    sc[i] = load_meta<SCHEME>(a.scale[0], mi);
    zr[i] = 0.f;
    if constexpr (!Q::sym) zr[i] = load_meta<SCHEME>(a.zero[0], mi);
  }
#pragma unroll
  for (int i = 0; i < N; ++i) {
    const int r = i * (64 / LPR) + lane / LPR;
    int c[Q::epl];
    unpack_codes<SCHEME>(w[i], c);
#pragma unroll
    for (int j = 0; j < Q::epl / 4; ++j)
      *reinterpret_cast<float4*>(rows + r * QP + lane % LPR * Q::epl + 4 * j) =
          make_float4(((float)c[4 * j] - zr[i]) * sc[i], ((float)c[4 * j + 1] - zr[i]) * sc[i],
                      ((float)c[4 * j + 2] - zr[i]) * sc[i], ((float)c[4 * j + 3] - zr[i]) * sc[i]);
  }
}

// NC = 2 or 4 consecutive dimensions from e0 (a multiple of NC) of a cached V row.
template <int SCHEME, int NC>
__device__ __forceinline__ void cached_v(const PrefillArgs& a, int64_t row, int D, int e0, float (&f)[NC]) {
  using Q = QScheme<SCHEME>;
  const char* p = reinterpret_cast<const char*>(a.codes[1]) + (row * D + e0) * Q::bits / 8;
  uint32_t w;
  if constexpr (NC * Q::bits == 32) w = *reinterpret_cast<const uint32_t*>(p);
  else if constexpr (NC * Q::bits == 16) w = *reinterpret_cast<const uint16_t*>(p);
  else w = *reinterpret_cast<const uint8_t*>(p);
  const int64_t mi = row * (D / a.group) + e0 / a.group;
  const float s = load_meta<SCHEME>(a.scale[1], mi);
  float z = 0.f;
  if constexpr (!Q::sym) z = load_meta<SCHEME>(a.zero[1], mi);
#pragma unroll
  for (int j = 0; j < NC; ++j) {
    const int b = (int)((w >> (Q::bits * j)) & ((1u << Q::bits) - 1u));
    const int c = Q::sym ? (b ^ (1 << (Q::bits - 1))) - (1 << (Q::bits - 1)) : b;
    f[j] = ((float)c - z) * s;
  }
}

template <int SCHEME, int DH>
__global__ __launch_bounds__(64 * kPfWaves, 2) void prefill_attend_kernel(PrefillArgs a) {
  constexpr int NC = DH / 32;            // dimensions of a lane in the second product
  constexpr int QP = DH + 4;             // row pitch in LDS: 16-byte reads of 16 rows touch every bank once
  __shared__ float buf[kPfWaves * kPfRows * QP];   // every wavefront's K tile, at the end its output
  __shared__ float stat[2][kPfWaves][kPfRows];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int half = lane >> 5, ln = lane & 31;
  const int b = blockIdx.x / a.n_kv, kvh = blockIdx.x % a.n_kv;
  // With a causal end the last rows see the most keys.  They start first; where all blocks are on the chip at
  // once, two to a compute unit, the second half of them starts with the shortest.
  const int late = ((int)gridDim.y + 1) / 2;
  const bool paired = gridDim.x * gridDim.y * gridDim.z <= 512u;
  const int tile = paired && (int)blockIdx.y >= late ? (int)blockIdx.y - late : (int)(gridDim.y - 1 - blockIdx.y);
  const int64_t r0 = (int64_t)tile * kPfRows;
  const int Hq = a.n_kv * a.rep, D = a.n_kv * DH;
  float* const krows = buf + wave * kPfRows * QP;

  float qf[DH / 2];                      // DH / 2 dimensions of row ln
  {
    const int64_t r = r0 + ln < a.n_rows ? r0 + ln : a.n_rows - 1;
    const float* p = a.q + (((int64_t)b * a.S + r / a.rep) * Hq + kvh * a.rep + r % a.rep) * DH + half * (DH / 2);
#pragma unroll
    for (int i = 0; i < DH / 8; ++i) {
      const float4 x = *reinterpret_cast<const float4*>(p + 4 * i);
      qf[4 * i] = x.x; qf[4 * i + 1] = x.y; qf[4 * i + 2] = x.z; qf[4 * i + 3] = x.w;
    }
  }

  int64_t cached = 0, base = 0;
  if (a.codes[0] != nullptr) {
    cached = a.fill[b] < a.max_cached ? a.fill[b] : a.max_cached;
    base = a.row_base[b];
  }
  const int my_query = r0 + ln < a.n_rows ? (int)((r0 + ln) / a.rep) : a.S - 1;
  const int64_t r_last = r0 + kPfRows < a.n_rows ? r0 + kPfRows - 1 : a.n_rows - 1;
  const int own = a.causal ? (int)(r_last / a.rep) + 1 : a.S;     // own keys some row of the block sees
  const int64_t tiles_cached = (cached + kPfKeys - 1) / kPfKeys;
  const int64_t n_tiles = tiles_cached + (own + kPfKeys - 1) / kPfKeys;
  const int64_t per = (n_tiles + a.n_split - 1) / a.n_split;
  const int64_t t_begin = per * blockIdx.z, t_end = t_begin + per < n_tiles ? t_begin + per : n_tiles;

  float m = -__builtin_inff(), l = 0.f;
  f32x16 acc[NC];
#pragma unroll
  for (int c = 0; c < NC; ++c)
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[c][i] = 0.f;

  for (int64_t t = t_begin + wave; t < t_end; t += kPfWaves) {
    const bool past = t < tiles_cached;
    const int64_t key0 = (past ? t : t - tiles_cached) * kPfKeys;
    const int64_t n_keys = past ? cached : own;
    // the tile's rows; rows past the end are read from the last one and masked
    const int last = n_keys - key0 < kPfKeys ? (int)(n_keys - key0) - 1 : kPfKeys - 1;
    const int64_t own0 = (((int64_t)b * a.S + key0) * a.n_kv + kvh) * DH;   // of the chunk's own rows
    wave_lds_exchange();                 // the reads of the tile before come first
    if (past) stage_cached_k<SCHEME, DH, QP>(a, base + key0, kvh, last, lane, krows);
    else stage_own_k<DH, QP>(a.k + own0, D, last, lane, krows);
    wave_lds_exchange();
    // V of keys 16 g + 4 half + (0..3) and 16 g + 8 + 4 half + (0..3): the first half of them is in flight
    // during the scores, the second during the softmax
    auto load_v = [&](int g, float (&vf)[8][NC]) {
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const int key = 16 * g + 8 * (i >> 2) + 4 * half + (i & 3);
        const int kv = key < last ? key : last;
        if (past) {
          cached_v<SCHEME, NC>(a, base + key0 + kv, D, kvh * DH + NC * ln, vf[i]);
        } else {
          const float* p = a.v + own0 + (kv * D + NC * ln);
          if constexpr (NC == 4) {
            const float4 x = *reinterpret_cast<const float4*>(p);
            vf[i][0] = x.x; vf[i][1] = x.y; vf[i][2] = x.z; vf[i][3] = x.w;
          } else {
            const float2 x = *reinterpret_cast<const float2*>(p);
            vf[i][0] = x.x; vf[i][1] = x.y;
          }
        }
      }
    };
    float va[8][NC], vb[8][NC];
    load_v(0, va);
    f32x16 s;
#pragma unroll
    for (int i = 0; i < 16; ++i) s[i] = 0.f;
    const float* kp = krows + ln * QP + half * (DH / 2);
#pragma unroll
    for (int i = 0; i < DH / 8; ++i) {
      const float4 x = *reinterpret_cast<const float4*>(kp + 4 * i);
      s = __builtin_amdgcn_mfma_f32_32x32x2f32(x.x, qf[4 * i], s, 0, 0, 0);
      s = __builtin_amdgcn_mfma_f32_32x32x2f32(x.y, qf[4 * i + 1], s, 0, 0, 0);
      s = __builtin_amdgcn_mfma_f32_32x32x2f32(x.z, qf[4 * i + 2], s, 0, 0, 0);
      s = __builtin_amdgcn_mfma_f32_32x32x2f32(x.w, qf[4 * i + 3], s, 0, 0, 0);
      if (i % 8 == 7) __builtin_amdgcn_sched_barrier(0);   // all of the K row in registers would not fit
    }
    load_v(1, vb);
    // s[i]: key key0 + 8 (i / 4) + 4 half + i % 4 of row ln, seen by the row if below `seen`
    const int64_t end = past || !a.causal || my_query + 1 > n_keys ? n_keys : my_query + 1;
    const int seen = end - key0 < kPfKeys ? (int)(end - key0) : kPfKeys;
    float tm = -__builtin_inff();
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      s[i] = 8 * (i >> 2) + 4 * half + (i & 3) < seen ? s[i] * a.scale_qk : -__builtin_inff();
      tm = fmaxf(tm, s[i]);
    }
    tm = fmaxf(tm, __shfl_xor(tm, 32, PIKV_WAVE));
    const float mn = fmaxf(m, tm);
    const float ref = mn == -__builtin_inff() ? 0.f : mn;         // nothing seen yet
    const float f = expf(m - ref);
    m = mn;
    l *= f;
#pragma unroll
    for (int c = 0; c < NC; ++c)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[c][i] *= f;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const float p = expf(s[i] - ref);
      l += p;
#pragma unroll
      for (int c = 0; c < NC; ++c) acc[c] = __builtin_amdgcn_mfma_f32_32x32x2f32(va[i][c], p, acc[c], 0, 0, 0);
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const float p = expf(s[8 + i] - ref);
      l += p;
#pragma unroll
      for (int c = 0; c < NC; ++c) acc[c] = __builtin_amdgcn_mfma_f32_32x32x2f32(vb[i][c], p, acc[c], 0, 0, 0);
    }
  }
  l += __shfl_xor(l, 32, PIKV_WAVE);

  // merge of the four wavefronts
  if (half == 0) { stat[0][wave][ln] = m; stat[1][wave][ln] = l; }
  __syncthreads();                       // also: every wavefront is done with its K tile
  float mx = -__builtin_inff();
#pragma unroll
  for (int w = 0; w < kPfWaves; ++w) mx = fmaxf(mx, stat[0][w][ln]);
  const float f = expf(m - (mx == -__builtin_inff() ? 0.f : mx));
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    float* o = buf + (wave * kPfRows + ln) * QP + NC * (8 * (i >> 2) + 4 * half + (i & 3));
#pragma unroll
    for (int c = 0; c < NC; ++c) o[c] = acc[c][i] * f;
  }
  __syncthreads();
  for (int i = threadIdx.x; i < kPfRows * DH; i += 64 * kPfWaves) {
    const int r = i / DH, d = i % DH;
    if (r0 + r >= a.n_rows) break;
    float mr = -__builtin_inff();
#pragma unroll
    for (int w = 0; w < kPfWaves; ++w) mr = fmaxf(mr, stat[0][w][r]);
    const float rr = mr == -__builtin_inff() ? 0.f : mr;
    float o = 0.f, lr = 0.f;
#pragma unroll
    for (int w = 0; w < kPfWaves; ++w) {
      o += buf[(w * kPfRows + r) * QP + d];
      lr += stat[1][w][r] * expf(stat[0][w][r] - rr);
    }
    if (a.n_split == 1) {
      const int64_t tq = (r0 + r) / a.rep;
      const int h = kvh * a.rep + (int)((r0 + r) % a.rep);
      a.out[(((int64_t)b * a.S + tq) * Hq + h) * DH + d] = o / lr;
    } else {
      float* p = a.part + (((int64_t)blockIdx.z * gridDim.x + blockIdx.x) * a.n_rows + r0 + r) * (DH + 2);
      p[d] = o;
      if (d == 0) { p[DH] = mr; p[DH + 1] = lr; }
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
  a.causal = causal; a.scale_qk = scale_qk;
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
