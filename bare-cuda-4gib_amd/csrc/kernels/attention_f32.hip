// Causal softmax attention over the paged float32 cache on the matrix cores (float operands and sums, no operand rounded): the
// attention of the 32-bit path.  Keys [page, kv_head, token, dim], values [page, kv_head, dim, token]; head sizes of a multiple
// of 16 up to 128 (beyond, the operands do not fit the registers), pages of a multiple of 4 tokens; attention_generic takes
// everything else.  A row at position p sees key
// j <= p with p - j < window (window 0: every key) and nothing else is read: pages outside may belong to nobody.
//
// Both kernels: a wave holds 16 rows (tokens x the query heads that share a key/value head) and takes keys 16 a block with
// 16x16x4 MFMAs, S^T = K Q^T, so that a lane holds, for its row, four keys of every 16 -- which is the operand of
// O^T += V^T P^T as it lies; running maximum and sum of a row in float, expf.
//
// attention_f32_kernel, requests that bring more than 16 rows: four waves with consecutive rows walk their keys together,
// KT a tile; the tile's keys and values come through registers, asked for a tile ahead, into padded LDS rows.  Bound by the
// matrix cores.  attention_f32_few_kernel, up to 16 rows (decode): eight waves share out a request's tiles of keys, straight from
// memory into operand order, and their sums meet in LDS; bound by the way to memory and back.  Which of the two a
// request's rows take depends on that request alone, and tiles lie at absolute positions: a row's bits do not depend on its
// neighbours in the batch.
//
// At TinyLlama's heads (32 over 4 of 64), one wave a row in plain FMA (attention_generic) -> this: a 1,000-token prompt's call
// 1,328 -> 98 us (2,048 tokens: 5,199 -> 252), one decoded token for each of 8 requests at 130 tokens 29 -> 11 us, at 1,000 152 -> 27.
#include <float.h>
#include <math.h>

#include "api.h"
#include "mfma.h"

namespace bc4g {
namespace {

constexpr int kRowsAWave = 16, kWavesAGroup = 4, kRowsAGroup = kRowsAWave * kWavesAGroup, kThreads = kWavesAGroup * kWave;
constexpr int kFewRows = 16, kFewWaves = 8;

struct AttnF32Args {
  const float* q;
  long q_row;
  const float *k_cache, *v_cache;
  const int32_t* block_table;
  int table_stride;
  const int32_t *seq_start, *seq_ctx;
  float* out;
  int n_heads, n_kv_heads, dim, page_tokens, page_shift, window, n_tiles;
  float scale;
};

__device__ inline floatx4 load_floats(const float* p) { return *reinterpret_cast<const floatx4*>(p); }
__device__ inline floatx4 no_floats() { return floatx4{0.f, 0.f, 0.f, 0.f}; }
// 0 if all four are finite, NaN otherwise
__device__ inline float finite_probe(floatx4 v) { return (v[0] * 0.f + v[1] * 0.f) + (v[2] * 0.f + v[3] * 0.f); }

// The float32 cache, as one key/value head of one request sees it.
struct Paged {
  const int32_t* table;
  int n_kv_heads, kvh, dim, page_tokens, page_shift;
  __device__ long region(int j, int& off) const {
    const int page = page_shift >= 0 ? j >> page_shift : j / page_tokens;
    off = j - page * page_tokens;
    return (static_cast<long>(table[page]) * n_kv_heads + kvh) * page_tokens * dim;
  }
  __device__ long key(int j, int d) const {
    int off;
    const long r = region(j, off);
    return r + static_cast<long>(off) * dim + d;
  }
  __device__ long value(int j, int d) const {
    int off;
    const long r = region(j, off);
    return r + static_cast<long>(d) * page_tokens + off;
  }
};

__device__ inline bool sees(int pos, int j, int window) { return j <= pos && (window <= 0 || pos - j < window); }

// One tile's scores to weights: running maximum m and sum l of the lane's row, sc[kb][i] the score of key j0 + 16 kb + 4 g + i
// before scaling, the weights in its place.  Returns what the sums so far are multiplied by.
template <int KB>
__device__ inline float softmax_tile(floatx4 (&sc)[KB], float& m, float& l, float scale, bool whole, int j0, int g, int pos, int window) {
  float top = m;
#pragma unroll
  for (int kb = 0; kb < KB; ++kb)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      float x = sc[kb][i] * scale;
      if (!whole && !sees(pos, j0 + 16 * kb + 4 * g + i, window)) x = -INFINITY;
      sc[kb][i] = x;
      top = fmaxf(top, x);
    }
  top = four_lanes_max(top);
  const float alpha = expf(m - top);
  m = top;
  float sum = 0.f;
#pragma unroll
  for (int kb = 0; kb < KB; ++kb)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      sc[kb][i] = expf(sc[kb][i] - top);
      sum += sc[kb][i];
    }
  l = l * alpha + sum;
  return alpha;
}

// DB: blocks of 16 dimensions (dim <= 16 DB), KT: keys of a tile.
template <int DB, int KT>
__global__ __launch_bounds__(kThreads, 2) void attention_f32_kernel(const AttnF32Args a) {
  constexpr int KB = KT / 16, KW = DB * 16 + 4, VW = KT + 4;                 // (rows padded: reads of 16 rows side by side meet different banks)
  constexpr int KP = DB * 4, VP = KT / 4;                                    // 16-byte pieces of a key's row, of a dimension's
  constexpr int N = KT * KP / kThreads;                                      // pieces a thread brings, of keys and of values alike
  static_assert(KT * KP % kThreads == 0 && DB * 16 * VP == KT * KP, "whole pieces a thread");
  extern __shared__ __align__(16) float attn_lds[];
  float* k_s = attn_lds;                                                     // [KT][KW]
  float* v_s = attn_lds + KT * KW;                                           // [DB * 16][VW]
  __shared__ int odd_values;                                                 // a tile with values that are not finite: its number + 1
  const int tid = threadIdx.x, lane = tid % kWave, wave = tid / kWave, c = lane % 16, g = lane / 16;
  const int kvh = blockIdx.x % a.n_kv_heads, tile = a.n_tiles - 1 - blockIdx.x / a.n_kv_heads, s = blockIdx.y;
  const int hg = a.n_heads / a.n_kv_heads, start = a.seq_start[s], ctx = a.seq_ctx[s];
  const int rows = (a.seq_start[s + 1] - start) * hg, r0 = tile * kRowsAGroup;
  if (rows <= kFewRows || r0 >= rows) return;
  const Paged cache{a.block_table + static_cast<long>(s) * a.table_stride, a.n_kv_heads, kvh, a.dim, a.page_tokens, a.page_shift};
  const int group_last = ctx + (min(r0 + kRowsAGroup, rows) - 1) / hg;       // the positions of the group's rows
  const int group_first = ctx + r0 / hg;
  const int lo = a.window > 0 && group_first - a.window + 1 > 0 ? group_first - a.window + 1 : 0;

  // this lane's row (a lane beyond the last row repeats it and is dropped at the end), and the range of the wave's positions
  const int row = min(r0 + wave * kRowsAWave + c, rows - 1);
  const bool live = r0 + wave * kRowsAWave + c < rows;
  const int head = kvh * hg + row % hg, pos = ctx + row / hg;
  const long token = start + row / hg;
  const int wave_first = ctx + min(r0 + wave * kRowsAWave, rows - 1) / hg, wave_last = ctx + min(r0 + wave * kRowsAWave + 15, rows - 1) / hg;
  const int wave_lo = a.window > 0 ? wave_first - a.window + 1 : 0;

  floatx4 qf[DB], o[DB];
#pragma unroll
  for (int b = 0; b < DB; ++b) {
    const int d = 16 * b + 4 * g;
    qf[b] = d < a.dim ? load_floats(a.q + token * a.q_row + static_cast<long>(head) * a.dim + d) : no_floats();
    o[b] = no_floats();
  }
  float m = -FLT_MAX, l = 0.f;                                               // (l: this lane's share of the row's sum)
  if (tid == 0) odd_values = 0;

  floatx4 k_next[N], v_next[N];
  auto fetch = [&](int j0) {
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const int idx = tid + i * kThreads, j = j0 + idx / KP, d = idx % KP * 4;
      k_next[i] = j >= lo && j <= group_last && d < a.dim ? load_floats(a.k_cache + cache.key(j, d)) : no_floats();
    }
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const int idx = tid + i * kThreads, j = j0 + idx % VP * 4, d = idx / VP;
      v_next[i] = j + 3 >= lo && j <= group_last && d < a.dim ? load_floats(a.v_cache + cache.value(j, d)) : no_floats();
    }
  };
  fetch(lo - lo % KT);
  for (int j0 = lo - lo % KT; j0 <= group_last; j0 += KT) {
    __syncthreads();                                                         // (the tile before has been read)
    float probe = 0.f;
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const int idx = tid + i * kThreads;
      *reinterpret_cast<floatx4*>(k_s + idx / KP * KW + idx % KP * 4) = k_next[i];
    }
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const int idx = tid + i * kThreads, j = j0 + idx % VP * 4;
      if (j < lo || j + 3 > group_last) {                                    // (nobody's tokens beside somebody's)
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (j + e < lo || j + e > group_last) v_next[i][e] = 0.f;
      }
      probe += finite_probe(v_next[i]);
      *reinterpret_cast<floatx4*>(v_s + idx / VP * VW + idx % VP * 4) = v_next[i];
    }
    if (!(probe == 0.f)) odd_values = j0 + 1;
    __syncthreads();
    if (j0 + KT <= group_last) fetch(j0 + KT);
    if (j0 > wave_last || j0 + KT <= wave_lo) continue;                      // (no row of this wave sees a key of the tile)

    floatx4 sc[KB];
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) sc[kb] = no_floats();
#pragma unroll
    for (int b = 0; b < DB; ++b) {
      floatx4 kf[KB];
#pragma unroll
      for (int kb = 0; kb < KB; ++kb) kf[kb] = load_floats(k_s + (16 * kb + c) * KW + 16 * b + 4 * g);
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int kb = 0; kb < KB; ++kb) sc[kb] = mfma_16x16x4(kf[kb][e], qf[b][e], sc[kb]);
    }
    // (a tile that every row of the wave sees whole needs no mask)
    const bool whole = j0 + KT - 1 <= wave_first && (a.window <= 0 || j0 > wave_last - a.window);
    const float alpha = softmax_tile<KB>(sc, m, l, a.scale, whole, j0, g, pos, a.window);
    if (__any(alpha != 1.0f)) {
#pragma unroll
      for (int b = 0; b < DB; ++b) o[b] *= alpha;
    }
    if (whole || odd_values != j0 + 1) {
#pragma unroll
      for (int kb = 0; kb < KB; ++kb) {
        floatx4 vf[DB];
#pragma unroll
        for (int b = 0; b < DB; ++b) vf[b] = load_floats(v_s + (16 * b + c) * VW + 16 * kb + 4 * g);
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
          for (int b = 0; b < DB; ++b) o[b] = mfma_16x16x4(vf[b][e], sc[kb][e], o[b]);
      }
    } else {
      // Values that are not finite, and rows that must not see them (a weight of zero would still make them NaN): key by key.
#pragma unroll
      for (int kb = 0; kb < KB; ++kb)
        for (int key = 0; key < 16; ++key) {
          const floatx4 w = sc[kb];
          const float mine = key % 4 == 0 ? w[0] : key % 4 == 1 ? w[1] : key % 4 == 2 ? w[2] : w[3];
          const float p = __shfl(mine, c + 16 * (key / 4), kWave);
          const bool seen = sees(pos, j0 + 16 * kb + key, a.window);
#pragma unroll
          for (int b = 0; b < DB; ++b)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
              const float v = v_s[(16 * b + 4 * g + i) * VW + 16 * kb + key];
              if (seen) o[b][i] = fmaf(p, v, o[b][i]);
            }
        }
    }
  }
  l = four_lanes_sum(l);
  if (!live) return;
  const float inv = 1.0f / l;
#pragma unroll
  for (int b = 0; b < DB; ++b) {
    const int d = 16 * b + 4 * g;
    if (d < a.dim) *reinterpret_cast<floatx4*>(a.out + (token * a.n_heads + head) * a.dim + d) = o[b] * inv;
  }
}

// KT keys of a wave's tile; tile t of a request (from position 0) is wave t % 8's.  AHEAD: a tile is asked for while the one
// before it is worked on, where two fit the registers.
template <int DB, int KT, bool AHEAD>
__global__ __launch_bounds__(kFewWaves * kWave) void attention_f32_few_kernel(const AttnF32Args a) {
  constexpr int KB = KT / 16, kPad = 17;
  extern __shared__ __align__(16) float few_lds[];                           // the waves' sums [kFewWaves][DB * 16][kPad]
  __shared__ float m_s[kFewWaves][16], l_s[kFewWaves][16];
  const int tid = threadIdx.x, lane = tid % kWave, c = lane % 16, g = lane / 16;
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int kvh = blockIdx.x, s = blockIdx.y;
  const int hg = a.n_heads / a.n_kv_heads, start = a.seq_start[s], ctx = a.seq_ctx[s];
  const int rows = (a.seq_start[s + 1] - start) * hg;
  if (rows <= 0 || rows > kFewRows) return;
  const Paged cache{a.block_table + static_cast<long>(s) * a.table_stride, a.n_kv_heads, kvh, a.dim, a.page_tokens, a.page_shift};
  const int last = ctx + (rows - 1) / hg;
  const int lo = a.window > 0 && ctx - a.window + 1 > 0 ? ctx - a.window + 1 : 0;
  const int row = min(c, rows - 1), head = kvh * hg + row % hg, pos = ctx + row / hg;
  const long token = start + row / hg;

  struct Tile {
    floatx4 k[KB][DB], v[KB][DB];
  };
  struct Places {                            // where a tile's keys or values lie, and whether they are there
    long at[KB];
    bool ok[KB];
  };
  auto key_places = [&](int j0) {
    Places p;
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) {
      const int j = j0 + 16 * kb + c;
      p.ok[kb] = j >= lo && j <= last;
      p.at[kb] = p.ok[kb] ? cache.key(j, 4 * g) : 0;
    }
    return p;
  };
  auto value_places = [&](int j0) {
    Places p;
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) {
      const int j = j0 + 16 * kb + 4 * g;
      p.ok[kb] = j + 3 >= lo && j <= last;
      p.at[kb] = p.ok[kb] ? cache.value(j, c) : 0;
    }
    return p;
  };
  auto fetch_keys = [&](Tile& t, const Places& places) {
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) {
      const bool ok = places.ok[kb];
      const float* p = a.k_cache + places.at[kb];
#pragma unroll
      for (int b = 0; b < DB; ++b) t.k[kb][b] = ok && 16 * b + 4 * g < a.dim ? load_floats(p + 16 * b) : no_floats();
    }
  };
  auto fetch_values = [&](Tile& t, const Places& places) {
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) {
      const bool ok = places.ok[kb];
      const float* p = a.v_cache + places.at[kb];
#pragma unroll
      for (int b = 0; b < DB; ++b)
        t.v[kb][b] = ok && 16 * b + c < a.dim ? load_floats(p + static_cast<long>(16 * b) * a.page_tokens) : no_floats();
    }
  };
  int j0 = (lo / KT - lo / KT % kFewWaves + wave) * KT;                      // this wave's first tile at or after lo's
  if (j0 < lo - lo % KT) j0 += kFewWaves * KT;
  Tile cur, nxt;
  // The first tile's places are looked up for both before either is asked for: loads come back in the order asked, and a look at the block table
  // behind the keys' loads waited for those (8 requests of 100 tokens, 32 heads of 128: 8.4 -> 8.0 us).  Later tiles' are looked up as they are
  // asked for: with both first 8 heads of 96 over three times 3,000 tokens took 109 us instead of 98, 32 of 128 over eight times 1,000 49 instead of 44.
  const Places first_keys = key_places(j0), first_values = value_places(j0);
  floatx4 qf[DB], o[DB];
#pragma unroll
  for (int b = 0; b < DB; ++b) {
    const int d = 16 * b + 4 * g;
    qf[b] = d < a.dim ? load_floats(a.q + token * a.q_row + static_cast<long>(head) * a.dim + d) : no_floats();
    o[b] = no_floats();
  }
  if (j0 <= last) {
    fetch_keys(cur, first_keys);
    if constexpr (AHEAD) fetch_values(cur, first_values);
  }
  bool first = true;

  float m = -FLT_MAX, l = 0.f;
  for (; j0 <= last; j0 += kFewWaves * KT) {
    const int next = j0 + kFewWaves * KT;
    if (AHEAD && next <= last) {
      fetch_keys(nxt, key_places(next));
      fetch_values(nxt, value_places(next));
    }
    floatx4 sc[KB];
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) sc[kb] = no_floats();
#pragma unroll
    for (int b = 0; b < DB; ++b)
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int kb = 0; kb < KB; ++kb) sc[kb] = mfma_16x16x4(cur.k[kb][b][e], qf[b][e], sc[kb]);
    if constexpr (!AHEAD) fetch_values(cur, first ? first_values : value_places(j0)), first = false;
    const bool whole = j0 + KT - 1 <= ctx && (a.window <= 0 || j0 > last - a.window);
    const float alpha = softmax_tile<KB>(sc, m, l, a.scale, whole, j0, g, pos, a.window);
#pragma unroll
    for (int b = 0; b < DB; ++b) o[b] *= alpha;
    bool odd = false;
    if (!whole) {
      float probe = 0.f;
#pragma unroll
      for (int kb = 0; kb < KB; ++kb) {
        const int j = j0 + 16 * kb + 4 * g;
#pragma unroll
        for (int b = 0; b < DB; ++b) {
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (j + e < lo || j + e > last) cur.v[kb][b][e] = 0.f;           // (nobody's tokens beside somebody's)
          probe += finite_probe(cur.v[kb][b]);
        }
      }
      odd = __any(!(probe == 0.f));
    }
    if (!odd) {
#pragma unroll
      for (int kb = 0; kb < KB; ++kb)
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
          for (int b = 0; b < DB; ++b) o[b] = mfma_16x16x4(cur.v[kb][b][e], sc[kb][e], o[b]);
    } else {                                                                 // (as in the kernel above)
#pragma unroll
      for (int kb = 0; kb < KB; ++kb)
#pragma unroll
        for (int e = 0; e < 4; ++e)
          for (int q = 0; q < 4; ++q) {
            const float p = __shfl(sc[kb][e], c + 16 * q, kWave);
            const bool seen = sees(pos, j0 + 16 * kb + 4 * q + e, a.window);
#pragma unroll
            for (int b = 0; b < DB; ++b)
#pragma unroll
              for (int i = 0; i < 4; ++i) {
                const float v = __shfl(cur.v[kb][b][e], 4 * g + i + 16 * q, kWave);
                if (seen) o[b][i] = fmaf(p, v, o[b][i]);
              }
          }
    }
    if (next <= last) {
      if constexpr (AHEAD) cur = nxt;
      else fetch_keys(cur, key_places(next));
    }
  }
  l = four_lanes_sum(l);
#pragma unroll
  for (int b = 0; b < DB; ++b)
#pragma unroll
    for (int i = 0; i < 4; ++i) few_lds[(wave * DB * 16 + 16 * b + 4 * g + i) * kPad + c] = o[b][i];
  if (g == 0) m_s[wave][c] = m, l_s[wave][c] = l;
  __syncthreads();
  for (int idx = tid; idx < rows * a.dim; idx += kFewWaves * kWave) {
    const int r = idx / a.dim, d = idx % a.dim;
    float top = m_s[0][r];
#pragma unroll
    for (int w = 1; w < kFewWaves; ++w) top = fmaxf(top, m_s[w][r]);
    float sum = 0.f, part = 0.f;
#pragma unroll
    for (int w = 0; w < kFewWaves; ++w) {
      const float by = expf(m_s[w][r] - top);
      sum = fmaf(l_s[w][r], by, sum);
      part = fmaf(few_lds[(w * DB * 16 + d) * kPad + r], by, part);
    }
    a.out[((static_cast<long>(start) + r / hg) * a.n_heads + kvh * hg + r % hg) * a.dim + d] = part * (1.0f / sum);
  }
}

template <int DB, int KT, int FEW_KT, bool AHEAD>
int launch_attention(const AttnF32Args& a, int n_seqs, bool many, bool few, hipStream_t s) {
  constexpr int kLds = (KT * (DB * 16 + 4) + DB * 16 * (KT + 4)) * 4, kFewLds = kFewWaves * DB * 16 * 17 * 4;
  auto kernel = attention_f32_kernel<DB, KT>;
  auto few_kernel = attention_f32_few_kernel<DB, FEW_KT, AHEAD>;
  static std::atomic<bool> raised{false};   // per instantiation: allow more than the default dynamic LDS
  if (!raised) {
    if (hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, kLds) != hipSuccess ||
        hipFuncSetAttribute(reinterpret_cast<const void*>(few_kernel), hipFuncAttributeMaxDynamicSharedMemorySize, kFewLds) != hipSuccess)
      return fail("attention_f32: cannot raise the dynamic LDS limit");
    raised = true;
  }
  if (many) kernel<<<dim3(static_cast<unsigned>(a.n_tiles) * a.n_kv_heads, n_seqs), kThreads, kLds, s>>>(a);
  if (few) few_kernel<<<dim3(a.n_kv_heads, n_seqs), kFewWaves * kWave, kFewLds, s>>>(a);
  return 0;
}

}  // namespace
}  // namespace bc4g

using namespace bc4g;

extern "C" int bc4g_attention_f32(const float* q, int q_stride, float* out, const float* k_cache, const float* v_cache, const int32_t* block_table,
                                  int table_stride, const int32_t* seq_start, const int32_t* seq_ctx, int n_seqs, int most_rows, int few,
                                  int n_heads, int n_kv_heads, int head_dim, int page_tokens, int window, float scale, void* stream) {
  BC4G_REQUIRE(n_seqs >= 0 && n_seqs <= 65535 && most_rows >= 0 && n_heads > 0 && n_kv_heads > 0 && n_heads % n_kv_heads == 0,
               "attention_f32: bad sizes S=%d rows=%d heads=%d/%d", n_seqs, most_rows, n_heads, n_kv_heads);
  BC4G_REQUIRE(head_dim > 0 && head_dim <= 128 && head_dim % 16 == 0, "attention_f32: head_dim=%d must be a multiple of 16 up to 128", head_dim);
  BC4G_REQUIRE(page_tokens > 0 && page_tokens % 4 == 0 && table_stride > 0 && window >= 0,
               "attention_f32: bad cache sizes page_tokens=%d table_stride=%d window=%d", page_tokens, table_stride, window);
  BC4G_REQUIRE(q && out && k_cache && v_cache && block_table && seq_start && seq_ctx && q_stride >= n_heads * head_dim && q_stride % 4 == 0,
               "attention_f32: a tensor is missing, or a row is shorter than its heads");
  BC4G_REQUIRE((reinterpret_cast<uintptr_t>(q) | reinterpret_cast<uintptr_t>(out) | reinterpret_cast<uintptr_t>(k_cache) |
                reinterpret_cast<uintptr_t>(v_cache)) % 16 == 0, "attention_f32: queries, caches and the output must lie on 16-byte boundaries");
  if (n_seqs == 0 || most_rows == 0) return 0;
  const int hg = n_heads / n_kv_heads;
  const long tiles = (static_cast<long>(most_rows) * hg + kRowsAGroup - 1) / kRowsAGroup;
  BC4G_REQUIRE(tiles * n_kv_heads <= 2147483647L, "attention_f32: too many tiles");
  int shift = -1;
  for (int b = 0; b < 31; ++b)
    if (page_tokens == 1 << b) shift = b;
  const AttnF32Args a{q, q_stride, k_cache, v_cache, block_table, table_stride, seq_start, seq_ctx, out, n_heads, n_kv_heads, head_dim,
                      page_tokens, shift, window, static_cast<int>(tiles), scale};
  const bool many = static_cast<long>(most_rows) * hg > kFewRows;
  hipStream_t s = static_cast<hipStream_t>(stream);
  int e = 0;
  if (head_dim <= 32) e = launch_attention<2, 64, 16, true>(a, n_seqs, many, few != 0, s);
  else if (head_dim <= 64) e = launch_attention<4, 64, 16, true>(a, n_seqs, many, few != 0, s);
  else e = launch_attention<8, 32, 16, false>(a, n_seqs, many, few != 0, s);
  if (e) return e;
  return check_launch("attention_f32");
}
