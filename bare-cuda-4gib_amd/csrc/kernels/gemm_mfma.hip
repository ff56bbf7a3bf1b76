// out[m, n] (+)= sum_k a[m, k] * w[n, k], bfloat16 operands, float accumulation on the matrix
// cores: the product of prompt portions (many rows).
//
// Both operands are contiguous in k.  A workgroup computes a tile of the output in k-steps of 64:
// the rows of a and of w that the tile needs are staged in LDS, every wave reads its fragments there
// and feeds 32x32x16 MFMAs.  Two forms:
//  - the operand tiles go from memory into LDS without passing registers (k a multiple of 64, operands on 16-byte
//    boundaries): gemm_mfma_halves_kernel for tiles of 256 x 256, gemm_mfma_turns_kernel for 256 x 192,
//    gemm_mfma_piped_kernel for 256 x 128, 128 x 128 and 128 x 64 (q|k|v), gemm_mfma_ahead_kernel for 64 x 64 -- and
//    gemm_mfma_direct_kernel for most of them where k is short (short_walk); whichever lets the busiest CU finish first, or two of them
//    side by side (parts_of).
//  - gemm_mfma_staged_kernel: through registers, 128 x 128 tiles; any k that is a multiple of 8.
// Every output element is accumulated over k in ascending order in both, whatever the number of
// rows and the tile: the same bits whichever form and tile a shape selects.  (Products that are added to the residual stream may be cut into
// parts of k by their callers, bc4g_gemm_mfma_parts and _large, whose sums are added up afterwards: other bits, by a rounding of float, and
// whether and into how many depends on the number of rows, up to 3,840 of them for 2,048 outputs.)
// Rows and columns beyond the matrix are not stored.
//
// What bounds these kernels: the loop over k is 85-90 % of a tile's time where k is long.  With all waves of a workgroup reading, waiting and
// multiplying together (gemm_mfma_direct_kernel) the matrix cores are busy 37 to 39 % of a launch (hardware counters); where two groups of waves
// take turns, one multiplying while the other reads, 64 % with many turns of 256 x 256 tiles (2,048 x 28,672 x 4,096), 48 % with
// 256 x 192 (2,048 x 11,264 x 2,048).  LDS has room: a quarter of its clocks, with 1 to 3 % of
// conflicts.  The waves spend 26 to 37 % of their time at the turns' barriers and 36 to 47 % until an instruction is done, and the whole chip's
// power sets the clock: MFMAs on random operands alone run at 1,670 of 2,500 TFLOP/s.  The rest is the stores after the loop, which all
// CUs issue at the same time.
//
// Workgroups are numbered so that those sharing rows of a and of w run on the same XCD at the same
// time (tile_of).
#include <math.h>

#include "api.h"
#include "mfma.h"

namespace bc4g {
namespace {

constexpr int kBM = 128, kBN = 128, kBK = 64;
constexpr int kLdsStride = kBK + 8;   // elements; 144 bytes
constexpr int kXcds = 8;

// kSwigluBf16: every 16 rows of w are eight gate rows and the eight up rows of the same outputs;
// out [m, n / 2] = silu(gate) * up.  A gate and its up lie eight columns apart in the product.
// kRopeKvBf16: w holds query, key and value heads with every head's rows in blocks of 16 (eight dimensions, then their
// rotation partners, which so lie eight columns apart in the product): queries are stored rotated, keys go rotated
// into their pages, values into theirs (operands straight into LDS only).
// kSwigluScaledBf16: the same for rows of a that lack their RMSNorm's common factor (a = bfloat16(residual * g), as the
// product that last added to the residual left it, with every row's sum of squares in parts): a row's sums are
// multiplied by 1 / sqrt(sum of squares / k + eps) before the activation (operands straight into LDS only).
// kSquaredReluBf16: out = max(sum, 0)^2, stored as bfloat16.
// kGegluBf16, kGegluScaledBf16: as the two SwiGLU epilogues, with the gelu written with tanh for the silu.
// kAccumF32 may add a number a column beside the product (bias).
enum Epilogue : int {
  kStoreBf16 = 0, kStoreF32 = 1, kAccumF32 = 2, kSwigluBf16 = 3, kRopeKvBf16 = 4, kSwigluScaledBf16 = 5, kSquaredReluBf16 = 6,
  kGegluBf16 = 7, kGegluScaledBf16 = 8
};
constexpr bool gated(int epi) { return epi == kSwigluBf16 || epi == kSwigluScaledBf16 || epi == kGegluBf16 || epi == kGegluScaledBf16; }
constexpr bool row_scaled(int epi) { return epi == kSwigluScaledBf16 || epi == kGegluScaledBf16; }
template <int EPI>
__device__ inline float gate_act(float z) { return EPI == kGegluBf16 || EPI == kGegluScaledBf16 ? gelu_tanh_quick(z) : silu_quick(z); }

__device__ inline float squared_relu(float v) {
  const float z = fmaxf(v, 0.f);
  return z * z;
}

constexpr int kPartSums = 8;  // chains a row's parts are added in: chain j takes parts j, j + 8, ... in ascending order, and the
                              // chains are added in order of j -- the order of the weight-streaming kernel, so the same factor
struct RowScaleArgs {
  const float* parts;         // [blocks][stride]: block b's share of every row's sum of squares
  int blocks, stride;
  float eps;
  const float* bias;          // kAccumF32: [n], joins every row's sums (null: none)
};
// a patch's rows' sums in LDS ([kPartSums][stride], from the patch's first row on) and what finishes them
struct RowScale {
  const float* sums = nullptr;
  int stride = 0;
  float inv_k = 0.f, eps = 0.f;
};

struct RopeKvArgs {
  const float2* table;        // [m, head_dim / 2] (cos, sin) of every row's position and pair (null: no rotation)
  const int32_t* slot_map;    // [m] page * page_tokens + offset
  bf16_t* k_cache;            // [pages, n_kv, page_tokens, d], or every [page_tokens, d] in fragment order
  bf16_t* v_cache;            // [pages, n_kv, d, page_tokens], or likewise
  int n_heads, n_kv_heads, head_dim, page_tokens, write_kv;
  int fragment_order;         // how the cache's pages are laid out (cache_fragment_order)
  unsigned per_head, per_page;         // for division by head_dim and page_tokens (reciprocal_of)
};

// Which tile a workgroup takes.  Workgroups are dealt to the 8 XCDs in turn, each with an L2 of its
// own: consecutive logical ids stay on one XCD and walk the output in bands of kBand rows of tiles,
// m fastest inside a band -- so the 32 tiles an XCD works on at one time are 8 x 4 of them, which
// share their rows of a and of w in that L2 (with all of m fastest, 8,192 rows were 32 tiles of one
// column, each with rows of a of its own: measured 807 -> 896 TFLOP/s for 8192 x 28672 x 4096).  Totals that are no multiple of 8 give the first XCDs
// one more; dealt out as they came instead, every XCD read all of a and w: 800 rows 2,560 x 2,048 (140 tiles) 19.6 -> 15.9 us, 700 rows
// q|k|v 2,688 x 1,536 (126) 17.5 -> 11.1, 4,096 x 4,096 (192, as before) 35.0.
constexpr int kBand = 8;
__device__ inline void tile_of(int block, int m_blocks, int n_blocks, int& bm, int& bn) {
  const int total = m_blocks * n_blocks, xcd = block % kXcds;
  const int logical = xcd * (total / kXcds) + min(xcd, total % kXcds) + block / kXcds;     // (the first total % kXcds of them have one more)
  const int per_band = kBand * n_blocks;
  const int first = (logical / per_band) * kBand;
  const int rows = min(kBand, m_blocks - first);
  const int in_band = logical % per_band;
  bm = first + in_band % rows;
  bn = in_band / rows;
}

// Stores ROWS x COLS floats (stride COLS + 4) from LDS with the epilogue, THREADS threads together.
template <int EPI, int THREADS, int ROWS, int COLS>
__device__ inline void store_patch(const float* patch, void* __restrict__ out, int m, int n, long m0, long n0, int tid,
                                   const RowScale& rs = RowScale{}, const float* bias = nullptr) {
  constexpr int kStride = COLS + 4;
  if constexpr (gated(EPI)) {
    // (a block of 16 columns -- eight gates, then their eight ups -- a thread: eight outputs, stored at once)
    const long n_out = n / 2;
    for (int c = tid; c < ROWS * (COLS / 16); c += THREADS) {
      const int row = c / (COLS / 16), col = (c % (COLS / 16)) * 16;
      const long gm = m0 + row, gn = n0 + col;
      if (gm >= m || gn >= n) continue;
      const float* src = patch + row * kStride + col;
      const floatx4 g0 = *reinterpret_cast<const floatx4*>(src), g1 = *reinterpret_cast<const floatx4*>(src + 4);
      const floatx4 u0 = *reinterpret_cast<const floatx4*>(src + 8), u1 = *reinterpret_cast<const floatx4*>(src + 12);
      float scale = 1.f;
      if constexpr (row_scaled(EPI)) {
        float ssq = 0.f;
#pragma unroll
        for (int j = 0; j < kPartSums; ++j) ssq += rs.sums[j * rs.stride + row];
        scale = 1.0f / sqrtf(ssq * rs.inv_k + rs.eps);
      }
      float v[8];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        v[e] = gate_act<EPI>(g0[e] * scale) * (u0[e] * scale);
        v[4 + e] = gate_act<EPI>(g1[e] * scale) * (u1[e] * scale);
      }
      bf16_t* dst = static_cast<bf16_t*>(out) + gm * n_out + (gn / 16) * 8;
      if (n_out % 8 == 0) {
        *reinterpret_cast<uint4*>(dst) = make_uint4(pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]), pack_bf16x2(v[4], v[5]), pack_bf16x2(v[6], v[7]));
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e) dst[e] = from_float<bf16_t>(v[e]);
      }
    }
  } else if ((EPI == kStoreBf16 || EPI == kSquaredReluBf16) && n % 8 == 0) {
    // (eight columns a thread, stored at once: 16-byte stores where 8-byte ones were, 108 -> 102 us for a wide product)
    for (int c = tid; c < ROWS * (COLS / 8); c += THREADS) {
      const int row = c / (COLS / 8), col = (c % (COLS / 8)) * 8;
      const long gm = m0 + row, gn = n0 + col;
      if (gm >= m || gn >= n) continue;
      floatx4 v0 = *reinterpret_cast<const floatx4*>(patch + row * kStride + col);
      floatx4 v1 = *reinterpret_cast<const floatx4*>(patch + row * kStride + col + 4);
      if constexpr (EPI == kSquaredReluBf16) {
#pragma unroll
        for (int e = 0; e < 4; ++e) v0[e] = squared_relu(v0[e]), v1[e] = squared_relu(v1[e]);
      }
      *reinterpret_cast<uint4*>(static_cast<bf16_t*>(out) + gm * n + gn) =
          make_uint4(pack_bf16x2(v0[0], v0[1]), pack_bf16x2(v0[2], v0[3]), pack_bf16x2(v1[0], v1[1]), pack_bf16x2(v1[2], v1[3]));
    }
  } else {
    const bool vec = n % 4 == 0;
    for (int c = tid; c < ROWS * (COLS / 4); c += THREADS) {
      const int row = c / (COLS / 4), col = (c % (COLS / 4)) * 4;
      const long gm = m0 + row, gn = n0 + col;
      if (gm >= m || gn >= n) continue;
      floatx4 v = *reinterpret_cast<const floatx4*>(patch + row * kStride + col);
      if constexpr (EPI == kSquaredReluBf16) {
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = squared_relu(v[e]);
      }
      if constexpr (EPI == kAccumF32) {
        if (bias != nullptr) {
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] += gn + e < n ? bias[gn + e] : 0.f;
        }
      }
      const long o = gm * n + gn;
      if (vec) {
        if constexpr (EPI == kStoreBf16 || EPI == kSquaredReluBf16) {
          uint2 pk;
          pk.x = static_cast<uint32_t>(bf16_bits_from_float(v[0])) | (static_cast<uint32_t>(bf16_bits_from_float(v[1])) << 16);
          pk.y = static_cast<uint32_t>(bf16_bits_from_float(v[2])) | (static_cast<uint32_t>(bf16_bits_from_float(v[3])) << 16);
          *reinterpret_cast<uint2*>(static_cast<bf16_t*>(out) + o) = pk;
        } else if constexpr (EPI == kStoreF32) {
          *reinterpret_cast<floatx4*>(static_cast<float*>(out) + o) = v;
        } else {
          floatx4* dst = reinterpret_cast<floatx4*>(static_cast<float*>(out) + o);
          const floatx4 old = *dst;
          *dst = floatx4{old[0] + v[0], old[1] + v[1], old[2] + v[2], old[3] + v[3]};
        }
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          if (gn + e >= n) break;
          if constexpr (EPI == kStoreBf16 || EPI == kSquaredReluBf16) static_cast<bf16_t*>(out)[o + e] = from_float<bf16_t>(v[e]);
          else if constexpr (EPI == kStoreF32) static_cast<float*>(out)[o + e] = v[e];
          else static_cast<float*>(out)[o + e] += v[e];
        }
      }
    }
  }
}

// x / by and what remains, x below 2^31, by a number prepared on the host, R = floor((2^32 - 1) / by): a true division by a number known at run
// time only is 25 instructions, of 64 bits over a hundred.  (R > 2^32 / by - 1 - 1 / by, so x R / 2^32 > x / by - 1: short by one at most.)
inline unsigned reciprocal_of(unsigned by) { return 0xffffffffu / by; }
__device__ inline int divide(int x, int by, unsigned reciprocal, int& rest) {
  unsigned q = __umulhi(static_cast<unsigned>(x), reciprocal), r = static_cast<unsigned>(x) - q * by;
  if (r >= static_cast<unsigned>(by)) r -= by, ++q;
  rest = static_cast<int>(r);
  return static_cast<int>(q);
}

// Where a patch's 32 rows go in the cache, a row a lane (and again in the upper lanes): the part of a key's or value's place that its row gives
// -- the rest comes from its column --, and from which rows on four consecutive tokens lie side by side in fragment order, a bit a row.
struct RowPlaces {
  long key, value;
  unsigned long long quads;
};
__device__ inline RowPlaces row_places(int slot, const RopeKvArgs& ra) {
  int off;
  const long page = divide(slot, ra.page_tokens, ra.per_page, off), first = page * ra.n_kv_heads * ra.page_tokens * ra.head_dim;
  RowPlaces r;
  r.key = first + (ra.fragment_order ? frag_k_offset(off, 0, ra.head_dim) : static_cast<long>(off) * ra.head_dim);
  r.value = first + (ra.fragment_order ? frag_v_offset(off, 0, ra.head_dim) : static_cast<long>(off));
  const bool follow = __shfl_down(slot, 1, kWave) == slot + 1 && __shfl_down(slot, 2, kWave) == slot + 2 && __shfl_down(slot, 3, kWave) == slot + 3;
  r.quads = __ballot(ra.fragment_order && slot % 4 == 0 && follow);
  return r;
}
__device__ inline long from_row(long v, int row) {
  const unsigned lo = __shfl(static_cast<unsigned>(v), row, kWave), hi = __shfl(static_cast<unsigned>(v >> 32), row, kWave);
  return static_cast<long>((static_cast<unsigned long>(hi) << 32) | lo);
}

// The q|k|v epilogue: a wave takes 32 x COLS floats (stride COLS + 4) from LDS, eight neighbouring columns a lane -- a block's eight
// dimensions, or their eight partners --, rotates them with what lies eight columns away in the patch, and stores queries to out
// [m, n_heads * head_dim], keys and values into their pages.  What bounds it is the chain of a lane's items and the vector ALU: with every
// item's place looked up and divided out by itself a tile of keys and values was 2 to 10 us longer than one of queries, and the product with it (us, weights
// from memory, before and now): 268 x 2,560 x 2,048 11.4 and 10.5, 1,000 23.8 and 20.5, 4,096 58 and 51; 2,048 x 6,144 x 4,096 104 and
// 99.5; 2,048 x 12,288 x 4,096 211 and 196, 4,096 363 and 323 (a plain store 184 and 310).
template <int COLS>
__device__ inline void store_patch_rope(const float* patch, bf16_t* __restrict__ out, int m, int n, long m0, long n0, int lane,
                                        const RopeKvArgs& ra, const RowPlaces& places) {
  constexpr int kRows = 32, kStride = COLS + 4;
  const int d = ra.head_dim, first_row = static_cast<int>(m0), first_col = static_cast<int>(n0);
  const long per_head = static_cast<long>(ra.page_tokens) * d;
  if (ra.fragment_order && first_col >= (ra.n_heads + ra.n_kv_heads) * d) {
    // A patch of value columns only, for a cache in fragment order, where four consecutive tokens of one dimension
    // lie side by side: a lane takes one column of four rows, and where those four tokens' places are four in a
    // row from a multiple of four on (a prompt portion's usually are) it stores them at once.
#pragma unroll
    for (int it = 0; it < kRows / 4 * COLS / kWave; ++it) {
      const int c = lane + it * kWave, col = c % COLS, row = (c / COLS) * 4;
      const int gm = first_row + row, gn = first_col + col;
      int dim;
      const int head = divide(min(gn, n - 1), d, ra.per_head, dim) - ra.n_heads - ra.n_kv_heads;
      const long column = head * per_head + (dim / 16) * 256 + (dim % 16) * 4;          // (frag_v_offset's share of the dimension)
      const float* mine = patch + row * kStride + col;
      const uint2 pk = make_uint2(pack_bf16x2(mine[0], mine[kStride]), pack_bf16x2(mine[2 * kStride], mine[3 * kStride]));
      const long at = from_row(places.value, row) + column;
      if (__all(gm + 3 < m && (places.quads >> row & 1))) {        // (the lanes together: what a lane asks of another is asked by all)
        if (gn < n) *reinterpret_cast<uint2*>(ra.v_cache + at) = pk;
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const long to = e == 0 ? at : from_row(places.value, row + e) + column;
          if (gm + e < m && gn < n) ra.v_cache[to].bits = static_cast<uint16_t>(e % 2 ? (e < 2 ? pk.x : pk.y) >> 16 : (e < 2 ? pk.x : pk.y));
        }
      }
    }
    return;
  }
  const bool caches = ra.write_kv && first_col + COLS > ra.n_heads * d;
  constexpr int kItems = kRows * (COLS / 8) / kWave, kTogether = kItems % 2 ? 1 : 2;       // items of a lane; whose angles are asked for together
#pragma unroll
  for (int i0 = 0; i0 < kItems; i0 += kTogether) {
    int row[kTogether], col[kTogether], head[kTogether], dim[kTogether];
    floatx4 cs[kTogether][4];                                  // (cos, sin) of two pairs each
#pragma unroll
    for (int u = 0; u < kTogether; ++u) {
      const int c = lane + (i0 + u) * kWave;
      row[u] = c / (COLS / 8), col[u] = c % (COLS / 8) * 8;
      head[u] = divide(min(first_col + col[u], n - 8), d, ra.per_head, dim[u]);
      if (ra.table != nullptr) {
        const floatx4* from = reinterpret_cast<const floatx4*>(ra.table + static_cast<long>(min(first_row + row[u], m - 1)) * (d / 2) + (dim[u] / 16) * 8);
#pragma unroll
        for (int e = 0; e < 4; ++e) cs[u][e] = from[e];
      }
    }
#pragma unroll
    for (int u = 0; u < kTogether; ++u) {
      const int gm = first_row + row[u], gn = first_col + col[u];
      const bool is_q = head[u] < ra.n_heads, is_v = head[u] >= ra.n_heads + ra.n_kv_heads;
      long key = 0, value = 0;
      if (caches) key = from_row(places.key, row[u]), value = from_row(places.value, row[u]);          // (by every lane)
      if (gm >= m || gn >= n || (!is_q && !ra.write_kv)) continue;
      float v[8];
      const float* mine = patch + row[u] * kStride + col[u];
      {
        const floatx4 v0 = *reinterpret_cast<const floatx4*>(mine), v1 = *reinterpret_cast<const floatx4*>(mine + 4);
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = v0[e], v[4 + e] = v1[e];
      }
      if (ra.table != nullptr && !is_v) {
        const bool first = dim[u] % 16 < 8;                    // a block's eight first halves of pairs; their partners lie 8 further
        const float* partner = first ? mine + 8 : mine - 8;
        const floatx4 o0 = *reinterpret_cast<const floatx4*>(partner), o1 = *reinterpret_cast<const floatx4*>(partner + 4);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const floatx4 a = cs[u][e];
          const float p0 = e < 2 ? o0[2 * e] : o1[2 * e - 4], p1 = e < 2 ? o0[2 * e + 1] : o1[2 * e - 3];
          v[2 * e] = first ? v[2 * e] * a[0] - p0 * a[1] : v[2 * e] * a[0] + p0 * a[1];
          v[2 * e + 1] = first ? v[2 * e + 1] * a[2] - p1 * a[3] : v[2 * e + 1] * a[2] + p1 * a[3];
        }
      }
      const uint4 pk = make_uint4(pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]), pack_bf16x2(v[4], v[5]), pack_bf16x2(v[6], v[7]));
      if (is_q) {
        *reinterpret_cast<uint4*>(out + static_cast<long>(gm) * (ra.n_heads * d) + gn) = pk;
      } else if (!is_v) {      // keys: [page][kv head][token][dim], or in fragment order: eight dimensions of 16 tokens together
        *reinterpret_cast<uint4*>(ra.k_cache + key + (head[u] - ra.n_heads) * per_head + (ra.fragment_order ? frag_k_offset(0, dim[u], d) : dim[u])) = pk;
      } else {                 // values are kept transposed: [page][kv head][dim][token], or in fragment order
        bf16_t* dst = ra.v_cache + value + (head[u] - ra.n_heads - ra.n_kv_heads) * per_head +
                      (ra.fragment_order ? frag_v_offset(0, dim[u], d) : static_cast<long>(dim[u]) * ra.page_tokens);
        const long step = ra.fragment_order ? 4 : ra.page_tokens;
#pragma unroll
        for (int e = 0; e < 8; ++e) dst[e * step].bits = static_cast<uint16_t>(e % 2 ? (&pk.x)[e / 2] >> 16 : (&pk.x)[e / 2]);
      }
    }
  }
}

// ---- operands through registers ---------------------------------------------------------------
// A workgroup of 4 waves computes a 128 x 128 tile.  A tile of each operand is staged in LDS as
// [128 rows][64 k] with rows padded to 144 bytes (which makes the 16-byte fragment reads of
// consecutive lanes cover all banks), in two buffers: while the waves feed MFMAs from one, the next
// k-step is written to the other and the one after it is in flight from memory, in registers.
// Each wave owns a 64 x 64 quarter (2 x 2 MFMA blocks).  Rows, columns and k beyond the matrix are
// read as zero.
struct StagedTile {
  bf16_t a[kBM][kLdsStride];
  bf16_t w[kBN][kLdsStride];
};

template <int EPI>
__global__ __launch_bounds__(256, 2) void gemm_mfma_staged_kernel(
    const bf16_t* __restrict__ a, const bf16_t* __restrict__ w, void* __restrict__ out, int m, int n, int k,
    int m_blocks, int n_blocks, const float* __restrict__ bias) {
  constexpr int SETS = 2, kRows = kBM, kThreads = 256;   // SETS register sets: SETS - 1 k-steps in flight while one is written
  constexpr int kChunkRows = kThreads / 8;           // rows one chunk of a thread's loads covers
  constexpr int kChunksA = kRows / kChunkRows, kChunksW = kBN / kChunkRows;
  typedef StagedTile Tile;
  __shared__ __align__(16) unsigned char lds_raw[sizeof(Tile) * 2];
  Tile* tiles = reinterpret_cast<Tile*>(lds_raw);
  const int tid = threadIdx.x, lane = tid % kWave, wave = tid / kWave;
  const int wm = wave / 2, wn = wave % 2;   // this wave's 64 x 64 part

  int bm, bn;
  tile_of(blockIdx.x, m_blocks, n_blocks, bm, bn);
  const long m0 = static_cast<long>(bm) * kRows, n0 = static_cast<long>(bn) * kBN;

  // global -> LDS: a tile's rows are 8 segments of 16 bytes; thread t moves segment t%8 of rows
  // t/8 + kChunkRows * i (chunk i of each operand; chunks 0..3 carry both where both have as many).
  const int seg = tid % 8, lrow = tid / 8;
  struct Staged {
    uint4 a[kChunksA], w[kChunksW];
  };
  const bf16_t* arow[kChunksA];
  const bf16_t* wrow[kChunksW];
  bool a_ok[kChunksA], w_ok[kChunksW];
#pragma unroll
  for (int i = 0; i < kChunksA; ++i) {
    const long gm = m0 + lrow + kChunkRows * i;
    a_ok[i] = gm < m;
    arow[i] = a + (a_ok[i] ? gm : 0) * k + seg * 8;
  }
#pragma unroll
  for (int i = 0; i < kChunksW; ++i) {
    const long gn = n0 + lrow + kChunkRows * i;
    w_ok[i] = gn < n;
    wrow[i] = w + (w_ok[i] ? gn : 0) * k + seg * 8;
  }
  static_assert(kChunksA == 4, "the loop below moves four chunks a k-step");
  auto load_chunk = [&](Staged& r, int kt, int i) {
    const int kk = kt * kBK;
    const bool k_ok = kk + seg * 8 < k;
    r.a[i] = (k_ok && a_ok[i]) ? load16(arow[i] + kk) : zero16();
    if (i < kChunksW) r.w[i] = (k_ok && w_ok[i]) ? load16(wrow[i] + kk) : zero16();
  };
  auto store_chunk = [&](const Staged& r, int buf, int i) {
    *reinterpret_cast<uint4*>(&tiles[buf].a[lrow + kChunkRows * i][seg * 8]) = r.a[i];
    if (i < kChunksW) *reinterpret_cast<uint4*>(&tiles[buf].w[lrow + kChunkRows * i][seg * 8]) = r.w[i];
  };

  floatx16 acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;

  const int frow = lane % 32, fk = (lane / 32) * 8;

  // Step s of k lives in register set s % SETS on its way from memory.  Iteration t multiplies
  // step t from LDS buffer t % 2; before its MFMAs the wave asks memory for step t + SETS (into the
  // set that step t left in the iteration before), and between its MFMAs it writes step t + 1 to
  // the other buffer, chunk by chunk -- so the memory pipeline, LDS and the matrix cores work at the
  // same time inside one wave, and no register is loaded in the iteration that stores it.
  // (The loop is unrolled over SETS sets x 2 buffers.)
  const int nk = (k + kBK - 1) / kBK;
  Staged r[SETS];
#pragma unroll
  for (int s = 0; s < SETS; ++s)
    if (s < nk) {
#pragma unroll
      for (int i = 0; i < 4; ++i) load_chunk(r[s], s, i);
    }
#pragma unroll
  for (int i = 0; i < 4; ++i) store_chunk(r[0], 0, i);
  if (nk > SETS) {
#pragma unroll
    for (int i = 0; i < 4; ++i) load_chunk(r[0], SETS, i);
  }
  lds_barrier();
  constexpr int kUnroll = SETS % 2 ? 2 * SETS : SETS;
  for (int kt = 0; kt < nk; kt += kUnroll) {
#pragma unroll
    for (int j = 0; j < kUnroll; ++j) {
      const int t = kt + j;
      if (t >= nk) break;
      const int cur = j % 2;
      const bool st = t + 1 < nk;
      // all the k-step's fragments are asked for at once: LDS answers in order, so the MFMAs of the
      // first slice start when its four reads are back while the other twelve are on their way
      uint4 fa[kBK / 16][2], fw[kBK / 16][2];
#pragma unroll
      for (int ks = 0; ks < kBK / 16; ++ks)
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          fa[ks][i] = *reinterpret_cast<const uint4*>(&tiles[cur].a[wm * 64 + i * 32 + frow][ks * 16 + fk]);
          fw[ks][i] = *reinterpret_cast<const uint4*>(&tiles[cur].w[wn * 64 + i * 32 + frow][ks * 16 + fk]);
        }
      __builtin_amdgcn_sched_group_barrier(0x100, 16, 0);   // the 16 LDS reads first
#pragma unroll
      for (int ks = 0; ks < kBK / 16; ++ks)
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
          for (int jj = 0; jj < 2; ++jj) acc[i][jj] = mfma_32x32x16(fa[ks][i], fw[ks][jj], acc[i][jj]);
      __builtin_amdgcn_sched_group_barrier(0x008, 16, 0);   // then the 16 MFMAs
      if (st) {
#pragma unroll
        for (int i = 0; i < 4; ++i) store_chunk(r[(j + 1) % SETS], 1 - cur, i);
      }
      if (t + 1 + SETS < nk) {
#pragma unroll
        for (int i = 0; i < 4; ++i) load_chunk(r[(j + 1) % SETS], t + 1 + SETS, i);
      }
      lds_barrier();
    }
  }

  // The tile goes out through LDS (as float [128][128 + 4]), so that a thread stores four
  // neighbouring columns of a row at once.  acc[i][j][r] is row wm*64 + i*32 + 8*(r/4) + 4*(lane/32)
  // + r%4 and column wn*64 + j*32 + lane%32 of the tile.
  constexpr int kOutStride = kBN + 4;
  static_assert(sizeof(float) * kBM * kOutStride <= sizeof(Tile) * 2, "the output tile must fit the operand buffers");
  float* tile_out = reinterpret_cast<float*>(lds_raw);
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r)
        tile_out[(wm * 64 + i * 32 + 8 * (r / 4) + 4 * (lane / 32) + r % 4) * kOutStride + wn * 64 + j * 32 + lane % 32] =
            acc[i][j][r];
  lds_barrier();
  store_patch<EPI, kThreads, kBM, kBN>(tile_out, out, m, n, m0, n0, tid, RowScale{}, bias);
}

// A tile goes out through LDS so that a thread stores several neighbouring columns of a row at once: every wave for itself,
// 32 rows of its part at a time through a patch of its own (no barrier).  acc[i][j][r] is row i 32 + 8 (r / 4) + 4 (lane / 32) + r % 4 and
// column j 32 + lane % 32 of the part, which begins at (m0, n0); part_sum: see row_scaled (the part's first row's sums, rows of a tile apart).
template <int EPI, int TM, int TN>
__device__ inline void store_part(const floatx16 (&acc)[TM][TN], float* patch, void* __restrict__ out, int m, int n, int k, long m0, long n0, int lane,
                                  const RopeKvArgs& ra, const RowScaleArgs& rows, const float* part_sum = nullptr, int tile_rows = 0) {
  constexpr int kStride = 32 * TN + 4;
  // (q|k|v: the rows' places, where the part has columns of keys or values)
  RowPlaces places{};
  int slot[TM];
  const bool caches = EPI == kRopeKvBf16 && ra.write_kv && n0 + 32 * TN > static_cast<long>(ra.n_heads) * ra.head_dim;
  if (caches) {
#pragma unroll
    for (int i = 0; i < TM; ++i) slot[i] = ra.slot_map[min(m0 + i * 32 + lane % 32, m - 1L)];
  }
#pragma unroll
  for (int i = 0; i < TM; ++i) {
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) patch[(8 * (r / 4) + 4 * (lane / 32) + r % 4) * kStride + j * 32 + lane % 32] = acc[i][j][r];
    if constexpr (EPI == kRopeKvBf16) {
      if (caches) places = row_places(slot[i], ra);
      store_patch_rope<32 * TN>(patch, static_cast<bf16_t*>(out), m, n, m0 + i * 32, n0, lane, ra, places);
    } else if constexpr (row_scaled(EPI))
      store_patch<EPI, kWave, 32, 32 * TN>(patch, out, m, n, m0 + i * 32, n0, lane,
                                           RowScale{part_sum + i * 32, tile_rows, 1.0f / static_cast<float>(k), rows.eps});
    else
      store_patch<EPI, kWave, 32, 32 * TN>(patch, out, m, n, m0 + i * 32, n0, lane, RowScale{}, rows.bias);
  }
}

// ---- operands straight into LDS ---------------------------------------------------------------
// The same product with the operand tiles going from memory into LDS without passing registers
// (global_load_lds_dwordx4: a wave's 64 lanes bring 16 bytes each to 1 KB of consecutive LDS), in a
// ring of STAGES buffers: step t + STAGES - 1 is asked for when step t's multiplication starts, one
// barrier a step.  No registers are spent on staging and no instruction on writing LDS, so twice
// the waves fit a CU, and the forms below are 15-30 % faster than those above on every shape measured
// (2048 x 11264 x 2048: 104 against 131 us; 2048 x 2048 x 5632: 52 against 74; 4096^3: 1,139 against
// 1,015 TFLOP/s).  What did not help: a deeper ring where the tiles fill the chip (three stages are
// slower than two; with fewer tiles than CUs a step is as long as a load takes, and four stages of a
// 64 x 64 tile halve that: 512 x 2048 x 5632 48 -> 28 us), raising the waves' priority around the MFMAs.
//
// The weight comes packed (the weight-streaming kernel's order) and its blocks are copied as they are: see the
// kernel.  The rows of x lie in LDS without padding, BK * 2 bytes each; the 16-byte segment s of row r lies in
// slot s ^ key(r) of its row, key(r) = (r / 2) % 8 for rows of 128 bytes and r % 16 for rows of 256.  A
// fragment read is served sixteen lanes (rows r .. r + 15, one segment) at a time from 64 banks of
// four bytes: two rows of 128 bytes share the banks' span, so the eight rows of one parity must lie
// in eight different slots (with r % 8 as the key rows r and r + 8 met in one bank: counted, half of
// all LDS cycles were conflicts).  A wave-wide load covers 1024 / (BK * 2) rows; which segment a lane
// brings follows from where its 16 bytes land.
//
// WM x WN waves take TM x TN MFMA blocks of 32 x 32 each.  An output element is added up over k in
// ascending order, as in the form above: the same bits whichever form the shape selects.
// k must be a multiple of BK; rows beyond m are read from the last row, blocks beyond n from the last block, and
// not stored.
template <int PER, int MAX>
__device__ inline void wait_for_stage(int later) {
  if constexpr (MAX == 0) {
    wait_loads<0>();
  } else {
    if (later >= MAX) wait_loads<PER * MAX>();
    else wait_for_stage<PER, MAX - 1>(later);
  }
}

template <int ROW_BYTES>
__device__ inline int slot_key(int row) {
  return ROW_BYTES == 128 ? (row >> 1) & 7 : row & 15;
}

template <int WM, int WN, int TM, int TN, int BK, int STAGES>
struct DirectShape {
  static constexpr int kRowsA = 32 * TM * WM, kRowsW = 32 * TN * WN, kRowBytes = BK * 2;
  static constexpr int kWaves = WM * WN, kThreads = 64 * kWaves;
  static constexpr int kStageBytes = (kRowsA + kRowsW) * kRowBytes;
  static constexpr int kPatchBytes = 32 * (32 * TN + 4) * 4;                   // a wave's 32 rows of output, as floats
  static constexpr int kLdsBytes = STAGES * kStageBytes > kWaves * kPatchBytes ? STAGES * kStageBytes : kWaves * kPatchBytes;
  static_assert(kLdsBytes <= 160 * 1024, "a workgroup's LDS");
  static_assert(kRowBytes == 128 || kRowBytes == 256, "rows of 128 or 256 bytes (the slot rule)");
};

// kSwigluScaledBf16: a tile's RA rows' sums of squares from their parts, a chain a thread (its loads all in flight
// together), beside the first operands' way into LDS.  (The compiler's wait for these loads knows nothing of the
// operands asked for before them and so waits for those too: loads return in the order asked.  By the loop's own
// waits, which count the operands' loads alone, these are done.)
template <int RA, int THREADS>
__device__ inline void sum_row_parts(float* part_sum, const RowScaleArgs& rows, int m, long m0, int tid) {
  static_assert(kPartSums * RA % THREADS == 0 && kPartSums * RA / 4 <= THREADS, "whole chains a thread");
  constexpr int kAhead = 16;              // parts of a chain asked for together: one way to memory and back for 128 parts
  // Four rows a thread where the parts' rows allow loads of 16 bytes (a tile begins at a multiple of 64 rows): a CU
  // takes a wave's load every 19 clocks or so, whatever its width, and a row a thread was 128 of them a tile of 64
  // rows and 128 parts -- a microsecond, with the operands' loads waiting among them.
  if (rows.stride % 4 == 0 && reinterpret_cast<uintptr_t>(rows.parts) % 16 == 0) {
    if (tid < kPartSums * RA / 4) {
      const int row = (tid % (RA / 4)) * 4, chain = tid / (RA / 4);
      const bool live = m0 + row < m;     // (then all four are within the stride, which is no less than m)
      const float* p = rows.parts + (live ? m0 + row : 0);
      floatx4 ss = {0.f, 0.f, 0.f, 0.f};
      for (int b0 = chain; b0 < rows.blocks; b0 += kAhead * kPartSums) {
        floatx4 part[kAhead];
#pragma unroll
        for (int i = 0; i < kAhead; ++i) {
          const int b = b0 + i * kPartSums;
          part[i] = live && b < rows.blocks ? *reinterpret_cast<const floatx4*>(p + static_cast<long>(b) * rows.stride)
                                            : floatx4{0.f, 0.f, 0.f, 0.f};
        }
#pragma unroll
        for (int i = 0; i < kAhead; ++i) ss += part[i];        // (in ascending order; a part that is not there adds 0)
      }
      *reinterpret_cast<floatx4*>(part_sum + chain * RA + row) = ss;
    }
  } else
#pragma unroll
  for (int turn = 0; turn < kPartSums * RA / THREADS; ++turn) {
    const int slot = turn * THREADS + tid, row = slot % RA, chain = slot / RA;
    const bool live = m0 + row < m;
    const float* p = rows.parts + (live ? m0 + row : 0);
    float ss = 0.f;
    for (int b0 = chain; b0 < rows.blocks; b0 += kAhead * kPartSums) {
      float part[kAhead];
#pragma unroll
      for (int i = 0; i < kAhead; ++i) {
        const int b = b0 + i * kPartSums;
        part[i] = live && b < rows.blocks ? p[static_cast<long>(b) * rows.stride] : 0.f;
      }
#pragma unroll
      for (int i = 0; i < kAhead; ++i) ss += part[i];          // (in ascending order; a part that is not there adds 0)
    }
    part_sum[slot] = ss;
  }
}

template <int EPI, int WM, int WN, int TM, int TN, int BK, int STAGES, int MINWG>
__global__ __launch_bounds__(64 * WM * WN, MINWG) void gemm_mfma_direct_kernel(
    const bf16_t* __restrict__ a, const bf16_t* __restrict__ w, void* __restrict__ out, int m, int n, int k, int m_blocks,
    int n_blocks, int n_first, const RopeKvArgs ra, const RowScaleArgs rows) {
  typedef DirectShape<WM, WN, TM, TN, BK, STAGES> S;
  constexpr int RA = S::kRowsA, RW = S::kRowsW, RB = S::kRowBytes, NW = S::kWaves;
  constexpr int kGroupRows = 1024 / RB;                    // rows a wave-wide load covers
  constexpr int GA = RA / kGroupRows, GW = RW / kGroupRows, PER = (GA + GW + NW - 1) / NW;
  extern __shared__ __align__(1024) unsigned char direct_lds[];
  const unsigned lds_base = static_cast<unsigned>(
      reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) unsigned char*)direct_lds));   // its LDS address
  const int tid = threadIdx.x, lane = tid % kWave;
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int wm = wave / WN, wn = wave % WN;
  int bm, bn;
  tile_of(blockIdx.x, m_blocks, n_blocks, bm, bn);
  const long m0 = static_cast<long>(bm) * RA, n0 = n_first + static_cast<long>(bn) * RW;
  const int nk = k / BK;
  // The weight comes in the order the weight-streaming kernel reads, so that a model keeps every weight once:
  // [n / 16][k / 32][64 lanes][8] -- blocks of 16 rows x 32 k, 1 KB each, the 16 bytes of row r and k 8 c .. 8 c + 7 at
  // ((r / 16) * (k / 32) + c / 4) * 1024 + ((c % 4) * 16 + r % 16) * 16 (rows beyond n are zeros).  A wave-wide load
  // brings one such block, 1 KB of consecutive memory to 1 KB of consecutive LDS, and the weight's part of a stage is
  // the tile's blocks as they lie in memory, [rows / 16][BK / 32][1 KB]: a fragment read (lane l: row l % 32, k-slot
  // l / 32) takes 16 consecutive rows' 16 bytes side by side, 256 bytes without a bank conflict, and its address is the
  // lane's own offset plus a constant for the slice (no key to fold in, as the rows of x need).
  static_assert(BK % 32 == 0 && RW % 16 == 0, "whole blocks of the packed weight");
  constexpr int kBlocksK = BK / 32;                              // blocks a row block brings every step
  constexpr size_t kPackedStep = static_cast<size_t>(kBlocksK) * 1024;
  static_assert(GW == RW / 16 * kBlocksK, "a wave-wide load of the weight is one block");
  const long w_row_blocks = (static_cast<long>(n) + 15) / 16;

  // the groups of rows (of x) and the blocks (of w) this wave brings every step (a spare turn repeats the last: the
  // same bytes to the same place), and which of a row's segments this lane's 16 bytes of x are
  const int lr = (lane * 16) / RB, ls = (lane * 16 % RB) / 16;
  const unsigned char* src[PER];
  unsigned dst[PER];
  bool piece_of_w[PER];
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    int g = wave + NW * i;
    if (g >= GA + GW) g = GA + GW - 1;
    const bool of_a = g < GA;
    if (of_a) {
      const int trow = g * kGroupRows + lr;
      const int seg = ls ^ slot_key<RB>(trow);
      long row = m0 + trow;
      if (row > m - 1) row = m - 1;
      src[i] = reinterpret_cast<const unsigned char*>(a + row * k) + seg * 16;
      dst[i] = g * 1024;
    } else {
      const int gw = g - GA;
      long block = n0 / 16 + gw / kBlocksK;
      if (block > w_row_blocks - 1) block = w_row_blocks - 1;
      src[i] = reinterpret_cast<const unsigned char*>(w) +
               (block * (k / 32) + gw % kBlocksK) * 1024 + lane * 16;
      dst[i] = RA * RB + gw * 1024;
    }
    piece_of_w[i] = !of_a;                  // (the same in all lanes of the wave)
  }
  auto ask = [&](int step) {
    const unsigned base = lds_base + (step % STAGES) * S::kStageBytes;
    const size_t at_a = static_cast<size_t>(step) * RB, at_w = static_cast<size_t>(step) * kPackedStep;   // once a step
#pragma unroll
    for (int i = 0; i < PER; ++i)
      load_to_lds_16(src[i] + (piece_of_w[i] ? at_w : at_a), __builtin_amdgcn_readfirstlane(base + dst[i]));
  };

  floatx16 acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;

#pragma unroll
  for (int s = 0; s < STAGES - 1; ++s)
    if (s < nk) ask(s);

  const int frow = lane % 32, fhalf = lane / 32;
  int aoff[TM], woff[TN], aswz[TM];
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    const int r = (wm * TM + i) * 32 + frow;
    aoff[i] = r * RB;
    aswz[i] = slot_key<RB>(r);
  }
#pragma unroll
  for (int j = 0; j < TN; ++j) {
    // row r's place in its block of 16, in the block row's first block of the stage; k-slot fhalf of a slice's two
    const int r = (wn * TN + j) * 32 + frow;
    woff[j] = RA * RB + (r / 16) * (kBlocksK * 1024) + (r % 16) * 16 + fhalf * 256;
  }
  constexpr int kSlices = BK / 16;
  uint4 fa[2][TM], fw[2][TN];
  auto read_fragments = [&](int set, const unsigned char* stage, int slice) {
    const int s = slice * 2 + fhalf;
    // the weight's k-slots 2 slice and 2 slice + 1: block (2 slice) / 4 of the row block, 256 bytes a slot in it
    const int w_slice = (slice / 2) * 1024 + (slice % 2) * 512;
#pragma unroll
    for (int i = 0; i < TM; ++i) fa[set][i] = *reinterpret_cast<const uint4*>(stage + aoff[i] + ((s ^ aswz[i]) * 16));
#pragma unroll
    for (int j = 0; j < TN; ++j) fw[set][j] = *reinterpret_cast<const uint4*>(stage + woff[j] + w_slice);
  };

  for (int t = 0; t < nk; ++t) {
    // step t has landed once only the steps asked for after it are outstanding
    wait_for_stage<PER, STAGES - 2>(min(nk - 1, t + STAGES - 2) - t);
    lds_barrier();          // everybody's part of step t is there, and nobody reads step t - 1 any more
    if (t + STAGES - 1 < nk) ask(t + STAGES - 1);
    const unsigned char* stage = direct_lds + (t % STAGES) * S::kStageBytes;
    read_fragments(0, stage, 0);
    __builtin_amdgcn_sched_group_barrier(0x100, TM + TN, 0);
#pragma unroll
    for (int ks = 0; ks < kSlices; ++ks) {
      // the next slice's fragments are asked for before this slice's MFMAs, which hide the wait (the
      // order is pinned: left alone, the compiler moves the reads down to where their registers come free)
      if (ks + 1 < kSlices) {
        read_fragments((ks + 1) % 2, stage, ks + 1);
        __builtin_amdgcn_sched_group_barrier(0x100, TM + TN, 0);
      }
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = mfma_32x32x16(fa[ks % 2][i], fw[ks % 2][j], acc[i][j]);
      __builtin_amdgcn_sched_group_barrier(0x008, TM * TN, 0);
    }
  }
  lds_barrier();            // the last step has been read: LDS is free for the output

  store_part<EPI, TM, TN>(acc, reinterpret_cast<float*>(direct_lds) + wave * (S::kPatchBytes / 4), out, m, n, k, m0 + wm * TM * 32,
                          n0 + wn * TN * 32, lane, ra, rows);
}

// ---- the same, two groups of waves in turns ------------------------------------------------------
// Eight waves, two on every SIMD: while four of them multiply, the other four read their next fragments and ask for operands; a
// barrier ends both and they change places.  (One barrier more at the start sets the second four half a turn behind.)  Fragments are
// waited for before the barrier, so whatever a group has read by the end of its turn may be written over from the turn after
// the other group's, and what has been asked for is waited for (by hand: wait_loads) in the turn before it is read, by the waves that
// asked, in time for both groups.  The parts of the output and their order over k are those of the kernel above.
#define BC4G_TURN(waits)                                   \
  do {                                                     \
    __builtin_amdgcn_sched_barrier(0);                     \
    asm volatile(waits "s_barrier" ::: "memory");          \
    __builtin_amdgcn_sched_barrier(0);                     \
  } while (0)
#define BC4G_READ "s_waitcnt lgkmcnt(0)\n\t"

// N loads of a wave to N KB of LDS side by side, load i from bases[i] (the same in every lane) plus each lane's offset.  The LDS address
// is set once and each load adds i * 1,024 bytes to it, and to its memory address, so its base is that much short of its place.  (The offset
// field reaches from -4,096 to 4,095: five loads count from the middle one's address.)
constexpr int kMaxLoads = 5;
template <int N, bool PAST = false>
__device__ inline void load_side_by_side(const void* const (&bases)[kMaxLoads], const unsigned (&off)[kMaxLoads], unsigned lds_address) {
  static_assert(N == 2 || N == 4 || N == 5, "loads a statement");
  static_assert(N == 4 || !PAST, "past the caches: four");
#define BC4G_LOAD(v, s, o) "global_load_lds_dwordx4 %" #v ", %" #s " offset:" #o "\n\t"
#define BC4G_LOAD_PAST(v, s, o) "global_load_lds_dwordx4 %" #v ", %" #s " offset:" #o " nt\n\t"
  if constexpr (PAST) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\t" BC4G_LOAD_PAST(1, 5, 0) BC4G_LOAD_PAST(2, 6, 1024) BC4G_LOAD_PAST(3, 7, 2048) BC4G_LOAD_PAST(4, 8, 3072)
                 ::"s"(lds_address), "v"(off[0]), "v"(off[1]), "v"(off[2]), "v"(off[3]), "s"(bases[0]), "s"(bases[1]), "s"(bases[2]), "s"(bases[3])
                 : "memory", "m0");
  } else if constexpr (N == 2) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\t" BC4G_LOAD(1, 3, 0) BC4G_LOAD(2, 4, 1024)
                 ::"s"(lds_address), "v"(off[0]), "v"(off[1]), "s"(bases[0]), "s"(bases[1]) : "memory", "m0");
  } else if constexpr (N == 4) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\t" BC4G_LOAD(1, 5, 0) BC4G_LOAD(2, 6, 1024) BC4G_LOAD(3, 7, 2048) BC4G_LOAD(4, 8, 3072)
                 ::"s"(lds_address), "v"(off[0]), "v"(off[1]), "v"(off[2]), "v"(off[3]), "s"(bases[0]), "s"(bases[1]), "s"(bases[2]), "s"(bases[3])
                 : "memory", "m0");
  } else {
    const void* b[5];
#pragma unroll
    for (int i = 0; i < 5; ++i) b[i] = static_cast<const unsigned char*>(bases[i]) + 2048;
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\t" BC4G_LOAD(1, 6, -2048) BC4G_LOAD(2, 7, -1024) BC4G_LOAD(3, 8, 0) BC4G_LOAD(4, 9, 1024)
                 BC4G_LOAD(5, 10, 2048)
                 ::"s"(lds_address + 2048), "v"(off[0]), "v"(off[1]), "v"(off[2]), "v"(off[3]), "v"(off[4]), "s"(b[0]), "s"(b[1]), "s"(b[2]),
                 "s"(b[3]), "s"(b[4]) : "memory", "m0");
  }
#undef BC4G_LOAD_PAST
#undef BC4G_LOAD
}

// 256 x 256: a wave's part is 128 x 64, and a step of 64 two turns: its first 64 rows by its columns, then the other 64.  So
// a turn is 16 MFMAs, its reads 16 of 1 KB (or 8: the weight's fragments stay), and the two stages of 64 KB are written over in pieces as
// they are read: the weight and the first rows of a step are asked for a step and a half before they are read, the other
// rows as well.  LDS: a stage is the first rows of both row parts, the other rows, then the weight likewise by columns.
// Against 16 waves that read and multiply together (weights from memory): 2,048 x 28,672 x 4,096 437 -> 387 us, 15,400 x 12,288 x 4,096
// 1,440 -> 1,210 (1,040 -> 1,280 TFLOP/s), 8,192^3 960 -> 800.  Four turns of eight MFMAs a step: 3-5 % slower; four waves of 128 x 128 on
// a SIMD each: 15-20 % slower; the waves' priority raised around the MFMAs: the same.
struct HalvesShape {
  static constexpr int kThreads = 512, kHalf = 16 * 1024, kStage = 4 * kHalf;
  static constexpr int kPatchBytes = 32 * (64 + 4) * 4, kLdsBytes = 2 * kStage;
  static_assert(8 * kPatchBytes <= kLdsBytes, "the output's patches take the stages' place");
};

template <int EPI>
__device__ __forceinline__ void halves_tile(const bf16_t* __restrict__ a, const bf16_t* __restrict__ w, void* __restrict__ out, int m, int n, int k,
                                            long m0, long n0, const RopeKvArgs& ra, const RowScaleArgs& rows) {
  typedef HalvesShape S;
  extern __shared__ __align__(1024) unsigned char direct_lds[];
  const unsigned lds_base = static_cast<unsigned>(
      reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) unsigned char*)direct_lds));
  const int tid = threadIdx.x, lane = tid % kWave;
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int wm = wave / 4, wn = wave % 4;
  const int nk = k / 64;

  // What this wave brings of a half of x: 16 of its 128 rows, in two loads (rows past m: the last).  Of a half of the weight: the step's
  // two blocks of one block row (past n: of the last), 2 KB of memory side by side.
  const unsigned char* abase = reinterpret_cast<const unsigned char*>(a + m0 * k);
  unsigned aoff[2][2];
  const unsigned char* wbase[2];
  const long w_row_blocks = (static_cast<long>(n) + 15) / 16;
#pragma unroll
  for (int h = 0; h < 2; ++h) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int hr = (2 * wave + i) * 8 + lane / 8;                 // row of the half,
      const int trow = (hr / 64) * 128 + h * 64 + hr % 64;          // of the tile
      const long row = min(static_cast<long>(m) - 1 - m0, static_cast<long>(trow));
      aoff[h][i] = static_cast<unsigned>(row * k * 2 + ((lane % 8) ^ slot_key<128>(hr)) * 16);
    }
    const long block = min(w_row_blocks - 1, n0 / 16 + (wave / 2) * 4 + h * 2 + wave % 2);
    wbase[h] = reinterpret_cast<const unsigned char*>(w) + block * (k / 32) * 1024;
  }
  auto ask = [&](const unsigned char* first, const unsigned char* second_less_1k, unsigned off0, unsigned off1, unsigned to) {
    const void* bases[kMaxLoads] = {first, second_less_1k};
    const unsigned off[kMaxLoads] = {off0, off1};
    load_side_by_side<2>(bases, off, to);
  };
  auto ask_a = [&](int step, int h) {
    const unsigned char* p = abase + static_cast<size_t>(step) * 128;
    ask(p, p - 1024, aoff[h][0], aoff[h][1], lds_base + (step & 1) * S::kStage + h * S::kHalf + wave * 2048);
  };
  auto ask_w = [&](int step, int h) {
    const unsigned char* p = wbase[h] + static_cast<size_t>(step) * 2048;
    ask(p, p, lane * 16, lane * 16, lds_base + (step & 1) * S::kStage + (2 + h) * S::kHalf + wave * 2048);
  };

  floatx16 acc[4][2];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;

  const int frow = lane % 32, fhalf = lane / 32;
  const unsigned char* aread = direct_lds + (wm * 64 + frow) * 128;
  const int akey = slot_key<128>(wm * 64 + frow);       // (the same 32 rows further)
  const unsigned char* wread = direct_lds + 2 * S::kHalf + (wn * 2 + frow / 16) * 2048 + (frow % 16) * 16 + fhalf * 256;
  uint4 fa[2][4], fw[2][4];
  auto read_a = [&](int buf, int h) {
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
      for (int i = 0; i < 2; ++i)
        fa[i][s] = *reinterpret_cast<const uint4*>(aread + buf * S::kStage + h * S::kHalf + i * 4096 + (((s * 2 + fhalf) ^ akey) * 16));
  };
  auto read_w = [&](int buf) {
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
      for (int h = 0; h < 2; ++h)
        fw[h][s] = *reinterpret_cast<const uint4*>(wread + buf * S::kStage + h * S::kHalf + (s / 2) * 1024 + (s % 2) * 512);
  };
  auto multiply = [&](int i0) {
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i0 + i][j] = mfma_32x32x16(fa[i][s], fw[j][s], acc[i0 + i][j]);
  };
  // A wave's loads in the order asked: ... W(t), first rows (t), other rows (t) ... in 4 + 2 + 2.  In the first turn of step t the
  // other rows of t are waited for (behind them: 6 of t + 1 and the 2 just asked for), in the second W and the first rows of t + 1
  // (behind them: 2 of t + 1 and the 6 of t + 2).
  auto step = [&](int t, int buf) {
    read_w(buf);
    read_a(buf, 0);
    if (t + 1 < nk) ask_a(t + 1, 1);
    if (t + 2 < nk) wait_loads<8>(); else wait_loads<0>();
    BC4G_TURN(BC4G_READ);
    multiply(0);
    BC4G_TURN("");
    read_a(buf, 1);
    if (t + 2 < nk) {
      ask_w(t + 2, 0), ask_w(t + 2, 1), ask_a(t + 2, 0);
      wait_loads<8>();
    } else {
      wait_loads<0>();
    }
    BC4G_TURN(BC4G_READ);
    multiply(2);
    BC4G_TURN("");
  };

  ask_w(0, 0), ask_w(0, 1), ask_a(0, 0), ask_a(0, 1);
  if (nk > 1) {
    ask_w(1, 0), ask_w(1, 1), ask_a(1, 0);
    wait_loads<8>();
  } else {
    wait_loads<0>();
  }
  BC4G_TURN("");
  if (wm == 1) BC4G_TURN("");
  for (int t = 0; t < nk; t += 2) {
    step(t, 0);
    if (t + 1 < nk) step(t + 1, 1);
  }
  if (wm == 0) BC4G_TURN("");
  lds_barrier();            // the last step has been read: LDS is free for the output
  store_part<EPI, 4, 2>(acc, reinterpret_cast<float*>(direct_lds) + wave * (S::kPatchBytes / 4), out, m, n, k, m0 + wm * 128, n0 + wn * 64, lane, ra,
                        rows);
}

template <int EPI>
__global__ __launch_bounds__(512, 2) void gemm_mfma_halves_kernel(const bf16_t* __restrict__ a, const bf16_t* __restrict__ w,
                                                                  void* __restrict__ out, int m, int n, int k, int m_blocks, int n_blocks,
                                                                  int n_first, const RopeKvArgs ra, const RowScaleArgs rows) {
  int bm, bn;
  tile_of(blockIdx.x, m_blocks, n_blocks, bm, bn);
  halves_tile<EPI>(a, w, out, m, n, k, bm * 256L, n_first + bn * 256L, ra, rows);
}

// A turn is a step of BK, in a ring of STAGES: 256 x 192 (steps of 32: what LDS holds five of).  Against gemm_mfma_direct_kernel, 2,048 x 11,264 x 2,048:
// 102 -> 96 us; with fragments slices ahead (piped_tile) 91 to 102, level.  (256 x 256 so: 5 % slower than in halves.)
template <int WM, int WN, int TM, int TN, int BK, int STAGES>
struct TurnsShape {
  static constexpr int kRowsA = 32 * TM * WM, kRowsW = 32 * TN * WN, kRowBytes = BK * 2;
  static constexpr int kThreads = 512, kStageBytes = (kRowsA + kRowsW) * kRowBytes;
  static constexpr int kPatchBytes = 32 * (32 * TN + 4) * 4;                   // a wave's 32 rows of output, as floats
  static constexpr int kLdsBytes = STAGES * kStageBytes > 8 * kPatchBytes ? STAGES * kStageBytes : 8 * kPatchBytes;
  static constexpr int kGroupsA = kRowsA * kRowBytes / 1024, kGroupsW = kRowsW * kRowBytes / 1024;
  static constexpr int kLoads = (kGroupsA + kGroupsW + 7) / 8;                 // a wave's a step
  static_assert(WM * WN == 8 && kLdsBytes <= 160 * 1024 && (BK == 32 || BK == 64) && STAGES >= 3, "eight waves, LDS, rows of 64 or 128 bytes");
};
// which 16-byte slot of its row a segment of x lies in (rows of 64 bytes: four of them share the banks' span)
template <int ROW_BYTES>
__device__ inline int turns_key(int row) {
  return ROW_BYTES == 64 ? (row >> 2) & 3 : slot_key<128>(row);
}

template <int EPI, int WM, int WN, int TM, int TN, int BK, int STAGES>
__device__ __forceinline__ void turns_tile(const bf16_t* __restrict__ a, const bf16_t* __restrict__ w, void* __restrict__ out, int m, int n, int k,
                                           long m0, long n0, const RopeKvArgs& ra, const RowScaleArgs& rows) {
  typedef TurnsShape<WM, WN, TM, TN, BK, STAGES> S;
  constexpr int RA = S::kRowsA, RW = S::kRowsW, RB = S::kRowBytes, N = S::kLoads, kBlocksK = BK / 32, kSlices = BK / 16;
  constexpr int kGroupRows = 1024 / RB;                    // rows of x a wave-wide load covers
  extern __shared__ __align__(1024) unsigned char direct_lds[];
  const unsigned lds_base = static_cast<unsigned>(
      reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) unsigned char*)direct_lds));
  const int tid = threadIdx.x, lane = tid % kWave;
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int wm = wave / WN, wn = wave % WN;
  const int nk = k / BK;

  // the N groups of rows (of x) or blocks (of w) this wave brings every step, side by side in LDS (waves past the last group bring
  // the last ones again: the same bytes to the same place); rows past m and blocks past n: the last
  const int g0 = min(wave * N, S::kGroupsA + S::kGroupsW - N);
  const unsigned char* base[kMaxLoads];
  unsigned off[kMaxLoads];
  int advance[kMaxLoads];
  const long w_row_blocks = (static_cast<long>(n) + 15) / 16;
#pragma unroll
  for (int i = 0; i < N; ++i) {
    const int g = g0 + i;
    if (g < S::kGroupsA) {
      const int trow = g * kGroupRows + lane * 16 / RB;
      const long row = min(static_cast<long>(m) - 1 - m0, static_cast<long>(trow));
      base[i] = reinterpret_cast<const unsigned char*>(a + m0 * k) - i * 1024;
      off[i] = static_cast<unsigned>(row * k * 2 + ((lane * 16 % RB / 16) ^ turns_key<RB>(trow)) * 16);
      advance[i] = RB;
    } else {
      const int gw = g - S::kGroupsA;
      const long block = min(w_row_blocks - 1, n0 / 16 + gw / kBlocksK);
      base[i] = reinterpret_cast<const unsigned char*>(w) + (block * (k / 32) + gw % kBlocksK) * 1024 - i * 1024;
      off[i] = lane * 16;
      advance[i] = kBlocksK * 1024;
    }
  }
  auto ask = [&](int slot) {                               // the next step's
    const void* from[kMaxLoads];
#pragma unroll
    for (int i = 0; i < N; ++i) from[i] = base[i], base[i] += advance[i];
    load_side_by_side<N>(from, off, lds_base + slot * S::kStageBytes + g0 * 1024);
  };

  floatx16 acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;

  const int frow = lane % 32, fhalf = lane / 32;
  const unsigned char* aread = direct_lds + (wm * TM * 32 + frow) * RB;
  const int akey = turns_key<RB>(frow);                    // (the same 32 rows further)
  const unsigned char* wread = direct_lds + RA * RB + (wn * TN * 2 + frow / 16) * (kBlocksK * 1024) + (frow % 16) * 16 + fhalf * 256;
  uint4 fa[TM][kSlices], fw[TN][kSlices];

#pragma unroll
  for (int s = 0; s < STAGES - 1; ++s)
    if (s < nk) ask(s);
  if (nk >= STAGES - 1) wait_loads<N * (STAGES - 2)>(); else wait_loads<0>();
  BC4G_TURN("");
  if (wave >= 4) BC4G_TURN("");
  int slot = 0, free_slot = STAGES - 1;                    // (both groups have read step t - 1 when one of them comes to step t)
  for (int t = 0; t < nk; ++t) {
#pragma unroll
    for (int s = 0; s < kSlices; ++s) {
#pragma unroll
      for (int j = 0; j < TN; ++j)
        fw[j][s] = *reinterpret_cast<const uint4*>(wread + slot * S::kStageBytes + j * 2 * kBlocksK * 1024 + (s / 2) * 1024 + (s % 2) * 512);
#pragma unroll
      for (int i = 0; i < TM; ++i)
        fa[i][s] = *reinterpret_cast<const uint4*>(aread + slot * S::kStageBytes + i * 32 * RB + (((s * 2 + fhalf) ^ akey) * 16));
    }
    if (t + STAGES - 1 < nk) {
      ask(free_slot);
      wait_loads<N * (STAGES - 2)>();                      // step t + 1 is there
    } else {
      wait_loads<0>();
    }
    BC4G_TURN(BC4G_READ);
#pragma unroll
    for (int s = 0; s < kSlices; ++s)
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = mfma_32x32x16(fa[i][s], fw[j][s], acc[i][j]);
    BC4G_TURN("");
    free_slot = slot;
    if (++slot == STAGES) slot = 0;
  }
  if (wave < 4) BC4G_TURN("");
  lds_barrier();            // the last step has been read: LDS is free for the output
  store_part<EPI, TM, TN>(acc, reinterpret_cast<float*>(direct_lds) + wave * (S::kPatchBytes / 4), out, m, n, k, m0 + wm * TM * 32,
                          n0 + wn * TN * 32, lane, ra, rows);
}
#undef BC4G_TURN
#undef BC4G_READ

template <int EPI, int WM, int WN, int TM, int TN, int BK, int STAGES>
__global__ __launch_bounds__(512, 2) void gemm_mfma_turns_kernel(const bf16_t* __restrict__ a, const bf16_t* __restrict__ w,
                                                                 void* __restrict__ out, int m, int n, int k, int m_blocks, int n_blocks,
                                                                 int n_first, const RopeKvArgs ra, const RowScaleArgs rows) {
  typedef TurnsShape<WM, WN, TM, TN, BK, STAGES> S;
  int bm, bn;
  tile_of(blockIdx.x, m_blocks, n_blocks, bm, bn);
  turns_tile<EPI, WM, WN, TM, TN, BK, STAGES>(a, w, out, m, n, k, static_cast<long>(bm) * S::kRowsA, n_first + static_cast<long>(bn) * S::kRowsW, ra, rows);
}

// ---- fragments slices ahead ----------------------------------------------------------------------
// Tiles of 256 x 128 and 128 x 128, and the 64 x 256 ones beside whole tiles: eight waves of 64 x 64, 64 x 32 or 32 x 64 (128 x 64 for q|k|v: 32 x 32).  Every wave goes by itself: a step of 64 k
// is four slices of 16, and while a slice's MFMAs run the wave reads the fragments of two slices on, so that it never waits for LDS; one barrier
// a step, when the last fragments of the step have been read, behind which its stage is asked for anew.  All loads of a step share two LDS addresses.
// What bounds it: with one tile a CU, the chain of 64 k / 64 steps at 0.33 us (128 x 128; 0.22 of it MFMAs) or 0.63 us (256 x 128; 0.43 of it
// MFMAs); with the chip full, its power.  Against all waves reading, waiting and multiplying together (256 x 128) and two groups of waves taking turns
// (128 x 128), which took 0.79 us and 0.38 us a step; weights from memory: 256 x 128 at 2,048 rows, 4,096 x 2,048 39.7 -> 31.6 us, 4,096 x 14,336
// 248 -> 215, 130 rows 28,672 x 4,096 68.4 -> 60.9; 128 x 128 at 300 rows, 2,048 x 2,048 18.7 -> 15.4, 1,000 rows 21.8 -> 18.7, 2,048 rows 2,048 x 5,632
// 56.8 -> 54.2.  Slower: one slice ahead (256 x 128 37), four waves of 64 x 64 on 128 x 128 (30.0 where eight take 26.2); and
// 256 x 256 so is, with its 16 waves or 128 x 64 a wave, no faster than waves taking turns.
template <int WM, int WN, int TM, int TN, int STAGES>
struct PipedShape {
  static constexpr int kRowsA = 32 * TM * WM, kRowsW = 32 * TN * WN, kWaves = WM * WN, kThreads = 64 * kWaves;
  static constexpr int kBytesA = kRowsA * 128, kStageBytes = kBytesA + kRowsW * 128;
  static constexpr int kPieceA = kRowsA / 8 / kWaves, kPieceW = kRowsW / 8 / kWaves, kPieces = kPieceA + kPieceW;
  static constexpr int kPatchBytes = 32 * (32 * TN + 4) * 4;
  static constexpr int kLdsBytes = STAGES * kStageBytes > kWaves * kPatchBytes ? STAGES * kStageBytes : kWaves * kPatchBytes;
  static_assert(kRowsA % (8 * kWaves) == 0 && kRowsW % (8 * kWaves) == 0 && kLdsBytes <= 160 * 1024, "whole loads a wave; a workgroup's LDS");
};

// The tile whose first row and column are m0 and n0 (the rows there are and whole blocks of them), over nk steps from first_step on.
template <int EPI, int WM, int WN, int TM, int TN, int STAGES>
__device__ __forceinline__ void piped_tile(const bf16_t* __restrict__ a, const bf16_t* __restrict__ w, void* __restrict__ out, int m, int n, int k, long m0,
                                           long n0, int first_step, int nk, const RopeKvArgs& ra, const RowScaleArgs& rows) {
  typedef PipedShape<WM, WN, TM, TN, STAGES> S;
  constexpr int kAhead = 2;
  extern __shared__ __align__(1024) unsigned char direct_lds[];
  const unsigned lds_base = static_cast<unsigned>(
      reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) unsigned char*)direct_lds));
  const int tid = threadIdx.x, lane = tid % kWave;
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int wm = wave / WN, wn = wave % WN;

  // What a wave brings every step: kPieceA times eight rows of x (past m: the last), and of the weight's block rows (past n: the last) the step's blocks.
  unsigned x_off[S::kPieceA], w_off[S::kPieceW];
  const unsigned char* x_base = scalar_address(a + m0 * k + first_step * 64L) - kPieceBias;
#pragma unroll
  for (int i = 0; i < S::kPieceA; ++i) {
    const int trow = (wave * S::kPieceA + i) * 8 + lane / 8;
    const long row = min(static_cast<long>(m) - 1 - m0, static_cast<long>(trow));
    x_off[i] = piece_offset<S::kPieceA>(i, static_cast<unsigned>(row * k * 2 + ((lane % 8) ^ slot_key<128>(trow)) * 16));
  }
  const long w_row_blocks = (static_cast<long>(n) + 15) / 16, first_block = min(w_row_blocks - 1, n0 / 16 + wave * S::kPieceW / 2);
  const unsigned char* w_base = scalar_address(reinterpret_cast<const unsigned char*>(w) + (first_block * (k / 32) + first_step * 2L) * 1024) - kPieceBias;
#pragma unroll
  for (int i = 0; i < S::kPieceW; ++i) {
    const long block = min(w_row_blocks - 1, n0 / 16 + (wave * S::kPieceW + i) / 2) - first_block;
    w_off[i] = piece_offset<S::kPieceW>(i, static_cast<unsigned>((block * (k / 32) + (wave * S::kPieceW + i) % 2) * 1024 + lane * 16));
  }
  // (past the last step: the last once more, so that the number of loads under way is known; it is not used)
  int left = nk - 1;
  auto ask = [&](int slot) {
    const unsigned to = lds_base + slot * S::kStageBytes;
    load_tile_pieces<S::kPieceA>(x_base, x_off, to + (wave * S::kPieceA + S::kPieceA / 2) * 1024);
    load_tile_pieces<S::kPieceW>(w_base, w_off, to + S::kBytesA + (wave * S::kPieceW + S::kPieceW / 2) * 1024);
    x_base += left > 0 ? 128 : 0, w_base += left > 0 ? 2048 : 0, --left;
  };
#pragma unroll
  for (int s = 0; s < STAGES; ++s) ask(s);

  floatx16 acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;

  const int frow = lane % 32, fhalf = lane / 32;
  const unsigned char* aread[4];
#pragma unroll
  for (int s = 0; s < 4; ++s) aread[s] = direct_lds + (wm * TM * 32 + frow) * 128 + (((s * 2 + fhalf) ^ slot_key<128>(frow)) * 16);
  const unsigned char* wread = direct_lds + S::kBytesA + (wn * TN * 2 + frow / 16) * 2048 + (frow % 16) * 16 + fhalf * 256;
  uint4 fa[4][TM], fw[4][TN];
  auto read = [&](int slot, int s) {
#pragma unroll
    for (int i = 0; i < TM; ++i) fa[s][i] = *reinterpret_cast<const uint4*>(aread[s] + slot * S::kStageBytes + i * 4096);
#pragma unroll
    for (int j = 0; j < TN; ++j) fw[s][j] = *reinterpret_cast<const uint4*>(wread + slot * S::kStageBytes + j * 4096 + (s / 2) * 1024 + (s % 2) * 512);
  };
  wait_loads<(STAGES - 1) * S::kPieces>();
  lds_barrier();
#pragma unroll
  for (int s = 0; s < kAhead; ++s) read(0, s);

  auto step = [&](int slot) {
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      __builtin_amdgcn_sched_barrier(0);
      if (s == 4 - kAhead) {                  // the next step's stage is there for all, and nobody reads this one's any more
        wait_loads<(STAGES - 2) * S::kPieces>();
        lds_barrier();
        ask(slot);
      }
      __builtin_amdgcn_sched_barrier(0);
      read(s + kAhead < 4 ? slot : (slot + 1) % STAGES, (s + kAhead) % 4);
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = mfma_32x32x16(fa[s][i], fw[s][j], acc[i][j]);
#pragma unroll
      for (int e = 0; e < TM * TN; ++e) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x100, (TM + TN + TM * TN - 1) / (TM * TN), 0);
      }
    }
  };
  for (int t = 0; t < nk; t += STAGES) {
#pragma unroll
    for (int u = 0; u < STAGES; ++u)
      if (u == 0 || t + u < nk) step(u);
  }
  wait_loads<0>();                            // (what was asked for past the last step)
  lds_barrier();                              // LDS is free for the output
  store_part<EPI, TM, TN>(acc, reinterpret_cast<float*>(direct_lds) + wave * (S::kPatchBytes / 4), out, m, n, k, m0 + wm * TM * 32, n0 + wn * TN * 32, lane,
                          ra, rows);
}

// gridDim.y > 1: k in that many equal parts, part y's sums in an output of its own, as below.
template <int EPI, int WM, int WN, int TM, int TN, int STAGES>
__global__ __launch_bounds__(64 * WM * WN, 2) void gemm_mfma_piped_kernel(const bf16_t* __restrict__ a, const bf16_t* __restrict__ w,
                                                                          void* __restrict__ out, int m, int n, int k, int m_blocks, int n_blocks,
                                                                          int n_first, const RopeKvArgs ra, const RowScaleArgs rows) {
  typedef PipedShape<WM, WN, TM, TN, STAGES> S;
  int bm, bn;
  tile_of(blockIdx.x, m_blocks, n_blocks, bm, bn);
  int first_step = 0, nk = k / 64;
  if constexpr (EPI == kStoreF32) {
    nk /= static_cast<int>(gridDim.y), first_step = static_cast<int>(blockIdx.y) * nk;
    out = static_cast<float*>(out) + static_cast<size_t>(blockIdx.y) * m * n;
  }
  piped_tile<EPI, WM, WN, TM, TN, STAGES>(a, w, out, m, n, k, static_cast<long>(bm) * S::kRowsA, n_first + static_cast<long>(bn) * S::kRowsW, first_step, nk,
                                          ra, rows);
}

// ---- rows beyond whole tiles, beside them ---------------------------------------------------------
// A portion of a prompt with decoded tokens beside it has a few rows more than whole tiles (270, 519): another row of large tiles is
// nearly all padding, and a whole turn of the chip where the tiles just fitted.  So the whole row tiles (256 x 256, or 128 x 128 with LARGE false) and, on the
// CUs they leave, 64 x 256 tiles of the rows that remain, in one launch; those come last and fill in.  Every element is added up as before.
// Weights from memory, gate-up products: 270 x 11,264 x 2,048 34.5 -> 23.2 us (176 tiles of 256 x 128 before, 176 of 128 x 128 and 44 of 64 x 256 now),
// 519 x 28,672 x 4,096 170 -> 139, 1,030 x 28,672 x 4,096 256 -> 210, 519 x 22,016 x 4,096 127 -> 106; a plain store, 270 x 12,288 x 4,096 66 -> 42.
typedef PipedShape<2, 4, 1, 2, 3> RestShape;
template <int EPI, bool LARGE>
__global__ __launch_bounds__(512, 2) void gemm_mfma_rest_kernel(const bf16_t* __restrict__ a, const bf16_t* __restrict__ w, void* __restrict__ out,
                                                                int m, int n, int k, int m_blocks, int n_blocks, const RopeKvArgs ra,
                                                                const RowScaleArgs rows) {
  constexpr int kRows = LARGE ? 256 : 128;
  const int whole = m_blocks * n_blocks, block = blockIdx.x;
  int bm, bn;
  if (block < whole) {
    tile_of(block, m_blocks, n_blocks, bm, bn);
    if constexpr (LARGE) halves_tile<EPI>(a, w, out, m, n, k, bm * 256L, bn * 256L, ra, rows);
    else piped_tile<EPI, 2, 4, 2, 1, 4>(a, w, out, m, n, k, bm * 128L, bn * 128L, 0, k / 64, ra, rows);
  } else {
    const int first = m_blocks * kRows, rest_cols = (n + RestShape::kRowsW - 1) / RestShape::kRowsW;
    tile_of(block - whole, (m - first + RestShape::kRowsA - 1) / RestShape::kRowsA, rest_cols, bm, bn);
    piped_tile<EPI, 2, 4, 1, 2, 3>(a, w, out, m, n, k, first + static_cast<long>(bm) * RestShape::kRowsA, static_cast<long>(bn) * RestShape::kRowsW, 0, k / 64, ra,
                                       rows);
  }
}

// ---- 64 x 64, fragments a step ahead --------------------------------------------------------------
// Few rows or few columns: fewer tiles than CUs, or one or two a CU, where a step is as long as its chain (barrier, ask, read, multiply): 580
// clocks of it with the kernel above, 128 of them MFMAs, whatever the ring's depth (four to nine stages, steps of 64 or 128: the same).  So all
// fragments of step t + 1 are read while step t multiplies, a wave's four loads of a step lie side by side in LDS (one LDS address a
// step: setting it anew waits for the load that uses it), and a stage may be asked for again as soon as its fragments are read: four stages
// are four steps ahead.  What bounds it now is what a CU can pull: 16 KB a step at 65 to 74 bytes a ns.  Weights from memory: 200 rows, 2,560 x
// 2,048 11.7 -> 10.6 us, 2,048 x 5,632 26.3 -> 24.0, 256 rows 2,048 x 4,096 21.0 -> 19.7; 64 rows and 11,264 x 2,048, which memory bounds: level.
// PAST: the weight past the caches (passes_by), where one tile of rows reads it: 64 rows 11,264 x 2,048 14.6 -> 13.5 us, 32 rows 13.5 -> 12.5.
//
// gridDim.y > 1: k is cut into that many equal parts (each whole steps), and part y's sums go to an output of its own,
// out + y * m * n (kStoreF32 only: whoever reads them adds the parts up in order).
struct AheadShape {
  static constexpr int kStages = 4, kStageBytes = 16 * 1024, kThreads = 256, kLdsBytes = kStages * kStageBytes;
  static constexpr int kPatchBytes = 32 * (32 + 4) * 4;
  static_assert(4 * kPatchBytes <= kLdsBytes, "the output's patches take the stages' place");
};

template <int EPI, bool PAST>
__global__ __launch_bounds__(256, 2) void gemm_mfma_ahead_kernel(const bf16_t* __restrict__ a, const bf16_t* __restrict__ w, void* __restrict__ out,
                                                                 int m, int n, int k, int m_blocks, int n_blocks, int n_first, const RopeKvArgs ra,
                                                                 const RowScaleArgs rows) {
  constexpr int kStages = AheadShape::kStages, kStageBytes = AheadShape::kStageBytes;
  extern __shared__ __align__(1024) unsigned char direct_lds[];
  const unsigned lds_base = static_cast<unsigned>(
      reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) unsigned char*)direct_lds));
  const int tid = threadIdx.x, lane = tid % kWave;
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int wm = wave / 2, wn = wave % 2;
  int bm, bn;
  tile_of(blockIdx.x, m_blocks, n_blocks, bm, bn);
  const long m0 = static_cast<long>(bm) * 64, n0 = n_first + static_cast<long>(bn) * 64;
  const int nk = k / 64 / static_cast<int>(gridDim.y);
  const size_t first_step = static_cast<size_t>(blockIdx.y) * nk;
  if constexpr (EPI == kStoreF32) out = static_cast<float*>(out) + static_cast<size_t>(blockIdx.y) * m * n;

  // What a wave brings every step, 4 KB: waves 0 and 1 half of the rows of x (past m: the last), 2 and 3 the two blocks of two of the
  // tile's four block rows of the weight (past n: of the last).
  const unsigned char* base[4];
  unsigned off[kMaxLoads];
  const unsigned step_bytes = wave < 2 ? 128 : 2048;
  const long w_row_blocks = (static_cast<long>(n) + 15) / 16;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    if (wave < 2) {
      const int trow = wave * 32 + i * 8 + lane / 8;
      const long row = min(static_cast<long>(m) - 1 - m0, static_cast<long>(trow));
      base[i] = reinterpret_cast<const unsigned char*>(a + m0 * k) + first_step * 128 - i * 1024;
      off[i] = static_cast<unsigned>(row * k * 2 + ((lane % 8) ^ slot_key<128>(trow)) * 16);
    } else {
      const long block = min(w_row_blocks - 1, n0 / 16 + (wave - 2) * 2 + i / 2);
      base[i] = reinterpret_cast<const unsigned char*>(w) + (block * (k / 32) + static_cast<long>(first_step) * 2 + i % 2) * 1024 - i * 1024;
      off[i] = lane * 16;
    }
  }
  auto ask = [&](int step) {                  // (in order: the bases go on by a step each time)
    const void* from[kMaxLoads] = {base[0], base[1], base[2], base[3]};
    const unsigned to = lds_base + (step % kStages) * kStageBytes + wave * 4096;
    if (PAST && wave >= 2) load_side_by_side<4, PAST>(from, off, to);
    else load_side_by_side<4>(from, off, to);
#pragma unroll
    for (int i = 0; i < 4; ++i) base[i] += step_bytes;
  };
#pragma unroll
  for (int s = 0; s < kStages; ++s)
    if (s < nk) ask(s);

  __shared__ __align__(16) float part_sum[row_scaled(EPI) ? kPartSums * 64 : 4];
  if constexpr (row_scaled(EPI)) sum_row_parts<64, 256>(part_sum, rows, m, m0, tid);

  floatx16 acc[1][1];
#pragma unroll
  for (int r = 0; r < 16; ++r) acc[0][0][r] = 0.f;

  const int frow = lane % 32, fhalf = lane / 32;
  const unsigned char* aread = direct_lds + (wm * 32 + frow) * 128;
  const int akey = slot_key<128>(wm * 32 + frow);
  const unsigned char* wread = direct_lds + 8192 + (wn * 2 + frow / 16) * 2048 + (frow % 16) * 16 + fhalf * 256;
  struct Fragments {
    uint4 a[4], w[4];
  };
  auto read = [&](Fragments& f, int step) {
    const int at = (step % kStages) * kStageBytes;
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      f.a[s] = *reinterpret_cast<const uint4*>(aread + at + (((s * 2 + fhalf) ^ akey) * 16));
      f.w[s] = *reinterpret_cast<const uint4*>(wread + at + (s / 2) * 1024 + (s % 2) * 512);
    }
  };
  // Step t from `now`, the fragments of t + 1 into `next`.  The barrier comes when this wave's loads of t + 1 have landed and its reads of
  // step t are back (lds_barrier waits for those): behind it everybody's part of t + 1 is there, and t's stage is free.
  // (No branch between the reads and the MFMAs, and the wait for the reads of t said in the compiler's own terms too: else it waits for all
  // reads before the first MFMA.)
  auto wait_lds_reads = []() { __builtin_amdgcn_s_waitcnt(63 >> 4 << 14 | 0 << 8 | 7 << 4 | 15); };      // lgkmcnt(0)
  auto multiply = [&](const Fragments& now) {
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int s = 0; s < 4; ++s) acc[0][0] = mfma_32x32x16(now.a[s], now.w[s], acc[0][0]);
    __builtin_amdgcn_sched_barrier(0);
  };
  auto turn = [&](int t, const Fragments& now, Fragments& next) {             // (t + kStages < nk)
    wait_loads<4 * (kStages - 2)>();
    wait_lds_reads();
    lds_barrier();
    ask(t + kStages);
    read(next, t + 1);
    multiply(now);
  };
  auto late_turn = [&](int t, const Fragments& now, Fragments& next) {        // (t + 1 < nk, nothing left to ask for)
    wait_for_stage<4, kStages - 2>(nk - 2 - t);
    wait_lds_reads();
    lds_barrier();
    read(next, t + 1);
    multiply(now);
  };
  Fragments even, odd;
  wait_for_stage<4, kStages - 1>(min(nk - 1, kStages - 1));
  lds_barrier();
  read(even, 0);
  int t = 0;
  for (; t + kStages + 1 < nk; t += 2) turn(t, even, odd), turn(t + 1, odd, even);
  if (t + kStages < nk) turn(t, even, odd), even = odd, ++t;
  for (; t + 2 < nk; t += 2) late_turn(t, even, odd), late_turn(t + 1, odd, even);
  if (t + 1 < nk) late_turn(t, even, odd), even = odd;
  multiply(even);
  lds_barrier();            // the last step has been read: LDS is free for the output
  store_part<EPI, 1, 1>(acc, reinterpret_cast<float*>(direct_lds) + wave * (AheadShape::kPatchBytes / 4), out, m, n, k, m0 + wm * 32, n0 + wn * 32, lane,
                        ra, rows, row_scaled(EPI) ? part_sum + wm * 32 : nullptr, 64);
}

// What a product's kernels get: n columns, of which this launch computes n_cols from n_first on (all of them: 0, n).
struct Operands {
  const bf16_t* a;
  const bf16_t* w;
  void* out;
  int m, n, k, n_first, n_cols;
  hipStream_t stream;
};

// Launches kernel on tiles of rows x cols, with more than the default dynamic LDS allowed (asked for once: `raised` is the caller's).
template <typename Kernel>
int launch_tiles(Kernel kernel, std::atomic<bool>& raised, int rows, int cols, int threads, int lds, const Operands& o, const RopeKvArgs& ra, const RowScaleArgs& scale,
                 int k_parts = 1) {
  if (!raised) {
    if (hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, lds) != hipSuccess)
      return fail("gemm_mfma: cannot raise the dynamic LDS limit");
    raised = true;
  }
  const long m_blocks = (o.m + rows - 1) / rows, n_blocks = (o.n_cols + cols - 1) / cols;
  kernel<<<dim3(static_cast<unsigned>(m_blocks * n_blocks), static_cast<unsigned>(k_parts)), dim3(threads), lds, o.stream>>>(
      o.a, o.w, o.out, o.m, o.n, o.k, static_cast<int>(m_blocks), static_cast<int>(n_blocks), o.n_first, ra, scale);
  return 0;
}

template <int EPI>
int launch_ahead(const Operands& o, const RopeKvArgs& ra, const RowScaleArgs& scale, int k_parts = 1) {
  static std::atomic<bool> raised{false}, raised_past{false};
  if (o.m <= 64 && passes_by(o.n, o.k, 2))
    return launch_tiles(gemm_mfma_ahead_kernel<EPI, true>, raised_past, 64, 64, AheadShape::kThreads, AheadShape::kLdsBytes, o, ra, scale, k_parts);
  return launch_tiles(gemm_mfma_ahead_kernel<EPI, false>, raised, 64, 64, AheadShape::kThreads, AheadShape::kLdsBytes, o, ra, scale, k_parts);
}

template <int EPI, int WM, int WN, int TM, int TN, int BK, int STAGES, int MINWG>
int launch_direct(const Operands& o, const RopeKvArgs& ra, const RowScaleArgs& scale) {
  typedef DirectShape<WM, WN, TM, TN, BK, STAGES> S;
  static std::atomic<bool> raised{false};
  return launch_tiles(gemm_mfma_direct_kernel<EPI, WM, WN, TM, TN, BK, STAGES, MINWG>, raised, S::kRowsA, S::kRowsW, S::kThreads, S::kLdsBytes, o, ra,
                      scale);
}

template <int EPI, int WM, int WN, int TM, int TN, int BK, int STAGES>
int launch_turns(const Operands& o, const RopeKvArgs& ra, const RowScaleArgs& scale) {
  typedef TurnsShape<WM, WN, TM, TN, BK, STAGES> S;
  static std::atomic<bool> raised{false};
  return launch_tiles(gemm_mfma_turns_kernel<EPI, WM, WN, TM, TN, BK, STAGES>, raised, S::kRowsA, S::kRowsW, S::kThreads, S::kLdsBytes, o, ra, scale);
}

template <int EPI, int WM, int WN, int TM, int TN, int STAGES>
int launch_piped(const Operands& o, const RopeKvArgs& ra, const RowScaleArgs& scale, int k_parts = 1) {
  typedef PipedShape<WM, WN, TM, TN, STAGES> S;
  static std::atomic<bool> raised{false};
  return launch_tiles(gemm_mfma_piped_kernel<EPI, WM, WN, TM, TN, STAGES>, raised, S::kRowsA, S::kRowsW, S::kThreads, S::kLdsBytes, o, ra, scale,
                      k_parts);
}

template <int EPI>
int launch_halves(const Operands& o, const RopeKvArgs& ra, const RowScaleArgs& scale) {
  static std::atomic<bool> raised{false};
  return launch_tiles(gemm_mfma_halves_kernel<EPI>, raised, 256, 256, HalvesShape::kThreads, HalvesShape::kLdsBytes, o, ra, scale);
}

// Which tile: the one with which the busiest CU finishes first.  A CU's tiles come one after the other, a turn of the chip each;
// a tile takes its steps of 64, each as long as the fuller the chip is (L2, memory and power are shared: us a step with few tiles on
// the chip and with one on every CU), a few us around them, and its stores.  All measured with the weights coming from memory, as they do
// inside a model (forty weights one after the other): a loop over one product finds its weights in the 256 MB cache before
// memory and flatters the small tiles and the short rings.  The model's times are within 5 % of those measured for 72 to 4,096 rows at
// outputs of 2,048 to 28,672 and k of 2,048 to 14,336 (one product after the other without a pause 1 % short to 7 % long at the median, 64 x 64
// 18 % long).  A function of (m, n, k) alone; every tile adds over k in the same order.
// That is what they were fitted to, and of 256 x 128 and 128 x 128 tiles, and of the 64 x 256 ones beside whole tiles (kRestForm), it is no more: these were walked by
// kernels whose waves go together or take turns, and gemm_mfma_piped_kernel, which walks them now, takes 0.55 / 0.84 and 0.31 / 0.52 us a step (kQkvForm).  kDirectForm still
// ranks the forms as measured then (256 x 128, 0.87 / 1.06, a little lower since); over 48 products the tiles it chooses take 0.944 of the time with the kernels of
// now, 1,025 rows of 4,096 x 14,336 189 -> 194 us and 270 rows of 28,672 x 4,096 90 -> 91 the other way.
struct DirectForm {
  int rows, cols;
  double us_a_step_few, us_a_step_full, us_around, us_stores;
  bool beside = false;          // four workgroups a CU, beside each other: us_a_step_full is the chip's for a tile a CU, us_a_step_few one tile's
};
// The last, 128 x 64 with room for two workgroups a CU, is for the q|k|v epilogue alone: what comes after the
// loop is long there (rotation, three destinations), and several workgroups a CU run it beside each other's loops
// (600 rows 2,560 x 2,048 12.9 us, in 64 x 64 tiles 15.4; 1,000 rows 1,536 x 1,024 8.6 and 10.6).
// That epilogue's products, up to kQkvMeasured outputs, have times of their own (kQkvForm; stores are the epilogue), fitted to 29 of 130 to 4,000 rows, 1,536 to 12,288
// outputs and k 768 to 4,096, weights from memory, every form of each, within 3 to 10 %: what is chosen takes 0.970 of what the plain stores' times and an
// epilogue's a form chose: 2,048 rows 2,560 x 2,048 34.3 -> 30.6 us (256 x 128), 6,144 x 4,096 98.1 -> 91.3 (256 x 256), 600 rows 2,560 x 2,048 15.1 -> 12.9;
// 1,300 rows 22.3 -> 24.0.
constexpr int kQkvMeasured = 20480;
constexpr int kDirectForms = 6;
constexpr DirectForm kDirectForm[kDirectForms] = {
    {256, 256, 1.12, 1.48, 4.0, 2.0}, {256, 192, 1.15, 1.40, 4.0, 1.5}, {256, 128, 0.80, 1.02, 4.0, 1.5},
    {128, 128, 0.50, 0.59, 3.5, 1.0}, {64, 64, 0.25, 0.27, 3.0, 0.25},  {128, 64, 0.67, 0.36, 8.5, 0.0, true}};
constexpr int kQkvForms = 7;
constexpr DirectForm kQkvForm[kQkvForms] = {
    {256, 256, 0.83, 1.30, 0.0, 15.7}, {256, 192, 0.73, 1.22, 0.0, 13.8}, {256, 128, 0.55, 0.84, 1.0, 9.0},
    {128, 128, 0.31, 0.52, 2.7, 3.4},  {64, 64, 0.165, 0.19, 3.9, 0.3},   {128, 64, 0.22, 0.31, 2.4, 0.9},
    {128, 128, 0.77, 1.02, 2.5, 3.0}};
// Their seventh: 128 x 128 in two stages, two workgroups a CU, which takes a second, partly filled turn of the chip beside the first; asked from an eighth of the chip beyond a
// turn up to two, where us_a_step_few and _full are both workgroups' with none and all CUs sharing.  2,560 x 2,048, 1,800 rows 33.2 -> 29.4 us, 3,200 rows 44.1 ->
// 37.7, 12,288 x 4,096, 600 rows 75.4 -> 67.9; with k 4,096 and 256 x 128 tiles on most CUs those are faster (1,000 rows 6,144 x 4,096 54.8, 66.9 so).
// Up to kBriefQkv most forms are other kernels (short_walk), whose epilogues the waves of a CU do not overlap: 2,048 rows 2,560 x 512 14.5 us in 128 x 64, 17.0 in what
// the table above chooses.
constexpr int kBriefQkv = 704;
constexpr DirectForm kBriefQkvForm[kDirectForms] = {
    {256, 256, 1.12, 1.48, 4.0, 24.5}, {256, 192, 1.15, 1.40, 4.0, 19.0}, {256, 128, 0.80, 1.02, 4.0, 12.5},
    {128, 128, 0.50, 0.59, 3.5, 6.3},  {64, 64, 0.25, 0.27, 3.0, 3.25},   {128, 64, 0.67, 0.36, 8.5, 2.0, true}};
const DirectForm& form_of(int form, bool qkv, int k) { return !qkv ? kDirectForm[form] : k <= kBriefQkv ? kBriefQkvForm[form] : kQkvForm[form]; }


double form_time(const DirectForm& form, int m, int n, int k) {
  const long tiles = static_cast<long>((m + form.rows - 1) / form.rows) * ((n + form.cols - 1) / form.cols), cus = compute_units();
  const long full = tiles / cus;
  const double last = static_cast<double>(tiles % cus) / static_cast<double>(cus), steps = k / 64;
  const double few = form.us_a_step_few, more = form.us_a_step_full - few, stores = form.us_stores;
  if (&form == &kQkvForm[kQkvForms - 1]) {
    const double shared = static_cast<double>(tiles - cus) / static_cast<double>(cus);
    return shared < 0.125 || shared > 1.0 ? 1e30 : form.us_around + steps * (few + more * shared) + stores;
  }
  if (form.beside) {
    const double chip = static_cast<double>(tiles) / static_cast<double>(cus) * (steps * form.us_a_step_full + stores), chain = steps * few + stores;
    return form.us_around + (chip > chain ? chip : chain);
  }
  return form.us_around + full * (steps * (few + more) + stores) + (last > 0.0 ? steps * (few + more * last) + stores : 0.0);
}

int direct_form(int m, int n, int k, bool long_epilogue, bool qkv) {
  int best = 0;
  double best_time = 0.0;
  for (int f = 0; f < (qkv && k > kBriefQkv ? kQkvForms : long_epilogue ? kDirectForms : kDirectForms - 1); ++f) {
    const double time = form_time(form_of(f, qkv, k), m, n, k);
    if (f == 0 || time < best_time) best = f, best_time = time;
  }
  return best;
}

// Rows beyond whole tiles beside them (gemm_mfma_rest_kernel): the 64 x 256 tiles' times, measured as the others' were, and the time of a launch that
// begins with `whole` tiles of a form and goes on with `rest` such: those first go to the CUs that the last turn of large tiles leaves.  (On
// what the chip shares a tile is a load by its size: four small ones are a 256 x 256.)
constexpr DirectForm kRestForm = {64, 256, 0.50, 0.62, 0.0, 1.0};
constexpr double kRestQkv = 2.0;       // (the q|k|v epilogue beyond plain stores)
double rest_time(const DirectForm& form, int whole, int rest, int k, bool qkv) {
  const int cus = compute_units(), steps = k / 64;
  const double load = whole + rest * static_cast<double>(kRestForm.rows * kRestForm.cols) / (form.rows * form.cols);
  const double fill = load < cus ? load / cus : 1.0;
  const double large = steps * (form.us_a_step_few + (form.us_a_step_full - form.us_a_step_few) * fill) + form.us_stores;
  const double small = steps * (kRestForm.us_a_step_few + (kRestForm.us_a_step_full - kRestForm.us_a_step_few) * fill) + kRestForm.us_stores +
                       (qkv ? kRestQkv : 0.0);
  const int full = whole / cus, busy = whole % cus;
  const double early = full * large, late = busy ? (full + 1) * large : early;
  // a turn of small tiles after the other, on the CUs free early and on those free late, whichever ends first
  int left = rest;
  double a = early + small, b = late + small, end = late;
  while (left > 0) {
    const bool first = busy == 0 || a <= b;
    left -= first ? cus - busy : busy;
    end = first ? a : b;
    (first ? a : b) += small;
  }
  // (with tiles waiting for CUs measured 3 to 8 % longer than this)
  return form.us_around + (end > late ? end : late) * (whole + rest > cus ? 1.05 : 1.0);
}

// How an output's columns are cut: the first n1 in tiles of `first`, the rest (if any) in tiles of `second`, one launch each.  Tiles that do not
// fill the last turn of the chip leave CUs idle for a whole tile (3,000 x 11,264 are 528 tiles of 256 x 256: 256, 256 and 16); columns that fill
// whole turns with large tiles, and smaller tiles for the others, leave less.  Every element is added up as before, by whichever tile.
// From k = 512 on (below, a launch is as long as a tile), and where it is 4 % and more by the model, a second launch counted with 6 us:
// weights from memory, 3,000 x 11,264 x 2,048 138 -> 125 us (10,752 columns in 256 x 256, 512 in 64 x 64), 1,500 x 11,264 x 2,048 76 -> 69 (the
// same), 2,300 x 2,048 x 5,632 80 -> 74 (128 x 128 and 64 x 64).
constexpr double kCutGap = 6.0;
// Or its rows: whole tiles of `first`, and the rows that remain in the same launch (rest_time; up to four turns of the chip, beyond them a turn more matters
// little).
// Over 11,000 products of 257 to 4,200 rows, 2,048 to 30,720 outputs and k 1,024 to 8,192 the times of cut columns and rows beyond are 3 % too long at
// the median and 20 % too long to 17 % too short at the ends, so forms within 5 % of each other are taken as it falls: what is chosen is 1.3 % slower on average
// than the fastest of the forms measured, and 0.05 % slower than whole tiles where it displaces them.  (With small tiles counted as large ones in
// the load and 8 us a cut more than 261 of them took another form: 236 gained 8 % by the change, 25 lost 5.)
struct Parts {
  int first, n1, second;
  bool rest;
};
Parts parts_of(int m, int n, int k, bool long_epilogue) {
  const bool qkv = long_epilogue && n <= kQkvMeasured;
  Parts best{direct_form(m, n, k, long_epilogue, qkv), n, 0, false};
  if (k < 512) return best;
  double best_time = 0.96 * form_time(form_of(best.first, qkv, k), m, n, k);
  for (int f = 0; f < 4; f += 3) {
    const DirectForm& form = form_of(f, qkv, k);
    const int row_tiles = m / form.rows, beyond = m % form.rows;
    const long whole = static_cast<long>(row_tiles) * ((n + form.cols - 1) / form.cols);
    if (whole == 0 || beyond == 0 || whole > 4L * compute_units()) continue;
    const int rest = (beyond + kRestForm.rows - 1) / kRestForm.rows * ((n + kRestForm.cols - 1) / kRestForm.cols);
    const double time = rest_time(form, static_cast<int>(whole), rest, k, qkv);
    if (time < best_time) best = Parts{f, n, 0, true}, best_time = time;
  }
  for (int f = 0; f < 4; ++f) {
    const DirectForm& form = form_of(f, qkv, k);
    const long rows = (m + form.rows - 1) / form.rows, cus = compute_units();
    for (long turns = rows * ((n + form.cols - 1) / form.cols) / cus; turns >= 1 && rows <= turns * cus; --turns) {
      const long n1 = turns * cus / rows * form.cols;
      if (n1 <= 0 || n1 >= n) continue;
      const int rest = n - static_cast<int>(n1), second = direct_form(m, rest, k, long_epilogue, qkv);
      const double time = form_time(form, m, static_cast<int>(n1), k) + form_time(form_of(second, qkv, k), m, rest, k) + kCutGap;
      if (time < best_time) best = Parts{f, static_cast<int>(n1), second, false}, best_time = time;
      break;      // (fewer turns of large tiles leave more for the small ones)
    }
  }
  return best;
}

template <int EPI, bool LARGE>
int launch_rest(const Operands& o, const RopeKvArgs& ra, const RowScaleArgs& scale) {
  constexpr int kRows = LARGE ? 256 : 128, kLds = LARGE ? HalvesShape::kLdsBytes : PipedShape<2, 4, 2, 1, 4>::kLdsBytes;
  static_assert(RestShape::kLdsBytes <= kLds, "both tiles in one workgroup's LDS");
  static std::atomic<bool> raised{false};
  auto kernel = gemm_mfma_rest_kernel<EPI, LARGE>;
  if (!raised) {
    if (hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, kLds) != hipSuccess)
      return fail("gemm_mfma: cannot raise the dynamic LDS limit");
    raised = true;
  }
  const int m_blocks = o.m / kRows, n_blocks = (o.n + kRows - 1) / kRows;
  const int rest = (o.m % kRows + RestShape::kRowsA - 1) / RestShape::kRowsA * ((o.n + RestShape::kRowsW - 1) / RestShape::kRowsW);
  kernel<<<dim3(m_blocks * n_blocks + rest), dim3(512), kLds, o.stream>>>(o.a, o.w, o.out, o.m, o.n, o.k, m_blocks, n_blocks, ra, scale);
  return 0;
}

// Up to which k a form is walked by gemm_mfma_direct_kernel: a short walk is mostly its beginning and its stores, which the kernels whose waves
// take turns (and the one that reads a step ahead) do with fewer waves or more barriers.  Kernel of before over this one, 40 to 1,800 tiles, k
// 128, 512 and 1,024: 256 x 256 0.82, 0.98 and 1.09 (adding 0.77, 0.90 and 0.98, at 1,536 1.06; gated 0.88, 1.06 and 1.18), 256 x 192 0.97, 1.05 and 1.10,
// 128 x 128 0.93, 0.99 and 1.02, 64 x 64 0.94, 1.00 and 1.06.  256 x 128 with 256 tiles: k 128 0.97, 256 1.02, 512 1.07, 1,024 1.11.
// 128 x 64: k 512 and 640 0.87 to 0.92, 1,024 1.09.
constexpr int short_walk(int form, int epi) {
  return form == 0 && epi == kAccumF32 ? 1024 : form == 0 && gated(epi) ? 384 : form == 1 ? 256 : form == 2 ? 128 : form == 5 ? 704 : 576;
}

template <int EPI>
int launch_form(int form, const Operands& o, const RopeKvArgs& ra, const RowScaleArgs& scale) {
  const bool brief = o.k <= short_walk(form, EPI);
  switch (form) {
    case 0: return brief ? launch_direct<EPI, 4, 4, 2, 2, 64, 2, 1>(o, ra, scale) : launch_halves<EPI>(o, ra, scale);
    case 1: return brief ? launch_direct<EPI, 4, 2, 2, 3, 64, 2, 1>(o, ra, scale) : launch_turns<EPI, 4, 2, 2, 3, 32, 5>(o, ra, scale);
    case 2: return brief ? launch_direct<EPI, 4, 2, 2, 2, 64, 3, 1>(o, ra, scale) : launch_piped<EPI, 4, 2, 2, 2, 3>(o, ra, scale);
    case 3: return brief ? launch_direct<EPI, 2, 4, 2, 1, 64, 4, 1>(o, ra, scale) : launch_piped<EPI, 2, 4, 2, 1, 4>(o, ra, scale);
    case 6:
      if constexpr (EPI == kRopeKvBf16) return launch_piped<EPI, 2, 4, 2, 1, 2>(o, ra, scale);
      else return fail("gemm_mfma: a form of the q|k|v product");
    case 5: return brief ? launch_direct<EPI, 2, 2, 2, 1, 64, 2, 4>(o, ra, scale) : launch_piped<EPI, 4, 2, 1, 1, 3>(o, ra, scale);
    default: return brief ? launch_direct<EPI, 2, 2, 1, 1, 64, 4, 2>(o, ra, scale) : launch_ahead<EPI>(o, ra, scale);
  }
}

template <int EPI>
int launch_direct_form(const bf16_t* ap, const bf16_t* wp, void* out, int m, int n, int k, hipStream_t s, const RopeKvArgs& ra = RopeKvArgs{},
                       const RowScaleArgs& scale = RowScaleArgs{}) {
  Operands o{ap, wp, out, m, n, k, 0, n, s};
  if constexpr (row_scaled(EPI)) {
    return launch_ahead<EPI>(o, ra, scale);      // (for a decode step's rows, where this is the tile anyway)
  } else {
    const Parts parts = parts_of(m, n, k, EPI == kRopeKvBf16);
    if (parts.rest) return parts.first == 0 ? launch_rest<EPI, true>(o, ra, scale) : launch_rest<EPI, false>(o, ra, scale);
    o.n_cols = parts.n1;
    if (int e = launch_form<EPI>(parts.first, o, ra, scale)) return e;
    if (parts.n1 == n) return 0;
    o.n_first = parts.n1, o.n_cols = n - parts.n1;
    return launch_form<EPI>(parts.second, o, ra, scale);
  }
}

bool direct_operands(const void* ap, const void* wp, int k) {
  // operands straight into LDS wherever k is whole steps of it and rows start on 16-byte boundaries
  return k % 64 == 0 && reinterpret_cast<uintptr_t>(ap) % 16 == 0 && reinterpret_cast<uintptr_t>(wp) % 16 == 0;
}

// w_packed: the weight in the weight-streaming kernel's order, for the kernel with operands straight into LDS (k in
// whole steps of 64, operands on 16-byte boundaries); else the weight by rows, for the kernel that stages its tiles
// through registers (any k that is a multiple of 8).
template <int EPI>
int launch_tiled(const bf16_t* ap, const bf16_t* wp, void* out, const float* bias, int m, int n, int k, hipStream_t s, int w_packed) {
  if (w_packed) {
    if (!direct_operands(ap, wp, k))
      return fail("gemm_mfma: a packed weight needs k in whole steps of 64 and operands on 16-byte boundaries (K=%d)", k);
    return launch_direct_form<EPI>(ap, wp, out, m, n, k, s, RopeKvArgs{}, RowScaleArgs{nullptr, 0, 0, 0.f, bias});
  }
  const long m_blocks = (m + kBM - 1) / kBM, n_blocks = (n + kBN - 1) / kBN;
  gemm_mfma_staged_kernel<EPI><<<dim3(static_cast<unsigned>(m_blocks * n_blocks)), dim3(256), 0, s>>>(
      ap, wp, out, m, n, k, static_cast<int>(m_blocks), static_cast<int>(n_blocks), bias);
  return 0;
}

int parts_of_product(const char* name, const void* a, const void* w, int w_packed, float* parts, int m, int n, int k, int k_parts, int tile_rows, void* stream) {
  BC4G_REQUIRE(m > 0 && n > 0 && k > 0 && k_parts >= 1 && k_parts <= 16 && k % (64 * k_parts) == 0 && direct_operands(a, w, k) &&
                   w_packed,
               "%s: K=%d must be %d times a multiple of 64, the weight packed and the operands on 16-byte boundaries "
               "(M=%d N=%d)", name, k, k_parts, m, n);
  BC4G_REQUIRE(((m + 63L) / 64) * ((n + 63L) / 64) <= 2147483647L, "%s: too many tiles", name);
  const Operands o{static_cast<const bf16_t*>(a), static_cast<const bf16_t*>(w), parts, m, n, k, 0, n, static_cast<hipStream_t>(stream)};
  const int e = tile_rows == 64    ? launch_ahead<kStoreF32>(o, RopeKvArgs{}, RowScaleArgs{}, k_parts)
                : tile_rows == 128 ? launch_piped<kStoreF32, 2, 4, 2, 1, 4>(o, RopeKvArgs{}, RowScaleArgs{}, k_parts)
                                   : launch_piped<kStoreF32, 4, 2, 2, 2, 3>(o, RopeKvArgs{}, RowScaleArgs{}, k_parts);
  return e ? e : check_launch(name);
}

}  // namespace
}  // namespace bc4g

using namespace bc4g;

extern "C" int bc4g_gemm_mfma(const void* a, const void* w, int w_packed, void* out, const float* bias, int epilogue, int m, int n, int k,
                              void* stream) {
  BC4G_REQUIRE(m >= 0 && n > 0 && k > 0 && k % 8 == 0, "gemm_mfma: K=%d must be a positive multiple of 8 (M=%d N=%d)",
               k, m, n);
  BC4G_REQUIRE(!bias || epilogue == kAccumF32, "gemm_mfma: only the adding epilogue takes a bias");
  if (m == 0) return 0;
  BC4G_REQUIRE(((m + 63L) / 64) * ((n + 63L) / 64) <= 2147483647L, "gemm_mfma: too many tiles");
  hipStream_t s = static_cast<hipStream_t>(stream);
  const bf16_t* ap = static_cast<const bf16_t*>(a);
  const bf16_t* wp = static_cast<const bf16_t*>(w);
  int e = 0;
  switch (epilogue) {
    case kStoreBf16: e = launch_tiled<kStoreBf16>(ap, wp, out, bias, m, n, k, s, w_packed); break;
    case kStoreF32: e = launch_tiled<kStoreF32>(ap, wp, out, bias, m, n, k, s, w_packed); break;
    case kAccumF32: e = launch_tiled<kAccumF32>(ap, wp, out, bias, m, n, k, s, w_packed); break;
    case kSquaredReluBf16: e = launch_tiled<kSquaredReluBf16>(ap, wp, out, bias, m, n, k, s, w_packed); break;
    case kSwigluBf16:
    case kGegluBf16:
      BC4G_REQUIRE(n % 16 == 0, "gemm_mfma: a gated product needs blocks of eight gate and eight up rows, N=%d is no multiple of 16", n);
      if (epilogue == kSwigluBf16) e = launch_tiled<kSwigluBf16>(ap, wp, out, bias, m, n, k, s, w_packed);
      else e = launch_tiled<kGegluBf16>(ap, wp, out, bias, m, n, k, s, w_packed);
      break;
    default: return fail("gemm_mfma: unknown epilogue %d", epilogue);
  }
  if (e) return e;
  return check_launch("gemm_mfma");
}

extern "C" int bc4g_gemm_mfma_swiglu_scaled(const void* a, const float* ssq_parts, int ssq_blocks, int ssq_stride, float eps,
                                            const void* w, int w_packed, void* out, int gelu, int m, int n, int k, void* stream) {
  BC4G_REQUIRE(m >= 0 && n > 0 && n % 16 == 0 && k > 0 && direct_operands(a, w, k) && w_packed,
               "gemm_mfma_swiglu_scaled: K=%d must be a multiple of 64, N=%d one of 16, the weight packed and the operands on 16-byte boundaries (M=%d)", k, n, m);
  BC4G_REQUIRE(ssq_parts != nullptr && ssq_blocks > 0 && ssq_stride >= m && eps >= 0.f,
               "gemm_mfma_swiglu_scaled: the sums of squares need %d parts of at least %d rows, and eps must not be negative", ssq_blocks, m);
  if (m == 0) return 0;
  BC4G_REQUIRE(((m + 63L) / 64) * ((n + 63L) / 64) <= 2147483647L, "gemm_mfma_swiglu_scaled: too many tiles");
  const bf16_t* ap = static_cast<const bf16_t*>(a);
  const bf16_t* wp = static_cast<const bf16_t*>(w);
  hipStream_t s = static_cast<hipStream_t>(stream);
  const RowScaleArgs rows{ssq_parts, ssq_blocks, ssq_stride, eps, nullptr};
  if (int e = gelu ? launch_direct_form<kGegluScaledBf16>(ap, wp, out, m, n, k, s, RopeKvArgs{}, rows)
                   : launch_direct_form<kSwigluScaledBf16>(ap, wp, out, m, n, k, s, RopeKvArgs{}, rows))
    return e;
  return check_launch("gemm_mfma_swiglu_scaled");
}

extern "C" int bc4g_gemm_mfma_parts(const void* a, const void* w, int w_packed, float* parts, int m, int n, int k, int k_parts,
                                    void* stream) {
  return parts_of_product("gemm_mfma_parts", a, w, w_packed, parts, m, n, k, k_parts, 64, stream);
}

extern "C" int bc4g_gemm_mfma_parts_large(const void* a, const void* w, int w_packed, float* parts, int m, int n, int k, int k_parts, int tile_rows,
                                          void* stream) {
  BC4G_REQUIRE(tile_rows == 128 || tile_rows == 256, "gemm_mfma_parts_large: tiles of %d rows (128 or 256)", tile_rows);
  return parts_of_product("gemm_mfma_parts_large", a, w, w_packed, parts, m, n, k, k_parts, tile_rows, stream);
}

extern "C" int bc4g_gemm_mfma_qkv(const void* a, const void* w, int w_packed, void* out, const float* table, const int32_t* slot_map,
                                  void* k_cache, void* v_cache, int m, int n, int k, int n_heads, int n_kv_heads,
                                  int head_dim, int page_tokens, int write_kv, void* stream) {
  BC4G_REQUIRE(m > 0 && n > 0 && k > 0 && direct_operands(a, w, k) && w_packed,
               "gemm_mfma_qkv: K=%d must be a multiple of 64, the weight packed and the operands on 16-byte boundaries (M=%d N=%d)", k, m, n);
  BC4G_REQUIRE(n_heads > 0 && n_kv_heads > 0 && head_dim > 0 && head_dim % 16 == 0 &&
                   static_cast<long>(n_heads + 2 * n_kv_heads) * head_dim == n,
               "gemm_mfma_qkv: %d + 2 x %d heads of %d (a multiple of 16) are not %d columns", n_heads, n_kv_heads, head_dim, n);
  BC4G_REQUIRE(!write_kv || (page_tokens > 0 && k_cache && v_cache && slot_map), "gemm_mfma_qkv: cache write asked for without a cache");
  BC4G_REQUIRE(((m + 63L) / 64) * ((n + 63L) / 64) <= 2147483647L, "gemm_mfma_qkv: too many tiles");
  RopeKvArgs ra{};
  ra.table = reinterpret_cast<const float2*>(table);
  ra.slot_map = slot_map;
  ra.k_cache = static_cast<bf16_t*>(k_cache);
  ra.v_cache = static_cast<bf16_t*>(v_cache);
  ra.n_heads = n_heads;
  ra.n_kv_heads = n_kv_heads;
  ra.head_dim = head_dim;
  ra.page_tokens = page_tokens;
  ra.per_head = reciprocal_of(static_cast<unsigned>(head_dim));
  ra.per_page = page_tokens > 0 ? reciprocal_of(static_cast<unsigned>(page_tokens)) : 0u;
  ra.write_kv = write_kv ? 1 : 0;
  ra.fragment_order = write_kv && cache_fragment_order(true, head_dim, page_tokens) ? 1 : 0;
  if (int e = launch_direct_form<kRopeKvBf16>(static_cast<const bf16_t*>(a), static_cast<const bf16_t*>(w), out, m, n, k,
                                              static_cast<hipStream_t>(stream), ra))
    return e;
  return check_launch("gemm_mfma_qkv");
}

extern "C" int bc4g_gemm_mfma_cut(const void* a, const void* w, int m, int n, int k, int qkv, int* first_cols, int* rows, int* cols, int* beyond) {
  BC4G_REQUIRE(first_cols && rows && cols && beyond && m > 0 && n > 0 && k > 0, "gemm_mfma_cut: sizes and four places for the answer");
  const Parts parts = direct_operands(a, w, k) ? parts_of(m, n, k, qkv != 0) : Parts{0, n, 0, false};
  const bool cut = parts.n1 < n;
  *first_cols = parts.n1, *rows = cut ? kQkvForm[parts.second].rows : 0, *cols = cut ? kQkvForm[parts.second].cols : 0, *beyond = parts.rest;
  return 0;
}

extern "C" int bc4g_gemm_mfma_tile(const void* a, const void* w, int m, int n, int k, int qkv, int* rows, int* cols) {
  BC4G_REQUIRE(rows != nullptr && cols != nullptr && m > 0 && n > 0 && k > 0, "gemm_mfma_tile: sizes and two places for the answer");
  if (direct_operands(a, w, k)) {
    const DirectForm& form = kQkvForm[parts_of(m, n, k, qkv != 0).first];
    *rows = form.rows, *cols = form.cols;
  } else {
    *rows = kBM, *cols = kBN;
  }
  return 0;
}
