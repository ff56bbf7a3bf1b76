// out[m, n] (+)= sum_k x[m, k] * w[n, k] in float32 on the matrix cores (v_mfma_f32_*_f32: float operands, float sums, no operand
// rounded anywhere): the products of the 32-bit path.  Operands lie by rows; k a multiple of 4, rows on 16-byte boundaries
// (gemm_generic takes what these refuse).  Both kernels add up k in the same order, eight shares from zero and the shares in
// order: a row's bits do not depend on how many rows came with it.
//
// gemm_f32_stream_kernel, few rows (a decode step), bound by reading w once.  A workgroup owns 16 rows of w (or eight gate
// rows and the eight up rows of the same outputs) and all of k, a share of it each of its 8 waves.  A wave's part of w and of x goes
// from memory into a ring of its own in LDS without passing registers -- whole cache lines of 128 bytes a row (lanes that read 16
// rows' 16 bytes straight into operand order keep the texture path busy four times as long), two steps of 32 k ahead and
// with no barrier; it reads its fragments there and feeds 16x16x4 MFMAs with w as the A operand.  The shares meet in LDS.
// Eight rows, weights from memory, plain float FMA (gemm_generic) -> this: 11,264 x 2,048 59 -> 17.2 us (5.4 TB/s), 2,048 x 5,632 82 -> 13.3,
// 2,048 x 2,048 32 -> 7.4; 64 rows 188 -> 55, 530 -> 23 and 196 -> 11.  With the attention of
// attention_f32.hip 32 decode steps of 8 requests after their prompts at TinyLlama's sizes take 213 -> 63 ms.
// What a decode step does between these products -- two norms a layer, the rotation and the cache write, each a launch of 3 to 5 us
// with next to nothing to do -- they do themselves: one that adds into the residual stream leaves, for the RMSNorm behind it, new
// residual * g and every row's sum of squares in parts, a workgroup's outputs each (emit); a product whose x was so prepared applies the
// rows' factor to its sums (ssq); and the q|k|v product holds a rotation's pairs in one workgroup (kRopeKv): a layer's eight
// launches are five, 72 -> 63 us of kernels (8 rows, TinyLlama's sizes); eight prompts of 24 to 100 tokens and 31 such steps 64.1 -> 60.5 ms.
// Parts of those sums that every wave asks for at once instead of two waves one after another, w past the caches and two steps ahead instead of
// three to eight: 8 rows, the q|k|v product 10.1 -> 8.7 us, gates and ups 20.7 -> 18.9, down 15.9 -> 14.4; 16 rows 10.9 -> 9.5, 27.2 -> 20.6, 18.6 -> 17.6; those
// prompts and steps 58.4 -> 53.6 ms.
//
// gemm_f32_tiled_kernel, many rows, bound by the matrix cores (157 TFLOP/s of float32 at the full clock).  A step's 32 k of the
// tile's rows of x and of w go straight into a ring of stages in LDS; the waves feed 32x32x2 MFMAs from there and keep
// two sets of sums, the share's and the total.  2,048 rows: 11,264 x 2,048 128 TFLOP/s, 2,048 x 5,632 129 (plain FMA: 54 and 50); 512 rows
// 104 and 84 (44 and 23).  With attention_f32.hip a 1,000-token prompt at TinyLlama's sizes takes 75 -> 20.5 ms.
#include <math.h>

#include "api.h"
#include "mfma.h"

namespace bc4g {
namespace {

constexpr int kWaves = 8;                     // of the few rows' kernel: one a share of k
constexpr int kThreads = kWaves * kWave;
constexpr int kStepK = 32;                    // floats of a row a step brings: one cache line
constexpr int kStepBytes = kStepK * 4;
constexpr int kRedPad = 17;
constexpr int kXcds = 8;

// kRopeKv (few rows only): w holds query, key and value heads; queries are stored rotated, keys go rotated into their pages, values into
// theirs.
enum Epilogue : int { kStore = 0, kAccum = 1, kSwiglu = 2, kGeglu = 3, kRopeKv = 4 };
constexpr bool gated(int epi) { return epi == kSwiglu || epi == kGeglu; }
constexpr bool paired(int epi) { return gated(epi) || epi == kRopeKv; }      // a workgroup's second eight rows of w belong to its first eight

// The activations as the elementwise kernel has them.
template <int EPI>
__device__ inline float gate_act(float g) {
  if constexpr (EPI == kGeglu) return 0.5f * g * (1.0f + tanhf(0.7978845608028654f * (g + 0.044715f * g * g * g)));
  return g / (1.0f + expf(-g));
}

struct RopeKv {
  const float2* table;      // [m, head_dim / 2] (cos, sin) (null: no rotation)
  const int32_t* slot_map;  // [m] page * page_tokens + offset
  float* k_cache;           // [pages, n_kv, page_tokens, d]
  float* v_cache;           // [pages, n_kv, d, page_tokens]
  int n_heads, n_kv_heads, head_dim, page_tokens, write_kv;
};
struct Args {
  const float* x;           // [m, k]
  const float* w;           // [n, k]; gated: n / 2 gate rows, then the up rows
  const float* bias;        // kAccum: [n] (null: none)
  float* out;               // [m, n], gated: [m, n / 2], kRopeKv: [m, n_heads * head_dim]
  int m, n, k;
  // the few rows' kernel: x is residual * g of an RMSNorm whose rows' sums of squares come in parts of 16 columns, [ssq_blocks][m], or
  // their halves, [ssq_blocks][m][2] (null: x as it is)
  const float* ssq = nullptr;
  int ssq_blocks = 0, ssq_halves = 0;
  float eps = 0.f;
  // kAccum there: what the RMSNorm behind needs (emit_g null: nothing)
  const float* emit_g = nullptr;      // [n]
  float* emit_x = nullptr;            // [m, n]
  float* emit_ssq = nullptr;          // [ceil(n / 16)][m], with eight outputs a workgroup [ceil(n / 16)][m][2]
  RopeKv rope = {};
};

// k is added up in eight shares of whole steps, each from zero, and the shares' sums in order: by both kernels, so that a row's
// bits do not depend on how many rows came with it.
constexpr int kShares = 8;
__host__ __device__ inline int steps_a_share(int k) { return ((k + kStepK - 1) / kStepK + kShares - 1) / kShares; }

// Where 16-byte segment s of row r of a step lies in the row's 128 bytes of LDS: s ^ key(r), so that the 16 rows' reads of one
// segment (two rows share the 64 banks' span) meet different banks.
__device__ inline int slot_key(int row) { return (row >> 1) & 7; }

// N wave-wide loads to N KB of consecutive LDS as one statement, load i from its own scalar base and lane offsets: the LDS
// address travels in m0, set once, and the loads' offset field (which moves the memory address too: taken off the base here)
// steps through the stretch.  The weights' pieces (the first; the first two of three and more) past the caches or through them.
template <int N, bool PAST>
__device__ inline void load_pieces_to_lds(const float* const (&bases)[N], const unsigned (&offsets)[N], unsigned lds_first) {
  static_assert(N == 2 || N == 3 || N == 4 || N == 6, "one or two pieces of weights and one, two or four of x");
  constexpr int kMid = N / 2;
  const void* b[N];
#pragma unroll
  for (int r = 0; r < N; ++r) {
    const uintptr_t bits = reinterpret_cast<uintptr_t>(bases[r]) - (r - kMid) * 1024;
    const unsigned lo = __builtin_amdgcn_readfirstlane(static_cast<unsigned>(bits));
    const unsigned hi = __builtin_amdgcn_readfirstlane(static_cast<unsigned>(bits >> 32));
    b[r] = reinterpret_cast<const void*>((static_cast<uintptr_t>(hi) << 32) | lo);
  }
  const unsigned mid = __builtin_amdgcn_readfirstlane(lds_first + kMid * 1024);
#define BC4G_PIECE(i, v, s) "global_load_lds_dwordx4 %" #v ", %" #s " offset:" #i "\n\t"
#define BC4G_WEIGHT(i, v, s, how) "global_load_lds_dwordx4 %" #v ", %" #s " offset:" #i how "\n\t"
#define BC4G_PIECES(pieces, ...) asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\t" pieces ::"s"(mid), __VA_ARGS__ : "memory", "m0")
#define BC4G_STEP(how)                                                                                                                           \
  if constexpr (N == 2)                                                                                                                          \
    BC4G_PIECES(BC4G_WEIGHT(-1024, 1, 3, how) BC4G_PIECE(0, 2, 4), "v"(offsets[0]), "v"(offsets[1]), "s"(b[0]), "s"(b[1]));                      \
  else if constexpr (N == 3)                                                                                                                     \
    BC4G_PIECES(BC4G_WEIGHT(-1024, 1, 4, how) BC4G_WEIGHT(0, 2, 5, how) BC4G_PIECE(1024, 3, 6), "v"(offsets[0]), "v"(offsets[1]),                \
                "v"(offsets[2]), "s"(b[0]), "s"(b[1]), "s"(b[2]));                                                                               \
  else if constexpr (N == 4)                                                                                                                     \
    BC4G_PIECES(BC4G_WEIGHT(-2048, 1, 5, how) BC4G_WEIGHT(-1024, 2, 6, how) BC4G_PIECE(0, 3, 7) BC4G_PIECE(1024, 4, 8), "v"(offsets[0]),         \
                "v"(offsets[1]), "v"(offsets[2]), "v"(offsets[3]), "s"(b[0]), "s"(b[1]), "s"(b[2]), "s"(b[3]));                                  \
  else                                                                                                                                           \
    BC4G_PIECES(BC4G_WEIGHT(-3072, 1, 7, how) BC4G_WEIGHT(-2048, 2, 8, how) BC4G_PIECE(-1024, 3, 9) BC4G_PIECE(0, 4, 10) BC4G_PIECE(1024, 5, 11) \
                    BC4G_PIECE(2048, 6, 12), "v"(offsets[0]), "v"(offsets[1]), "v"(offsets[2]), "v"(offsets[3]), "v"(offsets[4]),                \
                "v"(offsets[5]), "s"(b[0]), "s"(b[1]), "s"(b[2]), "s"(b[3]), "s"(b[4]), "s"(b[5]));
  if constexpr (PAST) {
    BC4G_STEP(" nt")
  } else {
    BC4G_STEP("")
  }
#undef BC4G_STEP
#undef BC4G_PIECES
#undef BC4G_WEIGHT
#undef BC4G_PIECE
}

// Which tile a workgroup takes: consecutive ones stay on one XCD (workgroups are dealt to the eight in turn) and walk the output
// in bands of eight rows of tiles, so that those on an XCD at one time share their rows of x and of w in its L2.
__device__ inline void tile_of(int block, int m_blocks, int n_blocks, int& bm, int& bn) {
  const int total = m_blocks * n_blocks;
  const int logical = total % kXcds == 0 ? (block % kXcds) * (total / kXcds) + block / kXcds : block;
  const int per_band = 8 * n_blocks, first = (logical / per_band) * 8, rows = min(8, m_blocks - first);
  bm = first + logical % per_band % rows;
  bn = logical % per_band / rows;
}

// Waits until only the loads of `later` steps of PER loads each are outstanding (they finish in order).
template <int PER, int MAX>
__device__ inline void wait_for_step(int later) {
  if constexpr (MAX == 0) {
    wait_loads<0>();
  } else {
    if (later >= MAX) wait_loads<PER * MAX>();
    else wait_for_step<PER, MAX - 1>(later);
  }
}

// What a product of few rows has to do with an RMSNorm: nothing, or it finishes one (ssq), or it prepares one (emit_g).  Each its own
// kernel: one with both in it cost a product without a norm 0.1 to 0.4 us (8 rows, 192 x 64 2.30 us with them in it and 2.19 without, 2,048 x 5,632
// 16.0 and 15.7).
enum Norm : int { kNoNorm = 0, kFinishes = 1, kPrepares = 2 };

// XR: rows of x a workgroup takes (blockIdx.y: which).  HALF: eight rows of w a workgroup instead of 16 (see launch_stream).  PAST: w past the caches.
template <int XR, int STAGES, int EPI, int NORM, bool HALF, bool PAST>
__global__ __launch_bounds__(kThreads) void gemm_f32_stream_kernel(const Args a) {
  constexpr int MT = (XR + 15) / 16, WP = HALF ? 1 : 2, PER = WP + XR / 8, kRing = PER * 1024;      // (WP: pieces of w a step)
  static_assert(!HALF || !paired(EPI), "half a block of a gated product would part gates and ups, of a rotated one a pair");
  extern __shared__ __align__(1024) unsigned char stream_lds[];
  const int lane = threadIdx.x % kWave;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int col = lane % 16, grp = lane / 16;
  const int k = a.k, row0 = blockIdx.y * XR, m = min(XR, a.m - row0);
  constexpr int kCols = paired(EPI) || HALF ? 8 : 16;        // outputs (pairs of them) of a workgroup
  const int n_out = paired(EPI) ? a.n / 2 : a.n;
  // kRopeKv: pairs 8 b .. of a head, b = blockIdx.x % (d / 16): dimensions 8 b .. and d / 2 further; n0 is the first's row of w
  const int head_dim = EPI == kRopeKv ? a.rope.head_dim : 16, head = EPI == kRopeKv ? blockIdx.x / (head_dim / 16) : 0;
  const int pair0 = EPI == kRopeKv ? blockIdx.x % (head_dim / 16) * 8 : 0;
  const int n0 = EPI == kRopeKv ? head * head_dim + pair0 : blockIdx.x * kCols;

  // this wave's steps of k
  const int per_wave = steps_a_share(k), first = wave * per_wave;
  const int n_steps = max(0, min((k + kStepK - 1) / kStepK, first + per_wave) - first);
  unsigned char* ring = stream_lds + wave * (STAGES * kRing);
  const unsigned ring_at = static_cast<unsigned>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) unsigned char*)ring));

  // Lane l of a load brings segment (l % 8) ^ key of the eight rows' row l / 8.  Rows beyond the matrix are read from its
  // last row (their results are not stored).
  const float* bases[PER];
  unsigned offsets[PER], back[PER];                          // (back: from a segment to its row's first one)
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const int r = (i < WP ? i : i - WP) * 8 + lane / 8, seg = (lane % 8) ^ slot_key(r);
    back[i] = seg * 16;
    if (i < WP) {                                            // (a load's eight rows of w lie together, from a scalar base)
      // (paired: the second eight rows as far from the first as the ups from the gates, or a pair's halves)
      const int last = EPI == kRopeKv ? a.n - 1 : n_out - 1;
      const int from = paired(EPI) ? n0 : min(n0 + i * 8, last);
      const int at = min(paired(EPI) ? n0 + lane / 8 : n0 + r, last);
      bases[i] = a.w + static_cast<long>(from + (gated(EPI) ? i * (a.n / 2) : EPI == kRopeKv ? i * (head_dim / 2) : 0)) * k + first * kStepK;
      offsets[i] = static_cast<unsigned>(at - from) * k * 4 + seg * 16;
    } else {
      bases[i] = a.x + static_cast<long>(row0) * k + first * kStepK;
      offsets[i] = static_cast<unsigned>(min(r, m - 1)) * k * 4 + seg * 16;
    }
  }
  // (the offsets before the loads below: a multiplication with a 64-bit addend takes whatever register is beside its own, and waits for it)
  if constexpr (EPI == kAccum || EPI == kRopeKv || NORM == kFinishes) {
#pragma unroll
    for (int i = 0; i < PER; ++i) asm volatile("" : "+v"(offsets[i])::"memory");
  }

  // What is added to is asked for now: item j of a thread is output (threadIdx.x + j * kThreads) of the workgroup's.  (Every load is made, from a
  // place that there is, and nothing is done with it before the walk: behind a branch, or for its sum, the compiler waits for it.)
  constexpr int kItems = (XR * kCols + kThreads - 1) / kThreads;
  float prev[kItems], bias[kItems], gain[kItems];
  if constexpr (EPI == kAccum) {
#pragma unroll
    for (int j = 0; j < kItems; ++j) {
      const int idx = threadIdx.x + j * kThreads, gn = min(n0 + idx % kCols, n_out - 1);
      prev[j] = a.out[static_cast<long>(row0 + min(idx / kCols, m - 1)) * n_out + gn];
      bias[j] = (a.bias != nullptr ? a.bias : a.out)[gn];
      if constexpr (NORM == kPrepares) gain[j] = a.emit_g[gn];
    }
  }
  // So are a prepared x's parts of the rows' sums of squares -- sixteen chains a row, chain c adding blocks c, c + 16, ... in that order, the
  // first kAhead of them (4,096 columns) asked for together, two chains a wave --, and a rotation's angles and the places in the cache.
  constexpr int kChains = 16, kAhead = 16, kWaveParts = 2 * kAhead * XR / kWave;
  static_assert(kChains == 2 * kWaves && 2 * XR <= kWave, "two chains a wave, a lane for each row of both");
  auto part_at = [&](int chain, int i, int row) {
    return static_cast<unsigned>(min(chain + i * kChains, a.ssq_blocks - 1) * a.m + row0 + min(row, m - 1)) * (1 + a.ssq_halves);
  };
  constexpr bool kPairs = XR == 8;                           // (as many rows as halves come with; of more rows they are read after the walk)
  float part[kWaveParts], second[kPairs ? kWaveParts : 1];   // (second: of a pair of halves, else the same once more)
  if constexpr (NORM == kFinishes) {
#pragma unroll
    for (int j = 0; j < kWaveParts; ++j) {
      const int idx = (j * kWave + lane) / XR;
      const float* from = a.ssq + part_at(2 * wave + idx / kAhead, idx % kAhead, lane % XR);
      part[j] = from[0];
      if constexpr (kPairs) second[j] = from[a.ssq_halves];
    }
  }
  float2 angle[kItems];
  int slot[kItems];
  const bool rotates = EPI == kRopeKv && a.rope.table != nullptr, writes = EPI == kRopeKv && a.rope.write_kv && head >= a.rope.n_heads;
  if constexpr (EPI == kRopeKv) {
#pragma unroll
    for (int j = 0; j < kItems; ++j) {
      const int idx = threadIdx.x + j * kThreads, row = min(idx / kCols, m - 1);
      angle[j] = (rotates ? a.rope.table : reinterpret_cast<const float2*>(a.x))[rotates ? (row0 + row) * (head_dim / 2) + pair0 + idx % kCols : 0];
      slot[j] = (writes ? a.rope.slot_map : reinterpret_cast<const int32_t*>(a.x))[writes ? row0 + row : 0];
    }
  }

  auto ask = [&](int s) {                                    // step s of this wave's
    const int k0 = (first + s) * kStepK;
    const float* b[PER];
    unsigned o[PER];
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      b[i] = bases[i] + s * kStepK;
      // (a segment beyond the row's end: its row's first, it is not used)
      o[i] = k0 + kStepK <= k || k0 * 4 + static_cast<int>(back[i]) < k * 4 ? offsets[i] : offsets[i] - back[i];
    }
    load_pieces_to_lds<PER, PAST>(b, o, ring_at + (s % STAGES) * kRing);
  };

  floatx4 acc[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t) acc[t] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int s = 0; s < STAGES; ++s)
    if (s < n_steps) ask(s);

  for (int s = 0; s < n_steps; ++s) {
    // The ring is one wave's and ordered by waits alone: a step's reads stay below the wait for its loads, and above the one
    // after which its place is filled anew.  (To the compiler a bare wait is no access to memory: it is told.)
    wait_for_step<PER, STAGES - 1>(min(n_steps - 1, s + STAGES - 1) - s);
    asm volatile("" ::: "memory");
    const unsigned char* at = ring + (s % STAGES) * kRing;
    const int k0 = (first + s) * kStepK;
    floatx4 wf[2], xf[MT][2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int seg = 4 * h + grp;
      const int wr = HALF ? col % 8 : col;                     // (the other eight rows repeat them, their sums are not used)
      wf[h] = *reinterpret_cast<const floatx4*>(at + wr * kStepBytes + ((seg ^ slot_key(wr)) * 16));
#pragma unroll
      for (int t = 0; t < MT; ++t) {
        const int r = (t * 16 + col) % XR;
        xf[t][h] = *reinterpret_cast<const floatx4*>(at + WP * 1024 + r * kStepBytes + ((seg ^ slot_key(r)) * 16));
      }
      if (k0 + kStepK > k && k0 + seg * 4 >= k) {
        wf[h] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int t = 0; t < MT; ++t) xf[t][h] = floatx4{0.f, 0.f, 0.f, 0.f};
      }
    }
    if (s + STAGES < n_steps) {
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");       // the reads are done: their place is filled anew
      ask(s + STAGES);
    }
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int t = 0; t < MT; ++t) acc[t] = mfma_16x16x4(wf[h][e], xf[t][h][e], acc[t]);
  }

  __shared__ float part_sum[NORM == kFinishes ? kChains : 1][NORM == kFinishes ? XR : 1];
  if constexpr (NORM == kFinishes) {
    // through the wave's own ring, which is free
    float* own = reinterpret_cast<float*>(ring);
    static_assert(kWaveParts * kWave * 4 <= STAGES * kRing, "the parts fit the ring");
#pragma unroll
    for (int j = 0; j < kWaveParts; ++j) {
      const int idx = (j * kWave + lane) / XR;
      float other = 0.f;
      if constexpr (kPairs) other = second[j];
      asm volatile("" : "+v"(part[j]), "+v"(other));
      if (!kPairs && a.ssq_halves) other = a.ssq[part_at(2 * wave + idx / kAhead, idx % kAhead, lane % XR) + 1];
      own[j * kWave + lane] = 2 * wave + idx / kAhead + idx % kAhead * kChains < a.ssq_blocks ? part[j] + (a.ssq_halves ? other : 0.f) : 0.f;
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    if (lane < 2 * XR) {
      const int chain = 2 * wave + lane / XR;
      float ss = 0.f;
#pragma unroll
      for (int i = 0; i < kAhead; ++i) ss += own[(lane / XR * kAhead + i) * XR + lane % XR];
      for (int i = kAhead; chain + i * kChains < a.ssq_blocks; ++i) {
        const float* from = a.ssq + part_at(chain, i, lane % XR);
        ss += from[0] + (a.ssq_halves ? from[1] : 0.f);
      }
      part_sum[chain][lane % XR] = ss;
    }
  }
  __syncthreads();                                           // the rings' place takes the waves' sums
  typedef float Red[MT][16][kRedPad];
  Red* red = reinterpret_cast<Red*>(stream_lds);
  static_assert(sizeof(Red) <= STAGES * kRing, "the sums fit the rings");
  // acc[t][r] is this wave's share of weight row 4 grp + r and row t * 16 + col
#pragma unroll
  for (int t = 0; t < MT; ++t)
#pragma unroll
    for (int r = 0; r < 4; ++r) red[wave][t][4 * grp + r][col] = acc[t][r];
  __syncthreads();
#pragma unroll
  for (int j = 0; j < kItems; ++j) {
    const int idx = threadIdx.x + j * kThreads, nl = idx % kCols, row = idx / kCols, gn = n0 + nl;
    const bool live = row < m && (EPI == kRopeKv || gn < n_out);
    if (NORM != kPrepares && !live) continue;                // (else the lanes exchange sums of squares)
    float sum = 0.f, up = 0.f;
    if (live) {
#pragma unroll
      for (int v = 0; v < kShares; ++v) sum += red[v][row / 16][nl][row % 16];
      if constexpr (paired(EPI)) {
#pragma unroll
        for (int v = 0; v < kShares; ++v) up += red[v][row / 16][nl + 8][row % 16];
      }
      if constexpr (NORM == kFinishes) {
        float ss = 0.f;
#pragma unroll
        for (int v = 0; v < kChains; ++v) ss += part_sum[v][row];
        const float scale = 1.0f / sqrtf(ss / static_cast<float>(k) + a.eps);
        sum *= scale;
        up *= scale;
      }
    }
    if constexpr (EPI == kRopeKv) {
      const RopeKv& r = a.rope;
      const bool is_v = head >= r.n_heads + r.n_kv_heads;
      asm volatile("" : "+v"(angle[j].x), "+v"(angle[j].y), "+v"(slot[j]));
      if (!rotates) angle[j] = make_float2(1.f, 0.f);
      const int i0 = pair0 + nl, i1 = i0 + head_dim / 2;
      const float lo = is_v ? sum : fmaf(sum, angle[j].x, -(up * angle[j].y)), hi = is_v ? up : fmaf(up, angle[j].x, sum * angle[j].y);
      if (head < r.n_heads) {
        float* to = a.out + (static_cast<long>(row0 + row) * r.n_heads + head) * head_dim;
        to[i0] = lo, to[i1] = hi;
      } else if (writes) {
        const int kvh = is_v ? head - r.n_heads - r.n_kv_heads : head - r.n_heads, off = slot[j] % r.page_tokens;
        float* to = (is_v ? r.v_cache : r.k_cache) +
                    (static_cast<long>(slot[j] / r.page_tokens) * r.n_kv_heads + kvh) * head_dim * r.page_tokens;
        if (is_v) to += off, to[static_cast<long>(i0) * r.page_tokens] = lo, to[static_cast<long>(i1) * r.page_tokens] = hi;
        else to += static_cast<long>(off) * head_dim, to[i0] = lo, to[i1] = hi;
      }
      continue;
    }
    const long at = static_cast<long>(row0 + row) * n_out + gn;
    if constexpr (EPI == kAccum) {
      asm volatile("" : "+v"(prev[j]), "+v"(bias[j]));
      const float nv = prev[j] + (a.bias != nullptr ? bias[j] : 0.f) + sum;
      if (live) a.out[at] = nv;
      if constexpr (NORM == kPrepares) {
        // the row's outputs of this workgroup lie in kCols neighbouring lanes
        float sq = live ? nv * nv : 0.f;
#pragma unroll
        for (int off = 1; off < kCols; off <<= 1) sq += __shfl_xor(sq, off, kWave);
        if (live) a.emit_x[at] = nv * gain[j];
        if (nl == 0 && row < m) {
          if constexpr (HALF) {
            float* to = a.emit_ssq + (static_cast<long>(blockIdx.x / 2) * a.m + row0 + row) * 2;
            to[blockIdx.x % 2] = sq;
            if (blockIdx.x % 2 == 0 && blockIdx.x + 1 == gridDim.x) to[1] = 0.f;      // (a last block that has no second half)
          } else {
            a.emit_ssq[static_cast<long>(blockIdx.x) * a.m + row0 + row] = sq;
          }
        }
      }
    } else if constexpr (gated(EPI)) {
      a.out[at] = gate_act<EPI>(sum) * up;
    } else {
      a.out[at] = sum;
    }
  }
}

template <int XR, int STAGES, int EPI, int NORM, bool HALF, bool PAST>
int launch_stream_kernel(const Args& a, hipStream_t s) {
  auto kernel = gemm_f32_stream_kernel<XR, STAGES, EPI, NORM, HALF, PAST>;
  constexpr int kLds = kWaves * STAGES * ((HALF ? 1 : 2) + XR / 8) * 1024;
  static_assert(kLds <= 160 * 1024, "a workgroup's LDS");
  static std::atomic<bool> raised{false};   // per instantiation: allow more than the default dynamic LDS
  if (!raised) {
    if (hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, kLds) != hipSuccess)
      return fail("gemm_f32: cannot raise the dynamic LDS limit");
    raised = true;
  }
  const int cols = paired(EPI) || HALF ? 8 : 16, n_out = paired(EPI) ? a.n / 2 : a.n;
  kernel<<<dim3((n_out + cols - 1) / cols, (a.m + XR - 1) / XR), kThreads, kLds, s>>>(a);
  return 0;
}

// Past the caches where one workgroup alone reads a part of w (64 rows, two workgroups a part: 11,264 x 2,048 54.4 us and 59.4 past them).
template <int XR, int STAGES, int EPI, int NORM, bool HALF = false>
int launch_stream_form(const Args& a, hipStream_t s) {
  return a.m <= XR && passes_by(a.n, a.k, 4) ? launch_stream_kernel<XR, STAGES, EPI, NORM, HALF, true>(a, s)
                                             : launch_stream_kernel<XR, STAGES, EPI, NORM, HALF, false>(a, s);
}

// Outputs a workgroup of few rows' kernel takes of a product that stores or adds.
int stream_cols(int m, int n) { return m <= 8 && 2 * ((n + 15) / 16) <= compute_units() ? 8 : 16; }

template <int EPI, int NORM = kNoNorm>
int launch_stream(const Args& a, hipStream_t s) {
  const int cols = paired(EPI) ? 8 : 16, n_out = paired(EPI) ? a.n / 2 : a.n;
  // Outputs that would leave every other CU idle: eight a workgroup, half the weights for each CU to bring and the
  // same sums.  A decode step's two such products, 2,048 x 2,048 and
  // 2,048 x 5,632, from memory, 8 rows, inside a step: 13.05 -> 11.7 us on average; 32 steps of 8 requests after their prompts 67.6 -> 63.5 ms.
  if constexpr (!paired(EPI)) {
    if (stream_cols(a.m, n_out) == 8) return launch_stream_form<8, 2, EPI, NORM, true>(a, s);
  }
  // Two steps ahead, so that a CU holds up to three workgroups: more of them in flight were slower in every product whose weights come from memory
  // (8 rows: 2,048 x 5,632 rings of 8 steps 16.5 us, of 4 15.3, of 2 14.5; 2,560 x 2,048 of 6 10.0, of 3 9.2, of 2 8.7; 16 rows 11,264 x 2,048 of 3
  // 26.6, of 2 20.7).
  if (a.m <= 8) return launch_stream_form<8, 2, EPI, NORM>(a, s);
  if (a.m <= 16) return launch_stream_form<16, 2, EPI, NORM>(a, s);
  return launch_stream_form<32, 2, EPI, NORM>(a, s);
}

// ---- many rows ----------------------------------------------------------------------------------

// WM x WN waves of TM x TN blocks of 32 x 32.  Gated: of a wave's blocks of columns the even ones are gate rows of w, the odd
// ones the up rows of the same outputs, which so meet in the same registers of the same lane.
template <int WM, int WN, int TM, int TN, int STAGES, int MINWG, int EPI>
__global__ __launch_bounds__(64 * WM * WN, MINWG) void gemm_f32_tiled_kernel(const Args a, int m_blocks, int n_blocks) {
  constexpr int RA = 32 * TM * WM, RW = 32 * TN * WN, NW = WM * WN, kStage = (RA + RW) * kStepBytes;
  constexpr int GA = RA / 8, GW = RW / 8, PER = (GA + GW) / NW;              // wave-wide loads a step: eight rows each
  static_assert((GA + GW) % NW == 0 && (!gated(EPI) || TN % 2 == 0), "whole loads a wave; gates beside ups");
  constexpr int kOut = gated(EPI) ? RW / 2 : RW;                             // columns of the output tile
  extern __shared__ __align__(1024) unsigned char tile_lds[];
  const unsigned lds_at = static_cast<unsigned>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) unsigned char*)tile_lds));
  const int lane = threadIdx.x % kWave;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int wm = wave / WN, wn = wave % WN, col = lane % 32, half = lane / 32;
  const int n_out = gated(EPI) ? a.n / 2 : a.n;
  int bm, bn;
  tile_of(blockIdx.x, m_blocks, n_blocks, bm, bn);
  const int m0 = bm * RA, n0 = bn * kOut;

  const unsigned char* src[PER];
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const int g = wave * PER + i, r = (g < GA ? g : g - GA) * 8 + lane / 8, seg = (lane % 8) ^ slot_key(r);
    long row;
    if (g < GA) {
      row = min(m0 + r, a.m - 1);
    } else if constexpr (gated(EPI)) {
      const int block = r / 32;                                              // (wave column block / TN, its block block % TN)
      row = min(n0 + (block / 2) * 32 + r % 32, n_out - 1) + (block % 2 ? n_out : 0);
    } else {
      row = min(n0 + r, n_out - 1);
    }
    src[i] = reinterpret_cast<const unsigned char*>((g < GA ? a.x : a.w) + row * a.k) + seg * 16;
  }
  auto ask = [&](int t) {
    const unsigned base = lds_at + (t % STAGES) * kStage + wave * PER * 1024;
    const size_t at = static_cast<size_t>(t) * kStepBytes;
#pragma unroll
    for (int i = 0; i < PER; ++i) load_to_lds_16(src[i] + at, __builtin_amdgcn_readfirstlane(base + i * 1024));
  };

  floatx16 acc[TM][TN], sum[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f, sum[i][j][r] = 0.f;
  const int n_steps = a.k / kStepK, share = steps_a_share(a.k);
#pragma unroll
  for (int s = 0; s < STAGES - 1; ++s)
    if (s < n_steps) ask(s);

  int left = share;                                          // steps until the share of k that is being added up ends
  for (int t = 0; t < n_steps; ++t) {
    wait_for_step<PER, STAGES - 2>(min(n_steps - 1, t + STAGES - 2) - t);
    lds_barrier();          // everybody's part of step t is there, and nobody reads step t - 1 any more
    if (t + STAGES - 1 < n_steps) ask(t + STAGES - 1);
    const unsigned char* at = tile_lds + (t % STAGES) * kStage;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      // segments 4 h + half and 4 h + 2 + half: with the first's element e and then the second's, an output adds up k in the
      // order of the few rows' kernel, four segments' element 0, then 1 ...
      floatx4 xf[TM][2], wf[TN][2];
#pragma unroll
      for (int i = 0; i < TM; ++i) {
        const int r = (wm * TM + i) * 32 + col;
#pragma unroll
        for (int p = 0; p < 2; ++p) xf[i][p] = *reinterpret_cast<const floatx4*>(at + r * kStepBytes + (((4 * h + 2 * p + half) ^ slot_key(r)) * 16));
      }
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        const int r = (wn * TN + j) * 32 + col;
#pragma unroll
        for (int p = 0; p < 2; ++p)
          wf[j][p] = *reinterpret_cast<const floatx4*>(at + RA * kStepBytes + r * kStepBytes + (((4 * h + 2 * p + half) ^ slot_key(r)) * 16));
      }
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int p = 0; p < 2; ++p)
#pragma unroll
          for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j)
              acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(xf[i][p][e], wf[j][p][e], acc[i][j], 0, 0, 0);
    }
    if (--left == 0) {
      left = share;
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) {
          sum[i][j] += acc[i][j];
#pragma unroll
          for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;
        }
    }
  }
  // [i][j][r] is row i 32 + 8 (r / 4) + 4 half + r % 4 and column j 32 + col of the wave's part: a store writes two rows'
  // 128 bytes
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; j += gated(EPI) ? 2 : 1) {
      const int gn = n0 + (gated(EPI) ? (wn * TN + j) / 2 : wn * TN + j) * 32 + col;
      if (gn >= n_out) continue;
      const float bias = EPI == kAccum && a.bias != nullptr ? a.bias[gn] : 0.f;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int gm = m0 + (wm * TM + i) * 32 + 8 * (r / 4) + 4 * half + r % 4;
        if (gm >= a.m) continue;
        float* to = a.out + static_cast<long>(gm) * n_out + gn;
        const float s = sum[i][j][r] + acc[i][j][r];
        if constexpr (EPI == kAccum) *to = *to + bias + s;
        else if constexpr (gated(EPI)) *to = gate_act<EPI>(s) * (sum[i][j + 1][r] + acc[i][j + 1][r]);
        else *to = s;
      }
    }
}

template <int WM, int WN, int TM, int TN, int STAGES, int MINWG, int EPI>
int launch_tiled_form(const Args& a, hipStream_t s) {
  auto kernel = gemm_f32_tiled_kernel<WM, WN, TM, TN, STAGES, MINWG, EPI>;
  constexpr int RA = 32 * TM * WM, RW = 32 * TN * WN, kLds = STAGES * (RA + RW) * kStepBytes;
  static_assert(kLds * MINWG <= 160 * 1024, "the workgroups' LDS");
  static std::atomic<bool> raised{false};   // per instantiation: allow more than the default dynamic LDS
  if (!raised) {
    if (hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, kLds) != hipSuccess)
      return fail("gemm_f32: cannot raise the dynamic LDS limit");
    raised = true;
  }
  const int n_out = gated(EPI) ? a.n / 2 : a.n, out = gated(EPI) ? RW / 2 : RW;
  const int m_blocks = (a.m + RA - 1) / RA, n_blocks = (n_out + out - 1) / out;
  kernel<<<m_blocks * n_blocks, 64 * WM * WN, kLds, s>>>(a, m_blocks, n_blocks);
  return 0;
}

// Which kernel and tile, by what each was measured to take (microseconds, the weights not in a cache; both add up k in the same
// order, so the choice moves no bit).  The few rows' kernel sustains 52 TFLOP/s once its rows are 32 a workgroup (64 rows x
// 2,048 x 5,632: 27 us; 64 x 11,264 x 2,048: 58).  The tiled one sustains 115 on all CUs (0.49 a CU's tile at a time) but no tile
// is faster than its chain of steps, 0.8 us each (65 to 256 rows x 2,048 x 5,632: 140 us whatever the rows, 128 rows x 2,560 x
// 2,048: 55): for 64 to about 250 rows of a narrow output the first is up to twice as fast, for wide ones and more rows the second.
constexpr int kTileForms = 3;
constexpr int kTileForm[kTileForms][2] = {{128, 128}, {64, 128}, {64, 64}};   // rows of x, rows of w

double stream_time(int m, int n, int k) { return 4.0 + 2.0e-6 * ((m + 31) / 32 * 32) * n * k / 52.0; }

int tile_form(int m, int n, int k, double& time) {
  int best = 0;
  for (int f = 0; f < kTileForms; ++f) {
    const long tiles = static_cast<long>((m + kTileForm[f][0] - 1) / kTileForm[f][0]) * ((n + kTileForm[f][1] - 1) / kTileForm[f][1]);
    const long turns = (tiles + compute_units() - 1) / compute_units();
    const double work = turns * 2.0e-6 * kTileForm[f][0] * kTileForm[f][1] * k * (1.0 + 0.05 * f) / 0.49;
    const double chain = 5.0 + 0.8 * (k / kStepK), t = work > chain ? work : chain;
    if (f == 0 || t < time) best = f, time = t;
  }
  return best;
}

template <int EPI>
int launch_tiled(const Args& a, int form, hipStream_t s) {
  switch (form) {
    case 0: return launch_tiled_form<2, 2, 2, 2, 2, 2, EPI>(a, s);
    case 1: return launch_tiled_form<2, 2, 1, 2, 3, 2, EPI>(a, s);
    default:
      if constexpr (gated(EPI)) return launch_tiled_form<2, 1, 1, 2, 3, 3, EPI>(a, s);
      else return launch_tiled_form<2, 2, 1, 1, 3, 3, EPI>(a, s);
  }
}

// The tiled kernel's form for a product, or -1: the few rows' kernel.
int tile_for(int m, int n, int k) {
  if (m <= 64 || k % kStepK != 0) return -1;
  double tiled;
  const int form = tile_form(m, n, k, tiled);
  return stream_time(m, n, k) < tiled ? -1 : form;
}

template <int EPI>
int launch(const Args& a, hipStream_t s) {
  const int form = tile_for(a.m, a.n, a.k);
  return form < 0 ? launch_stream<EPI>(a, s) : launch_tiled<EPI>(a, form, s);
}

}  // namespace
}  // namespace bc4g

using namespace bc4g;

extern "C" int bc4g_gemm_f32(const float* x, const float* w, const float* bias, float* out, int epilogue, int m, int n, int k, void* stream) {
  BC4G_REQUIRE(m >= 0 && n > 0 && k > 0 && k % 4 == 0 && k <= (1 << 24), "gemm_f32: bad sizes M=%d N=%d K=%d (K a multiple of 4)", m, n, k);
  BC4G_REQUIRE(reinterpret_cast<uintptr_t>(x) % 16 == 0 && reinterpret_cast<uintptr_t>(w) % 16 == 0, "gemm_f32: operands must lie on 16-byte boundaries");
  BC4G_REQUIRE((m + 31L) / 32 <= 65535 && ((m + 63L) / 64) * ((n + 31L) / 32) <= 2147483647L, "gemm_f32: M=%d N=%d are beyond the grid limit", m, n);
  BC4G_REQUIRE(!bias || epilogue == kAccum, "gemm_f32: only an adding product takes a bias");
  BC4G_REQUIRE(!gated(epilogue) || n % 2 == 0, "gemm_f32: a gated product has as many gate rows as up rows (N=%d)", n);
  if (m == 0) return 0;
  hipStream_t s = static_cast<hipStream_t>(stream);
  const Args a{x, w, bias, out, m, n, k};
  int e = 0;
  switch (epilogue) {
    case kStore: e = launch<kStore>(a, s); break;
    case kAccum: e = launch<kAccum>(a, s); break;
    case kSwiglu: e = launch<kSwiglu>(a, s); break;
    case kGeglu: e = launch<kGeglu>(a, s); break;
    default: return fail("gemm_f32: unknown epilogue %d", epilogue);
  }
  if (e) return e;
  return check_launch("gemm_f32");
}

namespace {
int few_rows(const char* what, const float* x, const float* w, int m, int n, int k) {
  BC4G_REQUIRE(m > 0 && m <= 64 && n > 0 && k > 0 && k % 4 == 0 && k <= (1 << 24), "%s: bad sizes M=%d N=%d K=%d (1 to 64 rows, K a multiple of 4)", what,
               m, n, k);
  BC4G_REQUIRE(x && w && reinterpret_cast<uintptr_t>(x) % 16 == 0 && reinterpret_cast<uintptr_t>(w) % 16 == 0,
               "%s: operands must lie on 16-byte boundaries", what);
  return 0;
}
}  // namespace

extern "C" int bc4g_gemm_f32_emit(const float* x, const float* w, const float* bias, float* residual, const float* g, float* emit_x, float* emit_ssq,
                                  int halves, int m, int n, int k, void* stream) {
  if (int e = few_rows("gemm_f32_emit", x, w, m, n, k)) return e;
  BC4G_REQUIRE((halves != 0) == (stream_cols(m, n) == 8), "gemm_f32_emit: the parts' shape does not fit M=%d N=%d", m, n);
  BC4G_REQUIRE(residual && g && emit_x && emit_ssq, "gemm_f32_emit: an operand is missing");
  Args a{x, w, bias, residual, m, n, k};
  a.emit_g = g, a.emit_x = emit_x, a.emit_ssq = emit_ssq;
  if (int e = launch_stream<kAccum, kPrepares>(a, static_cast<hipStream_t>(stream))) return e;
  return check_launch("gemm_f32_emit");
}

extern "C" int bc4g_gemm_f32_prenormed(const float* x, const float* ssq, int ssq_blocks, int ssq_halves, float eps, const float* w, float* out, int epilogue, int m, int n,
                                       int k, void* stream) {
  if (int e = few_rows("gemm_f32_prenormed", x, w, m, n, k)) return e;
  BC4G_REQUIRE(ssq && ssq_blocks > 0 && eps >= 0.f && out, "gemm_f32_prenormed: the rows' sums of squares come in %d parts", ssq_blocks);
  BC4G_REQUIRE(!gated(epilogue) || n % 2 == 0, "gemm_f32_prenormed: a gated product has as many gate rows as up rows (N=%d)", n);
  Args a{x, w, nullptr, out, m, n, k};
  a.ssq = ssq, a.ssq_blocks = ssq_blocks, a.ssq_halves = ssq_halves, a.eps = eps;
  hipStream_t s = static_cast<hipStream_t>(stream);
  int e = 0;
  switch (epilogue) {
    case kStore: e = launch_stream<kStore, kFinishes>(a, s); break;
    case kSwiglu: e = launch_stream<kSwiglu, kFinishes>(a, s); break;
    case kGeglu: e = launch_stream<kGeglu, kFinishes>(a, s); break;
    default: return fail("gemm_f32_prenormed: unknown epilogue %d", epilogue);
  }
  if (e) return e;
  return check_launch("gemm_f32_prenormed");
}

extern "C" int bc4g_gemm_f32_qkv(const float* x, const float* ssq, int ssq_blocks, int ssq_halves, float eps, const float* w, float* q, const float* table,
                                 const int32_t* slot_map, float* k_cache, float* v_cache, int m, int k, int n_heads, int n_kv_heads, int head_dim,
                                 int page_tokens, int write_kv, void* stream) {
  BC4G_REQUIRE(n_heads > 0 && n_kv_heads > 0 && head_dim > 0 && head_dim % 16 == 0 && (n_heads + 2L * n_kv_heads) * head_dim <= 2147483647L,
               "gemm_f32_qkv: %d + 2 x %d heads of %d (a multiple of 16)", n_heads, n_kv_heads, head_dim);
  const int n = (n_heads + 2 * n_kv_heads) * head_dim;
  if (int e = few_rows("gemm_f32_qkv", x, w, m, n, k)) return e;
  BC4G_REQUIRE(q && (ssq == nullptr || (ssq_blocks > 0 && eps >= 0.f)), "gemm_f32_qkv: an operand is missing");
  BC4G_REQUIRE(!write_kv || (page_tokens > 0 && k_cache && v_cache && slot_map), "gemm_f32_qkv: cache write asked for without a cache");
  Args a{x, w, nullptr, q, m, n, k};
  a.ssq = ssq, a.ssq_blocks = ssq_blocks, a.ssq_halves = ssq_halves, a.eps = eps;
  a.rope = RopeKv{reinterpret_cast<const float2*>(table), slot_map, k_cache, v_cache, n_heads, n_kv_heads, head_dim, page_tokens, write_kv ? 1 : 0};
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (int e = ssq ? launch_stream<kRopeKv, kFinishes>(a, s) : launch_stream<kRopeKv>(a, s)) return e;
  return check_launch("gemm_f32_qkv");
}

extern "C" int bc4g_gemm_f32_tile(int m, int n, int k, int* rows, int* cols) {
  BC4G_REQUIRE(rows != nullptr && cols != nullptr && m > 0 && n > 0 && k > 0, "gemm_f32_tile: sizes and two places for the answer");
  const int form = tile_for(m, n, k);
  *rows = form < 0 ? 0 : kTileForm[form][0], *cols = form < 0 ? 0 : kTileForm[form][1];
  return 0;
}
