// out[m, n] = sum_k x[m, k] * w[n, k] for few rows m (a decode step: m <= 64), bfloat16 weights.
//
// Two kernels, the same bits.  gemm_ring_kernel (below) brings weights and rows through rings in LDS and takes most products of k in whole steps of 64;
// gemm_skinny_kernel, the streaming kernel, takes them straight into registers, and serves every other k, operands off 16-byte boundaries, the
// fused norm of many or short rows, and the sizes at which it is the faster one (rings_are_slower).  What both do:
//
// The weights are read once: a workgroup owns
// 16 output columns n (16 rows of w) and all of k; its 8 waves split k between them, each wave
// feeding 16x16x32 MFMAs with w as the A operand and x as the B operand.  The weights come
// *packed in fragment order*: for every block of 16 rows and every k-step of 32, the 1 KB that a
// wave's 64 lanes load (lane l: row l % 16, k 8 * (l / 16) .. + 7) lies contiguous, blocks and
// k-steps in order -- so every load instruction reads eight whole cache lines and a wave walks
// straight through memory (rows past n and k past the matrix are stored as zeros).  Loads run
// ahead of the MFMAs that use them, by a batch of k-steps in registers or by as many stages as the rings have.  The waves' partial sums meet in LDS
// and are added in wave order, so a result does not depend on the number of rows or on timing.
// Where the weight blocks are few and the rows of x more than eight, two workgroups share a block,
// each with half of the rows of x (what a CU can pull through its cache bounds the kernel, so the
// pulling is spread).
//
// What comes in (XMODE; as the streaming kernel takes it):
//   plain    x is bfloat16 [m, k].  The B operand's own pattern (a lane group reads 16 bytes of
//            each of 16 rows) keeps the texture path busy four times as long as a load of whole
//            cache lines, and with 64 rows x is four times the weights' traffic: so x comes in row
//            by row (eight or sixteen lanes read a row's part of the batch) and is turned into
//            operand order through a buffer in LDS that belongs to the wave -- no barrier, and the
//            next batch's loads are in flight meanwhile.
//   normed   x is the float residual stream (rows taken through `rows` if given) and RMSNorm is
//            fused (up to 16 rows): while the first weights are already on their way, the
//            workgroup writes bf16(x * g) into LDS and sums x^2 per row; the MFMAs read their B
//            operand from LDS, and the row's rsqrt(mean(x^2) + eps) -- a factor common to the
//            whole row -- multiplies the finished sum.
//   prenormed  x is bfloat16(residual * g), written by the product that last added to the residual
//            (below), together with parts of every row's sum of squares: the row's scale is worked out
//            from the parts while the weights are on their way and multiplies the finished sum -- the
//            norm costs neither a kernel of its own nor the staging of the float rows.
// What goes out (EPI): bfloat16 or float stored; bfloat16 after max(., 0)^2 or xIELU (8 rows,
// 2,048 to 8,192: product with its norm inside 13.0 us and the activation behind it 5.5; normed before and activated here 8.8);
// float added into the residual stream; SwiGLU,
// when every 16 rows of w are eight gate rows followed by the eight up rows of the same outputs; or
// rotary positions and the cache write, when w holds query, key and value heads with every head's
// rows reordered in blocks of 16 (eight dimensions, then their rotation partners): queries are
// stored rotated, keys rotated into their page, values into theirs.  The epilogue that adds into the
// residual stream can prepare the RMSNorm that follows (emit): it also stores bfloat16(new residual * g)
// and, per row, the sum of squares over its 16 columns -- parts that the next product adds up in
// block order, so the result does not depend on timing.
#include <type_traits>
#include <math.h>

#include "api.h"
#include "mfma.h"

namespace bc4g {
namespace {

constexpr int kWaves = 8;
constexpr int kThreads = kWaves * kWave;
constexpr int kRedPad = 17;
constexpr int kStagePad = 8;     // bf16 elements appended to each staged row of x

enum Epilogue : int { kStoreBf16 = 0, kStoreF32 = 1, kAccumF32 = 2, kSwigluBf16 = 3, kRopeKvBf16 = 4, kSquaredReluBf16 = 6, kGegluBf16 = 7, kXieluBf16 = 8 };
// products whose weight holds blocks of eight gate rows and the eight up rows of the same outputs
constexpr bool gated(int epi) { return epi == kSwigluBf16 || epi == kGegluBf16; }

struct RopeKvArgs {
  const int32_t* positions;   // [m]
  const int32_t* slot_map;    // [m] page * page_tokens + offset
  bf16_t* k_cache;            // [pages, n_kv, page_tokens, d], or every [page_tokens, d] in fragment order
  bf16_t* v_cache;            // [pages, n_kv, d, page_tokens], or likewise
  int n_heads, n_kv_heads, head_dim, rotary_dim, page_tokens, write_kv;
  int fragment_order;         // how the cache's pages are laid out (cache_fragment_order)
  float theta;
};
enum XMode : int { kPlain = 0, kNormedG16 = 1, kNormedG32 = 2 };   // norm scale g in bfloat16 / float

struct SkinnyArgs {
  // (first, 64 bytes together, what the ring kernel needs before its first load: one trip for them)
  const void* x;            // bf16 [m, k], or float [*, k] in the normed modes
  const bf16_t* w;          // packed: [ceil(n / 16)][ceil(k / 32)][64 lanes][8]
  void* out;
  // prenormed x (plain mode): parts [ssq_blocks][ssq_stride] of the rows' sums of squares (null: x as it is)
  const float* ssq_parts;
  int m, n, k;
  int rows_per_block;       // plain mode: blockIdx.y takes rows y * rows_per_block .. of x and out (0: all rows)
  int chunk;                // ring kernel: a wave's part of k,
  int last_block;           // the last block of w,
  int part_stride;          // numbers from one part to the next, and where the last four of all parts begin
  int last_four;
  int x_row_bytes, g_f32;   // ring kernel, normed modes: LDS of a float row of x; whether g is float
  int ssq_blocks, ssq_stride;
  int ssq_halves;           // the parts are pairs, [ssq_blocks][ssq_stride][2]
  float eps;
  const int32_t* rows;      // normed modes: row m of the product reads x[rows[m]] (null: x[m])
  const void* g;            // normed modes: RMSNorm scale [k]
  int m_stage;              // normed modes: rows of x staged in LDS (m rounded up to 4)
  int halves;               // host: two workgroups a block (see launch)
  // kAccumF32: a number a column that joins every row's sums (null: none); kXieluBf16: the activation's two numbers
  const float* bias;
  // kAccumF32: what the RMSNorm after this product needs (emit_g null: nothing)
  const void* emit_g;       // [n] its scale, bfloat16 or float (emit_g_f32)
  bf16_t* emit_x;           // [m, n] bfloat16(new residual * g)
  float* emit_ssq;          // [ceil(n / 16)][emit_stride]: block b's part of row r's sum of squares (with halves [..][2]: of its halves)
  int emit_g_f32, emit_stride;
  RopeKvArgs rope;          // kRopeKvBf16 only
};

__device__ inline uint32_t pack2(float a, float b) {
  return static_cast<uint32_t>(bf16_bits_from_float(a)) | (static_cast<uint32_t>(bf16_bits_from_float(b)) << 16);
}

// Where the weight blocks are too few to occupy the CUs, the rows are shared out over blockIdx.y (plain mode): such a workgroup sees
// its own rows only, as if they were the whole batch.
template <int EPI>
__device__ inline SkinnyArgs own_rows(const SkinnyArgs& args) {
  SkinnyArgs a = args;
  if (args.rows_per_block > 0) {
    const long row0 = static_cast<long>(blockIdx.y) * args.rows_per_block;
    a.m = min(args.rows_per_block, args.m - static_cast<int>(row0));
    a.x = static_cast<const bf16_t*>(args.x) + row0 * args.k;
    if constexpr (EPI == kStoreBf16 || EPI == kSquaredReluBf16 || EPI == kXieluBf16) a.out = static_cast<bf16_t*>(args.out) + row0 * args.n;
    else if constexpr (gated(EPI)) a.out = static_cast<bf16_t*>(args.out) + row0 * (args.n / 2);
    else if constexpr (EPI == kRopeKvBf16) {
      a.out = static_cast<bf16_t*>(args.out) + row0 * args.rope.n_heads * args.rope.head_dim;
      a.rope.positions = args.rope.positions ? args.rope.positions + row0 : nullptr;
      a.rope.slot_map = args.rope.slot_map ? args.rope.slot_map + row0 : nullptr;
    } else a.out = static_cast<float*>(args.out) + row0 * args.n;
    if (args.ssq_parts) a.ssq_parts = args.ssq_parts + row0;
    if (EPI == kAccumF32 && args.emit_g) {
      a.emit_x = args.emit_x + row0 * args.n;
      a.emit_ssq = args.emit_ssq + row0;
    }
  }
  return a;
}

// What an output's thread has at hand before its sum is there.
struct Kept {
  float prev;                 // kAccumF32: what the sum is added to (with the bias),
  bool ask_g;                 // whether the next norm's scale is yet to be asked for (behind the store of the sum), or
  float g;                    // that scale
  float cs, sn;               // kRopeKvBf16: its pair's rotation ...
  int slot;                   // ... and place in the cache
  float xielu_p, xielu_q;
};

__device__ inline float emit_scale(const SkinnyArgs& a, int gn) {
  return a.emit_g_f32 ? static_cast<const float*>(a.emit_g)[gn] : to_float(static_cast<const bf16_t*>(a.emit_g)[gn]);
}

// The rotation of a pair (its lower dimension's place in the products' columns) at a position.
__device__ inline void pair_angle(const RopeKvArgs& r, int n0, int nl, int position, float& cs, float& sn) {
  const int pair = (n0 % r.head_dim) / 2 + nl;            // 8 * block + nl
  const float inv_freq = 1.0f / powf(r.theta, (2.0f * static_cast<float>(pair)) / static_cast<float>(r.head_dim));
  sincosf(static_cast<float>(position) * inv_freq, &sn, &cs);
}

// The finished sum of output nl of the block (or half block) at n0, row `row`, goes out; `partner` is that of output nl + 8 where those belong
// together.  in_block: the lane stands for a row and column of the block at all (the adding epilogue goes on with every lane: COLS
// neighbouring lanes, a row's, exchange sums of squares); live: and for a column and row that there are.
template <int EPI, int COLS, bool HALF>
__device__ inline void put_output(const SkinnyArgs& a, int n0, int wblock_index, int half, int row, int nl, bool in_block, bool live, float sum, float partner,
                                  const Kept& kept) {
  const int gn = n0 + nl;
  if constexpr (EPI == kStoreBf16) {
    static_cast<bf16_t*>(a.out)[static_cast<long>(row) * a.n + gn] = from_float<bf16_t>(sum);
  } else if constexpr (EPI == kSquaredReluBf16) {
    const float z = fmaxf(sum, 0.f);
    static_cast<bf16_t*>(a.out)[static_cast<long>(row) * a.n + gn] = from_float<bf16_t>(z * z);
  } else if constexpr (EPI == kXieluBf16) {
    const float z = to_float(from_float<bf16_t>(sum));       // as a kernel behind the product would find it
    static_cast<bf16_t*>(a.out)[static_cast<long>(row) * a.n + gn] = from_float<bf16_t>(xielu_f(z, kept.xielu_p, kept.xielu_q));
  } else if constexpr (EPI == kStoreF32) {
    static_cast<float*>(a.out)[static_cast<long>(row) * a.n + gn] = sum;
  } else if constexpr (EPI == kAccumF32) {
    const float nv = kept.prev + sum;
    if (live) static_cast<float*>(a.out)[static_cast<long>(row) * a.n + gn] = nv;
    if (a.emit_g != nullptr) {
      // for the RMSNorm that follows: bf16(new residual * g), and this block's part of the row's sum
      // of squares (a row's 16 columns, or eight of half a block, lie in as many neighbouring lanes)
      float sq = 0.f;
      if (live) {
        a.emit_x[static_cast<long>(row) * a.n + gn] = from_float<bf16_t>(nv * (kept.ask_g ? emit_scale(a, gn) : kept.g));
        sq = nv * nv;
      }
#pragma unroll
      for (int off = 1; off < COLS; off <<= 1) sq += __shfl_xor(sq, off, kWave);
      if (nl == 0 && in_block && row < a.m && wblock_index * 16 < a.n) a.emit_ssq[(static_cast<long>(wblock_index) * a.emit_stride + row) * (HALF ? 2 : 1) + half] = sq;
    }
  } else if constexpr (gated(EPI)) {
    // block b = n0 / 16 holds gates and ups of outputs 8b .. 8b + 7
    const long o = static_cast<long>(row) * (a.n / 2) + (n0 / 2 + nl);
    static_cast<bf16_t*>(a.out)[o] = from_float<bf16_t>((EPI == kGegluBf16 ? gelu_tanh_quick(sum) : silu_quick(sum)) * partner);
  } else {
    const RopeKvArgs& r = a.rope;
    const int d = r.head_dim;
    const int head = n0 / d, in_head = n0 % d + nl;         // the pair lies at in_head and in_head + 8
    float lo = sum, hi = partner;
    const bool is_v = head >= r.n_heads + r.n_kv_heads;
    if (r.rotary_dim > 0 && !is_v) {                        // (spelt out, so that every form of the kernels rounds alike)
      const float cs = kept.cs, sn = kept.sn, l0 = lo, h0 = hi;
      lo = fmaf(l0, cs, -(h0 * sn));
      hi = fmaf(h0, cs, l0 * sn);
    }
    if (head < r.n_heads) {
      bf16_t* q = static_cast<bf16_t*>(a.out) + (static_cast<long>(row) * r.n_heads + head) * d + in_head;
      q[0] = from_float<bf16_t>(lo);
      q[8] = from_float<bf16_t>(hi);
    } else if (r.write_kv) {
      const int kvh = is_v ? head - r.n_heads - r.n_kv_heads : head - r.n_heads;
      const int slot = kept.slot;
      const long page = slot / r.page_tokens, off = slot % r.page_tokens;
      const long region = (page * r.n_kv_heads + kvh) * d * r.page_tokens;
      if (r.fragment_order) {
        bf16_t* dst = (is_v ? r.v_cache : r.k_cache) + region;
        const int o = static_cast<int>(off);
        dst[is_v ? frag_v_offset(o, in_head, d) : frag_k_offset(o, in_head, d)] = from_float<bf16_t>(lo);
        dst[is_v ? frag_v_offset(o, in_head + 8, d) : frag_k_offset(o, in_head + 8, d)] = from_float<bf16_t>(hi);
      } else if (is_v) {
        bf16_t* dst = r.v_cache + region + in_head * r.page_tokens + off;
        dst[0] = from_float<bf16_t>(lo);
        dst[8L * r.page_tokens] = from_float<bf16_t>(hi);
      } else {
        bf16_t* dst = r.k_cache + region + off * d + in_head;
        dst[0] = from_float<bf16_t>(lo);
        dst[8] = from_float<bf16_t>(hi);
      }
    }
  }
}

// MT tiles of 16 rows of x; U k-steps of 32 a batch; ROWS: 16, or 8 where there are no more rows than that (plain x: half the
// loads and LDS writes for x); HALF: two workgroups share a weight block, each with eight of its outputs (see launch).
template <int MT, int EPI, int XMODE, int U, int ROWS = 16, bool HALF = false>
// (The normed form keeps to 80 registers, so that three workgroups share a CU and all the blocks of
// a 5,632 x 2 wide gate-up matrix are in flight at once.)
__global__ __launch_bounds__(kThreads, (XMODE != kPlain || (MT == 1 && U == 2)) ? 6 : U == 8 ? 2 : 4) void gemm_skinny_kernel(const SkinnyArgs args) {
  constexpr bool kNormed = XMODE != kPlain;
  // Every line of the arguments in one trip: left to itself the compiler asks for the norm's, in the second line, behind the first loads, and waits
  // for them there (one row, weights from memory: 768 x 768 after a prepared norm 3.20 and 3.07 us, 32,000 x 512 8.6 and 7.9).
  if constexpr (!kNormed) asm volatile("" ::"s"(args.m), "s"(args.ssq_blocks), "s"(args.ssq_stride), "s"(args.ssq_halves), "s"(args.eps));
  if constexpr (EPI == kAccumF32) asm volatile("" ::"s"(args.bias), "s"(args.emit_stride));
  const SkinnyArgs a = kNormed ? args : own_rows<EPI>(args);
  constexpr bool kTurned = !kNormed;                      // x reaches operand order through LDS
  constexpr int kPieces = 4 * U;                       // 16-byte pieces of a row in one batch of k-steps
  static_assert(!kNormed || MT == 1, "the fused norm handles one tile of rows");
  static_assert(ROWS == 16 || (ROWS == 8 && MT == 1 && !kNormed), "eight rows: one tile of plain rows");
  static_assert(!HALF || (MT == 1 && XMODE == kPlain && !gated(EPI) && EPI != kRopeKvBf16), "half blocks: few plain rows, unpaired outputs");
  static_assert(!kTurned || 64 % kPieces == 0, "a load instruction covers whole rows of a batch");
  static_assert(!kTurned || kPieces >= 8, "the buffer's swizzle (piece ^ row % 8) must stay inside a row's pieces");
  // The waves' partial sums, and before them (kTurned) every wave's buffer for x: the same memory.
  typedef float Red[MT][16][kRedPad];
  constexpr int kRedBytes = kWaves * static_cast<int>(sizeof(Red));
  constexpr int kTurnBytes = kTurned ? kWaves * MT * ROWS * kPieces * 16 : 0;
  __shared__ __align__(16) unsigned char pool[kRedBytes > kTurnBytes ? kRedBytes : kTurnBytes];
  Red* red = reinterpret_cast<Red*>(pool);
  __shared__ float ssq_row[16];
  extern __shared__ __align__(16) unsigned char stage_raw[];   // normed: bf16 [m_stage][k + kStagePad]
  const int lane = threadIdx.x % kWave;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);   // uniform: k ranges and bases stay scalar
  const int col = lane % 16, grp = lane / 16;
  const int wblock_index = HALF ? blockIdx.x / 2 : blockIdx.x, half = HALF ? blockIdx.x % 2 : 0;
  const int n0 = wblock_index * 16 + 8 * half;
  const int k = a.k, m = a.m;

  // every wave's part of k starts on a cache line of x (64 elements), whatever the number of rows:
  // the order of the additions, and so the rounding, is the same in every form of the kernel
  const int chunk = ((k + kWaves * 64 - 1) / (kWaves * 64)) * 64;
  const int k_begin = wave * chunk;
  const int k_end = min(k, k_begin + chunk);

  floatx4 acc[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t) acc[t] = floatx4{0.f, 0.f, 0.f, 0.f};

  // this workgroup's block of 16 rows in the packed weights: k-step ks at wblock + ks * 512 elements
  // (a scalar base and a 32-bit lane offset, so the loads of a batch differ in their scalar part only)
  const int ksteps_total = (k + 31) / 32;
  const bf16_t* wblock = a.w + static_cast<long>(wblock_index) * ksteps_total * (kWave * 8);
  // (half a block: the lanes of the other eight rows ask for what their neighbours ask for, and their results are not used)
  const int wlane = (HALF ? (lane & ~8) | (8 * half) : lane) * 8;

  // where this lane's B operand comes from
  const bf16_t* xptr[MT];
  bool xrow_ok[MT];
  const int stage_stride = k + kStagePad;
#pragma unroll
  for (int t = 0; t < MT; ++t) {
    const int row = t * 16 + col;
    xrow_ok[t] = row < m;
    if constexpr (kNormed) {
      xptr[t] = reinterpret_cast<const bf16_t*>(stage_raw) + static_cast<long>(min(row, a.m_stage - 1)) * stage_stride;
    } else {
      xptr[t] = static_cast<const bf16_t*>(a.x) + static_cast<long>(row) * k;
    }
  }

  // The float sums that the product is added to (the residual stream) are asked for now, not
  // after the weights: item j of a thread is output (threadIdx.x + j * kThreads) of the block.
  constexpr bool kPaired = gated(EPI) || EPI == kRopeKvBf16;   // columns nl and nl + 8 belong together
  constexpr int kCols = kPaired || HALF ? 8 : 16;
  constexpr int kAccItems = (MT * 16 * kCols + kThreads - 1) / kThreads;
  float prev[kAccItems];
  if constexpr (EPI == kAccumF32) {
#pragma unroll
    for (int j = 0; j < kAccItems; ++j) {
      const int idx = threadIdx.x + j * kThreads;
      const int row = idx / kCols, gn = n0 + idx % kCols;
      const bool live = idx < MT * 16 * kCols && row < m && gn < a.n;
      prev[j] = live ? static_cast<const float*>(a.out)[static_cast<long>(row) * a.n + gn] : 0.f;
      if (a.bias != nullptr && live) prev[j] += a.bias[gn];
    }
  }

  float xielu_p = 0.f, xielu_q = 0.f;
  if constexpr (EPI == kXieluBf16) xielu_p = softplus_f(a.bias[0]), xielu_q = 0.5f + softplus_f(a.bias[1]);

  // The rotation a thread will apply in the epilogue (its output's angle: position and pair are
  // known now) and the place in the cache it will write to are worked out while the weights are
  // on their way: item j of a thread is pair (threadIdx.x + j * kThreads) % 8 of row ... / 8.
  constexpr int kRopeItems = (MT * 128 + kThreads - 1) / kThreads;
  float rope_cs[kRopeItems], rope_sn[kRopeItems];
  int rope_slot[kRopeItems];
  if constexpr (EPI == kRopeKvBf16) {
    const RopeKvArgs& r = a.rope;
    const int head = n0 / r.head_dim;
    const bool is_v = head >= r.n_heads + r.n_kv_heads;
#pragma unroll
    for (int j = 0; j < kRopeItems; ++j) {
      const int idx = threadIdx.x + j * kThreads;
      const int row = idx / 8, nl = idx % 8;
      const bool live = idx < MT * 128 && row < m;
      rope_cs[j] = 1.f;
      rope_sn[j] = 0.f;
      if (live && r.rotary_dim > 0 && !is_v) {
        pair_angle(r, n0, nl, r.positions[row], rope_cs[j], rope_sn[j]);
      }
      rope_slot[j] = (live && head >= r.n_heads && r.write_kv) ? r.slot_map[row] : 0;
    }
  }

  // prenormed x: every row's sum of squares from its parts.  Eight threads a row, thread j adding
  // the parts of blocks j, j + 8, ... in ascending order; the eight sums meet in LDS and are added in
  // order of j after the product: the order of the additions, and so the rounding, is the same for
  // every number of rows.  (After the first weights have been asked for.)  How many parts a thread asks
  // for together: sixteen -- one way to memory and back for 128 parts instead of four -- where a workgroup has up to 8 rows, in the kernels
  // of four k-steps a turn and before gates (us, weights from memory, four and sixteen: 8 rows 4,096 x 2,720 8.4 and 8.0, 11,264 x 2,080 gated 12.6 and 11.9,
  // 12 rows as two workgroups of six 2,048 x 5,480 13.0 and 11.5), four otherwise (the other kernels of two k-steps a turn spill with more).
  constexpr int kPartSums = 8;
  __shared__ float part_sum[kPartSums][MT * 16];
  const bool prenormed = !kNormed && a.ssq_parts != nullptr;
  auto sum_parts = [&]() {
    if (prenormed && threadIdx.x < kPartSums * MT * 16) {
      const int row = threadIdx.x % (MT * 16), j0 = threadIdx.x / (MT * 16);
      float ss = 0.f;
      if (row < m) {
        const float* p = a.ssq_parts + row;
        auto chain = [&](auto ahead) {
          constexpr int kAhead = decltype(ahead)::value;
          for (int b0 = j0; b0 < a.ssq_blocks; b0 += kAhead * kPartSums) {
            float part[kAhead];
#pragma unroll
            for (int i = 0; i < kAhead; ++i) {
              const int b = b0 + i * kPartSums;
              part[i] = b < a.ssq_blocks ? p[static_cast<long>(b) * a.ssq_stride] : 0.f;
            }
#pragma unroll
            for (int i = 0; i < kAhead; ++i) ss += part[i];      // (in ascending order; a part that is not there adds 0)
          }
        };
        if (a.ssq_halves) {
          // (left by half blocks: the two halves of a part side by side, their sum the part itself)
          const float2* p2 = reinterpret_cast<const float2*>(a.ssq_parts) + row;
          constexpr int kAhead = 8;
          for (int b0 = j0; b0 < a.ssq_blocks; b0 += kAhead * kPartSums) {
            float2 part[kAhead];
#pragma unroll
            for (int i = 0; i < kAhead; ++i) {
              const int b = b0 + i * kPartSums;
              part[i] = b < a.ssq_blocks ? p2[static_cast<long>(b) * a.ssq_stride] : make_float2(0.f, 0.f);
            }
#pragma unroll
            for (int i = 0; i < kAhead; ++i) ss += part[i].x + part[i].y;
          }
        } else if ((U == 4 || gated(EPI)) && m <= 8) chain(std::integral_constant<int, 16>{});
        else chain(std::integral_constant<int, 4>{});
      }
      part_sum[j0][row] = ss;
    }
  };

  // kTurned: load i of a batch brings piece (i * 64 + lane) % kPieces of row (i * 64 + lane) / kPieces;
  // in the wave's buffer piece p of row r lies at r * kPieces + (p ^ (r % 8)), which keeps both the
  // row-wise writes and the operand-wise reads (16 rows at one piece) off each other's banks.
  constexpr int kRowsPerLoad = kTurned ? 64 / kPieces : 1;
  const int turn_row = lane / kPieces, turn_piece = lane % kPieces;
  const bf16_t* turn_src = static_cast<const bf16_t*>(a.x) + static_cast<long>(turn_row) * k + turn_piece * 8;
  uint4* turn = reinterpret_cast<uint4*>(pool) + wave * (MT * ROWS * kPieces);
  constexpr int kXLoads = kTurned ? MT * U * ROWS / 16 : 1;      // a batch's loads of x, kRowsPerLoad rows each

  struct Batch {
    uint4 w[U];
    uint4 x[kNormed ? 1 : MT][kNormed ? 1 : U];
  };
  // A batch that lies whole inside the wave's part of k can be loaded without a condition anywhere (rows past m read
  // the last row: their results are never stored).  The compiler counts outstanding loads by instruction: where a load
  // may be skipped it cannot know how many were issued after the ones it waits for and waits for all of them, and a
  // copy from one set of registers to the other waits for the load it copies -- every batch then waits for the batch
  // asked for just before it.  With 32 rows a workgroup, whole batches are loaded so and multiplied from the
  // registers they were loaded into, two a turn (us, weights from memory, without and so: 64 rows as two workgroups of 32 2,048 x 5,480 15.5 and 14.3, behind
  // a norm 18.3 and 15.6; 32 rows 11,264 x 2,080 gated 19.7 and 16.4); with 16 rows the plain loop is the faster one, and with 48 and 64 rows a workgroup
  // the second set of registers does not fit the 128 a wave has (spilled, a product took three times as long).
  constexpr bool kPingPong = MT == 2;
  const int last_row_offset = (m - 1) * k;              // (m <= 64 rows: an int)
  int turn_offset[kXLoads];
  if constexpr (kTurned) {
#pragma unroll
    for (int i = 0; i < kXLoads; ++i) turn_offset[i] = min((turn_row + i * kRowsPerLoad) * k, last_row_offset) + turn_piece * 8;
  }
  const bf16_t* xptr_any[MT];                           // (the row itself, or the last row for rows past m)
#pragma unroll
  for (int t = 0; t < MT; ++t) xptr_any[t] = (kNormed || xrow_ok[t]) ? xptr[t] : static_cast<const bf16_t*>(a.x) + last_row_offset;
  auto load_whole = [&](Batch& b, int k0) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      b.w[u] = load16(wblock + static_cast<long>(k0 / 32 + u) * (kWave * 8) + wlane);
      if constexpr (!kNormed && !kTurned) {
#pragma unroll
        for (int t = 0; t < MT; ++t) b.x[t][u] = load16(xptr_any[t] + k0 + 32 * u + 8 * grp);
      }
    }
    if constexpr (kTurned) {
#pragma unroll
      for (int i = 0; i < kXLoads; ++i) b.x[i / U][i % U] = load16(static_cast<const bf16_t*>(a.x) + turn_offset[i] + k0);
    }
  };
  auto load = [&](Batch& b, int k0) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int kk = k0 + 32 * u + 8 * grp;
      const bool ok = kk < k_end;
      b.w[u] = k0 + 32 * u < k_end ? load16(wblock + static_cast<long>(k0 / 32 + u) * (kWave * 8) + wlane) : zero16();
      if constexpr (!kNormed && !kTurned) {
#pragma unroll
        for (int t = 0; t < MT; ++t) b.x[t][u] = (ok && xrow_ok[t]) ? load16(xptr[t] + kk) : zero16();
      }
    }
    if constexpr (kTurned) {
      const bool k_ok = k0 + turn_piece * 8 < k_end;
#pragma unroll
      for (int i = 0; i < kXLoads; ++i) {
        const bool ok = k_ok && turn_row + i * kRowsPerLoad < m;
        b.x[i / U][i % U] = ok ? load16(turn_src + static_cast<long>(i * kRowsPerLoad) * k + k0) : zero16();
      }
    }
  };
  auto compute = [&](const Batch& b, int k0) {
    if constexpr (kTurned) {
#pragma unroll
      for (int i = 0; i < kXLoads; ++i) {
        const int row = turn_row + i * kRowsPerLoad;
        turn[row * kPieces + (turn_piece ^ (row % 8))] = b.x[i / U][i % U];
      }
      // the wave's own lanes wrote what its lanes now read: LDS serves a wave's accesses in order
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
#pragma unroll
      for (int t = 0; t < MT; ++t) {
        uint4 xb;
        if constexpr (kNormed) {
          const int kk = k0 + 32 * u + 8 * grp;
          xb = kk < k_end ? *reinterpret_cast<const uint4*>(xptr[t] + kk) : zero16();
        } else if constexpr (kTurned) {
          xb = turn[(t * 16 + (ROWS == 8 ? col % 8 : col)) * kPieces + ((4 * u + grp) ^ (col % 8))];
        } else {
          xb = b.x[t][u];
        }
        acc[t] = mfma_16x16x32(b.w[u], xb, acc[t]);
      }
    }
    if constexpr (kTurned) {                             // read before the next batch is written
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
  };

  constexpr int kStep = 32 * U;
  Batch cur, nxt;

  if constexpr (kNormed) {
    // Stage bf16(x * g): wave w takes rows w, w + 8; a lane takes 8 elements of each 512.  The
    // loads of x and g are issued first and the first weights right after them: loads come back
    // in the order they were issued, so the (cached) x arrives while the weights are on their way.
    // (two pieces a round, 1,024 elements of a row; with a float scale one: two spilled, 8 rows 32,000 x 2,048 38.6 -> 32.9 us,
    // one row 31.8 -> 28.2, 8 rows 128,256 x 4,096 253 -> 221)
    constexpr int kStageIters = XMODE == kNormedG32 ? 1 : 2;
    bf16_t* stage = reinterpret_cast<bf16_t*>(stage_raw);
    bool first = true;
    for (int row = wave; row < a.m_stage; row += kWaves) {
      float ss = 0.f;
      const bool live = row < m;
      const long src = (live && a.rows) ? a.rows[row] : row;
      const float* xr = static_cast<const float*>(a.x) + src * k;
      for (int kb = 0; kb < k; kb += 512 * kStageIters) {
        uint4 x0[kStageIters], x1[kStageIters], g0[kStageIters], g1[kStageIters];
#pragma unroll
        for (int it = 0; it < kStageIters; ++it) {
          const int kk = kb + it * 512 + lane * 8;
          const bool ok = live && kk < k;
          x0[it] = ok ? load16(xr + kk) : zero16();
          x1[it] = ok ? load16(xr + kk + 4) : zero16();
          if constexpr (XMODE == kNormedG16) {
            g0[it] = ok ? load16(static_cast<const bf16_t*>(a.g) + kk) : zero16();
          } else {
            g0[it] = ok ? load16(static_cast<const float*>(a.g) + kk) : zero16();
            g1[it] = ok ? load16(static_cast<const float*>(a.g) + kk + 4) : zero16();
          }
        }
        if (first) {                                       // the first weights follow the first x
          if (k_begin < k_end) load(cur, k_begin);
          first = false;
        }
#pragma unroll
        for (int it = 0; it < kStageIters; ++it) {
          const int kk = kb + it * 512 + lane * 8;
          if (kk >= k) continue;
          const float xv[8] = {__uint_as_float(x0[it].x), __uint_as_float(x0[it].y), __uint_as_float(x0[it].z),
                               __uint_as_float(x0[it].w), __uint_as_float(x1[it].x), __uint_as_float(x1[it].y),
                               __uint_as_float(x1[it].z), __uint_as_float(x1[it].w)};
          float gv[8];
          if constexpr (XMODE == kNormedG16) {
            const uint32_t gr[4] = {g0[it].x, g0[it].y, g0[it].z, g0[it].w};
#pragma unroll
            for (int i = 0; i < 4; ++i) {
              gv[2 * i] = __uint_as_float(gr[i] << 16);
              gv[2 * i + 1] = __uint_as_float(gr[i] & 0xffff0000u);
            }
          } else {
            const uint32_t gr[8] = {g0[it].x, g0[it].y, g0[it].z, g0[it].w, g1[it].x, g1[it].y, g1[it].z, g1[it].w};
#pragma unroll
            for (int i = 0; i < 8; ++i) gv[i] = __uint_as_float(gr[i]);
          }
          ss = add_squares(xv, kb + it > 0, ss);
          *reinterpret_cast<uint4*>(stage + static_cast<long>(row) * stage_stride + kk) =
              make_uint4(pack2(xv[0] * gv[0], xv[1] * gv[1]), pack2(xv[2] * gv[2], xv[3] * gv[3]),
                         pack2(xv[4] * gv[4], xv[5] * gv[5]), pack2(xv[6] * gv[6], xv[7] * gv[7]));
        }
      }
      ss = wave_sum(ss);
      if (lane == 0 && row < 16) ssq_row[row] = ss;
    }
    if (first && k_begin < k_end) load(cur, k_begin);      // a wave without a row to stage
    lds_barrier();                                         // (the weights stay in flight)
  } else {
    if (k_begin < k_end) load(cur, k_begin);
    sum_parts();
  }

  int k0 = k_begin;
  while (kPingPong && k0 + 3 * kStep <= k_end) {
    load_whole(nxt, k0 + kStep);
    compute(cur, k0);
    load_whole(cur, k0 + 2 * kStep);
    compute(nxt, k0 + kStep);
    k0 += 2 * kStep;
  }
  for (; k0 < k_end; k0 += kStep) {
    const int next = k0 + kStep;
    if (kPingPong && next + kStep <= k_end) load_whole(nxt, next);
    else if (next < k_end) load(nxt, next);
    compute(cur, k0);
    if (next < k_end) cur = nxt;
  }

  if constexpr (kTurned) __syncthreads();               // the partial sums take the buffers' place
  // acc[t][r] is the partial sum for output column n0 + 4*grp + r and row t*16 + col
#pragma unroll
  for (int t = 0; t < MT; ++t)
#pragma unroll
    for (int r = 0; r < 4; ++r) red[wave][t][4 * grp + r][col] = acc[t][r];
  __syncthreads();

  constexpr int kItems = (MT * 16 * kCols + kThreads - 1) / kThreads;
#pragma unroll
  for (int j = 0; j < kItems; ++j) {
    const int idx = threadIdx.x + j * kThreads;
    const int nl = idx % kCols, row = idx / kCols;
    const int gn = n0 + nl;
    const bool live = idx < MT * 16 * kCols && row < m && gn < a.n;
    // (the adding epilogue goes on with every lane: its lanes may have sums of squares to exchange)
    if (EPI != kAccumF32 && !live) continue;
    float sum = 0.f, partner = 0.f;
    if (live) {
#pragma unroll
      for (int wv = 0; wv < kWaves; ++wv) sum += red[wv][row / 16][nl][row % 16];
      if constexpr (kPaired) {
#pragma unroll
        for (int wv = 0; wv < kWaves; ++wv) partner += red[wv][row / 16][nl + 8][row % 16];
      }
    }
    if (kNormed || prenormed) {
      float ssq = 0.f;
      if (live) {
        if (prenormed) {
#pragma unroll
          for (int j2 = 0; j2 < kPartSums; ++j2) ssq += part_sum[j2][row];
        } else {
          ssq = ssq_row[row];
        }
      }
      const float scale = live ? 1.0f / sqrtf(ssq / static_cast<float>(k) + a.eps) : 0.f;
      sum *= scale;
      partner *= scale;
    }
    put_output<EPI, kCols, HALF>(a, n0, wblock_index, half, row, nl, idx < MT * 16 * kCols, live, sum, partner,
                                 Kept{EPI == kAccumF32 ? prev[j] : 0.f, EPI == kAccumF32, 0.f, EPI == kRopeKvBf16 ? rope_cs[j] : 1.f, EPI == kRopeKvBf16 ? rope_sn[j] : 0.f,
                                      EPI == kRopeKvBf16 ? rope_slot[j] : 0, xielu_p, xielu_q});
  }
}

// ---- plain rows through private rings in LDS -----------------------------------------------------
// k a multiple of 64, operands on 16-byte boundaries: the forms above with x and the weights going from memory into LDS without passing
// registers (global_load_lds_dwordx4), in a ring of S stages that belongs to one wave -- so there is no barrier in the walk, only the wave's own
// waits, counted by hand, and what is in flight is what LDS holds (64 to 144 KB a CU) and not what registers are left for.  A stage is KS
// values of k: ROWS rows of x, 128 bytes each (64 with KS 32), the 16-byte pieces XOR-placed so that a fragment read meets no bank conflict, and
// the NB blocks of the weight as they lie in memory.  As soon as a stage's fragments are in registers it is asked for again, before they are multiplied.
// Waves, their parts of k, the MFMA and the order of the sums are those of the kernel above: the same bits.  Arithmetic in front of the first load
// counts: 24 waves a CU share four SIMDs, and with integer divisions there an 11,264 x 2,048 product of 8 rows took 0.4 us more.
//
// What bounds it: a launch and the first trip to memory, 3 to 3.5 us, then the memory's rate for the weights and, with 16 rows and more, what a
// CU pulls of x through its cache (105 to 120 bytes a ns from L2; with x turned through registers it was 65 of both together).  Weights
// from memory, us, kernel above and this: 8 rows 2,048 x 2,048 4.39 and 4.07, 2,048 x 5,632 7.74 and 6.81, 11,264 x 2,048 10.84 and 9.90, 28,672 x 4,096
// 41.4 and 39.3; 16 rows 2,048 x 5,632 9.18 and 7.66, 4,096 x 4,096 10.6 and 8.4, 4,096 x 11,008 26.1 and 19.0, 22,016 x 4,096 37.5 and 35.5; 32 rows
// 4,096 x 11,008 30.1 and 23.4; 64 rows 2,048 x 2,048 6.53 and 5.95, 4,096 x 4,096 14.9 and 12.5.  With weights past the caches (launch_ring) less again:
// one row 32,000 x 2,048 23.9 -> 21.7 (6 TB/s), 8 rows 11,264 x 2,048 10.6 -> 10.4, 28,672 x 4,096 39.5 -> 36.8, 16 rows 44.4 -> 40.1.
// With the norm fused (NORMED: x the float stream, up to eight rows) x and the norm's scale come into LDS once, ahead of the first weights; one wave
// takes a row's sum of squares, in the order of rmsnorm_prepare and of the kernel above, then every wave turns its part of k into bfloat16(x * g) in
// its place, and the rings hold weights only.  One row 2,560 x 2,048 6.23 and 5.36, 4,096 x 4,096 12.7 and 9.8, 11,264 x 2,048 11.6 and 11.2, 22,016 x 4,096
// 40.1 and 36.5; four rows 4,096 x 4,096 12.9 and 11.6.
template <int ROWS, int NB, int KS, int S, bool NORMED = false>
struct RingShape {
  static constexpr bool kHalf = NB == 0;                      // half a block: two workgroups share one
  static constexpr int kTiles = (ROWS + 15) / 16, kBlocks = kHalf ? 1 : NB;
  static constexpr int kXLoads = NORMED ? 0 : ROWS * KS / 512, kWLoads = kHalf ? KS / 64 : NB * KS / 32, kLoads = kXLoads + kWLoads;
  static constexpr int kStageBytes = kLoads * 1024, kRingBytes = kWaves * S * kStageBytes;
  static constexpr int kRedBytes = kWaves * kBlocks * kTiles * 16 * kRedPad * 4;
  static constexpr int kLdsBytes = kRingBytes > kRedBytes ? kRingBytes : kRedBytes;
  static_assert(kLdsBytes <= 152 * 1024 && S * kLoads < 64, "a workgroup's LDS beside what else it keeps there, and a wait's count");
  static_assert((KS == 64 && ROWS % 8 == 0) || (KS == 32 && ROWS % 16 == 0), "whole loads of x");
  static_assert(ROWS == 8 || ROWS % 16 == 0, "eight rows or whole tiles");
  static_assert(!NORMED || (ROWS == 8 && !kHalf && KS == 64), "the fused norm: eight rows, whole blocks");
};

// N loads of 1 KB to N KB of LDS side by side, load i from bases[i] (the same in every lane) + off[i]; past the caches or through them.
template <int N, bool PAST>
__device__ inline void ring_loads(const unsigned char* const* bases, const unsigned* off, unsigned lds_address) {
  // (the LDS address is set once, to the middle of the stretch: the offset field reaches 4 KB either way, and moves the memory address too)
  constexpr int kMid = N / 2;
  const void* b[N];
#pragma unroll
  for (int i = 0; i < N; ++i) {
    const uintptr_t bits = reinterpret_cast<uintptr_t>(bases[i]) - (i - kMid) * 1024;
    const unsigned lo = __builtin_amdgcn_readfirstlane(static_cast<unsigned>(bits)), hi = __builtin_amdgcn_readfirstlane(static_cast<unsigned>(bits >> 32));
    b[i] = reinterpret_cast<const void*>((static_cast<uintptr_t>(hi) << 32) | lo);
  }
  const unsigned mid = __builtin_amdgcn_readfirstlane(lds_address + kMid * 1024);
#define BC4G_LOAD(v, s, o, how) "global_load_lds_dwordx4 %" #v ", %" #s " offset:" #o how "\n\t"
#define BC4G_RING(loads, ...) asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\t" loads ::"s"(mid), __VA_ARGS__ : "memory", "m0")
#define BC4G_RINGS(how)                                                                                                                          \
  if constexpr (N == 1) BC4G_RING(BC4G_LOAD(1, 2, 0, how), "v"(off[0]), "s"(b[0]));                                                              \
  else if constexpr (N == 2)                                                                                                                     \
    BC4G_RING(BC4G_LOAD(1, 3, -1024, how) BC4G_LOAD(2, 4, 0, how), "v"(off[0]), "v"(off[1]), "s"(b[0]), "s"(b[1]));                              \
  else if constexpr (N == 3)                                                                                                                     \
    BC4G_RING(BC4G_LOAD(1, 4, -1024, how) BC4G_LOAD(2, 5, 0, how) BC4G_LOAD(3, 6, 1024, how), "v"(off[0]), "v"(off[1]), "v"(off[2]), "s"(b[0]),  \
              "s"(b[1]), "s"(b[2]));                                                                                                             \
  else {                                                                                                                                         \
    static_assert(N == 4, "loads a statement");                                                                                                  \
    BC4G_RING(BC4G_LOAD(1, 5, -2048, how) BC4G_LOAD(2, 6, -1024, how) BC4G_LOAD(3, 7, 0, how) BC4G_LOAD(4, 8, 1024, how), "v"(off[0]),           \
              "v"(off[1]), "v"(off[2]), "v"(off[3]), "s"(b[0]), "s"(b[1]), "s"(b[2]), "s"(b[3]));                                                \
  }
  if constexpr (PAST) {
    BC4G_RINGS(" nt")
  } else {
    BC4G_RINGS("")
  }
#undef BC4G_RINGS
#undef BC4G_RING
#undef BC4G_LOAD
}

// Lane i's 4 bytes to lds_address + 4 i.
__device__ inline void load_to_lds_4(const void* global, unsigned lds_address) {
  asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dword %0, off" ::"v"(global), "s"(lds_address) : "memory", "m0");
}

// Until all but the loads of the last `later` stages of LOADS (MOST such at most) have come; no access to LDS moves over it.
template <int LOADS, int MOST>
__device__ inline void ring_wait(int later) {
  if constexpr (MOST == 0) {
    asm volatile("" ::: "memory");
    wait_loads<0>();
    asm volatile("" ::: "memory");
  } else if (later >= MOST) {
    asm volatile("" ::: "memory");
    wait_loads<LOADS * MOST>();
    asm volatile("" ::: "memory");
  } else {
    ring_wait<LOADS, MOST - 1>(later);
  }
}

// (PAST: the weights past the caches.  Chosen while a step is asked for it cost 0.3 us a product.)
template <int EPI, int ROWS, int NB, int KS, int S, bool NORMED, bool PAST>
__global__ __launch_bounds__(kThreads, 2) void gemm_ring_kernel(const SkinnyArgs args) {
  typedef RingShape<ROWS, NB, KS, S, NORMED> P;
  constexpr bool kHalf = P::kHalf, kPaired = gated(EPI) || EPI == kRopeKvBf16;
  static_assert(!kHalf || (ROWS <= 16 && !kPaired), "half blocks: few rows, unpaired outputs");
  constexpr int TM = P::kTiles, TB = P::kBlocks, kSteps = KS / 32, kPartSums = 8;
  extern __shared__ __align__(128) unsigned char ring_lds[];
  __shared__ float part_sum[kPartSums][ROWS];                                // (normed modes: the rows' sums of squares)
  __shared__ int places[EPI == kRopeKvBf16 ? kWaves : 1][2][kWave];          // positions and cache slots, every wave's own
  const SkinnyArgs a = NORMED ? args : own_rows<EPI>(args);
  const int lane = threadIdx.x % kWave, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int col = lane % 16, grp = lane / 16;
  const int m = a.m, k = a.k;
  auto lds_address = [](const void* p) { return static_cast<unsigned>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) const unsigned char*)p)); };
  const int first_block = kHalf ? blockIdx.x / 2 : blockIdx.x * TB, half = kHalf ? blockIdx.x % 2 : 0;

  // Item j of a thread is output nl of block b and row `row` of number threadIdx.x + j * kThreads.  What it needs beside its sum is asked for before the
  // operands and used after the walk.  (Little arithmetic before the first operands: with 24 waves a CU every instruction of it is 40 clocks.)
  constexpr int kCols = kPaired || kHalf ? 8 : 16, kAll = TB * TM * 16 * kCols, kItems = (kAll + kThreads - 1) / kThreads;
  auto item = [&](int j, int& nl, int& b, int& row) {
    const int idx = threadIdx.x + j * kThreads;
    nl = idx % kCols, b = idx / kCols % TB, row = idx / (kCols * TB);
    return idx < kAll;
  };
  float prev[kItems], bias[kItems];
  typedef uint32_t uint32_any __attribute__((aligned(2)));
  uint32_t g[kItems];
  float cs[kItems], sn[kItems];
  int slot[kItems];
  if constexpr (EPI == kAccumF32) {
    // (every load is made, from a place that there is, whether it is needed or not: behind a branch the compiler waits for it)
#pragma unroll
    for (int j = 0; j < kItems; ++j) {
      int nl, b, row;
      item(j, nl, b, row);
      const unsigned gn = min((first_block + b) * 16 + 8 * half + nl, a.n - 1), at = min(row, m - 1) * a.n + gn;
      prev[j] = static_cast<const float*>(a.out)[at];
      bias[j] = (a.bias != nullptr ? a.bias : static_cast<const float*>(a.out))[gn];
      // (of a bfloat16 scale the column's and the one before it; the first column's and the one after)
      const unsigned char* scale = static_cast<const unsigned char*>(a.emit_g != nullptr ? a.emit_g : a.out);
      g[j] = *reinterpret_cast<const uint32_any*>(scale + (a.emit_g_f32 ? 4 * gn : 2 * max(gn, 1u) - 2));
    }
  }
  int src = lane;                             // normed modes: lane r's row of x
  if constexpr (NORMED) {
    if (a.rows != nullptr) src = a.rows[min(lane, m - 1)];
  }
  if constexpr (EPI == kRopeKvBf16) {
    if (a.rope.rotary_dim > 0) load_to_lds_4(a.rope.positions + min(lane, m - 1), lds_address(&places[wave][0][0]));
    if (a.rope.write_kv) load_to_lds_4(a.rope.slot_map + min(lane, m - 1), lds_address(&places[wave][1][0]));
  }

  // prenormed x: wave j adds up chain j of every row's parts, parts j, j + 8, ... in ascending order.  A part's numbers of ROWS rows (pairs of
  // them, where half blocks left it) lie side by side: four of them a lane, 2^shift lanes a part, up to 256 parts (128 pairs) asked for before the walk.
  // (Past the last part, or the last of its rows that the call names -- the parts may be those of more rows, and the call's their last --: the last four,
  // turned into place after the walk.)
  constexpr int kHeld = ROWS <= 8 ? 1 : ROWS / 8;
  typedef float floatx4_any __attribute__((ext_vector_type(4), aligned(4)));
  const bool prenormed = EPI != kAccumF32 && !NORMED && a.ssq_parts != nullptr, pairs = ROWS == 8 && a.ssq_halves;
  const int shift = ROWS == 8 ? 1 + a.ssq_halves : ROWS == 16 ? 2 : 3, parts_a_load = kWave >> shift;
  const int part_stride = a.part_stride;
  const int first_row = a.rows_per_block > 0 ? static_cast<int>(blockIdx.y) * a.rows_per_block : 0, last_four = a.last_four - first_row;
  auto part_at = [&](int h) {
    return min(wave + kPartSums * (h * parts_a_load + (lane >> shift)), a.ssq_blocks - 1) * part_stride + (lane & ((1 << shift) - 1)) * 4;
  };
  floatx4 held[kHeld];
  if constexpr (EPI != kAccumF32 && !NORMED) {
    const float* parts = prenormed ? a.ssq_parts : static_cast<const float*>(a.x);
#pragma unroll
    for (int h = 0; h < kHeld; ++h) held[h] = *reinterpret_cast<const floatx4_any*>(parts + static_cast<unsigned>(prenormed ? min(part_at(h), last_four) : 0));
  }

  // this wave's part of k, and where its lanes' bytes of a stage come from
  const int k_begin = wave * a.chunk, steps = max(0, min(k - k_begin, a.chunk)) / static_cast<unsigned>(KS);
  const unsigned char* mine = ring_lds + wave * (S * P::kStageBytes);
  const unsigned ring = static_cast<unsigned>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) const unsigned char*)mine));
  constexpr int kRowBytes = KS * 2, kPieces = KS / 8, kLoadRows = kWave / kPieces;
  auto key = [](int row) { return KS == 64 ? (row >> 1) & 7 : (row >> 2) & 3; };      // piece p of a row lies at p ^ key
  unsigned x_off[NORMED ? 1 : P::kXLoads], w_off[P::kWLoads];
#pragma unroll
  for (int i = 0; i < P::kXLoads; ++i) {
    const int row = i * kLoadRows + lane / kPieces;                                    // (rows past m: the last)
    x_off[i] = static_cast<unsigned>(min(row, m - 1)) * k * 2 + ((lane % kPieces) ^ key(row)) * 16;
  }
  // (half a block: its eight rows' 16 bytes of four k-slots side by side, 128 bytes each, of two k-steps a load)
#pragma unroll
  for (int i = 0; i < P::kWLoads; ++i) w_off[i] = kHalf ? lane / 32 * 1024 + lane % 32 / 8 * 256 + (8 * half + lane % 8) * 16 : lane * 16;
  const unsigned char* w_at[TB];
#pragma unroll
  for (int b = 0; b < TB; ++b)
    w_at[b] = reinterpret_cast<const unsigned char*>(a.w) +
              (static_cast<size_t>(min(first_block + b, a.last_block)) * (static_cast<unsigned>(k) / 32) + static_cast<unsigned>(k_begin) / 32) * 1024;
  const unsigned char* x_at = static_cast<const unsigned char*>(a.x) + static_cast<unsigned>(k_begin) * 2;
  auto ask = [&](int t) {
    const unsigned to = ring + (t % S) * P::kStageBytes;
    const unsigned char *xs[NORMED ? 1 : P::kXLoads], *ws[P::kWLoads];
#pragma unroll
    for (int i = 0; i < P::kWLoads; ++i)
      ws[i] = (kHalf ? w_at[0] + i * 2048 : w_at[i / kSteps] + i % kSteps * 1024) + static_cast<size_t>(t) * (kSteps * 1024);
#pragma unroll
    for (int i = 0; i < P::kXLoads; ++i) xs[i] = x_at + static_cast<size_t>(t) * kRowBytes;
    ring_loads<P::kWLoads, PAST>(ws, w_off, to);
    if constexpr (!NORMED) ring_loads<P::kXLoads, false>(xs, x_off, to + P::kWLoads * 1024);
  };

  // normed modes: x and g in pieces of 1 KB, piece p by wave p % 8 (lanes past the row's end: its last 16 bytes)
  unsigned char *rows_lds = ring_lds + P::kLdsBytes, *scale_lds = rows_lds + m * a.x_row_bytes;
  if constexpr (NORMED) {
    for (int at = wave * 1024; at < k * 4; at += kWaves * 1024) {
      const unsigned from = min(at + lane * 16, k * 4 - 16);
#pragma unroll
      for (int r = 0; r < 8; ++r)
        if (r < m)
          load_to_lds_16(static_cast<const unsigned char*>(a.x) + static_cast<size_t>(__builtin_amdgcn_readlane(src, r)) * (static_cast<unsigned>(k) * 4), from,
                         lds_address(rows_lds + r * a.x_row_bytes + at));
    }
    const int g_bytes = a.g_f32 ? 4 * k : 2 * k;
    for (int at = wave * 1024; at < g_bytes; at += kWaves * 1024)
      load_to_lds_16(a.g, static_cast<unsigned>(min(at + lane * 16, g_bytes - 16)), lds_address(scale_lds + at));
  }
#pragma unroll
  for (int s = 0; s < S; ++s)
    if (s < steps) ask(s);

  floatx4 acc[TM][TB];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int b = 0; b < TB; ++b) acc[i][b] = floatx4{0.f, 0.f, 0.f, 0.f};
  // (while the operands are on their way)
  float xielu_p = 0.f, xielu_q = 0.f;
  if constexpr (EPI == kXieluBf16) xielu_p = softplus_f(a.bias[0]), xielu_q = 0.5f + softplus_f(a.bias[1]);
  if constexpr (EPI == kRopeKvBf16) {
    ring_wait<P::kLoads, S>(min(S, steps));
#pragma unroll
    for (int j = 0; j < kItems; ++j) {
      int nl, b, row;
      const bool in_block = item(j, nl, b, row);
      const int n0 = (first_block + b) * 16, head = n0 / a.rope.head_dim;
      const bool live = in_block && row < m && n0 < a.n;
      cs[j] = 1.f, sn[j] = 0.f;
      if (live && a.rope.rotary_dim > 0 && head < a.rope.n_heads + a.rope.n_kv_heads) pair_angle(a.rope, n0, nl, places[wave][0][row], cs[j], sn[j]);
      slot[j] = live && head >= a.rope.n_heads && a.rope.write_kv ? places[wave][1][row] : 0;
    }
  }

  if constexpr (NORMED) {
    ring_wait<P::kLoads, S>(min(S, steps));
    lds_barrier();                              // (the weights stay in flight)
    if (wave < m) {
      // row `wave`: lane l takes elements 8 l .. 8 l + 7 of every 512
      float ss = 0.f;
      for (int kk = lane * 8; kk < k; kk += 512) {
        const float* p = reinterpret_cast<const float*>(rows_lds + wave * a.x_row_bytes) + kk;
        const floatx4 v0 = *reinterpret_cast<const floatx4*>(p), v1 = *reinterpret_cast<const floatx4*>(p + 4);
        const float v[8] = {v0[0], v0[1], v0[2], v0[3], v1[0], v1[1], v1[2], v1[3]};
        ss = add_squares(v, kk >= 512, ss);
      }
      ss = wave_sum(ss);
      if (lane == 0) part_sum[0][wave] = ss;
    }
    lds_barrier();
    // bfloat16(x * g) to the beginning of this wave's part: four numbers a lane, a piece of four rows read before anything is written over it
    for (int at = lane * 16; at < steps * KS * 4; at += 1024) {
      floatx4 scale;
      if (a.g_f32) {
        scale = *reinterpret_cast<const floatx4*>(scale_lds + k_begin * 4 + at);
      } else {
        const uint2 raw = *reinterpret_cast<const uint2*>(scale_lds + k_begin * 2 + at / 2);
        scale = floatx4{__uint_as_float(raw.x << 16), __uint_as_float(raw.x & 0xffff0000u), __uint_as_float(raw.y << 16), __uint_as_float(raw.y & 0xffff0000u)};
      }
      for (int r0 = 0; r0 < m; r0 += 4) {
        floatx4 v[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) v[r] = *reinterpret_cast<const floatx4*>(rows_lds + min(r0 + r, m - 1) * a.x_row_bytes + k_begin * 4 + at);
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int row = min(r0 + r, m - 1);
          *reinterpret_cast<uint2*>(rows_lds + row * a.x_row_bytes + k_begin * 4 + (at / 2 ^ row * 16)) =
              make_uint2(pack_bf16x2(v[r][0] * scale[0], v[r][1] * scale[1]), pack_bf16x2(v[r][2] * scale[2], v[r][3] * scale[3]));
        }
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
  }

  auto wait_lds_reads = []() { __builtin_amdgcn_s_waitcnt(63 >> 4 << 14 | 0 << 8 | 7 << 4 | 15); };      // lgkmcnt(0)
  const int read_row = ROWS == 8 ? col % 8 : col;
  const unsigned char* normed_row = rows_lds + min(read_row, m - 1) * a.x_row_bytes + k_begin * 4;
  const int normed_key = grp * 16 ^ min(read_row, m - 1) * 16;
  for (int t = 0; t < steps; ++t) {
    ring_wait<P::kLoads, S - 1>(min(steps - 1 - t, S - 1));
    __builtin_amdgcn_sched_barrier(0);
    const unsigned char* stage = mine + (t % S) * P::kStageBytes;
    uint4 fx[kSteps][TM], fw[kSteps][TB];
#pragma unroll
    for (int u = 0; u < kSteps; ++u) {
#pragma unroll
      for (int b = 0; b < TB; ++b) fw[u][b] = load16(kHalf ? stage + u * 512 + grp * 128 + col % 8 * 16 : stage + (b * kSteps + u) * 1024 + lane * 16);
#pragma unroll
      for (int i = 0; i < TM; ++i)
        fx[u][i] = NORMED ? load16(normed_row + ((t * 128 + u * 64) ^ normed_key))
                          : load16(stage + P::kWLoads * 1024 + (i * 16 + read_row) * kRowBytes + ((u * 4 + grp) ^ key(read_row)) * 16);
    }
    __builtin_amdgcn_sched_barrier(0);
    wait_lds_reads();                         // in registers: the stage may be written over
    __builtin_amdgcn_sched_barrier(0);
    if (t + S < steps) ask(t + S);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < kSteps; ++u)
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int b = 0; b < TB; ++b) acc[i][b] = mfma_16x16x32(fw[u][b], fx[u][i], acc[i][b]);
    __builtin_amdgcn_sched_barrier(0);
  }

  if (prenormed) {
    // through the wave's own ring, which is free; a part that is not there adds 0
    unsigned char* own = ring_lds + wave * (S * P::kStageBytes);
#pragma unroll
    for (int h = 0; h < kHeld; ++h) {
      floatx4 v = held[h];
      if (m < ROWS) {                                                                     // (only then a load of the last parts may end past them)
        const int turn = max(0, part_at(h) - last_four);
        if (turn & 1) v = floatx4{v[1], v[2], v[3], v[3]};
        if (turn & 2) v = floatx4{v[2], v[3], v[3], v[3]};
      }
      if (wave + kPartSums * (h * parts_a_load + (lane >> shift)) >= a.ssq_blocks) v = floatx4{0.f, 0.f, 0.f, 0.f};
      *reinterpret_cast<floatx4*>(own + (h * kWave + lane) * 16) = v;
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    const int row = lane % ROWS, in_chain = (a.ssq_blocks - wave + kPartSums - 1) / kPartSums;
    float ss = 0.f;
    if (pairs) {
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const float2 one = *reinterpret_cast<const float2*>(own + (i * ROWS + row) * 8);
        ss += one.x + one.y;
      }
    } else {
#pragma unroll
      for (int i = 0; i < 16; ++i) ss += *reinterpret_cast<const float*>(own + (i * ROWS + row) * 4);
      if (in_chain > 16) {
#pragma unroll
        for (int i = 16; i < 32; ++i) ss += *reinterpret_cast<const float*>(own + (i * ROWS + row) * 4);
      }
    }
    // Of more than 256 parts (128 pairs; rows of more than 4,096) the others, eight a chain asked for together: one after the other each was a trip of its own
    // behind the walk.  us, weights from memory, the streaming kernel, so and together: 2,048 x 14,336, 12 rows 22.9, 32.3 and 19.5; 4,096 x 14,336, 48 rows 44.7,
    // 50.4 and 37.2; 10,240 x 8,192 gated, 8 rows 36.0, 38.1 and 31.6.  (Sixteen together take the registers of the third workgroup of a CU.)
    constexpr int kTogether = 8;
    for (int i0 = pairs ? 16 : 32; i0 < in_chain; i0 += kTogether) {
      float one[kTogether], other[kTogether];
#pragma unroll
      for (int i = 0; i < kTogether; ++i) {
        const float* p = a.ssq_parts + static_cast<long>(wave + kPartSums * min(i0 + i, in_chain - 1)) * part_stride + (pairs ? 2 : 1) * min(row, m - 1);
        one[i] = p[0], other[i] = p[pairs ? 1 : 0];
      }
#pragma unroll
      for (int i = 0; i < kTogether; ++i) ss += i0 + i < in_chain ? (pairs ? one[i] + other[i] : one[i]) : 0.f;
    }
    if (lane < ROWS) part_sum[wave][row] = ss;
  }
  __syncthreads();                            // the partial sums take the rings' place
  typedef float Red[TB][TM][16][kRedPad];
  Red* red = reinterpret_cast<Red*>(ring_lds);
#pragma unroll
  for (int b = 0; b < TB; ++b)
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) red[wave][b][i][4 * grp + r][col] = acc[i][b][r];
  __syncthreads();

#pragma unroll
  for (int j = 0; j < kItems; ++j) {
    int nl, b, row;
    const bool in_block = item(j, nl, b, row);
    const int n0 = (first_block + b) * 16 + 8 * half;
    const bool live = in_block && row < m && n0 + nl < a.n;
    if (EPI != kAccumF32 && !live) continue;            // (the adding epilogue goes on with every lane)
    float sum = 0.f, partner = 0.f;
    if (live) {
#pragma unroll
      for (int v = 0; v < kWaves; ++v) sum += red[v][b][row / 16][nl][row % 16];
      if constexpr (kPaired) {
#pragma unroll
        for (int v = 0; v < kWaves; ++v) partner += red[v][b][row / 16][nl + 8][row % 16];
      }
      if (NORMED || prenormed) {
        float ssq = NORMED ? part_sum[0][row] : 0.f;
        if constexpr (!NORMED) {
#pragma unroll
          for (int c = 0; c < kPartSums; ++c) ssq += part_sum[c][row];
        }
        const float scale = 1.0f / sqrtf(ssq / static_cast<float>(k) + a.eps);
        sum *= scale;
        partner *= scale;
      }
    }
    Kept kept{0.f, false, 0.f, 1.f, 0.f, 0, xielu_p, xielu_q};
    if constexpr (EPI == kAccumF32) {
      asm volatile("" : "+v"(prev[j]), "+v"(bias[j]), "+v"(g[j]));            // (nothing done with them before the walk, where it would wait for them)
      kept.prev = a.bias != nullptr ? prev[j] + bias[j] : prev[j];
      kept.g = __uint_as_float(a.emit_g_f32 ? g[j] : n0 + nl > 0 ? g[j] & 0xffff0000u : g[j] << 16);
    }
    if constexpr (EPI == kRopeKvBf16) kept.cs = cs[j], kept.sn = sn[j], kept.slot = slot[j];
    put_output<EPI, kCols, kHalf>(a, n0, first_block + b, half, row, nl, in_block, live, sum, partner, kept);
  }
}

// LDS of a float row, in whole loads, and of all that the normed modes keep beside the rings
int ring_row_bytes(int k) { return (k * 4 + 1023) / 1024 * 1024; }
int ring_norm_bytes(int m, int k, bool g_f32) { return m * ring_row_bytes(k) + (g_f32 ? ring_row_bytes(k) : (k * 2 + 1023) / 1024 * 1024); }
constexpr int kRingNormBytes = 80 * 1024;     // of those at most

template <int EPI, int ROWS, int NB, int KS, int S, bool NORMED, bool PAST>
int launch_ring_form(const SkinnyArgs& a, int row_groups, hipStream_t s) {
  typedef RingShape<ROWS, NB, KS, S, NORMED> P;
  auto kernel = gemm_ring_kernel<EPI, ROWS, NB, KS, S, NORMED, PAST>;
  static std::atomic<bool> raised{false};
  if (!raised) {
    if (hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, P::kLdsBytes + (NORMED ? kRingNormBytes : 0)) !=
        hipSuccess)
      return fail("gemm_skinny: cannot raise the dynamic LDS limit");
    raised = true;
  }
  const int blocks = (a.n + 15) / 16;
  const dim3 grid(P::kHalf ? 2 * blocks : (blocks + NB - 1) / NB, row_groups);
  SkinnyArgs b = a;
  b.rows_per_block = row_groups > 1 ? (a.m + row_groups - 1) / row_groups : 0;
  b.chunk = (a.k + kWaves * 64 - 1) / (kWaves * 64) * 64;
  b.last_block = blocks - 1;
  b.part_stride = a.ssq_stride * (a.ssq_halves ? 2 : 1);
  b.last_four = (a.ssq_blocks - 1) * b.part_stride + a.m * (a.ssq_halves ? 2 : 1) - 4;
  b.x_row_bytes = NORMED ? ring_row_bytes(a.k) : 0;
  kernel<<<grid, dim3(kThreads), P::kLdsBytes + (NORMED ? ring_norm_bytes(a.m, a.k, a.g_f32) : 0), s>>>(b);
  return check_launch("gemm_skinny");
}

// Past the caches where one group of rows reads the weight: another would find it gone (64 rows 2,048 x 5,632, two groups: in a step 2 % slower).
template <int EPI, int ROWS, int NB, int KS, int S, bool NORMED = false>
int launch_ring(const SkinnyArgs& a, int row_groups, hipStream_t s) {
  return row_groups == 1 && passes_by(a.n, a.k, 2) ? launch_ring_form<EPI, ROWS, NB, KS, S, NORMED, true>(a, row_groups, s)
                                                   : launch_ring_form<EPI, ROWS, NB, KS, S, NORMED, false>(a, row_groups, s);
}

constexpr int kSplitMinRows = 8;

// Which rows a workgroup takes, how many blocks of outputs, and how deep its rings are: by what was measured for 1 to 64 rows, outputs of 2,048 to 28,672
// and k of 2,048 to 11,008 (us, weights from memory).  With at most a workgroup a CU the rings fill LDS; with more of them, two or three share a CU
// (11,264 x 2,048, 8 rows: rings of two stages 9.90, of four 11.7; 28,672 x 4,096: of three 39.3, of four 41.9).  More than eight rows go to two
// workgroups where the blocks are at most half the CUs: each pulls half of x, and the weight comes once more from L2 (16 rows 2,048 x 5,632
// 7.7 and 9.2; but 2,560 x 2,048 5.3 and 5.0).  Wider outputs of 16 rows and more take two or three blocks a workgroup, which so reads x once for all of them
// (32 rows 11,264 x 2,048: three blocks 12.6, one 13.9; 64 rows 4,096 x 11,008: two 28.5, one 35.6 and above).
template <int EPI>
int launch_rings(const SkinnyArgs& a, hipStream_t s) {
  const int blocks = (a.n + 15) / 16, cus = compute_units();
  if (a.m <= kSplitMinRows) {
    if constexpr (EPI == kAccumF32 || EPI == kStoreF32 || EPI == kStoreBf16)
      if (a.halves) return launch_ring<EPI, 8, 0, 64, 4>(a, 1, s);
    if (blocks <= cus) return launch_ring<EPI, 8, 1, 64, 4>(a, 1, s);
    return a.k < 4096 ? launch_ring<EPI, 8, 1, 64, 2>(a, 1, s) : launch_ring<EPI, 8, 1, 64, 3>(a, 1, s);
  }
  if (a.m <= 16) {
    if (2 * blocks <= cus) return launch_ring<EPI, 8, 1, 64, 4>(a, 2, s);
    if (blocks <= cus) return launch_ring<EPI, 16, 1, 64, 4>(a, 1, s);
    return 2 * blocks <= 3 * cus ? launch_ring<EPI, 16, 2, 64, 3>(a, 1, s) : launch_ring<EPI, 16, 1, 64, 2>(a, 1, s);
  }
  if (a.m <= 32) {
    if (2 * blocks <= cus) return launch_ring<EPI, 16, 1, 64, 4>(a, 2, s);
    if (blocks <= cus) return launch_ring<EPI, 32, 1, 64, 3>(a, 1, s);
    return blocks <= 2 * cus ? launch_ring<EPI, 32, 2, 64, 2>(a, 1, s) : launch_ring<EPI, 32, 3, 32, 2>(a, 1, s);
  }
  if (2 * blocks <= cus) return launch_ring<EPI, 32, 1, 64, 3>(a, 2, s);
  return blocks <= cus ? launch_ring<EPI, 32, 2, 64, 2>(a, 2, s) : launch_ring<EPI, 32, 3, 32, 2>(a, 2, s);
}

// The same with the norm fused.
template <int EPI>
int launch_normed_rings(const SkinnyArgs& a, hipStream_t s) {
  if ((a.n + 15) / 16 <= compute_units()) return launch_ring<EPI, 8, 1, 64, 4, true>(a, 1, s);
  return a.k < 4096 ? launch_ring<EPI, 8, 1, 64, 2, true>(a, 1, s) : launch_ring<EPI, 8, 1, 64, 3, true>(a, 1, s);
}

// Up to eight rows that fit LDS beside the rings, and for wide outputs beside those of two other workgroups of the CU (one from k = 4,096 on): with
// fewer of them there the kernel above is faster (four rows 11,264 x 2,048 12.5 and 13.1).  Below k = 2,048 too, where fewer waves than eight fetch all of x
// (2,048 x 1,024: one row 4.33 and 4.53, eight 4.91 and 5.71; 2,048 x 2,048: 6.17 and 5.26, 6.82 and 6.74).
bool normed_ring_operands(const SkinnyArgs& a) {
  const int most = (a.n + 15) / 16 <= compute_units() ? kRingNormBytes : a.k < 4096 ? 20 * 1024 : 28 * 1024;
  return a.k % 64 == 0 && a.k >= 2048 && a.m <= 8 && ring_norm_bytes(a.m, a.k, a.g_f32) <= most &&
         reinterpret_cast<uintptr_t>(a.x) % 16 == 0 && reinterpret_cast<uintptr_t>(a.g) % 16 == 0 && reinterpret_cast<uintptr_t>(a.w) % 16 == 0;
}

// What the rings take: the loads bring 16 bytes from 16-byte boundaries, a stage is 64 values of k, parts of a norm are read four numbers at a time and the
// next norm's scale two.
bool ring_operands(const SkinnyArgs& a) {
  return a.k % 64 == 0 && (a.ssq_parts == nullptr || (a.ssq_blocks - 1L) * a.ssq_stride + a.m >= 4) && (a.emit_g == nullptr || a.n > 1) &&
         reinterpret_cast<uintptr_t>(a.x) % 16 == 0 && reinterpret_cast<uintptr_t>(a.w) % 16 == 0;
}

// Which of those the streaming kernel takes all the same, because it is the faster one for them (the same bits from either).  us, weights from memory,
// streaming kernel and rings:
// - more than 32 rows and more than one and a half blocks a CU (beyond two the tiled kernel takes the product): the rings' two groups of rows are then
//   more workgroups than run at once.  48 rows 8,000 x 1,024 8.0 and 10.7, 7,168 x 4,096 21.9 and 26.7, 64 rows 25.7 and 28.3; but 6,144 x 4,096 25.4 and 17.8.
// - wide outputs of a short k: a workgroup's walk is one or two stages, and its rings only make a launch of many workgroups longer.  Up to 8 rows, from three
//   blocks a CU on: k up to 512, but for a gated product behind a prepared norm, and plain stores up to 768 (128,256 x 512 behind a norm, one row 22.9 and 29.7,
//   gated 30.6 and 30.3; 32,000 x 512 8 rows 8.4 and 10.0; 32,000 x 768 stored, one row 10.1 and 10.3, behind a norm 13.2 and 11.8; 12,288 x 512 4.76 and 4.75).
//   Four blocks a CU behind a norm also at 1,024: 8 rows 8.2 and 8.8.  9 to 16 rows, from two blocks a CU on: k up to 512 (128,256 x 512 26.1 and 37.8, 12,288 x 512
//   behind a norm 5.1 and 6.3; but 8,192 x 512 4.7 and 4.4), up to 1,024 what neither adds nor rotates nor finishes a norm before gates (32,000 x 768 stored 11.7 and
//   13.6, rotated 17.7 and 16.1, gated behind a norm 15.5 and 15.1; 32,000 x 1,152 16.0 and 16.3).
// - small weights of a k that gives a wave two stages: one trip and a second through LDS.  k from 576 to 1,024 and up to 640 numbers of k times blocks a CU, up to 32
//   rows (9 to 16 where the rows are shared out), what neither adds nor rotates (one row 768 x 768 2.44 and 2.67, 2,304 x 768 2.98 and 3.13, behind a norm
//   3.31 and 3.53, 24 rows 4.17 and 4.62; but rotated 4.78 and 4.34, added 3.65 and 3.56; 3,072 x 1,024 3.50 and 3.30, 4,096 x 768 3.45 and 3.28).
// - a norm to finish for more than 16 rows of k up to 512: more parts of sums of squares than operands (24 rows 4,096 x 256 3.35 and 3.70, 48 rows 512 x 512 3.45 and
//   3.65; rotated 4.52 and 4.48).
bool rings_are_slower(int epilogue, int m, int n, int k, bool finishes_norm) {
  const int blocks = (n + 15) / 16, cus = compute_units();
  if (m > 32 && 2 * blocks > 3 * cus) return true;
  const bool adds = epilogue == kAccumF32, rotates = epilogue == kRopeKvBf16, gates_normed = gated(epilogue) && finishes_norm;
  const bool plain = !adds && !rotates, shared_out = m <= kSplitMinRows || m > 16 || 2 * blocks <= cus;
  if (plain && m <= 32 && shared_out && k > 512 && k <= 1024 && static_cast<long>(blocks) * k <= 640L * cus) return true;
  if (finishes_norm && !rotates && m > 16 && k <= 512) return true;
  if (m > kSplitMinRows && m <= 16 && blocks > 2 * cus) return k <= 512 || (k <= 1024 && !adds && !rotates && !gates_normed);
  if (m <= kSplitMinRows && blocks > 3 * cus) {
    if (k <= 512) return !gates_normed;
    if (adds || rotates || gated(epilogue)) return false;
    return finishes_norm ? k > 768 && k <= 1024 && blocks <= 4 * cus : k <= 768;
  }
  return false;
}

constexpr int kMaxStageBytes = 96 * 1024;

template <int EPI, int XMODE>
int launch(const SkinnyArgs& a, hipStream_t s) {
  const int mt = (a.m + 15) / 16;
  dim3 grid((a.n + 15) / 16), block(kThreads);
  if constexpr (XMODE != kPlain) {
    if (mt != 1) return fail("gemm_skinny: the fused norm takes at most 16 rows, got %d", a.m);
    const size_t stage = static_cast<size_t>(a.m_stage) * (a.k + kStagePad) * 2;
    if (stage > kMaxStageBytes) return fail("gemm_skinny: %d rows of k=%d do not fit the staging buffer", a.m, a.k);
    if (normed_ring_operands(a)) return launch_normed_rings<EPI>(a, s);
    auto kernel = gemm_skinny_kernel<1, EPI, XMODE, 4>;
    static std::atomic<bool> raised{false};   // per instantiation: allow more than the default dynamic LDS
    if (!raised) {
      if (hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                              kMaxStageBytes) != hipSuccess)
        return fail("gemm_skinny: cannot raise the dynamic LDS limit");
      raised = true;
    }
    kernel<<<grid, block, stage, s>>>(a);
  } else {
    if (ring_operands(a) && !rings_are_slower(EPI, a.m, a.n, a.k, a.ssq_parts != nullptr)) return launch_rings<EPI>(a, s);
    // Every workgroup reads all its rows of x, and what a CU can pull through its cache is what bounds
    // the kernel once x is as large as the block's weights (16 rows).  Where the weight blocks are
    // few (up to one a CU: n = 4,096), two workgroups share a block's rows: each pulls half of
    // x, and the block's weights are read twice, once of it from L2 (us, weights from memory, one and two: 2,048 x 5,480 16 rows 10.8 and 9.6, 32 rows 15.2 and
    // 10.6, 64 rows 22.5 and 14.3; 32 rows 2,048 x 1,024 4.8 and 3.7; not at 16 rows of wider ones, 2,720 x 1,376 4.9 and 5.5).
    SkinnyArgs b = a;
    int tiles = mt;
    if (a.m > kSplitMinRows && static_cast<int>(grid.x) <= compute_units()) {
      b.rows_per_block = (a.m + 1) / 2;
      tiles = (b.rows_per_block + 15) / 16;
      grid.y = 2;
    }
    if (a.m <= kSplitMinRows) {
      // Few rows.  What bounds a weight of few blocks (2,048 x 5,480: 128 of 175 KB) is how many of its bytes are on their way
      // at once, so with at most three blocks for every four CUs a wave asks for eight k-steps together (two workgroups of
      // four would not share a CU anyway), and with at most a block for every other CU and a long k two workgroups
      // share a block, each with eight of its outputs (b.halves; the lanes of the other eight rows repeat
      // theirs, the same sums in the same order).  us, weights from memory, four k-steps and eight: 2,048 x 5,480 one row 8.8 and 7.5, 8 rows 9.0 and 8.3, 2,720 x 1,376
      // behind a norm, one row 5.1 and 4.7; whole blocks and halves: 2,048 x 5,480 one row 7.8 and 7.5, 8 rows 9.2 and 8.3, 1,024 x 5,480 8.0 and 6.9.
      // (A wide product's many workgroups, more than two a CU: with fewer k-steps in flight each they
      // need half the registers, and all of them are on the CUs at once.  Four k-steps and two: 8 rows 11,264 x 2,080 behind a norm, gated, 15.5 and 11.9, one row
      // 32,000 x 512 9.4 and 7.3.)
      const int blocks = static_cast<int>(grid.x);
      // A last batch of eight that four would hold -- every k up to 1,024, where it is the only one, and 2,049 to 3,072 -- adds
      // nothing but work for zeros: four there (8 rows: 1,024 x 1,024 3.84 us with eight, 3.34 with four).
      const int last = (a.k + kWaves * 64 - 1) / (kWaves * 64) * 2 % 8;
      const bool eights = last == 0 || last > 4;
      if constexpr (EPI == kAccumF32 || EPI == kStoreF32 || EPI == kStoreBf16) {
        if (b.halves) {
          grid.x *= 2;
          if (eights) gemm_skinny_kernel<1, EPI, XMODE, 8, 8, true><<<grid, block, 0, s>>>(b);
          else gemm_skinny_kernel<1, EPI, XMODE, 4, 8, true><<<grid, block, 0, s>>>(b);
          return check_launch("gemm_skinny");
        }
      }
      if (blocks > 2 * compute_units()) gemm_skinny_kernel<1, EPI, XMODE, 2, 8><<<grid, block, 0, s>>>(b);
      else if (eights && 4 * blocks <= 3 * compute_units()) gemm_skinny_kernel<1, EPI, XMODE, 8, 8><<<grid, block, 0, s>>>(b);
      else gemm_skinny_kernel<1, EPI, XMODE, 4, 8><<<grid, block, 0, s>>>(b);
      return check_launch("gemm_skinny");
    }
    switch (tiles) {
      // k-steps per batch chosen so that two batches of operands fit 128 registers (two workgroups a CU)
      case 1:
        // (a wide product's many workgroups: as above; 16 rows 32,000 x 512 behind a norm 12.1 and 9.0)
        if (static_cast<int>(grid.x) > 2 * compute_units()) gemm_skinny_kernel<1, EPI, XMODE, 2><<<grid, block, 0, s>>>(b);
        else gemm_skinny_kernel<1, EPI, XMODE, 4><<<grid, block, 0, s>>>(b);
        break;
      case 2: gemm_skinny_kernel<2, EPI, XMODE, 2><<<grid, block, 0, s>>>(b); break;
      case 3: gemm_skinny_kernel<3, EPI, XMODE, 2><<<grid, block, 0, s>>>(b); break;
      case 4: gemm_skinny_kernel<4, EPI, XMODE, 2><<<grid, block, 0, s>>>(b); break;
      default: return fail("gemm_skinny: M=%d is beyond 64 rows", a.m);
    }
  }
  return check_launch("gemm_skinny");
}

template <int XMODE>
int launch_epilogue(SkinnyArgs& a, int epilogue, hipStream_t s) {
  switch (epilogue) {
    case kStoreBf16: return launch<kStoreBf16, XMODE>(a, s);
    case kStoreF32: return launch<kStoreF32, XMODE>(a, s);
    case kSquaredReluBf16: return launch<kSquaredReluBf16, XMODE>(a, s);
    case kAccumF32:
      if constexpr (XMODE == kPlain) return launch<kAccumF32, XMODE>(a, s);
      else return fail("gemm_skinny: adding into the stream that is being normed is not supported");
    case kSwigluBf16: return launch<kSwigluBf16, XMODE>(a, s);
    case kGegluBf16: return launch<kGegluBf16, XMODE>(a, s);
    case kRopeKvBf16: return launch<kRopeKvBf16, XMODE>(a, s);
    default: return fail("gemm_skinny: unknown epilogue %d", epilogue);
  }
}

int check_common(const char* what, int m, int max_m, int n, int k, int epilogue) {
  BC4G_REQUIRE(m >= 0 && m <= max_m, "%s: M=%d must be at most %d", what, m, max_m);
  BC4G_REQUIRE(n > 0 && k > 0 && k % 8 == 0, "%s: K=%d must be a positive multiple of 8 (N=%d)", what, k, n);
  BC4G_REQUIRE(!gated(epilogue) || n % 16 == 0,
               "%s: a gated product needs blocks of eight gate and eight up rows, N=%d is no multiple of 16", what, n);
  return 0;
}

int check_rope(const char* what, const RopeKvArgs& r, int n) {
  BC4G_REQUIRE(r.n_heads > 0 && r.n_kv_heads > 0 && r.head_dim > 0 && r.head_dim % 16 == 0,
               "%s: bad head sizes %d/%d x %d (head_dim must be a multiple of 16)", what, r.n_heads, r.n_kv_heads,
               r.head_dim);
  BC4G_REQUIRE(n == (r.n_heads + 2 * r.n_kv_heads) * r.head_dim, "%s: N=%d is not (heads + 2 kv heads) * head_dim", what, n);
  BC4G_REQUIRE(r.rotary_dim == 0 || (r.rotary_dim == r.head_dim && r.positions && r.theta > 0.f),
               "%s: the rotation must cover the whole head (rotary_dim %d, head_dim %d)", what, r.rotary_dim, r.head_dim);
  BC4G_REQUIRE(!r.write_kv || (r.slot_map && r.k_cache && r.v_cache && r.page_tokens > 0),
               "%s: cache write asked for without a cache", what);
  return 0;
}

}  // namespace
}  // namespace bc4g

using namespace bc4g;

namespace bc4g {
namespace {
SkinnyArgs plain_args(const void* x, const void* w, void* out, int m, int n, int k) {
  SkinnyArgs a{};
  a.x = x;
  a.w = static_cast<const bf16_t*>(w);
  a.out = out;
  a.m = m;
  a.n = n;
  a.k = k;
  return a;
}

int check_parts(const char* what, const float* ssq_parts, int ssq_blocks, int ssq_stride, int ssq_halves, int m, float eps) {
  BC4G_REQUIRE(ssq_parts != nullptr && ssq_blocks > 0 && ssq_stride >= m, "%s: the sums of squares need %d parts of at least %d rows",
               what, ssq_blocks, m);
  // (where more rows are shared out over workgroups, a row's parts are counted in single numbers)
  BC4G_REQUIRE(!ssq_halves || m <= kSplitMinRows, "%s: half blocks leave parts of at most %d rows, not of %d", what, kSplitMinRows, m);
  BC4G_REQUIRE(eps >= 0.f, "%s: eps must not be negative", what);
  return 0;
}
}  // namespace
}  // namespace bc4g

extern "C" int bc4g_gemm_skinny(const void* x, const void* w, void* out, const float* bias, int epilogue, int m, int n, int k,
                                int halves, void* stream) {
  if (int e = check_common("gemm_skinny", m, 64, n, k, epilogue)) return e;
  BC4G_REQUIRE(epilogue != kRopeKvBf16, "gemm_skinny: use bc4g_gemm_skinny_qkv for the rotary epilogue");
  BC4G_REQUIRE(!bias || epilogue == kAccumF32, "gemm_skinny: only the adding epilogue takes a bias");
  BC4G_REQUIRE(!halves || (m <= kSplitMinRows && epilogue <= kAccumF32), "gemm_skinny: half blocks take at most %d rows and epilogues 0 to 2", kSplitMinRows);
  if (m == 0) return 0;
  SkinnyArgs a = plain_args(x, w, out, m, n, k);
  a.bias = bias;
  a.halves = halves;
  return launch_epilogue<kPlain>(a, epilogue, static_cast<hipStream_t>(stream));
}

// out (bfloat16) = xielu(x w^T), pq its two numbers.  With ssq_parts x is bfloat16(residual * g), as in bc4g_gemm_skinny_prenormed.
extern "C" int bc4g_gemm_skinny_xielu(const void* x, const float* ssq_parts, int ssq_blocks, int ssq_stride, float eps, const void* w,
                                      void* out, const float* pq, int m, int n, int k, void* stream) {
  if (int e = check_common("gemm_skinny_xielu", m, 64, n, k, kXieluBf16)) return e;
  BC4G_REQUIRE(x && w && out && pq, "gemm_skinny_xielu: a tensor is missing");
  if (ssq_parts)
    if (int e = check_parts("gemm_skinny_xielu", ssq_parts, ssq_blocks, ssq_stride, 0, m, eps)) return e;
  if (m == 0) return 0;
  SkinnyArgs a = plain_args(x, w, out, m, n, k);
  a.bias = pq;
  a.ssq_parts = ssq_parts;
  a.ssq_blocks = ssq_blocks;
  a.ssq_stride = ssq_stride;
  a.eps = eps;
  return launch<kXieluBf16, kPlain>(a, static_cast<hipStream_t>(stream));
}

// out (the float residual stream, [m, n]) += x w^T + bias (null: none), and what the RMSNorm after it needs: emit_x
// [m, n] = bfloat16(new residual * g) and emit_ssq [ceil(n / 16)][emit_stride], block b's part of
// every row's sum of squares.
extern "C" int bc4g_gemm_skinny_emit(const void* x, const void* w, float* out, const float* bias, const void* g, int g_dtype, void* emit_x,
                                     float* emit_ssq, int emit_stride, int m, int n, int k, int halves, void* stream) {
  if (int e = check_common("gemm_skinny_emit", m, 64, n, k, kAccumF32)) return e;
  BC4G_REQUIRE(g && emit_x && emit_ssq && emit_stride >= m, "gemm_skinny_emit: the norm's scale and both outputs are needed");
  BC4G_REQUIRE(g_dtype == kBF16 || g_dtype == kF32, "gemm_skinny_emit: unknown norm scale dtype %d", g_dtype);
  BC4G_REQUIRE(!halves || m <= kSplitMinRows, "gemm_skinny_emit: half blocks take at most %d rows", kSplitMinRows);
  if (m == 0) return 0;
  SkinnyArgs a = plain_args(x, w, out, m, n, k);
  a.bias = bias;
  a.emit_g = g;
  a.emit_g_f32 = g_dtype == kF32 ? 1 : 0;
  a.emit_x = static_cast<bf16_t*>(emit_x);
  a.emit_ssq = emit_ssq;
  a.emit_stride = emit_stride;
  a.halves = halves;
  return launch<kAccumF32, kPlain>(a, static_cast<hipStream_t>(stream));
}

// x is bfloat16(residual * g) and ssq_parts the parts of the rows' sums of squares, as
// bc4g_gemm_skinny_emit leaves them: out = rmsnorm(residual) w^T with the epilogues of bc4g_gemm_skinny
// except the adding one.
extern "C" int bc4g_gemm_skinny_prenormed(const void* x, const float* ssq_parts, int ssq_blocks, int ssq_stride, int ssq_halves, float eps,
                                          const void* w, void* out, int epilogue, int m, int n, int k, void* stream) {
  if (int e = check_common("gemm_skinny_prenormed", m, 64, n, k, epilogue)) return e;
  if (int e = check_parts("gemm_skinny_prenormed", ssq_parts, ssq_blocks, ssq_stride, ssq_halves, m, eps)) return e;
  BC4G_REQUIRE(epilogue != kAccumF32 && epilogue != kRopeKvBf16, "gemm_skinny_prenormed: epilogue %d is not supported here",
               epilogue);
  if (m == 0) return 0;
  SkinnyArgs a = plain_args(x, w, out, m, n, k);
  a.ssq_parts = ssq_parts;
  a.ssq_blocks = ssq_blocks;
  a.ssq_stride = ssq_stride;
  a.ssq_halves = ssq_halves ? 1 : 0;
  a.eps = eps;
  return launch_epilogue<kPlain>(a, epilogue, static_cast<hipStream_t>(stream));
}

// Whether a product of aligned operands whose norm is not fused goes through rings in LDS (rings: 1) or to the streaming kernel (0).
extern "C" int bc4g_gemm_skinny_rings(int m, int n, int k, int epilogue, int finishes_norm, int* rings) {
  if (int e = check_common("gemm_skinny_rings", m, 64, n, k, epilogue)) return e;
  BC4G_REQUIRE(rings != nullptr, "gemm_skinny_rings: a place for the answer");
  *rings = k % 64 == 0 && !rings_are_slower(epilogue, m, n, k, finishes_norm != 0) ? 1 : 0;
  return 0;
}

extern "C" int bc4g_weight_passes(int n, int k, int bytes_a_number, int* passes) {
  BC4G_REQUIRE(n > 0 && k > 0 && bytes_a_number > 0 && passes != nullptr, "weight_passes: sizes and a place for the answer");
  *passes = passes_by(n, k, bytes_a_number) ? 1 : 0;
  return 0;
}

extern "C" int bc4g_gemm_skinny_normed(const float* x, const int32_t* rows, const void* g, int g_dtype,
                                       float eps, const void* w, void* out, int epilogue, int m, int n, int k,
                                       void* stream) {
  if (int e = check_common("gemm_skinny_normed", m, 16, n, k, epilogue)) return e;
  BC4G_REQUIRE(epilogue != kAccumF32 && epilogue != kRopeKvBf16, "gemm_skinny_normed: epilogue %d is not supported here",
               epilogue);
  if (m == 0) return 0;
  SkinnyArgs a = plain_args(x, w, out, m, n, k);
  a.rows = rows;
  a.g = g;
  a.g_f32 = g_dtype == kF32 ? 1 : 0;
  a.m_stage = ((m + 3) / 4) * 4;
  a.eps = eps;
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (g_dtype == kBF16) return launch_epilogue<kNormedG16>(a, epilogue, s);
  if (g_dtype == kF32) return launch_epilogue<kNormedG32>(a, epilogue, s);
  return fail("gemm_skinny_normed: unknown norm scale dtype %d", g_dtype);
}

// The query/key/value product of a decode step with rotary positions and the cache write in its
// epilogue.  x: bfloat16 [m, k] (g null) -- with ssq_parts given it is bfloat16(residual * g) and the
// rows' scales come from the parts, as in bc4g_gemm_skinny_prenormed -- or the float residual stream
// with RMSNorm fused (g given, m <= 16).  q_out: bfloat16 [m, n_heads * head_dim], rotated, in the
// reordered head layout.
extern "C" int bc4g_gemm_skinny_qkv(const void* x, const void* g, int g_dtype, float eps, const float* ssq_parts,
                                    int ssq_blocks, int ssq_stride, int ssq_halves, const void* w, void* q_out,
                                    const int32_t* positions, const int32_t* slot_map, void* k_cache, void* v_cache,
                                    int m, int k, int n_heads, int n_kv_heads, int head_dim, int rotary_dim,
                                    float theta, int page_tokens, int write_kv, void* stream) {
  RopeKvArgs r{positions, slot_map, static_cast<bf16_t*>(k_cache), static_cast<bf16_t*>(v_cache), n_heads, n_kv_heads,
               head_dim, rotary_dim, page_tokens, write_kv,
               cache_fragment_order(true, head_dim, page_tokens) ? 1 : 0, theta};
  const int n = (n_heads + 2 * n_kv_heads) * head_dim;
  if (int e = check_common("gemm_skinny_qkv", m, g ? 16 : 64, n, k, kRopeKvBf16)) return e;
  if (int e = check_rope("gemm_skinny_qkv", r, n)) return e;
  BC4G_REQUIRE(!(g && ssq_parts), "gemm_skinny_qkv: the norm is either fused or prepared, not both");
  if (ssq_parts) {
    if (int e = check_parts("gemm_skinny_qkv", ssq_parts, ssq_blocks, ssq_stride, ssq_halves, m, eps)) return e;
  }
  if (m == 0) return 0;
  hipStream_t s = static_cast<hipStream_t>(stream);
  SkinnyArgs a = plain_args(x, w, q_out, m, n, k);
  a.g = g;
  a.g_f32 = g_dtype == kF32 ? 1 : 0;
  a.m_stage = g ? ((m + 3) / 4) * 4 : 0;
  a.eps = eps;
  a.rope = r;
  a.ssq_parts = ssq_parts;
  a.ssq_blocks = ssq_blocks;
  a.ssq_stride = ssq_stride;
  a.ssq_halves = ssq_halves ? 1 : 0;
  if (!g) return launch<kRopeKvBf16, kPlain>(a, s);
  if (g_dtype == kBF16) return launch<kRopeKvBf16, kNormedG16>(a, s);
  if (g_dtype == kF32) return launch<kRopeKvBf16, kNormedG32>(a, s);
  return fail("gemm_skinny_qkv: unknown norm scale dtype %d", g_dtype);
}
