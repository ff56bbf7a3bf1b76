// Choosing tokens on the device, one workgroup of 16 waves a row of logits: greedy, by temperature, and by top-k / top-p.
//
// The law with filters (the reference's, engine/src/sampler.cpp:63-104): weights w_i = exp((l_i - max) / T) in float; the
// tokens in the order of falling weight, lower id first among equal weights; the k likeliest are kept; of
// those, the fewest whose running sum reaches top_p times their total; the token drawn is the first of the
// kept ones at which u times their total minus the running sum turns negative.
//
// No sort of the row.  A float weight's bit pattern rises with its value, so each of the three questions -- where does
// the count reach k, where does the running sum reach top_p of the total, where does it pass u of the kept
// mass -- is a search in a histogram over the patterns' leading bits, 64 buckets an octave: the bucket in which the answer
// lies, and then the bucket's tokens put in order (each counts the keys before its own) with a running sum over them.
// A bucket of more than 512 tokens -- flat rows of a large vocabulary -- is first looked at by its next 11 bits in the same way.
// Where the first question's bucket and those above it hold up to 512 tokens -- a model's peaked rows, a small top-k of a row that
// is not flat there -- these are put in order at once and answer all three.  A bucket's mass is kept as the integer sum of its
// tokens' mantissas (they share the exponent), added with integer atomics: exact, and the same in every run whatever order the
// adds arrive in.
// Rows whose answers lie among more tokens of all but one weight than that, or below 2^-32 of the likeliest, go by walks down the
// patterns' digits: a histogram over the top 8 bits (the exponent) of the tokens in question, the bucket in which the answer lies,
// then the next 8 bits of that bucket's tokens, and so on over four levels to one exact pattern; tokens that share it are told apart by id.
// The sums over buckets are doubles.  (Sums in another order than the host's one-by-one walk over a sorted list: a boundary may
// move by one token when u falls within rounding of it.)
//
// A CU takes 64 lanes' instructions a clock, so what a row costs is the number of passes over its tokens times the instructions a
// token takes in each, and the barriers between them: a vocabulary of up to 32,768 is read once and its patterns stay in LDS.
// 64 rows of 32,000 tokens, a mixture of limits, two in five of them flat: 26 us, 32 with the rows that have none beside them in one launch (before,
// with walks for every question and every row's candidates listed in the order of their ids: 73, and 16 for the others' launch).
// A whole choice, 8 rows of 128,256 at temperature 5 with a top-p of 0.95: 526 us so, 609 with walks for buckets of more than 512 tokens,
// 157 with their next bits; 262,144 at temperature 1 and 0.9: 938, 1,184 and 227.
#include <float.h>
#include <math.h>

#include <mutex>

#include "api.h"
#include "common.h"

namespace bc4g {
namespace {

constexpr int kThreads = 1024;
constexpr int kWaves = kThreads / kWave;
constexpr int kBuckets = 256;
constexpr int kMaxHeld = 32768;              // tokens whose patterns go into LDS when they are first read (128 KB)
constexpr int kRoom = kMaxHeld + 4096;       // 32-bit words of LDS a row has: the patterns, and beside them the buckets' sums or the sorted tokens
// A bucket's count rides in the top bits of its mantissa sum, one atomic add for both, where the vocabulary
// leaves room: 2^19 tokens of 24-bit mantissas sum to less than 2^43.  (Beyond, an add each.)
constexpr int kCountShift = 44;
constexpr int kMaxPacked = 1 << 19;

enum { kByCount = 0, kByMassGe = 1, kByMassGt = 2 };

// A prefix of a row's tokens in the law's order.
struct Prefix {
  long long bits;   // every token whose weight's pattern is above this one (-1: every token), and
  int ties;         // this many of the tokens with exactly this pattern, lowest ids first
  double mass;      // the sum of its weights (negative: not known yet)
};

struct Shared {
  unsigned int cnt[kBuckets];
  unsigned long long msum[kBuckets];
  float red_v[kWaves];
  double red_d[kWaves];
  unsigned int red_u[kWaves];
  __align__(16) int wave_cnt[kWaves];
  // a walk's state: the wave that walks a level's buckets writes it between barriers, all read it after
  unsigned int prefix;         // the digits settled so far
  unsigned int above_count;    // tokens of the universe strictly above the bucket in question
  double above_mass;
  double target;
  double total;                // the universe's mass, where a walk had to work it out
  int done;
  int found;                   // the walk's answer: found, pattern, how many of its tokens count, how many there are
  long long res_bits;
  int res_ties;
  int res_count;
  int listed;                  // tokens gathered
  int first_ge, first_gt;      // places found in the sorted tokens
  int bucket;                  // a question's answer among the fine buckets: which, what lies above it, how many tokens it holds
  unsigned int bucket_above;
  double bucket_mass;
  int bucket_count;
  int alone_level;             // (>= 0: the answer is the one token of the bucket settled at this level; its pattern is looked up)
  int hit;
};

__device__ inline unsigned int mantissa(unsigned int b) {
  return (b >> 23) ? ((b & 0x7fffffu) | 0x800000u) : (b & 0x7fffffu);
}
__device__ inline double scaled(unsigned long long msum, unsigned int exponent) {
  // msum * 2^(exponent - 150) (a denormal's exponent counts as 1): the power of two built from its bits, the product exact
  const long long power = static_cast<long long>(static_cast<int>(exponent ? exponent : 1u) - 150 + 1023) << 52;
  return static_cast<double>(msum) * __longlong_as_double(power);
}
__device__ inline double value_of(long long bits) {
  return static_cast<double>(__uint_as_float(static_cast<unsigned int>(bits)));
}
__device__ inline bool reached(int mode, unsigned int k, double target, unsigned int count, double mass) {
  return mode == kByCount ? count >= k : mode == kByMassGe ? mass >= target : mass > target;
}

// How many of c tokens of one weight, after `above`, it takes to reach the goal: 1 .. c.
__device__ int ties_needed(int mode, unsigned int k, double target, unsigned int above_count, double above_mass,
                           double val, int c) {
  int r;
  if (mode == kByCount) {
    r = static_cast<int>(k - above_count);
  } else {
    if (!(val > 0.0)) return reached(mode, k, target, 0, above_mass) ? 1 : c;
    double need = (target - above_mass) / val;
    need = need < 0.0 ? 0.0 : need > static_cast<double>(c) ? static_cast<double>(c) : need;
    r = mode == kByMassGe ? static_cast<int>(ceil(need)) : static_cast<int>(floor(need)) + 1;
    r = r < 1 ? 1 : r > c ? c : r;
    for (int turn = 0; turn < 4 && r > 1 && reached(mode, k, target, 0, above_mass + (r - 1) * val); ++turn) --r;
    for (int turn = 0; turn < 4 && r < c && !reached(mode, k, target, 0, above_mass + r * val); ++turn) ++r;
  }
  return r < 1 ? 1 : r > c ? c : r;
}

// A row's tokens, their patterns from LDS or worked out from the logits.  each(f): f(pattern, id) for every token that is this
// thread's.
struct Cached {
  const unsigned int* bits;
  int n;
  __device__ bool packed() const { return true; }
  __device__ unsigned int at(int i) const { return bits[i]; }
  template <typename F>
  __device__ inline void each(F f) const {
    for (int base = 4 * threadIdx.x; base < n; base += 4 * kThreads) {
      const uint4 four = *reinterpret_cast<const uint4*>(bits + base);
      const unsigned int b[4] = {four.x, four.y, four.z, four.w};
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (base + e < n) f(b[e], base + e);
    }
  }
};
struct Logits {
  const float* logits;
  int n;
  float row_max, inv_t;
  __device__ bool packed() const { return n <= kMaxPacked; }
  __device__ unsigned int bits_of(float l) const { return __float_as_uint(expf((l - row_max) * inv_t)); }
  __device__ unsigned int at(int i) const { return bits_of(logits[i]); }
  template <typename F>
  __device__ inline void each(F f) const {
    // (eight loads are on their way together: a load from memory takes hundreds of clocks, and four waves a SIMD hide few)
    constexpr int kAhead = 8;
    for (int base = threadIdx.x; base < n; base += kAhead * kThreads) {
      float l[kAhead];
#pragma unroll
      for (int j = 0; j < kAhead; ++j) l[j] = base + j * kThreads < n ? logits[base + j * kThreads] : 0.f;
#pragma unroll
      for (int j = 0; j < kAhead; ++j)
        if (base + j * kThreads < n) f(bits_of(l[j]), base + j * kThreads);
    }
  }
};

constexpr int kHeldTurns = kMaxHeld / (4 * kThreads);

__device__ inline unsigned int wave_scan_u32(unsigned int v, int lane) {
#pragma unroll
  for (int off = 1; off < kWave; off <<= 1) {
    const unsigned int up = __shfl_up(v, off, kWave);
    if (lane >= off) v += up;
  }
  return v;
}
__device__ inline double wave_scan_f64(double v, int lane) {
#pragma unroll
  for (int off = 1; off < kWave; off <<= 1) {
    const double up = __shfl_up(v, off, kWave);
    if (lane >= off) v += up;
  }
  return v;
}

// Walks `universe` (those of the row's tokens that belong to it) in the law's order until the goal is reached: a
// count of k tokens, or a running sum that reaches (kByMassGe) or passes (kByMassGt) a target -- `goal` itself, or
// that fraction of the universe's mass where `of_total` (the mass is then left in sh.total).  Leaves in sh: found
// (0: the universe ends first), res_bits / res_ties (the prefix that reaches the goal ends with the res_ties-th of
// the res_count tokens of this pattern), above_count / above_mass (what lies above that pattern).
// Every thread of the workgroup calls it.
//
// A level's buckets are walked by one wave, four buckets a lane from the top down: every lane adds up its own,
// a running sum over the lanes gives each what lies above it, and the first lane in which the goal is reached
// settles the bucket.
template <typename R>
__device__ void walk(Shared& sh, const R& row, int vocab, const Prefix& universe, int mode, unsigned int k, double goal,
                     bool of_total) {
  constexpr int kShift[4] = {23, 15, 7, 0};
  constexpr unsigned int kMask[4] = {0xffu, 0xffu, 0xffu, 0x7fu};
  constexpr int kPerLane = kBuckets / kWave;
  const int tid = threadIdx.x, lane = tid % kWave;
  const bool packed = row.packed();
  if (tid == 0) {
    sh.prefix = 0;
    sh.above_count = 0;
    sh.above_mass = 0.0;
    sh.done = 0;
    sh.found = 0;
    sh.alone_level = -1;
  }
  for (int level = 0; level < 4; ++level) {
    for (int i = tid; i < kBuckets; i += kThreads) {
      sh.cnt[i] = 0;
      sh.msum[i] = 0;
    }
    __syncthreads();
    const unsigned int prefix = sh.prefix;
    // a thread's tokens in a row that fall into one bucket are added as one (most of a row shares few exponents)
    int cur = -1;
    unsigned int run_count = 0;
    unsigned long long run_sum = 0;
    auto add_run = [&](int bucket) {
      if (packed) {
        atomicAdd(&sh.msum[bucket], (static_cast<unsigned long long>(run_count) << kCountShift) + run_sum);
      } else {
        atomicAdd(&sh.cnt[bucket], run_count);
        atomicAdd(&sh.msum[bucket], run_sum);
      }
    };
    const bool bounded = universe.bits >= 0;
    const unsigned int floor_bits = static_cast<unsigned int>(universe.bits);
    row.each([&](unsigned int b, int) {
      if (bounded && b <= floor_bits) return;
      if (level > 0 && (b >> kShift[level - 1]) != prefix) return;
      const int bucket = static_cast<int>((b >> kShift[level]) & kMask[level]);
      if (bucket != cur) {
        if (cur >= 0) add_run(cur);
        cur = bucket, run_count = 0, run_sum = 0;
      }
      ++run_count;
      run_sum += mantissa(b);
    });
    if (cur >= 0) add_run(cur);
    __syncthreads();
    if (tid < kWave) {
      const unsigned int exponent = level == 0 ? 0u : prefix >> (23 - kShift[level - 1]);
      const int top = static_cast<int>(kMask[level]);
      unsigned int c[kPerLane];
      double m[kPerLane];
      unsigned int lane_count = 0;
      double lane_mass = 0.0;
#pragma unroll
      for (int j = 0; j < kPerLane; ++j) {
        const int b = top - (lane * kPerLane + j);
        const unsigned long long sum = b >= 0 ? sh.msum[b] : 0ull;
        c[j] = packed ? static_cast<unsigned int>(sum >> kCountShift) : b >= 0 ? sh.cnt[b] : 0u;
        m[j] = c[j] ? scaled(packed ? sum & ((1ull << kCountShift) - 1ull) : sum, level == 0 ? static_cast<unsigned int>(b) : exponent)
                    : 0.0;
        lane_count += c[j];
        lane_mass += m[j];
      }
      const unsigned int with_count = wave_scan_u32(lane_count, lane);
      const double with_mass = wave_scan_f64(lane_mass, lane);
      const unsigned int others_count = __shfl_up(with_count, 1, kWave);
      const double others_mass = __shfl_up(with_mass, 1, kWave);
      double target = sh.target;
      if (level == 0) {
        target = goal;
        if (of_total) {
          double total = __shfl(with_mass, kWave - 1, kWave);
          if (universe.ties > 0) total += universe.ties * value_of(universe.bits);
          target = goal * total;
          if (lane == 0) sh.total = total;
        }
        if (lane == 0) sh.target = target;
      }
      unsigned int above_count = sh.above_count + (lane ? others_count : 0u);
      double above_mass = sh.above_mass + (lane ? others_mass : 0.0);
      // in this lane's buckets: the first in which the goal is reached, and the last that holds anything
      int chosen = -1, last = -1;
      unsigned int last_count = above_count;
      double last_mass = above_mass;
#pragma unroll
      for (int j = 0; j < kPerLane; ++j) {
        if (!c[j] || chosen >= 0) continue;
        last = j, last_count = above_count, last_mass = above_mass;
        if (reached(mode, k, target, above_count + c[j], above_mass + m[j])) {
          chosen = j;
        } else {
          above_count += c[j];
          above_mass += m[j];
        }
      }
      const unsigned long long crossing = __ballot(chosen >= 0), holding = __ballot(last >= 0);
      int settler = -1;                     // the lane that settles this level, and its bucket
      if (crossing != 0ull) {
        settler = __ffsll(static_cast<long long>(crossing)) - 1;
      } else if (level > 0 && holding != 0ull) {
        // the bucket as a whole reached the goal and its parts one by one fall a rounding short: its last token does
        settler = 63 - __clzll(static_cast<long long>(holding));
        chosen = last, above_count = last_count, above_mass = last_mass;
      }
      if (settler < 0) {
        // the universe's own tokens are through; it may end with some of the tokens of one more pattern
        if (lane == kWave - 1) {
          sh.above_count = above_count;
          sh.above_mass = above_mass;
          sh.done = 1;
          if (universe.ties > 0) {
            const double val = value_of(universe.bits);
            if (reached(mode, k, target, above_count + universe.ties, above_mass + universe.ties * val)) {
              sh.found = 1;
              sh.res_bits = universe.bits;
              sh.res_count = 0;            // (how many tokens there are of this pattern is not known here)
              sh.res_ties = ties_needed(mode, k, target, above_count, above_mass, val, universe.ties);
            }
          }
        }
      } else if (lane == settler) {
        const unsigned int bucket = static_cast<unsigned int>(top - (lane * kPerLane + chosen));
        const unsigned int settled = level == 0 ? bucket : (prefix << (kShift[level - 1] - kShift[level])) | bucket;
        const int count = static_cast<int>(c[chosen]);
        sh.prefix = settled;
        sh.above_count = above_count;
        sh.above_mass = above_mass;
        sh.res_count = count;
        if (level == 3) {
          sh.done = 1;
          sh.found = 1;
          sh.res_bits = settled;
          sh.res_ties = ties_needed(mode, k, target, above_count, above_mass, value_of(settled), count);
        } else if (count == 1) {
          // one token in the bucket: it is the answer, whatever its other digits are
          sh.done = 1;
          sh.found = 1;
          sh.res_ties = 1;
          sh.alone_level = level;
        }
      }
    }
    __syncthreads();
    if (sh.done) break;
  }
  const int alone_level = sh.alone_level;
  if (alone_level >= 0) {
    const unsigned int digits = sh.prefix;
    const bool bounded = universe.bits >= 0;
    const unsigned int floor_bits = static_cast<unsigned int>(universe.bits);
    row.each([&](unsigned int b, int) {
      if ((!bounded || b > floor_bits) && (b >> kShift[alone_level]) == digits) sh.res_bits = b;
    });
    __syncthreads();
  }
}

// Tokens in 2,048 buckets in the law's order, all tokens of a bucket with one exponent, so that its mass is the sum of their mantissas,
// exactly.  Thread t owns buckets 2 t and 2 t + 1 from then on, with what lies above them.
constexpr int kFine = 2 * kThreads;
struct Fine {
  unsigned int count[2], above[2];
  double mass[2], above_mass[2];
  double total;
};
// The whole row's: 64 buckets an octave from 1 down to 2^-32, and all below that in the last one, whose mass is summed as it comes.
struct Octaves {
  static constexpr bool kLow = true;
  __device__ int bucket(unsigned int b) const {
    const int i = 0x1fc0 - static_cast<int>(b >> 17);
    return i < 0 ? 0 : i < kFine ? i : kFine - 1;
  }
  __device__ unsigned int exponent(int i) const { return (0x1fc0u - i) >> 6; }
};
// One of those buckets', whose patterns begin with the bits of `first`: by the next 11 bits.
struct Within {
  static constexpr bool kLow = false;
  unsigned int first;
  __device__ int bucket(unsigned int b) const { return (b ^ first) >> 17 ? -1 : 0x7ff - static_cast<int>((b >> 6) & 0x7ff); }
  __device__ unsigned int exponent(int) const { return first >> 23; }
};
// above, above_mass: what lies above the tokens in question.
template <typename R, typename B>
__device__ Fine look(Shared& sh, const R& row, const B& by, unsigned int above, double above_mass, unsigned long long* sums) {
  const int tid = threadIdx.x, lane = tid % kWave, wave = tid / kWave;
  const bool packed = row.packed();                   // (else the counts stand behind the sums)
  unsigned int* counts = reinterpret_cast<unsigned int*>(sums + kFine);
  sums[2 * tid] = sums[2 * tid + 1] = 0;
  if (!packed) counts[2 * tid] = counts[2 * tid + 1] = 0;
  __syncthreads();
  double low = 0.0;
  row.each([&](unsigned int b, int) {
    const int bucket = by.bucket(b);
    if (!B::kLow && bucket < 0) return;
    atomicAdd(&sums[bucket], (packed ? 1ull << kCountShift : 0ull) + mantissa(b));
    if (!packed) atomicAdd(&counts[bucket], 1u);
    if (B::kLow && bucket == kFine - 1) low += static_cast<double>(__uint_as_float(b));
  });
  if constexpr (B::kLow) {
#pragma unroll
    for (int off = kWave / 2; off > 0; off >>= 1) low += __shfl_xor(low, off, kWave);
    if (lane == 0) sh.red_d[wave] = low;
  }
  __syncthreads();
  Fine f;
  if constexpr (B::kLow) {
    low = 0.0;
    for (int w = 0; w < kWaves; ++w) low += sh.red_d[w];
  }
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const unsigned long long sum = sums[2 * tid + j];
    f.count[j] = packed ? static_cast<unsigned int>(sum >> kCountShift) : counts[2 * tid + j];
    f.mass[j] = B::kLow && 2 * tid + j == kFine - 1 ? low
                : f.count[j] ? scaled(packed ? sum & ((1ull << kCountShift) - 1ull) : sum, by.exponent(2 * tid + j)) : 0.0;
  }
  const unsigned int with_count = wave_scan_u32(f.count[0] + f.count[1], lane);
  const double with_mass = wave_scan_f64(f.mass[0] + f.mass[1], lane);
  __syncthreads();
  if (lane == kWave - 1) sh.red_u[wave] = with_count, sh.red_d[wave] = with_mass;
  const unsigned int lanes_count = __shfl_up(with_count, 1, kWave);
  const double lanes_mass = __shfl_up(with_mass, 1, kWave);
  __syncthreads();
  f.total = 0.0;
  for (int w = 0; w < kWaves; ++w) {
    if (w < wave) above += sh.red_u[w], above_mass += sh.red_d[w];
    f.total += sh.red_d[w];
  }
  f.above[0] = above + (lane ? lanes_count : 0u);
  f.above_mass[0] = above_mass + (lane ? lanes_mass : 0.0);
  f.above[1] = f.above[0] + f.count[0];
  f.above_mass[1] = f.above_mass[0] + f.mass[0];
  return f;
}

// The bucket in which a goal is reached (as walk's modes have it; kFine: in none), what lies above it and how many tokens it holds.
struct Found {
  int bucket, count;
  unsigned int above;
  double mass;
};
__device__ Found find_bucket(Shared& sh, const Fine& f, int mode, unsigned int k, double target) {
  if (threadIdx.x == 0) sh.bucket = kFine;
  __syncthreads();
#pragma unroll
  for (int j = 0; j < 2; ++j)
    if (f.count[j] && reached(mode, k, target, f.above[j] + f.count[j], f.above_mass[j] + f.mass[j])) {
      atomicMin(&sh.bucket, 2 * static_cast<int>(threadIdx.x) + j);
      break;
    }
  __syncthreads();
#pragma unroll
  for (int j = 0; j < 2; ++j)
    if (sh.bucket == 2 * static_cast<int>(threadIdx.x) + j)
      sh.bucket_above = f.above[j], sh.bucket_mass = f.above_mass[j], sh.bucket_count = static_cast<int>(f.count[j]);
  __syncthreads();
  const Found found = {sh.bucket, sh.bucket_count, sh.bucket_above, sh.bucket_mass};
  __syncthreads();
  return found;
}

// Few enough tokens to be put in order among which a goal is reached: those with patterns lo .. hi, and what lies above them.
constexpr int kFew = 512;
struct Spot {
  unsigned int lo, hi, above;
  int count;
  double mass;
};
enum { kNowhere = 0, kThere = 1, kTooMany = 2 };     // (kNowhere: also below the patterns from `floor` on, or in the last bucket of all)
// looked: whether the row was looked at again, which takes the place of what was sorted.
template <typename R>
__device__ int find_spot(Shared& sh, const R& row, const Fine& fine, int mode, unsigned int k, double target, unsigned int floor,
                         unsigned long long* room, Spot& spot, bool& looked) {
  looked = false;
  Found at = find_bucket(sh, fine, mode, k, target);
  if (at.bucket >= kFine - 1) return kNowhere;
  const unsigned int first = (0x1fc0u - at.bucket) << 17;
  spot.lo = first, spot.hi = at.bucket == 0 ? 0xffffffffu : first | 0x1ffffu;
  if (spot.hi < floor) return kNowhere;
  if (at.count > kFew) {
    looked = true;
    const Fine part = look(sh, row, Within{first}, at.above, at.mass, room);
    at = find_bucket(sh, part, mode, k, target);
    if (at.bucket == kFine || at.count > kFew) return kTooMany;
    spot.lo = first | (0x7ffu - at.bucket) << 6, spot.hi = spot.lo | 0x3fu;
  }
  spot.above = at.above, spot.count = at.count, spot.mass = at.mass;
  return kThere;
}

// Where this thread's `mine` items go among those of all the workgroup's threads, in the order of the threads, and
// how many there are of all.  Every thread calls it (two barriers).
__device__ inline void place_among(Shared& sh, unsigned int mine, int& place, int& all) {
  static_assert(kWaves == 16, "the waves' counts are read as four int4");
  const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
  const unsigned int with_mine = wave_scan_u32(mine, lane);
  if (lane == kWave - 1) sh.wave_cnt[wave] = static_cast<int>(with_mine);
  __syncthreads();
  int before = 0;
  all = 0;
#pragma unroll
  for (int q = 0; q < kWaves / 4; ++q) {
    const int4 c = reinterpret_cast<const int4*>(sh.wave_cnt)[q];
    before += (4 * q < wave ? c.x : 0) + (4 * q + 1 < wave ? c.y : 0) + (4 * q + 2 < wave ? c.z : 0) + (4 * q + 3 < wave ? c.w : 0);
    all += c.x + c.y + c.z + c.w;
  }
  place = before + static_cast<int>(with_mine - mine);
  __syncthreads();
}

// The id of the r-th of the tokens, in the order of the ids, whose weight has this pattern; into sh.hit.
template <typename R>
__device__ void locate(Shared& sh, const R& whole, unsigned int bits, int r) {
  int seen = 0;
  for (int base = 0; base < whole.n; base += kThreads) {
    const int i = base + threadIdx.x;
    const bool match = i < whole.n && whole.at(i) == bits;
    int place, all;
    place_among(sh, match ? 1u : 0u, place, all);
    if (match && seen + place + 1 == r) sh.hit = i;
    seen += all;
    if (seen >= r) break;
  }
}

// The tokens with patterns lo .. hi, up to kFew of them, in the law's order: their keys (a weight's pattern above, the id's
// complement below) in `room` + kFew, and returns this thread's running sum, up to and with the token of its number, from `above` on.
template <typename R>
__device__ double sort_few(Shared& sh, const R& row, unsigned int lo, unsigned int hi, double above, unsigned long long* room, int& n) {
  unsigned long long* keys = room;
  unsigned long long* sorted = room + kFew;
  int* rank = reinterpret_cast<int*>(room + 2 * kFew);
  const int tid = threadIdx.x, lane = tid % kWave, wave = tid / kWave;
  if (tid == 0) sh.listed = 0, sh.first_ge = kFew, sh.first_gt = kFew;
  if (tid < kFew) rank[tid] = 0;
  __syncthreads();
  row.each([&](unsigned int b, int i) {
    if (b < lo || b > hi) return;
    const int at = atomicAdd(&sh.listed, 1);
    if (at < kFew) keys[at] = static_cast<unsigned long long>(b) << 32 | static_cast<unsigned int>(~i);
  });
  __syncthreads();
  n = min(sh.listed, kFew);
  // every key counts those before it; where there are few, several threads share a key's count
  int width = kWave;
  while (width < n) width *= 2;
  const int parts = kThreads / width, mine = tid % width, part = tid / width, each = (n + parts - 1) / parts;
  if (mine < n) {
    const unsigned long long key = keys[mine];
    int before = 0;
    const int end = min(n, (part + 1) * each);
#pragma unroll 4
    for (int j = part * each; j < end; ++j) before += keys[j] > key ? 1 : 0;
    if (before) atomicAdd(&rank[mine], before);
  }
  __syncthreads();
  if (tid < n) sorted[rank[tid]] = keys[tid];
  __syncthreads();
  double mass = 0.0;
  if (tid < kFew) {
    mass = wave_scan_f64(tid < n ? value_of(static_cast<long long>(sorted[tid] >> 32)) : 0.0, lane);
    if (lane == kWave - 1) sh.red_d[wave] = mass;
  }
  __syncthreads();
  for (int w = 0; w < wave && w < kFew / kWave; ++w) above += sh.red_d[w];
  mass += above;
  if (tid < n) reinterpret_cast<double*>(keys)[tid] = mass;   // (the keys have been put in order)
  __syncthreads();
  return mass;
}
// The first of the sorted tokens below `end` at which a running sum reaches (ge) or passes the target; end - 1 if none does.
__device__ int first_at(int& place, double mass, bool ge, double target, int end) {
  const int tid = threadIdx.x;
  const unsigned long long over = __ballot(tid < end && (ge ? mass >= target : mass > target));
  if (over != 0ull && tid % kWave == 0) atomicMin(&place, tid + __ffsll(static_cast<long long>(over)) - 1);
  __syncthreads();
  return min(place, end - 1);
}

// The three questions by walks over the row, whatever its weights.
template <typename R>
__device__ int draw_by_walks(Shared& sh, const R& row, unsigned int k, double p, double u) {
  const int vocab = row.n;
  const Prefix everything = {-1, 0, -1.0};
  Prefix kept = everything;
  // the k likeliest; of those, the fewest that reach top_p of their total; the first of those at which the running sum
  // passes u of their mass; and, where rounding keeps that from being reached, the last of the row's tokens
  int question = k < static_cast<unsigned int>(vocab) ? 0 : p < 1.0 ? 1 : 2;
  for (;;) {
    const bool of_total = question > 0 && question < 3 && kept.mass < 0.0;
    const double share = question == 1 ? p : u;
    walk(sh, row, vocab, question == 3 ? everything : kept, question == 0 || question == 3 ? kByCount : question == 1 ? kByMassGe : kByMassGt,
         question == 3 ? static_cast<unsigned int>(vocab) : k, of_total ? share : share * kept.mass, of_total);
    const bool found = sh.found;
    const long long bits = sh.res_bits;
    const int ties = sh.res_ties;
    const double mass = sh.above_mass, all = sh.total;
    __syncthreads();
    if (question < 2) {
      if (found) kept = {bits, ties, mass + ties * value_of(bits)};
      else if (question == 1 && of_total) kept.mass = all;      // (rounding left the sum a hair short: everything is kept)
      question = question == 0 && p < 1.0 ? 1 : 2;
      continue;
    }
    if (!found && question == 2 && !(kept.bits >= 0 && kept.ties > 0)) {
      question = 3;
      continue;
    }
    const bool of_kept = !found && question == 2;               // (rounding again: the last of the kept tokens)
    locate(sh, row, static_cast<unsigned int>(of_kept ? kept.bits : bits), of_kept ? kept.ties : ties);
    __syncthreads();
    return sh.hit;
  }
}

template <typename R>
__device__ int draw_from(Shared& sh, const R& row, int top_k, double p, double u, unsigned long long* room) {
  const int vocab = row.n;
  const bool count_first = top_k > 0 && top_k < vocab;
  const unsigned int k = count_first ? static_cast<unsigned int>(top_k) : static_cast<unsigned int>(vocab);
  const Fine fine = look(sh, row, Octaves{}, 0u, 0.0, room);
  // Where the first question's answer lies.  (In the last bucket, which holds many exponents, or among more tokens than can be put
  // in order: the general way.)
  Spot at;
  bool looked;
  if (find_spot(sh, row, fine, count_first ? kByCount : kByMassGe, k, p * fine.total, 0u, room, at, looked) != kThere)
    return draw_by_walks(sh, row, k, p, u);
  const unsigned long long* sorted = room + kFew;
  const double* upto = reinterpret_cast<const double*>(room);
  const bool all = at.above + static_cast<unsigned int>(at.count) <= static_cast<unsigned int>(kFew);
  if (all) at.hi = 0xffffffffu, at.above = 0, at.mass = 0.0;        // (with every token above it)
  int n;
  double mass = sort_few(sh, row, at.lo, at.hi, at.mass, room, n);
  int kept = count_first ? min(static_cast<int>(k - at.above), n) : n;     // of the sorted tokens
  double kept_mass = upto[kept - 1];
  // A later question's answer lies above the sorted tokens or, rounding included, among them.  False: by walks.
  auto go_on = [&](int mode, double target) {
    if (all) return true;
    Spot there;
    const int found = find_spot(sh, row, fine, mode, 0u, target, at.lo, room, there, looked);
    if (found == kTooMany) return false;
    const bool earlier = found == kThere && there.lo > at.lo;
    if (earlier) at = there;
    if (earlier || looked) mass = sort_few(sh, row, at.lo, at.hi, at.mass, room, n);
    if (earlier) kept = n;
    return true;
  };
  if (p < 1.0) {
    const double target = p * (count_first ? kept_mass : fine.total);
    if (count_first && !go_on(kByMassGe, target)) return draw_by_walks(sh, row, k, p, u);
    kept = first_at(sh.first_ge, mass, true, target, kept) + 1;
    kept_mass = upto[kept - 1];
  }
  const double target = u * kept_mass;
  if (!go_on(kByMassGt, target)) return draw_by_walks(sh, row, k, p, u);
  return static_cast<int>(~static_cast<unsigned int>(sorted[first_at(sh.first_gt, mass, false, target, kept)]));
}

// HELD: the vocabulary's patterns fit LDS beside the few candidates' keys.
template <bool HELD>
__device__ int draw_filtered(Shared& sh, const float* logits, int vocab, float temperature, double u, int top_k, double p, unsigned int* room) {
  const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
  float v = -FLT_MAX;
  const bool by_four = vocab % 4 == 0 && reinterpret_cast<uintptr_t>(logits) % 16 == 0;
  auto four_at = [&](int first) {                   // four logits from `first` on (below the vocabulary), -FLT_MAX beyond its end
    if (by_four) return *reinterpret_cast<const float4*>(logits + first);
    return make_float4(logits[first], first + 1 < vocab ? logits[first + 1] : -FLT_MAX, first + 2 < vocab ? logits[first + 2] : -FLT_MAX,
                       first + 3 < vocab ? logits[first + 3] : -FLT_MAX);
  };
  float4 l[kHeldTurns];
  for (int begin = 0; begin < vocab; begin += kMaxHeld) {
#pragma unroll
    for (int j = 0; j < kHeldTurns; ++j) {
      const int first = begin + (j * kThreads + threadIdx.x) * 4;
      l[j] = first < vocab ? four_at(first) : make_float4(-FLT_MAX, -FLT_MAX, -FLT_MAX, -FLT_MAX);
    }
#pragma unroll
    for (int j = 0; j < kHeldTurns; ++j) v = fmaxf(fmaxf(fmaxf(v, l[j].x), fmaxf(l[j].y, l[j].z)), l[j].w);
  }
  v = wave_max(v);
  if (lane == 0) sh.red_v[wave] = v;
  __syncthreads();
  v = sh.red_v[0];
  for (int w = 1; w < kWaves; ++w) v = fmaxf(v, sh.red_v[w]);
  const Logits row{logits, vocab, v, 1.0f / temperature};
  if (threadIdx.x == 0) sh.hit = 0;
  if constexpr (HELD) {                             // (the logits are still in registers)
#pragma unroll
    for (int j = 0; j < kHeldTurns; ++j)
      *reinterpret_cast<uint4*>(room + (j * kThreads + threadIdx.x) * 4) =
          make_uint4(row.bits_of(l[j].x), row.bits_of(l[j].y), row.bits_of(l[j].z), row.bits_of(l[j].w));
    return draw_from(sh, Cached{room, vocab}, top_k, p, u, reinterpret_cast<unsigned long long*>(room + kMaxHeld));
  } else {
    return draw_from(sh, row, top_k, p, u, reinterpret_cast<unsigned long long*>(room));
  }
}

// ---- temperature sampling --------------------------------------------------
// The law: weights w_i = exp((l_i - max) / T) in float, summed in double; the token is the first i,
// in vocabulary order, at which u * total - (w_0 + ... + w_i) turns negative.  One workgroup a row.
// The vocabulary is cut into groups of 512 consecutive tokens, a lane holding eight in a row (more
// beyond 2,097,152 tokens, so that the groups' sums fit LDS): a lane sums its own tokens in order
// without a word to its neighbours (sums of doubles across lanes go through the LDS crossbar, which
// sixteen waves share), a wave then a group; every pass over the row reads whole cache lines.  The
// groups' sums, a running sum over them (one wave, 64 groups a step) and a last look inside the one
// group where the target is crossed find the token.
// (Sums in another order than the host's one-by-one walk: a boundary may move by one token when u
// falls within rounding of it.)
constexpr int kSampleMaxGroups = 4096;
constexpr int kSamplePerLane = 8;           // consecutive tokens a lane holds of a group
constexpr int kSampleAhead = 4;             // loads of 16 bytes (pairs of them in the second pass) a thread has in flight

__device__ inline void better(float& v, int& i, float ov, int oi) {
  if (ov > v || (ov == v && oi < i)) {
    v = ov;
    i = oi;
  }
}

__device__ inline double wave_sum_f64(double v) {
#pragma unroll
  for (int off = kWave / 2; off > 0; off >>= 1) v += __shfl_xor(v, off, kWave);
  return v;
}
// Thread 0 writes the token to `to`.  group_sum: kSampleMaxGroups doubles, then the running sums up to and with each group.
__device__ void draw_unfiltered(Shared& sh, const float* row, int vocab, float temp, double u, double* group_sum, int32_t* to) {
  float* best_v = sh.red_v;
  int* best_i = sh.wave_cnt;
  const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;

  // the maximum and where it stands first
  float v = -FLT_MAX;
  int idx = vocab;
  // in fours where the row starts on 16 bytes and the vocabulary is a multiple of four
  const bool by_four = vocab % 4 == 0 && reinterpret_cast<uintptr_t>(row) % 16 == 0;
  if (by_four) {
    const float4* row4 = reinterpret_cast<const float4*>(row);
    const int n4 = vocab / 4;
    for (int at = threadIdx.x; at < n4; at += kSampleAhead * kThreads) {
      float4 t[kSampleAhead];               // the loads first, so that they are in flight together
#pragma unroll
      for (int j = 0; j < kSampleAhead; ++j) {
        const int i4 = at + j * kThreads;
        t[j] = i4 < n4 ? row4[i4] : make_float4(0.f, 0.f, 0.f, 0.f);
      }
#pragma unroll
      for (int j = 0; j < kSampleAhead; ++j) {
        const int i4 = at + j * kThreads;
        if (i4 < n4) {
          better(v, idx, t[j].x, 4 * i4);
          better(v, idx, t[j].y, 4 * i4 + 1);
          better(v, idx, t[j].z, 4 * i4 + 2);
          better(v, idx, t[j].w, 4 * i4 + 3);
        }
      }
    }
  } else {
    for (int at = threadIdx.x; at < vocab; at += kThreads) better(v, idx, row[at], at);
  }
#pragma unroll
  for (int off = kWave / 2; off > 0; off >>= 1) better(v, idx, __shfl_xor(v, off, kWave), __shfl_xor(idx, off, kWave));
  if (lane == 0) {
    best_v[wave] = v;
    best_i[wave] = idx;
  }
  __syncthreads();
  float row_max = best_v[0];
  int best = best_i[0];
  for (int w = 1; w < kWaves; ++w) better(row_max, best, best_v[w], best_i[w]);
  const int arg = best < vocab ? best : 0;
  if (!(temp > 0.f)) {
    if (threadIdx.x == 0) *to = arg;
    return;
  }
  const float inv_t = 1.0f / temp;
  const int per_lane = max(kSamplePerLane, (vocab + kWave * kSampleMaxGroups - 1) / (kWave * kSampleMaxGroups));
  const int group_size = kWave * per_lane;
  const int n_groups = (vocab + group_size - 1) / group_size;
  auto lane_weight_sum = [&](int g) {      // this lane's tokens of group g, in order
    double s = 0.0;
    const int first = g * group_size + lane * per_lane;
    for (int j = 0; j < per_lane; ++j) {
      const int i = first + j;
      if (i < vocab) s += static_cast<double>(expf((row[i] - row_max) * inv_t));
    }
    return s;
  };
  if (by_four && per_lane == kSamplePerLane) {        // a wave's groups at once: their loads are in flight together
    static_assert(kSamplePerLane == 8, "two loads of four a lane");
    for (int g0 = wave; g0 < n_groups; g0 += kWaves * kSampleAhead) {
      float4 t[kSampleAhead][2];
#pragma unroll
      for (int j = 0; j < kSampleAhead; ++j) {
        const int first = (g0 + j * kWaves) * group_size + lane * kSamplePerLane;
#pragma unroll
        for (int h = 0; h < 2; ++h)
          t[j][h] = first + 4 * h < vocab ? *reinterpret_cast<const float4*>(row + first + 4 * h) : make_float4(0.f, 0.f, 0.f, 0.f);
      }
#pragma unroll
      for (int j = 0; j < kSampleAhead; ++j) {
        const int g = g0 + j * kWaves;
        const int first = g * group_size + lane * kSamplePerLane;
        double s = 0.0;                     // the order of lane_weight_sum: the look inside a group sums the same
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          if (first + 4 * h < vocab) {
            s += static_cast<double>(expf((t[j][h].x - row_max) * inv_t));
            s += static_cast<double>(expf((t[j][h].y - row_max) * inv_t));
            s += static_cast<double>(expf((t[j][h].z - row_max) * inv_t));
            s += static_cast<double>(expf((t[j][h].w - row_max) * inv_t));
          }
        }
        s = wave_sum_f64(s);
        if (lane == 0 && g < n_groups) group_sum[g] = s;
      }
    }
  } else {
    for (int g = wave; g < n_groups; g += kWaves) {
      const double s = wave_sum_f64(lane_weight_sum(g));
      if (lane == 0) group_sum[g] = s;
    }
  }
  __syncthreads();
  if (wave != 0) return;

  // one wave: running sums over the groups, 64 at a step; then the first group they cross the target in
  double carry = 0.0;
  for (int c = 0; c < n_groups; c += kWave) {
    const int g = c + lane;
    const double incl = carry + wave_scan_f64(g < n_groups ? group_sum[g] : 0.0, lane);
    if (g < n_groups) group_sum[g] = incl;
    carry = __shfl(incl, kWave - 1, kWave);
  }
  const double target = u * carry;
  int found = n_groups;
  for (int c = 0; c < n_groups && found == n_groups; c += kWave) {
    const int g = c + lane;
    const unsigned long long over = __ballot(g < n_groups && target - group_sum[g] < 0.0);
    if (over != 0ull) found = c + __ffsll(static_cast<long long>(over)) - 1;
  }
  int result = arg;        // rounding may leave the target a hair above zero after the last token
  if (found < n_groups) {
    const double before = found > 0 ? group_sum[found - 1] : 0.0;
    const double mine = lane_weight_sum(found);
    const double upto = before + wave_scan_f64(mine, lane);              // with this lane's tokens
    const unsigned long long over = __ballot(target - upto < 0.0);
    if (over != 0ull) {
      const int at = __ffsll(static_cast<long long>(over)) - 1;          // the lane whose tokens cross it
      double left = target - (upto - mine);
      const int first = found * group_size + lane * per_lane;
      int hit = min(vocab - 1, first + per_lane - 1);
      for (int j = 0; j < per_lane; ++j) {
        const int i = first + j;
        if (i >= vocab) break;
        left -= static_cast<double>(expf((row[i] - row_max) * inv_t));
        if (left < 0.0) {
          hit = i;
          break;
        }
      }
      result = __shfl(hit, at, kWave);
    }
  }
  if (lane == 0) *to = result;
}


// What the rows of a launch ask for, in its arguments: nothing to bring to the device before it.
constexpr int kChooseRows = 64;
struct ChooseArgs {
  double u[kChooseRows], top_p[kChooseRows];
  float temperature[kChooseRows];
  int top_k[kChooseRows];
};
// The same on the device, for any number of rows: entry i is logits row rows[i] (null: row i).
struct ChooseLists {
  const int32_t* rows;
  const float* temperature;
  const double* u;
  const int32_t* top_k;
  const double* top_p;
};

// One row's token to `to`.  HELD: as draw_filtered has it.
template <bool HELD>
__device__ inline void choose_row(Shared& sh, const float* from, int vocab, float temperature, double u, int top_k, double top_p, bool filtered,
                                  unsigned int* room, int32_t* to) {
  if (filtered) {
    const int token = draw_filtered<HELD>(sh, from, vocab, temperature, u, top_k, top_p, room);
    if (threadIdx.x == 0) *to = token;
  } else {
    draw_unfiltered(sh, from, vocab, temperature, u, reinterpret_cast<double*>(room), to);
  }
}
__host__ __device__ inline bool limited(float temperature, int top_k, double top_p, int vocab) {
  return temperature > 0.f && ((top_k > 0 && top_k < vocab) || top_p < 1.0);
}

// LIMITS false: no row has a limit -- a kernel without the other law's registers and scratch memory (64 rows of 32,000 15.5 us; with that law
// compiled in beside it, 21.8 in a serving step).
template <bool HELD, bool LIMITS>
__global__ __launch_bounds__(kThreads) void choose_kernel(const float* __restrict__ logits, int32_t* __restrict__ out, int vocab,
                                                                          const ChooseArgs a) {
  __shared__ Shared sh;
  extern __shared__ __align__(16) unsigned int room[];
  const int row = blockIdx.x;
  const float* from = logits + static_cast<size_t>(row) * vocab;
  if constexpr (LIMITS) {
    choose_row<HELD>(sh, from, vocab, a.temperature[row], a.u[row], a.top_k[row], a.top_p[row],
                     limited(a.temperature[row], a.top_k[row], a.top_p[row], vocab), room, out + row);
  } else {
    draw_unfiltered(sh, from, vocab, a.temperature[row], a.u[row], reinterpret_cast<double*>(room), out + row);
  }
}

// kNone: no row has a limit (a kernel of its own, of half the registers, so that two workgroups share a CU: a choice of 512
// rows of 32,000 198 us, 242 with the law with filters beside it); kSome: those that have; kEvery: every row by the law with filters, whatever its limits.
enum Limits : int { kNone = 0, kSome = 1, kEvery = 2 };

template <bool HELD, bool LIMITS>
__global__ __launch_bounds__(kThreads, LIMITS ? 4 : 8) void choose_listed_kernel(const float* __restrict__ logits, int32_t* __restrict__ out, int vocab,
                                                                 const ChooseLists a, int limits) {
  __shared__ Shared sh;
  extern __shared__ __align__(16) unsigned int room[];
  const int i = blockIdx.x, row = a.rows ? a.rows[i] : i;
  const float* from = logits + static_cast<size_t>(row) * vocab;
  if constexpr (LIMITS) {
    choose_row<HELD>(sh, from, vocab, a.temperature[i], a.u[i], a.top_k[i], a.top_p[i],
                     limits == kEvery || limited(a.temperature[i], a.top_k[i], a.top_p[i], vocab), room, out + row);
  } else {
    draw_unfiltered(sh, from, vocab, a.temperature[i], a.u[i], reinterpret_cast<double*>(room), out + row);
  }
}

// LDS of a workgroup: with the vocabulary's patterns, a CU to itself; without, room for two on a CU.
constexpr int kHeldBytes = kRoom * 4, kPlainBytes = kSampleMaxGroups * 8;
static_assert((kRoom - kMaxHeld) * 4 >= 3 * kFew * 8 && (kRoom - kMaxHeld) * 4 >= kFine * 8 && kPlainBytes >= (kRoom - kMaxHeld) * 4,
              "the sorted tokens, the buckets, and in a mixed launch a plain row's sums over groups");
static_assert(kPlainBytes >= kFine * 12, "the buckets with counts of their own");

int raise_room() {
  static std::once_flag once;
  static hipError_t raised = hipSuccess;
  std::call_once(once, [] {
    const void* kernels[] = {reinterpret_cast<const void*>(choose_listed_kernel<true, true>), reinterpret_cast<const void*>(choose_kernel<true, true>)};
    for (const void* kernel : kernels)
      if (raised == hipSuccess) raised = hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, kHeldBytes);
  });
  if (raised != hipSuccess) return fail("sampling: cannot raise the dynamic LDS limit to %d bytes", kHeldBytes);
  return 0;
}

int choose_listed(const char* what, const float* logits, const ChooseLists& lists, int32_t* out, int n, int vocab, Limits limits, hipStream_t s) {
  if (int e = raise_room()) return e;
  if (limits == kNone) choose_listed_kernel<false, false><<<n, kThreads, kPlainBytes, s>>>(logits, out, vocab, lists, limits);
  else if (vocab <= kMaxHeld) choose_listed_kernel<true, true><<<n, kThreads, kHeldBytes, s>>>(logits, out, vocab, lists, limits);
  else choose_listed_kernel<false, true><<<n, kThreads, kPlainBytes, s>>>(logits, out, vocab, lists, limits);
  return check_launch(what);
}

}  // namespace
}  // namespace bc4g

using namespace bc4g;

extern "C" int bc4g_sample(const float* logits, const float* temperature, const double* u, int32_t* out,
                           int n_rows, int vocab, void* stream) {
  BC4G_REQUIRE(n_rows >= 0 && vocab > 0, "sample: bad sizes rows=%d V=%d", n_rows, vocab);
  if (n_rows == 0) return 0;
  return choose_listed("sample", logits, ChooseLists{nullptr, temperature, u, nullptr, nullptr}, out, n_rows, vocab, kNone,
                       static_cast<hipStream_t>(stream));
}

// For each of n rows: draws the token of logits row rows[i] by the law above with temperature[i] (> 0), the
// uniform number u[i] in [0, 1), top_k[i] (0 or >= vocab: no limit) and top_p[i] (>= 1: no limit), into
// out[rows[i]].  logits: float [*, vocab], contiguous.
extern "C" int bc4g_sample_filtered(const float* logits, const int32_t* rows, const float* temperature, const double* u,
                                    const int32_t* top_k, const double* top_p, int32_t* out, int n, int vocab,
                                    void* stream) {
  BC4G_REQUIRE(n >= 0 && vocab > 0, "sample_filtered: bad sizes rows=%d V=%d", n, vocab);
  if (n == 0) return 0;
  return choose_listed("sample_filtered", logits, ChooseLists{rows, temperature, u, top_k, top_p}, out, n, vocab, kEvery,
                       static_cast<hipStream_t>(stream));
}

extern "C" int bc4g_choose_listed(const float* logits, const float* temperature, const double* u, const int32_t* top_k, const double* top_p,
                                  int32_t* out, int n_rows, int vocab, void* stream) {
  BC4G_REQUIRE(n_rows >= 0 && vocab > 0 && logits && temperature && u && !top_k == !top_p && out,
               "choose: bad sizes rows=%d V=%d, or a tensor is missing", n_rows, vocab);
  if (n_rows == 0) return 0;
  return choose_listed("choose", logits, ChooseLists{nullptr, temperature, u, top_k, top_p}, out, n_rows, vocab, top_k ? kSome : kNone,
                       static_cast<hipStream_t>(stream));
}

// temperature, u, top_k and top_p lie on the host.
extern "C" int bc4g_choose(const float* logits, const float* temperature, const double* u, const int32_t* top_k, const double* top_p,
                           int32_t* out, int n_rows, int vocab, void* stream) {
  BC4G_REQUIRE(n_rows >= 0 && n_rows <= kChooseRows && vocab > 0 && logits && temperature && u && top_k && top_p && out,
               "choose: bad sizes rows=%d (at most %d) V=%d, or a tensor is missing", n_rows, kChooseRows, vocab);
  if (n_rows == 0) return 0;
  if (int e = raise_room()) return e;
  hipStream_t s = static_cast<hipStream_t>(stream);
  ChooseArgs a{};
  bool filtered = false;
  for (int i = 0; i < n_rows; ++i) {
    a.temperature[i] = temperature[i], a.u[i] = u[i], a.top_k[i] = top_k[i], a.top_p[i] = top_p[i];
    filtered = filtered || limited(temperature[i], top_k[i], top_p[i], vocab);
  }
  if (!filtered) choose_kernel<false, false><<<n_rows, kThreads, kPlainBytes, s>>>(logits, out, vocab, a);
  else if (vocab <= kMaxHeld) choose_kernel<true, true><<<n_rows, kThreads, kHeldBytes, s>>>(logits, out, vocab, a);
  else choose_kernel<false, true><<<n_rows, kThreads, kPlainBytes, s>>>(logits, out, vocab, a);
  return check_launch("choose");
}
