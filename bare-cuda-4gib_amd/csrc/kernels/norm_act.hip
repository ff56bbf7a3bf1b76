// A norm that is added to the residual stream (the second norm of a layer whose sublayers are normed on both
// sides), the xIELU activation, and a gated unit with clamped branches.  One instantiation per storage type; all arithmetic in float.
#include <math.h>

#include "api.h"
#include "common.h"

namespace bc4g {
namespace {

constexpr int kBlock = 256;


// x[r, :] += y[r, :] * rsqrt(mean(y[r]^2) + eps) * w.  The row of y is read twice (the second time from the cache).
template <typename TY>
__global__ __launch_bounds__(kBlock) void rmsnorm_add_kernel(float* __restrict__ x, const TY* __restrict__ y,
                                                             const float* __restrict__ w, int hidden, float eps) {
  __shared__ float scratch[16];
  const TY* yr = y + static_cast<size_t>(blockIdx.x) * hidden;
  float* xr = x + static_cast<size_t>(blockIdx.x) * hidden;
  float ss = 0.f;
  for (int i = threadIdx.x; i < hidden; i += kBlock) {
    const float v = to_float(yr[i]);
    ss += v * v;
  }
  const float scale = 1.0f / sqrtf(block_sum(ss, scratch) / static_cast<float>(hidden) + eps);
  for (int i = threadIdx.x; i < hidden; i += kBlock) xr[i] += to_float(yr[i]) * scale * w[i];
}

__device__ inline void load_eight(const float* p, float (&v)[8]) {
  const float4 a = *reinterpret_cast<const float4*>(p), b = *reinterpret_cast<const float4*>(p + 4);
  v[0] = a.x, v[1] = a.y, v[2] = a.z, v[3] = a.w, v[4] = b.x, v[5] = b.y, v[6] = b.z, v[7] = b.w;
}
__device__ inline void load_eight(const bf16_t* p, float (&v)[8]) {
  const uint4 b = *reinterpret_cast<const uint4*>(p);
  const unsigned w[4] = {b.x, b.y, b.z, b.w};
#pragma unroll
  for (int e = 0; e < 4; ++e) v[2 * e] = __uint_as_float(w[e] << 16), v[2 * e + 1] = __uint_as_float(w[e] & 0xffff0000u);
}
__device__ inline void store_eight(float* p, const float (&v)[8]) {
  *reinterpret_cast<float4*>(p) = make_float4(v[0], v[1], v[2], v[3]);
  *reinterpret_cast<float4*>(p + 4) = make_float4(v[4], v[5], v[6], v[7]);
}
__device__ inline void store_eight(bf16_t* p, const float (&v)[8]) {
  unsigned w[4];
#pragma unroll
  for (int e = 0; e < 4; ++e)
    w[e] = static_cast<unsigned>(bf16_bits_from_float(v[2 * e])) | (static_cast<unsigned>(bf16_bits_from_float(v[2 * e + 1])) << 16);
  *reinterpret_cast<uint4*>(p) = make_uint4(w[0], w[1], w[2], w[3]);
}

enum Following : int { kNothing = 0, kNorm = 1, kPrepared = 2 };

// The same for widths that are a multiple of 8 and at most 2,048 * CHUNKS, on 16-byte boundaries, the same bits -- and what reads
// the stream next, of the new x.  kNorm: its RMSNorm, out[r, :] = x[r, :] * rsqrt(mean(x[r]^2) + next_eps) * next_w.  kPrepared: what the
// streaming product that absorbs that norm takes instead, out[r, :] = x[r, :] * next_w in bfloat16 and ssq[r] = the sum of x[r]^2.
// A decode step's few rows leave a workgroup a row that does nothing but wait, so everything a row needs is asked for at once
// and held in registers: 8 rows of 2,048 in a step 4.4 to 5.0 us where two passes over the row took 7.6, and 4.7 with what the product after it
// takes, whose norm was a launch of 4.2 us (from a launch to the next in a graph 2.75 us, two passes 3.83).
// Every sum is taken in the order of the kernel whose place this takes, so that the choice of kernel moves no bit: y's
// by the threads of the kernel above (neighbouring elements in neighbouring threads: the row is turned through LDS), a
// norm's in the order of the norm kernel's own, a prepared one's in the order of the product that absorbs a norm (gemm_skinny.hip:
// one wave, a lane eight elements of each 512).
template <typename TY, typename TN, typename TO, int CHUNKS, int NEXT>
__global__ __launch_bounds__(kBlock) void rmsnorm_add_rows_kernel(float* __restrict__ x, const TY* __restrict__ y, const float* __restrict__ w,
                                                                  int hidden, float eps, const TN* __restrict__ next_w, TO* __restrict__ out,
                                                                  float* __restrict__ ssq, float next_eps) {
  __shared__ float scratch[2][16];
  __shared__ __align__(16) float turned[CHUNKS * kBlock * 8];
  const size_t at = static_cast<size_t>(blockIdx.x) * hidden;
  float yv[CHUNKS][8], xv[CHUNKS][8], wv[CHUNKS][8], nv[NEXT ? CHUNKS : 1][8];
#pragma unroll
  for (int c = 0; c < CHUNKS; ++c) {
    const int i = (c * kBlock + threadIdx.x) * 8;
#pragma unroll
    for (int e = 0; e < 8; ++e) yv[c][e] = 0.f;
    if (i < hidden) {
      load_eight(y + at + i, yv[c]);
      load_eight(x + at + i, xv[c]);
      load_eight(w + i, wv[c]);
      if constexpr (NEXT) load_eight(next_w + i, nv[c]);
    }
  }
#pragma unroll
  for (int c = 0; c < CHUNKS; ++c) store_eight(turned + (c * kBlock + threadIdx.x) * 8, yv[c]);
  __syncthreads();
  // (fmaf: of an unrolled sum the compiler may join the second product with the first instead of the other way round)
  float ss = 0.f;
#pragma unroll
  for (int j = 0; j < CHUNKS * 8; ++j) {
    const float v = turned[j * kBlock + threadIdx.x];          // (zeros beyond the row)
    ss = fmaf(v, v, ss);
  }
  const float scale = 1.0f / sqrtf(block_sum(ss, scratch[0]) / static_cast<float>(hidden) + eps);
  ss = 0.f;
#pragma unroll
  for (int c = 0; c < CHUNKS; ++c) {
    const int i = (c * kBlock + threadIdx.x) * 8;
    if (i >= hidden) continue;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      xv[c][e] += yv[c][e] * scale * wv[c][e];
      if constexpr (NEXT == kNorm) ss += xv[c][e] * xv[c][e];
    }
    store_eight(x + at + i, xv[c]);
    if constexpr (NEXT == kPrepared) {
      float o[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) o[e] = xv[c][e] * nv[c][e];
      store_eight(out + at + i, o);
      store_eight(turned + i, xv[c]);                          // (y has been summed)
    }
  }
  if constexpr (NEXT == kNorm) {
    const float next_scale = 1.0f / sqrtf(block_sum(ss, scratch[1]) / static_cast<float>(hidden) + next_eps);
#pragma unroll
    for (int c = 0; c < CHUNKS; ++c) {
      const int i = (c * kBlock + threadIdx.x) * 8;
      if (i >= hidden) continue;
      float o[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) o[e] = xv[c][e] * next_scale * nv[c][e];
      store_eight(out + at + i, o);
    }
  }
  if constexpr (NEXT == kPrepared) {
    __syncthreads();
    if (threadIdx.x >= kWave) return;
#pragma unroll
    for (int j = 0; j < CHUNKS * 4; ++j) {
      const int i = (j * kWave + threadIdx.x) * 8;
      if (i >= hidden) continue;
      float v[8];
      load_eight(turned + i, v);
      ss = add_squares(v, j > 0, ss);
    }
    ss = wave_sum(ss);
    if (threadIdx.x == 0) ssq[blockIdx.x] = ss;
  }
}

// What a streaming product that absorbs an RMSNorm takes (kPrepared above) of rows of the stream as they lie: out[r, :] = x[rows[r], :] * w in
// bfloat16 and ssq[r] = the row's sum of squares, in that product's order.  Every workgroup of the product that absorbs the norm itself stages all
// the rows again; wide outputs pay more for that than for this launch (ops.LinearPlan.norms_apart has both sides).  A wave a row: a row does
// nothing but wait, so eight pieces of 512 elements are asked for together, without a condition (those past the row are its first again).
template <typename TN>
__global__ __launch_bounds__(kWave) void rmsnorm_prepare_kernel(const float* __restrict__ x, const int32_t* __restrict__ rows,
                                                                const TN* __restrict__ w, bf16_t* __restrict__ out, float* __restrict__ ssq, int hidden) {
  constexpr int kAhead = 8, kPiece = kWave * 8;
  const float* xr = x + static_cast<size_t>(rows ? rows[blockIdx.x] : blockIdx.x) * hidden;
  bf16_t* to = out + static_cast<size_t>(blockIdx.x) * hidden;
  float ss = 0.f;
  for (int i0 = threadIdx.x * 8; i0 < hidden; i0 += kAhead * kPiece) {
    float xv[kAhead][8], wv[kAhead][8];
#pragma unroll
    for (int j = 0; j < kAhead; ++j) {
      const int i = i0 + j * kPiece < hidden ? i0 + j * kPiece : 0;
      load_eight(xr + i, xv[j]);
      load_eight(w + i, wv[j]);
    }
#pragma unroll
    for (int j = 0; j < kAhead; ++j) {
      const int i = i0 + j * kPiece;
      if (i >= hidden) continue;
      ss = add_squares(xv[j], i >= kPiece, ss);
      float o[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) o[e] = xv[j][e] * wv[j][e];
      store_eight(to + i, o);
    }
  }
  ss = wave_sum(ss);
  if (threadIdx.x == 0) ssq[blockIdx.x] = ss;
}

// An RMSNorm and the causal convolution that is added to it, for rows that are one request's only one of the step (a decode step):
// h = the norm of x[r] as the norm kernel leaves it, out[r] = h + (bias + sum_j w[j] tail[j] + w[TAPS - 1] h), and the request's tail
// moves on by h.  What the two kernels would compute, bit for bit; widths as above.  8 rows of 2,048: 4.5 us where the
// two took 11.5, the second of them four trips to memory one after the other.
// ADD: what the sublayer before left to be added comes first, x[r] += y[r] * rsqrt(mean(y[r]^2) + add_eps) * add_w (a launch of 4 us between
// two layers of a step that has next to nothing to do), in the order of rmsnorm_add_rows_kernel, the same bits.
struct AddFirst {
  const float* y;
  const float* w;
  float eps;
};
template <typename TN, typename T, int CHUNKS, int TAPS, bool ADD>
__global__ __launch_bounds__(kBlock) void rmsnorm_conv_rows_kernel(float* __restrict__ x, const TN* __restrict__ norm_w, float eps,
                                                                   const float* __restrict__ w, const float* __restrict__ bias,
                                                                   T* __restrict__ out, T* __restrict__ state,
                                                                   const int32_t* __restrict__ slots, int hidden, const AddFirst add) {
  __shared__ float scratch[16];
  const size_t at = static_cast<size_t>(blockIdx.x) * hidden;
  T* tail = state + static_cast<size_t>(slots[blockIdx.x]) * (TAPS - 1) * hidden;
  float xv[CHUNKS][8], nv[CHUNKS][8], tv[CHUNKS][TAPS - 1][8], wv[CHUNKS][TAPS][8], bv[CHUNKS][8];
#pragma unroll
  for (int c = 0; c < CHUNKS; ++c) {
    const int i = (c * kBlock + threadIdx.x) * 8;
#pragma unroll
    for (int e = 0; e < 8; ++e) xv[c][e] = bv[c][e] = 0.f;
    if (i < hidden) {
      load_eight(x + at + i, xv[c]);
      load_eight(norm_w + i, nv[c]);
#pragma unroll
      for (int j = 0; j < TAPS; ++j) load_eight(w + static_cast<size_t>(j) * hidden + i, wv[c][j]);
#pragma unroll
      for (int j = 0; j < TAPS - 1; ++j) load_eight(tail + static_cast<size_t>(j) * hidden + i, tv[c][j]);
      if (bias != nullptr) load_eight(bias + i, bv[c]);
    }
  }
  if constexpr (ADD) {
    __shared__ float add_scratch[16];
    __shared__ __align__(16) float turned[CHUNKS * kBlock * 8];
    float yv[CHUNKS][8], av[CHUNKS][8];
#pragma unroll
    for (int c = 0; c < CHUNKS; ++c) {
      const int i = (c * kBlock + threadIdx.x) * 8;
#pragma unroll
      for (int e = 0; e < 8; ++e) yv[c][e] = av[c][e] = 0.f;
      if (i < hidden) {
        load_eight(add.y + at + i, yv[c]);
        load_eight(add.w + i, av[c]);
      }
    }
#pragma unroll
    for (int c = 0; c < CHUNKS; ++c) store_eight(turned + (c * kBlock + threadIdx.x) * 8, yv[c]);
    __syncthreads();
    float sq = 0.f;
#pragma unroll
    for (int j = 0; j < CHUNKS * 8; ++j) {
      const float v = turned[j * kBlock + threadIdx.x];        // (zeros beyond the row)
      sq = fmaf(v, v, sq);
    }
    const float by = 1.0f / sqrtf(block_sum(sq, add_scratch) / static_cast<float>(hidden) + add.eps);
#pragma unroll
    for (int c = 0; c < CHUNKS; ++c) {
      const int i = (c * kBlock + threadIdx.x) * 8;
      if (i >= hidden) continue;
#pragma unroll
      for (int e = 0; e < 8; ++e) xv[c][e] += yv[c][e] * by * av[c][e];
      store_eight(x + at + i, xv[c]);
    }
  }
  float ss = 0.f;
#pragma unroll
  for (int c = 0; c < CHUNKS; ++c)
#pragma unroll
    for (int e = 0; e < 8; ++e) ss += xv[c][e] * xv[c][e];
  const float scale = 1.0f / sqrtf(block_sum(ss, scratch) / static_cast<float>(hidden) + eps);
#pragma unroll
  for (int c = 0; c < CHUNKS; ++c) {
    // (h is a number of its own, as it is when it goes through memory: its product joins no later addition)
#pragma clang fp contract(off)
    const int i = (c * kBlock + threadIdx.x) * 8;
    if (i >= hidden) continue;
    float h[8], o[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      h[e] = to_float(from_float<T>(xv[c][e] * scale * nv[c][e]));
      float acc = bv[c][e];
#pragma unroll
      for (int j = 0; j < TAPS - 1; ++j) acc = fmaf(wv[c][j][e], tv[c][j][e], acc);
      o[e] = fmaf(wv[c][TAPS - 1][e], h[e], acc) + h[e];
    }
    store_eight(out + at + i, o);
#pragma unroll
    for (int j = 0; j + 1 < TAPS - 1; ++j) store_eight(tail + static_cast<size_t>(j) * hidden + i, tv[c][j + 1]);
    store_eight(tail + static_cast<size_t>(TAPS - 2) * hidden + i, h);
  }
}

template <typename T>
__global__ void xielu_kernel(const T* __restrict__ in, T* __restrict__ out, const float* __restrict__ pq, long total) {
  const float ap = softplus_f(pq[0]), aq = 0.5f + softplus_f(pq[1]);
  const long stride = static_cast<long>(blockDim.x) * gridDim.x;
  for (long i = blockIdx.x * static_cast<long>(blockDim.x) + threadIdx.x; i < total; i += stride) {
    const float z = to_float(in[i]);
    out[i] = from_float<T>(xielu_f(z, ap, aq));
  }
}

// The same, eight elements a thread in pieces of 16 bytes (bfloat16), for sizes that are whole pieces.
__global__ void xielu_pieces_kernel(const uint4* __restrict__ in, uint4* __restrict__ out, const float* __restrict__ pq, long pieces) {
  const float ap = softplus_f(pq[0]), aq = 0.5f + softplus_f(pq[1]);
  const long stride = static_cast<long>(blockDim.x) * gridDim.x;
  for (long i = blockIdx.x * static_cast<long>(blockDim.x) + threadIdx.x; i < pieces; i += stride) {
    const uint4 v = in[i];
    unsigned w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      float z[2] = {__uint_as_float(w[e] << 16), __uint_as_float(w[e] & 0xffff0000u)};
#pragma unroll
      for (int j = 0; j < 2; ++j) z[j] = xielu_f(z[j], ap, aq);
      w[e] = static_cast<unsigned>(bf16_bits_from_float(z[0])) | (static_cast<unsigned>(bf16_bits_from_float(z[1])) << 16);
    }
    out[i] = make_uint4(w[0], w[1], w[2], w[3]);
  }
}

// out[t, i] = g sigmoid(slope g) (u + 1) with g = min(gate, limit), u = clamp(up, -limit, limit); gu [T, 2 I]: a row's
// gates, then its ups.
template <typename T>
__global__ void clamped_glu_kernel(const T* __restrict__ gu, T* __restrict__ out, float limit, float slope, long total, int inter) {
  const long stride = static_cast<long>(blockDim.x) * gridDim.x;
  for (long i = blockIdx.x * static_cast<long>(blockDim.x) + threadIdx.x; i < total; i += stride) {
    const long r = i / inter;
    const int c = static_cast<int>(i - r * inter);
    const float g = fminf(to_float(gu[r * 2 * inter + c]), limit);
    const float u = fminf(fmaxf(to_float(gu[r * 2 * inter + inter + c]), -limit), limit);
    out[i] = from_float<T>(g / (1.0f + expf(-slope * g)) * (u + 1.0f));
  }
}

// The same for bfloat16 and I a multiple of 8: a thread takes eight neighbouring outputs, in pieces of 16 bytes.
__global__ void clamped_glu_pieces_kernel(const bf16_t* __restrict__ gu, bf16_t* __restrict__ out, float limit, float slope,
                                          long pieces, int inter) {
  const int per_row = inter / 8;
  const long stride = static_cast<long>(blockDim.x) * gridDim.x;
  for (long i = blockIdx.x * static_cast<long>(blockDim.x) + threadIdx.x; i < pieces; i += stride) {
    const long r = i / per_row;
    const int c = static_cast<int>(i - r * per_row) * 8;
    const uint4 gv = *reinterpret_cast<const uint4*>(gu + r * 2 * inter + c);
    const uint4 uv = *reinterpret_cast<const uint4*>(gu + r * 2 * inter + inter + c);
    const unsigned gw[4] = {gv.x, gv.y, gv.z, gv.w}, uw[4] = {uv.x, uv.y, uv.z, uv.w};
    unsigned o[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      float res[2];
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const float g = fminf(__uint_as_float(j ? gw[e] & 0xffff0000u : gw[e] << 16), limit);
        const float u = fminf(fmaxf(__uint_as_float(j ? uw[e] & 0xffff0000u : uw[e] << 16), -limit), limit);
        res[j] = g / (1.0f + expf(-slope * g)) * (u + 1.0f);
      }
      o[e] = static_cast<unsigned>(bf16_bits_from_float(res[0])) | (static_cast<unsigned>(bf16_bits_from_float(res[1])) << 16);
    }
    *reinterpret_cast<uint4*>(out + r * inter + c) = make_uint4(o[0], o[1], o[2], o[3]);
  }
}

// z Phi(z), the exact gelu: 0.5 z (1 + erf(z / sqrt 2)).
template <typename T>
__global__ void gelu_kernel(const T* __restrict__ in, T* __restrict__ out, long total) {
  const long stride = static_cast<long>(blockDim.x) * gridDim.x;
  for (long i = blockIdx.x * static_cast<long>(blockDim.x) + threadIdx.x; i < total; i += stride) {
    const float z = to_float(in[i]);
    out[i] = from_float<T>(0.5f * z * (1.0f + erff(z * 0.70710678118654752440f)));
  }
}

// max(z, 0)^2, element by element; PIECE elements a thread (16 bytes; 1: any count).
template <typename T, int PIECE>
__global__ void squared_relu_kernel(const T* in, T* out, long total) {      // (out may be in)
  const long stride = static_cast<long>(blockDim.x) * gridDim.x * PIECE;
  for (long i = (blockIdx.x * static_cast<long>(blockDim.x) + threadIdx.x) * PIECE; i < total; i += stride) {
    __align__(16) T piece[PIECE];
    if (PIECE == 1) piece[0] = in[i];
    else *reinterpret_cast<uint4*>(piece) = *reinterpret_cast<const uint4*>(in + i);
#pragma unroll
    for (int e = 0; e < PIECE; ++e) {
      const float z = fmaxf(to_float(piece[e]), 0.f);
      piece[e] = from_float<T>(z * z);
    }
    if (PIECE == 1) out[i] = piece[0];
    else *reinterpret_cast<uint4*>(out + i) = *reinterpret_cast<const uint4*>(piece);
  }
}

// z = cap tanh(z / cap) in place, four elements a thread (V 1: any count).
template <int V>
__global__ void softcap_kernel(float* __restrict__ z, float cap, long total) {
  const float inv = 1.0f / cap;
  const long stride = static_cast<long>(blockDim.x) * gridDim.x * V;
  for (long i = (blockIdx.x * static_cast<long>(blockDim.x) + threadIdx.x) * V; i < total; i += stride) {
    if (V == 4) {
      const float4 v = *reinterpret_cast<const float4*>(z + i);
      *reinterpret_cast<float4*>(z + i) = make_float4(cap * tanhf(v.x * inv), cap * tanhf(v.y * inv), cap * tanhf(v.z * inv),
                                                      cap * tanhf(v.w * inv));
    } else {
      z[i] = cap * tanhf(z[i] * inv);
    }
  }
}

int grid_for(long total) {
  const long g = (total + kBlock - 1) / kBlock;
  return static_cast<int>(g < 1 ? 1 : (g > 65535 ? 65535 : g));
}

// out[t] = h[t] + (h[t - 1] - h[t]) * mix with h = (x * rsqrt(mean(x^2) + eps) * w rounded to the output's type): an RMS
// norm and the token shift behind it in one pass.  A workgroup is one row; it works out the row before once more from
// the stream (that row is in the cache) instead of waiting for it.  A request's first row of the step reads its state
// (the h of its last row so far; zeros when it was admitted), and the same workgroup -- so nobody reads what another
// writes -- leaves the h of the request's last row of this step there.  V elements a thread and trip (4 where the width
// and the addresses allow: 16-byte loads, all of a pass in flight together).
template <int V> struct Pack { float v[V]; };
template <int V> __device__ inline Pack<V> load_pack(const float* p) {
  Pack<V> r;
  if (V == 4) { const float4 f = *reinterpret_cast<const float4*>(p); r.v[0] = f.x, r.v[1 % V] = f.y, r.v[2 % V] = f.z, r.v[3 % V] = f.w; }
  else r.v[0] = p[0];
  return r;
}
template <int V> __device__ inline Pack<V> load_pack(const bf16_t* p) {
  Pack<V> r;
  if (V == 4) {
    const uint2 b = *reinterpret_cast<const uint2*>(p);
    r.v[0] = __uint_as_float(b.x << 16), r.v[1 % V] = __uint_as_float(b.x & 0xffff0000u);
    r.v[2 % V] = __uint_as_float(b.y << 16), r.v[3 % V] = __uint_as_float(b.y & 0xffff0000u);
  } else r.v[0] = to_float(p[0]);
  return r;
}
template <int V> __device__ inline void store_pack(float* p, const Pack<V>& r) {
  if (V == 4) *reinterpret_cast<float4*>(p) = make_float4(r.v[0], r.v[1 % V], r.v[2 % V], r.v[3 % V]);
  else p[0] = r.v[0];
}
template <int V> __device__ inline void store_pack(bf16_t* p, const Pack<V>& r) {
  if (V == 4) {
    uint2 b;
    b.x = bf16_bits_from_float(r.v[0]) | (static_cast<uint32_t>(bf16_bits_from_float(r.v[1 % V])) << 16);
    b.y = bf16_bits_from_float(r.v[2 % V]) | (static_cast<uint32_t>(bf16_bits_from_float(r.v[3 % V])) << 16);
    *reinterpret_cast<uint2*>(p) = b;
  } else p[0] = from_float<bf16_t>(r.v[0]);
}

template <typename TO, int V>
__global__ __launch_bounds__(kBlock) void rmsnorm_shift_kernel(const float* __restrict__ x, const float* __restrict__ w,
                                                               const float* __restrict__ mix, TO* __restrict__ out,
                                                               TO* __restrict__ state, const int32_t* __restrict__ row_seq,
                                                               const int32_t* __restrict__ seq_start,
                                                               const int32_t* __restrict__ seq_slots, int hidden, float eps) {
  __shared__ float scratch[3][16];
  const int row = blockIdx.x, seq = row_seq[row];
  const int first = seq_start[seq], last = seq_start[seq + 1] - 1;
  const bool from_state = row == first;                     // (the same for every thread of the workgroup)
  const float* xr = x + static_cast<size_t>(row) * hidden;
  const float* xo = from_state ? x + static_cast<size_t>(last) * hidden : xr - hidden;   // the other row this workgroup norms
  const bool other = !from_state || last != row;
  float ss = 0.f, so = 0.f;
#pragma unroll 4
  for (int i = V * threadIdx.x; i < hidden; i += V * kBlock) {
    const Pack<V> a = load_pack<V>(xr + i), b = other ? load_pack<V>(xo + i) : a;
#pragma unroll
    for (int e = 0; e < V; ++e) ss = fmaf(a.v[e], a.v[e], ss), so = fmaf(b.v[e], b.v[e], so);
  }
  const float rs = 1.0f / sqrtf(block_sum(ss, scratch[0]) / static_cast<float>(hidden) + eps);
  const float ro = 1.0f / sqrtf(block_sum(so, scratch[1]) / static_cast<float>(hidden) + eps);
  TO* st = state + static_cast<size_t>(seq_slots[seq]) * hidden;
  TO* orow = out + static_cast<size_t>(row) * hidden;
#pragma unroll 4
  for (int i = V * threadIdx.x; i < hidden; i += V * kBlock) {
    const Pack<V> a = load_pack<V>(xr + i), b = other ? load_pack<V>(xo + i) : a, wi = load_pack<V>(w + i), mi = load_pack<V>(mix + i);
    Pack<V> before, h, o, keep;
    if (from_state) before = load_pack<V>(st + i);
#pragma unroll
    for (int e = 0; e < V; ++e) {
      h.v[e] = to_float(from_float<TO>(a.v[e] * rs * wi.v[e]));
      const float ho = to_float(from_float<TO>(b.v[e] * ro * wi.v[e]));      // the row before, or the request's last
      if (!from_state) before.v[e] = ho;
      o.v[e] = fmaf(before.v[e] - h.v[e], mi.v[e], h.v[e]);
      keep.v[e] = ho;
    }
    if (from_state) store_pack<V>(st + i, keep);
    store_pack<V>(orow + i, o);
  }
}

}  // namespace
}  // namespace bc4g

using namespace bc4g;

namespace bc4g {
namespace {
bool on_16(const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; }
}  // namespace
}  // namespace bc4g

extern "C" int bc4g_rmsnorm_add(float* x, const void* y, int y_dtype, const float* w, const void* next_w, int next_w_dtype, float next_eps,
                                void* out, int out_dtype, float* ssq, int n_rows, int hidden, float eps, void* stream) {
  BC4G_REQUIRE(n_rows >= 0 && hidden > 0 && x && y && w && !next_w == !out, "rmsnorm_add: bad arguments rows=%d H=%d", n_rows, hidden);
  BC4G_REQUIRE((y_dtype == kF32 || y_dtype == kBF16) && (!out || ((next_w_dtype == kF32 || next_w_dtype == kBF16) && (out_dtype == kF32 || out_dtype == kBF16))),
               "rmsnorm_add: unknown dtypes y=%d next=%d out=%d", y_dtype, next_w_dtype, out_dtype);
  BC4G_REQUIRE(!ssq || (out && out_dtype == kBF16), "rmsnorm_add: a prepared norm is bfloat16 rows and their sums of squares");
  const bool rows = hidden % 8 == 0 && hidden <= 8192 && on_16(x) && on_16(y) && on_16(w) && on_16(next_w) && on_16(out);
  BC4G_REQUIRE(!out || rows, "rmsnorm_add: the norm after it takes widths of a multiple of 8 up to 8192 on 16-byte boundaries (H=%d)", hidden);
  if (n_rows == 0) return 0;
  hipStream_t s = static_cast<hipStream_t>(stream);
  // (a narrow row leaves most threads of the one without an element: 8 rows of 64 2.24 us by the scalar kernel, 2.49 held in registers;
  // at 512 they are level, 2.57, and 8 rows of 2,048 take 3.83 and 2.75; from a launch to the next in a graph)
  if (!rows || (!out && hidden < 512)) {
    if (y_dtype == kF32) rmsnorm_add_kernel<float><<<n_rows, kBlock, 0, s>>>(x, static_cast<const float*>(y), w, hidden, eps);
    else rmsnorm_add_kernel<bf16_t><<<n_rows, kBlock, 0, s>>>(x, static_cast<const bf16_t*>(y), w, hidden, eps);
    return check_launch("rmsnorm_add");
  }
  const int chunks = (hidden + 2047) / 2048;
#define BC4G_ADD_ROWS(TY, TN, TO, C, NEXT)                                                                                              \
  rmsnorm_add_rows_kernel<TY, TN, TO, C, NEXT><<<n_rows, kBlock, 0, s>>>(x, static_cast<const TY*>(y), w, hidden, eps,                 \
                                                                         static_cast<const TN*>(next_w), static_cast<TO*>(out), ssq, next_eps)
#define BC4G_ADD(TY, TN, TO, NEXT)                                   \
  do {                                                               \
    if (chunks == 1) BC4G_ADD_ROWS(TY, TN, TO, 1, NEXT);             \
    else if (chunks == 2) BC4G_ADD_ROWS(TY, TN, TO, 2, NEXT);        \
    else BC4G_ADD_ROWS(TY, TN, TO, 4, NEXT);                         \
  } while (0)
#define BC4G_ADD_NEXT(TY)                                                                   \
  do {                                                                                      \
    if (!out) BC4G_ADD(TY, float, float, kNothing);                                         \
    else if (ssq && next_w_dtype == kF32) BC4G_ADD(TY, float, bf16_t, kPrepared);           \
    else if (ssq) BC4G_ADD(TY, bf16_t, bf16_t, kPrepared);                                  \
    else if (next_w_dtype == kF32 && out_dtype == kF32) BC4G_ADD(TY, float, float, kNorm);  \
    else if (next_w_dtype == kF32) BC4G_ADD(TY, float, bf16_t, kNorm);                      \
    else if (out_dtype == kF32) BC4G_ADD(TY, bf16_t, float, kNorm);                         \
    else BC4G_ADD(TY, bf16_t, bf16_t, kNorm);                                               \
  } while (0)
  if (y_dtype == kF32) BC4G_ADD_NEXT(float);
  else BC4G_ADD_NEXT(bf16_t);
#undef BC4G_ADD_NEXT
#undef BC4G_ADD
#undef BC4G_ADD_ROWS
  return check_launch("rmsnorm_add");
}

extern "C" int bc4g_rmsnorm_prepare(const float* x, const int32_t* rows, const void* w, int w_dtype, void* out, float* ssq, int n_rows, int hidden,
                                    void* stream) {
  BC4G_REQUIRE(n_rows >= 0 && hidden > 0 && hidden % 8 == 0 && x && w && out && ssq && on_16(x) && on_16(w) && on_16(out),
               "rmsnorm_prepare: bad arguments rows=%d H=%d (a multiple of 8, everything on 16-byte boundaries)", n_rows, hidden);
  BC4G_REQUIRE(w_dtype == kF32 || w_dtype == kBF16, "rmsnorm_prepare: unknown dtype %d of the scale", w_dtype);
  if (n_rows == 0) return 0;
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (w_dtype == kF32) rmsnorm_prepare_kernel<float><<<n_rows, kWave, 0, s>>>(x, rows, static_cast<const float*>(w), static_cast<bf16_t*>(out), ssq, hidden);
  else rmsnorm_prepare_kernel<bf16_t><<<n_rows, kWave, 0, s>>>(x, rows, static_cast<const bf16_t*>(w), static_cast<bf16_t*>(out), ssq, hidden);
  return check_launch("rmsnorm_prepare");
}

extern "C" int bc4g_rmsnorm_conv(float* x, const float* add_y, const float* add_w, float add_eps, const void* norm_w, int norm_w_dtype, float eps,
                                 const float* w, const float* bias, void* out, void* state, int dtype, const int32_t* slots, int n_rows, int hidden,
                                 int taps, void* stream) {
  BC4G_REQUIRE(n_rows >= 0 && hidden > 0 && hidden % 8 == 0 && hidden <= 4096 && taps >= 2 && taps <= 4,
               "rmsnorm_conv: rows=%d of H=%d (a multiple of 8, at most 4096) with %d taps (2 to 4)", n_rows, hidden, taps);
  BC4G_REQUIRE(x && norm_w && w && out && state && slots && on_16(x) && on_16(norm_w) && on_16(w) && on_16(bias) && on_16(out) && on_16(state),
               "rmsnorm_conv: a tensor is missing, or not on a 16-byte boundary");
  BC4G_REQUIRE(!add_y == !add_w && on_16(add_y) && on_16(add_w), "rmsnorm_conv: what is added first is rows and their norm's scale, on 16-byte boundaries");
  BC4G_REQUIRE((norm_w_dtype == kF32 || norm_w_dtype == kBF16) && (dtype == kF32 || dtype == kBF16), "rmsnorm_conv: unknown dtypes w=%d out=%d", norm_w_dtype, dtype);
  if (n_rows == 0) return 0;
  hipStream_t s = static_cast<hipStream_t>(stream);
  const AddFirst add{add_y, add_w, add_eps};
#define BC4G_NORM_CONV_ADD(TN, T, C, TAPS, ADD)                                                                                            \
  rmsnorm_conv_rows_kernel<TN, T, C, TAPS, ADD><<<n_rows, kBlock, 0, s>>>(x, static_cast<const TN*>(norm_w), eps, w, bias, static_cast<T*>(out), \
                                                                          static_cast<T*>(state), slots, hidden, add)
#define BC4G_NORM_CONV(TN, T, C, TAPS)                         \
  do {                                                         \
    if (add_y) BC4G_NORM_CONV_ADD(TN, T, C, TAPS, true);       \
    else BC4G_NORM_CONV_ADD(TN, T, C, TAPS, false);            \
  } while (0)
#define BC4G_NORM_TAPS(TN, T, C)                       \
  do {                                                 \
    if (taps == 2) BC4G_NORM_CONV(TN, T, C, 2);        \
    else if (taps == 3) BC4G_NORM_CONV(TN, T, C, 3);   \
    else BC4G_NORM_CONV(TN, T, C, 4);                  \
  } while (0)
#define BC4G_NORM_WIDTH(TN, T)                         \
  do {                                                 \
    if (hidden <= 2048) BC4G_NORM_TAPS(TN, T, 1);      \
    else BC4G_NORM_TAPS(TN, T, 2);                     \
  } while (0)
  if (norm_w_dtype == kF32 && dtype == kF32) BC4G_NORM_WIDTH(float, float);
  else if (norm_w_dtype == kF32) BC4G_NORM_WIDTH(float, bf16_t);
  else if (dtype == kF32) BC4G_NORM_WIDTH(bf16_t, float);
  else BC4G_NORM_WIDTH(bf16_t, bf16_t);
#undef BC4G_NORM_WIDTH
#undef BC4G_NORM_TAPS
#undef BC4G_NORM_CONV
#undef BC4G_NORM_CONV_ADD
  return check_launch("rmsnorm_conv");
}

extern "C" int bc4g_xielu(const void* in, void* out, int dtype, const float* pq, long total, void* stream) {
  BC4G_REQUIRE(total >= 0 && in && out && pq, "xielu: bad arguments (%ld elements)", total);
  if (total == 0) return 0;
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (dtype == kF32) xielu_kernel<float><<<grid_for(total), kBlock, 0, s>>>(static_cast<const float*>(in), static_cast<float*>(out), pq, total);
  else if (dtype == kBF16 && total % 8 == 0 && reinterpret_cast<uintptr_t>(in) % 16 == 0 && reinterpret_cast<uintptr_t>(out) % 16 == 0)
    xielu_pieces_kernel<<<grid_for(total / 8), kBlock, 0, s>>>(static_cast<const uint4*>(in), static_cast<uint4*>(out), pq, total / 8);
  else if (dtype == kBF16) xielu_kernel<bf16_t><<<grid_for(total), kBlock, 0, s>>>(static_cast<const bf16_t*>(in), static_cast<bf16_t*>(out), pq, total);
  else return fail("xielu: unknown dtype %d", dtype);
  return check_launch("xielu");
}

extern "C" int bc4g_clamped_glu(const void* gu, void* out, int dtype, float limit, float slope, int n_rows, int inter, void* stream) {
  BC4G_REQUIRE(n_rows >= 0 && inter > 0 && gu && out && gu != out, "clamped_glu: bad arguments rows=%d I=%d", n_rows, inter);
  if (n_rows == 0) return 0;
  hipStream_t s = static_cast<hipStream_t>(stream);
  const long total = static_cast<long>(n_rows) * inter;
  if (dtype == kF32) clamped_glu_kernel<float><<<grid_for(total), kBlock, 0, s>>>(static_cast<const float*>(gu), static_cast<float*>(out), limit, slope, total, inter);
  else if (dtype == kBF16 && inter % 8 == 0 && reinterpret_cast<uintptr_t>(gu) % 16 == 0 && reinterpret_cast<uintptr_t>(out) % 16 == 0)
    clamped_glu_pieces_kernel<<<grid_for(total / 8), kBlock, 0, s>>>(static_cast<const bf16_t*>(gu), static_cast<bf16_t*>(out), limit, slope, total / 8, inter);
  else if (dtype == kBF16) clamped_glu_kernel<bf16_t><<<grid_for(total), kBlock, 0, s>>>(static_cast<const bf16_t*>(gu), static_cast<bf16_t*>(out), limit, slope, total, inter);
  else return fail("clamped_glu: unknown dtype %d", dtype);
  return check_launch("clamped_glu");
}

extern "C" int bc4g_gelu(const void* in, void* out, int dtype, long total, void* stream) {
  BC4G_REQUIRE(total >= 0 && in && out, "gelu: bad arguments total=%ld", total);
  if (total == 0) return 0;
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (dtype == kF32) gelu_kernel<float><<<grid_for(total), kBlock, 0, s>>>(static_cast<const float*>(in), static_cast<float*>(out), total);
  else if (dtype == kBF16) gelu_kernel<bf16_t><<<grid_for(total), kBlock, 0, s>>>(static_cast<const bf16_t*>(in), static_cast<bf16_t*>(out), total);
  else return fail("gelu: unknown dtype %d", dtype);
  return check_launch("gelu");
}

extern "C" int bc4g_squared_relu(const void* in, void* out, int dtype, long total, void* stream) {
  BC4G_REQUIRE(total >= 0 && in && out, "squared_relu: bad arguments (%ld elements)", total);
  if (total == 0) return 0;
  hipStream_t s = static_cast<hipStream_t>(stream);
  const int piece = dtype == kF32 ? 4 : 8;      // elements in 16 bytes
  const bool pieces = total % piece == 0 && reinterpret_cast<uintptr_t>(in) % 16 == 0 && reinterpret_cast<uintptr_t>(out) % 16 == 0;
#define BC4G_RELU2(T, P) \
  squared_relu_kernel<T, P><<<grid_for(total / P), kBlock, 0, s>>>(static_cast<const T*>(in), static_cast<T*>(out), total)
  if (dtype == kF32) { if (pieces) BC4G_RELU2(float, 4); else BC4G_RELU2(float, 1); }
  else if (dtype == kBF16) { if (pieces) BC4G_RELU2(bf16_t, 8); else BC4G_RELU2(bf16_t, 1); }
  else return fail("squared_relu: unknown dtype %d", dtype);
#undef BC4G_RELU2
  return check_launch("squared_relu");
}

extern "C" int bc4g_softcap(float* z, float cap, long total, void* stream) {
  BC4G_REQUIRE(total >= 0 && z && cap > 0.f, "softcap: bad arguments (%ld elements, cap %g)", total, cap);
  if (total == 0) return 0;
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (total % 4 == 0 && reinterpret_cast<uintptr_t>(z) % 16 == 0) softcap_kernel<4><<<grid_for(total / 4), kBlock, 0, s>>>(z, cap, total);
  else softcap_kernel<1><<<grid_for(total), kBlock, 0, s>>>(z, cap, total);
  return check_launch("softcap");
}

extern "C" int bc4g_rmsnorm_shift(const float* x, const float* w, const float* mix, void* out, void* state, int dtype,
                                  const int32_t* row_seq, const int32_t* seq_start, const int32_t* seq_slots, int n_rows,
                                  int hidden, float eps, void* stream) {
  BC4G_REQUIRE(n_rows >= 0 && hidden > 0 && x && w && mix && out && state && row_seq && seq_start && seq_slots,
               "rmsnorm_shift: bad arguments rows=%d H=%d", n_rows, hidden);
  if (n_rows == 0) return 0;
  hipStream_t s = static_cast<hipStream_t>(stream);
  const bool four = hidden % 4 == 0 && reinterpret_cast<uintptr_t>(x) % 16 == 0 && reinterpret_cast<uintptr_t>(w) % 16 == 0 &&
                    reinterpret_cast<uintptr_t>(mix) % 16 == 0 && reinterpret_cast<uintptr_t>(out) % 16 == 0 &&
                    reinterpret_cast<uintptr_t>(state) % 16 == 0;
#define BC4G_SHIFT(T, V)                                                                                                    \
  rmsnorm_shift_kernel<T, V><<<n_rows, kBlock, 0, s>>>(x, w, mix, static_cast<T*>(out), static_cast<T*>(state), row_seq, seq_start, \
                                                      seq_slots, hidden, eps)
  if (dtype == kF32) { if (four) BC4G_SHIFT(float, 4); else BC4G_SHIFT(float, 1); }
  else if (dtype == kBF16) { if (four) BC4G_SHIFT(bf16_t, 4); else BC4G_SHIFT(bf16_t, 1); }
  else return fail("rmsnorm_shift: unknown dtype %d", dtype);
#undef BC4G_SHIFT
  return check_launch("rmsnorm_shift");
}
