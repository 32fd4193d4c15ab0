// GroupNorm over a spatially sharded input: the per-(sample, group) partial sums that
// the ranks add up, the normalise + affine pass, and the backward partials and pass.
// x is (N, C, S) contiguous (S = product of the local spatial extents); a group is
// C / G consecutive channels, so the elements of one (sample, group) are one contiguous
// span. Everything is HBM-bound: 16-byte loads, fp32 accumulation, block partials that a
// second small kernel adds up in a fixed order: the same call gives the same bits. (The one atomic, gn_resident_kernel's list,
// says which launch writes a chunk. Both write it by the same formulas, from the same statistics.)
//
// Passes over the tensor. Sharded: forward two (the moments of every group from ONE pass, centred on a
// sample of the block's own elements; normalise + affine), backward two (the sums; the input
// gradient), both from x and the statistics, x_hat recomputed in fp32 on the way. x_hat itself
// is only written for a caller that asks for it (jg_gn_apply with x_norm, jg_gn_partial_bwd,
// jg_gn_bwd_apply): it is rounded, and the backward is less exact from it. A step whose backward takes x
// keeps a copy of it (jg_gn_apply_keep, jg_gn_forward_keep), which the pass that writes y writes beside it: the caller
// may change x before the backward. A tensor that one rank holds whole is read once each way (gn_resident_kernel):
// 8 x 64 x 1024^2 bf16, 8 groups (1.07 GB a tensor), forward + backward 1.16 ms = 5.6 TB/s over six tensors, what a copy
// reaches; two launches each way that read it twice took 1.80 ms over nine. A second read out of the last-level
// cache is not what saves: both passes in one launch, the second one a few units behind, took 1.60 ms (that cache delivers
// 7 TB/s where memory delivers 6).
// Rows and spans start anywhere (S need not be a multiple of 8): a block takes the whole 16-byte
// words of its range as vectors and the elements before the first and behind the last one by one.
//
// Reference behaviour restated here:
//   jigsaw/modules/normalization/_functional.py:352-385 (forward: sum, centred squares, apply)
//   jigsaw/modules/normalization/_functional.py:431-468 (backward)
#include <algorithm>
#include <type_traits>

#include "jg_common.h"

namespace {

constexpr int kThreads = 256;
constexpr long long kChunk = 32768;  // elements a block reduces
constexpr int kMaxChunks = 64;

template <int DT>
struct Elem;
template <>
struct Elem<JG_F32> {
  typedef float T;
  static constexpr int VEC = 4;
  __device__ static __forceinline__ float up(float v) { return v; }
  __device__ static __forceinline__ float down(float v) { return v; }
};
template <>
struct Elem<JG_BF16> {
  typedef uint16_t T;
  static constexpr int VEC = 8;
  __device__ static __forceinline__ float up(uint16_t v) { return jg::bf16_to_f32(v); }
  __device__ static __forceinline__ uint16_t down(float v) { return __builtin_bit_cast(uint16_t, (__bf16)v); }
};
template <>
struct Elem<JG_F16> {
  typedef _Float16 T;
  static constexpr int VEC = 8;
  __device__ static __forceinline__ float up(_Float16 v) { return (float)v; }
  __device__ static __forceinline__ _Float16 down(float v) { return (_Float16)v; }
};

template <int DT>
struct alignas(16) Pack {
  typename Elem<DT>::T v[Elem<DT>::VEC];
};

template <int DT>
__device__ __forceinline__ void load_vec(const typename Elem<DT>::T* p, float out[Elem<DT>::VEC]) {
  const Pack<DT> q = *reinterpret_cast<const Pack<DT>*>(p);
#pragma unroll
  for (int t = 0; t < Elem<DT>::VEC; ++t) out[t] = Elem<DT>::up(q.v[t]);
}
template <int DT>
__device__ __forceinline__ void store_vec(typename Elem<DT>::T* p, const float in[Elem<DT>::VEC]) {
  Pack<DT> q;
#pragma unroll
  for (int t = 0; t < Elem<DT>::VEC; ++t) q.v[t] = Elem<DT>::down(in[t]);
  *reinterpret_cast<Pack<DT>*>(p) = q;
}

// The elements [lo, hi) of a tensor over the threads of a block: quad(i, step) for 4 vectors at i, i + step, ..
// (four loads in flight per thread), vec(i) for one, one(i) for single elements. vec_ok: the tensors start on 16 bytes.
template <int V, typename QUAD, typename VEC, typename ONE>
__device__ __forceinline__ void for_range(long long lo, long long hi, bool vec_ok, QUAD quad, VEC vec, ONE one) {
  long long b0 = (lo + V - 1) / V * V, b1 = hi / V * V;
  if (!vec_ok || b1 <= b0) b0 = b1 = hi;  // all of it one by one
  constexpr long long step = (long long)kThreads * V;
  long long i = b0 + (long long)threadIdx.x * V;
  for (; i + 3 * step < b1; i += 4 * step) quad(i, step);
  for (; i < b1; i += step) vec(i);
  for (long long j = lo + threadIdx.x; j < b0; j += kThreads) one(j);
  for (long long j = b1 + threadIdx.x; j < hi; j += kThreads) one(j);
}

// Sum of two per-thread values over the block, fixed order; valid in thread 0.
__device__ __forceinline__ void block_sum2(float& a, float& b) {
  __shared__ float red[2][kThreads / 64];
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    a += __shfl_xor(a, o, 64);
    b += __shfl_xor(b, o, 64);
  }
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if (lane == 0) {
    red[0][wave] = a;
    red[1][wave] = b;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    a = (red[0][0] + red[0][1]) + (red[0][2] + red[0][3]);
    b = (red[1][0] + red[1][1]) + (red[1][2] + red[1][3]);
  }
}

// Chunk b % chunks of unit b / chunks of `len` elements, as absolute element indices.
__device__ __forceinline__ void chunk_range(unsigned b, long long len, int chunks, long long chunk_len, long long* unit, long long* lo,
                                            long long* hi) {
  *unit = b / chunks;
  const long long from = (b % chunks) * chunk_len;
  *lo = *unit * len + (from < len ? from : len);
  *hi = *unit * len + (from + chunk_len < len ? from + chunk_len : len);
}

// The sums of MODE over the elements [lo, hi), valid in thread 0:
// MODE 0: a = sum x                      over a chunk of a (sample, group) span
// MODE 1: a = sum (x - m)^2              "
// MODE 2: a = sum g, b = sum g * y       over a chunk of a (sample, channel) row
// MODE 3: a = sum g, b = sum g * (y - m) * rs
template <int DT, int MODE>
__device__ __forceinline__ void chunk_sums(const typename Elem<DT>::T* __restrict__ x, const typename Elem<DT>::T* __restrict__ y, float m,
                                           float rs, long long lo, long long hi, bool vec_ok, float& a, float& b) {
  constexpr int V = Elem<DT>::VEC;
  a = b = 0.0f;
  auto add = [&](float v, float w) {
    if (MODE == 0) {
      a += v;
    } else if (MODE == 1) {
      const float d = v - m;
      a += d * d;
    } else {
      a += v;
      b += v * (MODE == 3 ? w - m : w);
    }
  };
  auto vecs = [&](long long i, long long step, auto count) {
    float v[count()][V], w[count()][V];
#pragma unroll
    for (int q = 0; q < count(); ++q) {
      load_vec<DT>(x + i + q * step, v[q]);
      if (MODE >= 2) load_vec<DT>(y + i + q * step, w[q]);
    }
#pragma unroll
    for (int q = 0; q < count(); ++q)
#pragma unroll
      for (int t = 0; t < V; ++t) add(v[q][t], MODE >= 2 ? w[q][t] : 0.0f);
  };
  for_range<V>(lo, hi, vec_ok, [&](long long i, long long step) { vecs(i, step, std::integral_constant<int, 4>{}); },
               [&](long long i) { vecs(i, 0, std::integral_constant<int, 1>{}); },
               [&](long long i) { add(Elem<DT>::up(x[i]), MODE >= 2 ? Elem<DT>::up(y[i]) : 0.0f); });
  block_sum2(a, b);
  if (MODE == 3) b *= rs;
}

// chunk_sums of chunk b % chunks of unit b / chunks (MODE 3: a unit is a row of the (sample, group) unit / channels_per_group).
// Partials at part[blockIdx.x * 2 + {0, 1}].
template <int DT, int MODE>
__global__ __launch_bounds__(kThreads) void gn_reduce_kernel(float* __restrict__ part,
                                                             const typename Elem<DT>::T* __restrict__ x,
                                                             const typename Elem<DT>::T* __restrict__ y,
                                                             const float* __restrict__ mean, const float* __restrict__ rstd,
                                                             int channels_per_group, long long len,
                                                             int chunks, long long chunk_len, bool vec_ok) {
  long long unit, lo, hi;
  chunk_range(blockIdx.x, len, chunks, chunk_len, &unit, &lo, &hi);
  const float m = MODE == 1 ? mean[unit] : MODE == 3 ? mean[unit / channels_per_group] : 0.0f;
  float a, b;
  chunk_sums<DT, MODE>(x, y, m, MODE == 3 ? rstd[unit / channels_per_group] : 1.0f, lo, hi, vec_ok, a, b);
  if (threadIdx.x == 0) {
    part[(size_t)blockIdx.x * 2 + 0] = a;
    part[(size_t)blockIdx.x * 2 + 1] = b;
  }
}

// Moments of the elements [lo, hi) in one pass: (mean, sum of squares about it), valid in thread 0. The sums are centred
// on the mean of the first (up to) 256 elements, so that the square of the mean does not swamp the variance.
template <int DT>
__device__ __forceinline__ float2 chunk_moments(const typename Elem<DT>::T* __restrict__ x, long long lo, long long hi, bool vec_ok) {
  constexpr int V = Elem<DT>::VEC;
  __shared__ float centre_s;
  const long long n = hi - lo;
  float first = (long long)threadIdx.x < n ? Elem<DT>::up(x[lo + threadIdx.x]) : 0.0f, none = 0.0f;
  block_sum2(first, none);
  if (threadIdx.x == 0) centre_s = n > 0 ? first / (float)(n < kThreads ? n : kThreads) : 0.0f;
  __syncthreads();
  const float centre = centre_s;
  float a = 0.0f, b = 0.0f;
  auto add = [&](float v) {
    const float d = v - centre;
    a += d;
    b += d * d;
  };
  auto vecs = [&](long long i, long long step, auto count) {
    float v[count()][V];
#pragma unroll
    for (int q = 0; q < count(); ++q) load_vec<DT>(x + i + q * step, v[q]);
#pragma unroll
    for (int q = 0; q < count(); ++q)
#pragma unroll
      for (int t = 0; t < V; ++t) add(v[q][t]);
  };
  for_range<V>(lo, hi, vec_ok, [&](long long i, long long step) { vecs(i, step, std::integral_constant<int, 4>{}); },
               [&](long long i) { vecs(i, 0, std::integral_constant<int, 1>{}); }, [&](long long i) { add(Elem<DT>::up(x[i])); });
  block_sum2(a, b);
  const float shift = n > 0 ? a / (float)n : 0.0f;
  return make_float2(centre + shift, n > 0 ? fmaxf(b - a * shift, 0.0f) : 0.0f);
}

// chunk_moments of chunk b % chunks of unit b / chunks
template <int DT>
__global__ __launch_bounds__(kThreads) void gn_moments_kernel(float* __restrict__ part, const typename Elem<DT>::T* __restrict__ x,
                                                              long long len, int chunks, long long chunk_len, bool vec_ok) {
  long long unit, lo, hi;
  chunk_range(blockIdx.x, len, chunks, chunk_len, &unit, &lo, &hi);
  const float2 v = chunk_moments<DT>(x, lo, hi, vec_ok);
  if (threadIdx.x == 0) {
    part[(size_t)blockIdx.x * 2 + 0] = v.x;
    part[(size_t)blockIdx.x * 2 + 1] = v.y;
  }
}

// The chunks' moments of a unit combined (one wavefront a unit, a lane a chunk, in double): mean, the centred square
// sum, and what a caller wants of count_sum = (count, sum) pairs and rstd = 1 / sqrt(sq / count + eps).
__global__ __launch_bounds__(64) void gn_moments_finish_kernel(float* mean, float* sq, float* count_sum, float* rstd,
                                                               const float* __restrict__ part, long long len, int chunks,
                                                               long long chunk_len, float eps) {
  const int u = blockIdx.x, k = threadIdx.x;
  double n = 0.0, m = 0.0, s = 0.0;
  if (k < chunks) {
    const long long from = k * chunk_len;
    n = (double)(from >= len ? 0 : from + chunk_len < len ? chunk_len : len - from);
    m = part[((size_t)u * chunks + k) * 2];
    s = part[((size_t)u * chunks + k) * 2 + 1];
  }
  auto total = [](double v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
  };
  const double mu = total(n * m) / (double)len, d = m - mu;
  const double all = total(s + n * d * d);
  if (k != 0) return;
  mean[u] = (float)mu;
  if (sq != nullptr) sq[u] = (float)all;
  if (rstd != nullptr) rstd[u] = 1.0f / sqrtf((float)(all / (double)len) + eps);
  if (count_sum != nullptr) {
    count_sum[2 * u] = (float)len;
    count_sum[2 * u + 1] = (float)(mu * (double)len);
  }
}
static_assert(kMaxChunks <= 64, "a lane per chunk");

// out0[u] (and out1[u]) = sum over the chunks of unit u, in chunk order
__global__ __launch_bounds__(kThreads) void gn_finish_kernel(float* __restrict__ out0, float* __restrict__ out1,
                                                             const float* __restrict__ part, long long units,
                                                             int chunks) {
  const long long u = (long long)blockIdx.x * kThreads + threadIdx.x;
  if (u >= units) return;
  float a = 0.0f, b = 0.0f;
  for (int k = 0; k < chunks; ++k) {
    a += part[((size_t)u * chunks + k) * 2 + 0];
    b += part[((size_t)u * chunks + k) * 2 + 1];
  }
  out0[u] = a;
  if (out1 != nullptr) out1[u] = b;
}

__device__ __forceinline__ void store_as(void* p, long long i, float v, int dtype) {
  if (dtype == JG_F32) static_cast<float*>(p)[i] = v;
  else if (dtype == JG_BF16) static_cast<uint16_t*>(p)[i] = jg::f32_to_bf16(v);
  else static_cast<_Float16*>(p)[i] = (_Float16)v;
}

// From the chunk partials (sum g, sum g * x_norm) of every row (n, c), a wavefront per result, fixed order:
//   blocks [0, N*G):       sums[n][grp] = (sum_c w[c] sum g, sum_c w[c] sum g * x_norm)
//   blocks [N*G, N*G + C): gb[c] = sum_n sum g, gw[c] = sum_n sum g * x_norm (dtype `wdtype`)
// sum0 / sum1: where the two sums of a group go, `stride` floats between groups.
template <int DT>
__global__ __launch_bounds__(64) void gn_bwd_finish_kernel(float* __restrict__ sum0, float* __restrict__ sum1, int stride,
                                                           void* gw, void* gb, int wdtype, const float* __restrict__ part,
                                                           const typename Elem<DT>::T* __restrict__ weight, long long N,
                                                           int C, int G, int chunks) {
  const int cpg = C / G;
  const bool group = blockIdx.x < N * G;
  const long long u = group ? blockIdx.x : blockIdx.x - N * G;
  const long long items = (group ? cpg : N) * (long long)chunks;  // (row, chunk) pairs of this result
  float s0 = 0.0f, s1 = 0.0f;
  for (long long i = threadIdx.x; i < items; i += 64) {
    const long long r = i / chunks, k = i - r * chunks;
    const long long row = group ? u * cpg + r : r * C + u;  // rows of a group are consecutive
    const float w = group && weight != nullptr ? Elem<DT>::up(weight[row % C]) : 1.0f;
    const float2 v = *reinterpret_cast<const float2*>(part + (row * chunks + k) * 2);
    s0 += w * v.x;
    s1 += w * v.y;
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    s0 += __shfl_xor(s0, o, 64);
    s1 += __shfl_xor(s1, o, 64);
  }
  if (threadIdx.x != 0) return;
  if (group) {
    sum0[u * stride] = s0;
    sum1[u * stride] = s1;
  } else {
    if (gb != nullptr) store_as(gb, u, s0, wdtype);
    if (gw != nullptr) store_as(gw, u, s1, wdtype);
  }
}

// What an apply pass reads and writes (a block: chunk b % chunks of row (n, c) = b / chunks)
struct ApplyArgs {
  void* out;         // y / gx
  void* out_norm;    // forward: x_norm, or NULL
  void* out_kept;    // forward: x once more, or NULL
  const void* in;    // x / g
  const void* in2;   // backward: x_norm (FROM_X: x)
  const float* mean; // forward and FROM_X
  const float* rstd;
  const float* gsum; // backward, `stride` floats between groups
  const float* gxsum;
  int stride;
  const float* cnt;  // backward: elements of every group, or NULL: `count` of each
  float count;
  const void* weight;
  const void* bias;
  int C, G;
};

// y and gx of an element, for every kernel that writes them. The fused products are spelled out: left to the compiler, two
// kernels may round the same expression differently, and which of two launches writes a chunk depends on timing.
// x_norm is rounded to the compute dtype and y computed from the rounded value, as the reference computes y from the x_norm tensor.
// fp16: `rounded` keeps the compiler from one instruction that multiplies, adds and rounds to 16 bits (v_fma_mixlo_f16), which it
// uses in one kernel and not in the other and which rounds once where fp32 and then fp16 round twice.
template <int DT>
__device__ __forceinline__ float rounded(float v) {
  if (DT == JG_F16) asm("" : "+v"(v));
  return v;
}
template <int DT>
__device__ __forceinline__ float normalised(float x, float m, float rs) {
  return Elem<DT>::up(Elem<DT>::down(rounded<DT>((x - m) * rs)));
}
template <int DT>
__device__ __forceinline__ float output(float x_norm, float w, float b) {
  return rounded<DT>(__builtin_fmaf(x_norm, w, b));
}
// rstd (g w - q1 - x_norm q2) with the factors of a row worked out beforehand: three roundings an element (relative error of
// an fp32 gradient 5.1e-8 where the terms one after the other gave 6.0e-8)
struct GradFactors {
  float g, d, one;
};
// from_x: elements d = x - mean, otherwise x_norm
__device__ __forceinline__ GradFactors grad_factors(float rs, float w, float q1, float q2, bool from_x) {
  return GradFactors{rs * w, from_x ? rs * (rs * q2) : rs * q2, rs * q1};
}
template <int DT>
__device__ __forceinline__ float input_gradient(float g, float d, const GradFactors& f) {
  return rounded<DT>(__builtin_fmaf(g, f.g, -__builtin_fmaf(d, f.d, f.one)));
}

// Forward:  x_norm = (x - mean) * rstd, y = x_norm * w[c] + b[c]
// Backward: gx = rstd * (g * w[c] - gsum / cnt - x_norm * gxsum / cnt); FROM_X: x_norm from x as in the forward, unrounded
// for the elements [lo, hi) of a row of channel c, with q1 = gsum / cnt, q2 = gxsum / cnt
template <int DT, bool BWD, bool FROM_X>
__device__ __forceinline__ void apply_range(const ApplyArgs& p, int c, float m, float rs, float q1, float q2, long long lo, long long hi, bool vec_ok) {
  typedef typename Elem<DT>::T T;
  constexpr int V = Elem<DT>::VEC;
  const float w = p.weight != nullptr ? Elem<DT>::up(static_cast<const T*>(p.weight)[c]) : 1.0f;
  const float bv = (!BWD && p.bias != nullptr) ? Elem<DT>::up(static_cast<const T*>(p.bias)[c]) : 0.0f;
  const T* in = static_cast<const T*>(p.in);
  const T* in2 = static_cast<const T*>(p.in2);
  T* out = static_cast<T*>(p.out);
  T* norm = static_cast<T*>(p.out_norm);
  T* kept = static_cast<T*>(p.out_kept);
  auto forward = [&](float v, float& xn) {  // (y, x_norm)
    xn = normalised<DT>(v, m, rs);
    return output<DT>(xn, w, bv);
  };
  const GradFactors f = grad_factors(rs, w, q1, q2, FROM_X);
  auto backward = [&](float g, float x) { return input_gradient<DT>(g, FROM_X ? x - m : x, f); };
  auto vecs = [&](long long i, long long step, auto count) {
    float v[count()][V], x[count()][V];
#pragma unroll
    for (int q = 0; q < count(); ++q) {
      load_vec<DT>(in + i + q * step, v[q]);
      if (BWD) load_vec<DT>(in2 + i + q * step, x[q]);
    }
#pragma unroll
    for (int q = 0; q < count(); ++q) {
      if (!BWD && kept != nullptr) store_vec<DT>(kept + i + q * step, v[q]);
#pragma unroll
      for (int t = 0; t < V; ++t) v[q][t] = BWD ? backward(v[q][t], x[q][t]) : forward(v[q][t], x[q][t]);
      if (!BWD && norm != nullptr) store_vec<DT>(norm + i + q * step, x[q]);
      store_vec<DT>(out + i + q * step, v[q]);
    }
  };
  for_range<V>(lo, hi, vec_ok, [&](long long i, long long step) { vecs(i, step, std::integral_constant<int, 4>{}); },
               [&](long long i) { vecs(i, 0, std::integral_constant<int, 1>{}); },
               [&](long long i) {
                 const float v = Elem<DT>::up(in[i]);
                 float xn = BWD ? Elem<DT>::up(in2[i]) : 0.0f;
                 const float r = BWD ? backward(v, xn) : forward(v, xn);
                 if (!BWD && norm != nullptr) norm[i] = Elem<DT>::down(xn);
                 if (!BWD && kept != nullptr) kept[i] = in[i];
                 out[i] = Elem<DT>::down(r);
               });
}

template <int DT, bool BWD, bool FROM_X>
__global__ __launch_bounds__(kThreads) void gn_apply_kernel(ApplyArgs p, long long S, int chunks, long long chunk_len, bool vec_ok) {
  long long row, lo, hi;
  // Last block first: the pass before read the tensors from front to back, so that their ends are what the last-level
  // cache still holds.
  chunk_range(gridDim.x - 1 - blockIdx.x, S, chunks, chunk_len, &row, &lo, &hi);
  const int c = (int)(row % p.C);
  const long long seg = row / p.C * p.G + c / (p.C / p.G);
  const float m = BWD && !FROM_X ? 0.0f : p.mean[seg], rs = p.rstd[seg];
  const float inv = BWD ? 1.0f / (p.cnt != nullptr ? p.cnt[seg] : p.count) : 0.0f;
  const float q1 = BWD ? p.gsum[seg * p.stride] * inv : 0.0f, q2 = BWD ? p.gxsum[seg * p.stride] * inv : 0.0f;
  apply_range<DT, BWD, FROM_X>(p, c, m, rs, q1, q2, lo, hi, vec_ok);
}

// ---- both passes over a tensor that one rank holds whole, in one launch, the tensor read once ----
// A block keeps a chunk of a row in registers, publishes the chunk's partials (forward: mean and centred squares; backward:
// the two sums), waits for those of the whole (sample, group) and writes its part of y or gx from the registers.
// The blocks of a unit do run at the same time on a chip that is free, and nothing depends on it: a wait ends after `polls`
// polls, the block then puts its chunk on a list and is gone, and a second launch, which finds every partial there, reads
// the chunks of the list again (none, as a rule). Once more than half of the blocks have given up, the chip is taken to have
// less room than a unit needs, where waiting only keeps the rest of the unit away, and the others wait less (kPollsStarved).
// A partial and the fact that it is there are one 8-byte word, written and read as one (kEmpty: not yet there), so that no
// fence and no write-back of an L2 lies between the two halves.
constexpr unsigned long long kEmpty = ~0ull;
// A poll takes 0.8 us, a wait on a free chip 5 to 30 us: of the 16384 blocks of 8 x 64 x 1024^2 forward none gave up within 96
// polls, 17 to 180 within 64, a tenth within 48, nine tenths within 8. What more than half of the blocks gave up for has to be
// longer than that too, or blocks go on giving up by themselves once the chip is free again. Beside a kernel of another stream
// that holds n compute units for about 3 ms, forward / backward, us (128 and 48 : 256, and 8 for everybody after the first block that
// gave up); a single chunk on the list took 1.74 / 2.95 ms by the latter rule and takes 0.59 / 0.57:
//   8 x 64 x 1024^2           n = 0  580 / 580 : 578 / 581   150  993 / 2409 : 1021 / 3896   200  1675 / 3884 : 2592 / 591 and
//   (for 20 ms) 1158 / 2508 : 2627 / 3956
//   2 x 64 x 512^2, 2 groups      0   40 / 49 : 39 / 52      150   89 / 315 : 91 / 342       200   355 / 533 : 293 / 463
constexpr unsigned kPolls = 128, kPollsStarved = 48;
constexpr unsigned kOwnChoice = ~0u;  // for `polls`: as the interface has it, a whole group a block where that covers the tensor, else kPolls
constexpr long long kStreamed = 1ll << 27;  // bytes of a tensor that goes past the last-level cache
constexpr int kMaxPartials = 2 * kThreads;  // partials of a unit: every block of the unit adds them up again

struct ResidentArgs {
  unsigned long long* slot;   // a word for every chunk of every row
  unsigned long long* result; // a word for every unit: (mean, rstd) or (q1, q2)
  unsigned* left;             // how many chunks are on the list
  unsigned* list;
  unsigned chunks, partials;  // of a row; of a unit = cpg * chunks
  unsigned polls;
  long long S, chunk_len;
  float* mean;                // forward: written, backward: read
  float* rstd;
  float eps;
};

__global__ __launch_bounds__(kThreads) void gn_resident_clear_kernel(unsigned long long* slot, unsigned* left, long long n) {
  const long long i = (long long)blockIdx.x * kThreads + threadIdx.x;
  if (i < n) slot[i] = kEmpty;
  if (i == 0) *left = 0;
}

__device__ __forceinline__ void publish(unsigned long long* slot, float a, float b) {
  auto word = [](float v) { return v != v ? 0x7fc00000u : __float_as_uint(v); };  // no NaN that reads as kEmpty
  __hip_atomic_store(slot, (unsigned long long)word(b) << 32 | word(a), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// The word of a slot, polled up to `polls` times
__device__ __forceinline__ unsigned long long await(const unsigned long long* slot, unsigned polls) {
  unsigned long long v;
  while ((v = __hip_atomic_load(slot, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) == kEmpty) {
    if (--polls == 0) break;
    __builtin_amdgcn_s_sleep(4);
  }
  return v;
}
__device__ __forceinline__ float2 pair_of(unsigned long long v) {
  return make_float2(__uint_as_float((unsigned)v), __uint_as_float((unsigned)(v >> 32)));
}

// Sum of a per-thread value over kThreads threads, in every one of them; fixed order. PARTS: how many such parts the block has
template <typename T, int PARTS = 1>
__device__ __forceinline__ T block_total(T v) {
  __shared__ T all[PARTS * kThreads / 64];
  T* const red = all + (PARTS > 1 ? threadIdx.x / kThreads * (kThreads / 64) : 0);
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) all[threadIdx.x >> 6] = v;
  __syncthreads();
  return (red[0] + red[1]) + (red[2] + red[3]);
}

template <int PARTS = 1>
__device__ __forceinline__ float2 block_total2(float a, float b) {
  __shared__ float2 all[PARTS * kThreads / 64];
  float2* const red = all + (PARTS > 1 ? threadIdx.x / kThreads * (kThreads / 64) : 0);
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    a += __shfl_xor(a, o, 64);
    b += __shfl_xor(b, o, 64);
  }
  __syncthreads();
  if ((threadIdx.x & 63) == 0) all[threadIdx.x >> 6] = make_float2(a, b);
  __syncthreads();
  return make_float2((red[0].x + red[1].x) + (red[2].x + red[3].x), (red[0].y + red[1].y) + (red[2].y + red[3].y));
}

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// An element of a 4-byte word
template <int DT>
struct Word {
  typename Elem<DT>::T v[4 / sizeof(typename Elem<DT>::T)];
};
template <int DT>
__device__ __forceinline__ float up_of(uint32_t w, int e) {
  if (DT == JG_BF16) return __uint_as_float(e == 0 ? w << 16 : w & 0xffff0000u);
  return Elem<DT>::up(__builtin_bit_cast(Word<DT>, w).v[e]);
}
// The same, worked out where it is written: the compiler would keep the elements of the first use for the second one, in
// twice the registers that the words take
template <int DT>
__device__ __forceinline__ float up_again(uint32_t w, int e) {
  float f;
  if (DT == JG_F32) f = __uint_as_float(w);
  else if (DT == JG_BF16 && e == 0) asm volatile("v_lshlrev_b32 %0, 16, %1" : "=v"(f) : "v"(w));
  else if (DT == JG_BF16) asm volatile("v_and_b32 %0, 0xffff0000, %1" : "=v"(f) : "v"(w));
  else if (e == 0) asm volatile("v_cvt_f32_f16 %0, %1" : "=v"(f) : "v"(w));
  else asm volatile("v_cvt_f32_f16_sdwa %0, %1 dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:WORD_1" : "=v"(f) : "v"(w));
  return f;
}
// A buffer of `bytes` bytes: loads beyond it give zeros, stores beyond it do nothing. Stores of 16 bytes take no scalar
// offset: behind one that does, the compiler puts no wait state before an instruction that writes the stored registers
// again, and the new value was stored now and then.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t buffer_of(const void* p, int bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, bytes, 0x00020000);
}

// Vectors of a tensor a thread keeps: 64 registers in all, so that four blocks (1024 on the chip, 64 MB) fit a compute unit:
// two units of 8 x 1024^2 bf16 elements backward, one of which loads while the other one waits or writes. 48 registers and
// five blocks: 797 / 946 us where 64 took 699 / 819; 80 registers, which divide such a row less evenly, 722 / 827.
template <bool BWD>
constexpr int kHeld = BWD ? 8 : 16;
// Up to this many partials every block of a unit adds them up itself: one hop less (8 x 32 x 512^2, 64 chunks a unit: 73
// instead of 78 us forward). Beyond it the block of the last chunk does, and the others wait for one word: with all of them
// polling all partials the polls were a quarter of the traffic (512 chunks a unit: 752 instead of 575 us backward).
constexpr unsigned kDirect = 64;

// Chunk t = (unit, chunk k of the unit): channel c, elements [lo, hi)
struct HeldRange {
  unsigned unit, k;
  int c;
  long long lo, hi;
};
__device__ __forceinline__ HeldRange held_range(const ResidentArgs& q, const ApplyArgs& p, unsigned t) {
  const unsigned unit = t / q.partials, k = t - unit * q.partials, r = k / q.chunks;
  const int cpg = p.C / p.G;
  const long long base = ((long long)unit * cpg + r) * q.S, from = (k - r * q.chunks) * q.chunk_len;
  return HeldRange{unit, k, (int)(unit % p.G) * cpg + (int)r, base + (from < q.S ? from : q.S),
                   base + (from + q.chunk_len < q.S ? from + q.chunk_len : q.S)};
}

// Statistics of unit u from its partials; false: some were not there after `polls`. Forward: mean and 1 / sqrt(variance + eps),
// in double over the chunks; backward: the unit's q1 and q2.
template <int DT, bool BWD>
__device__ __forceinline__ bool held_statistics(const ResidentArgs& q, const ApplyArgs& p, unsigned u, unsigned polls, float& m, float& rs,
                                                float& q1, float& q2) {
  typedef typename Elem<DT>::T T;
  const int cpg = p.C / p.G, tid = threadIdx.x;
  const unsigned long long* slot = q.slot + (size_t)u * q.partials;
  float2 v[kMaxPartials / kThreads];
  bool missing = false;
#pragma unroll
  for (int i = 0; i < kMaxPartials / kThreads; ++i) {
    const unsigned j = tid + i * kThreads;
    v[i] = make_float2(0.0f, 0.0f);
    if (j >= q.partials) continue;
    const unsigned long long word = await(slot + j, polls);
    missing |= word == kEmpty;
    v[i] = pair_of(word);
  }
  if (__builtin_amdgcn_readfirstlane(__syncthreads_or(missing)) != 0) return false;
  q1 = q2 = 0.0f;
  if (BWD) {
    m = q.mean[u];
    rs = q.rstd[u];
#pragma unroll
    for (int i = 0; i < kMaxPartials / kThreads; ++i) {
      const unsigned j = tid + i * kThreads;
      if (j >= q.partials) continue;
      const float w = p.weight != nullptr ? Elem<DT>::up(static_cast<const T*>(p.weight)[(u % p.G) * cpg + j / q.chunks]) : 1.0f;
      q1 += w * v[i].x;
      q2 += w * v[i].y;
    }
    const float inv = 1.0f / p.count;
    const float2 sums = block_total2(q1, q2);
    q1 = sums.x * inv;
    q2 = sums.y * inv;
  } else {
    double n[kMaxPartials / kThreads], sum = 0.0, dev = 0.0;
#pragma unroll
    for (int i = 0; i < kMaxPartials / kThreads; ++i) {
      const unsigned j = tid + i * kThreads;
      const long long from = (j % q.chunks) * q.chunk_len;
      n[i] = j >= q.partials || from >= q.S ? 0.0 : (double)(from + q.chunk_len < q.S ? q.chunk_len : q.S - from);
      sum += n[i] * v[i].x;
    }
    const double mu = block_total(sum) / (double)p.count;
#pragma unroll
    for (int i = 0; i < kMaxPartials / kThreads; ++i) dev += v[i].y + n[i] * (v[i].x - mu) * (v[i].x - mu);
    m = (float)mu;
    rs = 1.0f / sqrtf((float)(block_total(dev) / (double)p.count) + q.eps);
  }
  return true;
}

// The same from the partials of a unit in LDS (at most kWhole), with the roundings of held_statistics: its tree over the lanes is (0 + 2) + (1 + 3)
constexpr int kWhole = 4;
template <int DT, bool BWD>
__device__ __forceinline__ void whole_statistics(const ResidentArgs& q, const ApplyArgs& p, unsigned u, const float2 v[kWhole], float& m, float& rs,
                                                 float& q1, float& q2) {
  typedef typename Elem<DT>::T T;
  q1 = q2 = 0.0f;
  if (BWD) {
    const int cpg = p.C / p.G;
    float a[kWhole], b[kWhole];
#pragma unroll
    for (unsigned j = 0; j < kWhole; ++j) {
      const bool there = j < q.partials;
      const float w = there && p.weight != nullptr ? Elem<DT>::up(static_cast<const T*>(p.weight)[(u % p.G) * cpg + j / q.chunks]) : 1.0f;
      a[j] = there ? __builtin_fmaf(w, v[j].x, 0.0f) : 0.0f;
      b[j] = there ? __builtin_fmaf(w, v[j].y, 0.0f) : 0.0f;
    }
    const float inv = 1.0f / p.count;
    rs = q.rstd[u];
    q1 = ((a[0] + a[2]) + (a[1] + a[3])) * inv;
    q2 = ((b[0] + b[2]) + (b[1] + b[3])) * inv;
  } else {
    double n[kWhole], sum[kWhole], dev[kWhole];
#pragma unroll
    for (unsigned j = 0; j < kWhole; ++j) {
      const long long from = (j % q.chunks) * q.chunk_len;
      n[j] = j >= q.partials || from >= q.S ? 0.0 : (double)(from + q.chunk_len < q.S ? q.chunk_len : q.S - from);
      sum[j] = j < q.partials ? n[j] * v[j].x : 0.0;
    }
    const double mu = ((sum[0] + sum[2]) + (sum[1] + sum[3])) / (double)p.count;
#pragma unroll
    for (unsigned j = 0; j < kWhole; ++j) dev[j] = j < q.partials ? v[j].y + n[j] * (v[j].x - mu) * (v[j].x - mu) : 0.0;
    m = (float)mu;
    rs = 1.0f / sqrtf((float)(((dev[0] + dev[2]) + (dev[1] + dev[3])) / (double)p.count) + q.eps);
  }
}

// STREAM: loads and stores that leave nothing in the last-level cache, for tensors that do not fit there
// WHOLE: a block has a part of kThreads threads for each chunk of its unit (blockIdx.x), up to kWhole of them: the partials meet in LDS,
// nobody waits for another block, and neither the words nor the list are wanted. One launch forward where there are three,
// two backward: a short step is bound by the host, which takes 3 to 4 us a launch (forward and backward of 4 x 64 x 259 x 83 bf16 in
// 32 groups and of smaller tensors, us: 78 with six launches, 66 with three). On the GPU alone, blocks that wait : WHOLE: 8 x 8 x 16384 in 8 groups 12.5 : 7.6
// and 10.4 : 7.7 forward and backward, 4 x 64 x 21497 in 32 15.5 : 11.6 and 13.2 : 13.1, 4 x 64 x 32768 in 16 (four full chunks a group) 18.2 : 16.8 forward; few
// groups of four full chunks keep fewer compute units busy, for less than what the host saves: 4 x 32 x 32768 in 8 14.4 : 15.3
template <int DT, bool BWD, bool STREAM, bool WHOLE>
__global__ __launch_bounds__(WHOLE ? kWhole * kThreads : kThreads, 4) void gn_resident_kernel(ResidentArgs q, ApplyArgs p) {
  typedef typename Elem<DT>::T T;
  constexpr int V = Elem<DT>::VEC, E = 4 / sizeof(T), R = kHeld<BWD>, kAux = STREAM ? 2 : 0;  // 2: non-temporal
  constexpr int PARTS = WHOLE ? kWhole : 1;
  const int tid = threadIdx.x % kThreads;
  const unsigned me = WHOLE ? blockIdx.x * q.partials + __builtin_amdgcn_readfirstlane(threadIdx.x / kThreads) : blockIdx.x;
  const T* in = static_cast<const T*>(p.in);
  const T* in2 = static_cast<const T*>(p.in2);
  const HeldRange r = held_range(q, p, me);
  float m = BWD ? q.mean[r.unit] : 0.0f, rs, q1, q2;

  // the chunk into registers: whole vectors, and the elements before the first and behind the last one, one a thread
  const long long b0 = (r.lo + V - 1) / V * V, b1 = r.hi / V * V > b0 ? r.hi / V * V : b0;
  const int bytes = (int)(b1 - b0) * (int)sizeof(T), at = tid * 16;
  u32x4 a[R], b[BWD ? R : 1];
  const auto from = buffer_of(in + b0, bytes), from2 = buffer_of((BWD ? in2 : in) + b0, bytes);
#pragma unroll
  for (int i = 0; i < R; ++i) {
    a[i] = __builtin_amdgcn_raw_buffer_load_b128(from, at, i * kThreads * 16, kAux);
    if (BWD) b[i] = __builtin_amdgcn_raw_buffer_load_b128(from2, at, i * kThreads * 16, kAux);
  }
  const int single = tid < V ? tid : (int)(b1 - r.lo) + tid - 64;  // from r.lo on
  const bool has_single = tid < V ? single < (int)(b0 - r.lo) && single < (int)(r.hi - r.lo) : tid >= 64 && single < (int)(r.hi - r.lo);
  const float sa = has_single ? Elem<DT>::up((in + r.lo)[single]) : 0.0f, sb = BWD && has_single ? Elem<DT>::up((in2 + r.lo)[single]) : 0.0f;

  // its partials
  float2 part = make_float2(0.0f, 0.0f);
  if (BWD) {
#pragma unroll
    for (int i = 0; i < R; ++i) {
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int e = 0; e < V; ++e) {
        const float g = up_of<DT>(a[i][e / E], e % E);
        part.x += g;
        part.y += g * (up_of<DT>(b[i][e / E], e % E) - m);
      }
    }
    part.x += sa;
    part.y += sa * (sb - m);
    part = block_total2<PARTS>(part.x, part.y);
    part.y *= q.rstd[r.unit];
  } else {
    const float n = (float)(r.hi - r.lo);
    float sum = sa;
#pragma unroll
    for (int i = 0; i < R; ++i) {
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int e = 0; e < V; ++e) sum += up_of<DT>(a[i][e / E], e % E);
    }
    const float all = block_total<float, PARTS>(sum);
    part.x = n > 0.0f ? all / n : 0.0f;
    float dev = has_single ? (sa - part.x) * (sa - part.x) : 0.0f;
#pragma unroll
    for (int i = 0; i < R; ++i)
      if (at + i * kThreads * 16 < bytes)
#pragma unroll
        for (int e = 0; e < V; ++e) {
          const float d = up_again<DT>(a[i][e / E], e % E) - part.x;
          dev += d * d;
        }
    part.y = block_total<float, PARTS>(dev);
  }
  if (WHOLE) {
    __shared__ float2 parts[kWhole];
    if (tid == 0) parts[r.k] = part;
    if (BWD && tid == 0) publish(q.slot + me, part.x, part.y);  // for the parameter gradients
    __syncthreads();
    whole_statistics<DT, BWD>(q, p, r.unit, parts, m, rs, q1, q2);
  } else {
    if (tid == 0) publish(q.slot + blockIdx.x, part.x, part.y);

    __shared__ unsigned long long word_s;
    const bool adds = q.partials <= kDirect || r.k == q.partials - 1;
    const unsigned gave_up = __hip_atomic_load(q.left, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const unsigned polls = gave_up > (blockIdx.x + q.partials) / 2 && q.polls > kPollsStarved ? kPollsStarved : q.polls;
    bool there;
    if (adds) {
      there = held_statistics<DT, BWD>(q, p, r.unit, polls, m, rs, q1, q2);
      if (there && tid == 0 && q.partials > kDirect) publish(q.result + r.unit, BWD ? q1 : m, BWD ? q2 : rs);
    } else {
      if (tid == 0) word_s = await(q.result + r.unit, polls);
      __syncthreads();
      const unsigned lo = __builtin_amdgcn_readfirstlane((unsigned)word_s), hi = __builtin_amdgcn_readfirstlane((unsigned)(word_s >> 32));
      there = (lo & hi) != ~0u;
      const float v0 = __uint_as_float(lo), v1 = __uint_as_float(hi);
      if (BWD) q1 = v0, q2 = v1, rs = q.rstd[r.unit];
      else m = v0, rs = v1;
    }
    if (!there) {
      if (tid == 0) q.list[__hip_atomic_fetch_add(q.left, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)] = blockIdx.x;
      return;
    }
  }
  if (!BWD && r.k == 0 && tid == 0) {
    q.mean[r.unit] = m;
    q.rstd[r.unit] = rs;
  }
  T* out = static_cast<T*>(p.out);
  T* kept = static_cast<T*>(p.out_kept);
  const float w = p.weight != nullptr ? Elem<DT>::up(static_cast<const T*>(p.weight)[r.c]) : 1.0f;
  const float bv = !BWD && p.bias != nullptr ? Elem<DT>::up(static_cast<const T*>(p.bias)[r.c]) : 0.0f;
  const GradFactors f = grad_factors(rs, w, q1, q2, true);
  auto result = [&](float v, float x) {
    if (BWD) return input_gradient<DT>(v, x - m, f);
    return output<DT>(normalised<DT>(v, m, rs), w, bv);
  };
  const auto to = buffer_of(out + b0, bytes), to_kept = buffer_of((kept != nullptr ? kept : out) + b0, bytes);
#pragma unroll
  for (int i = 0; i < R; ++i) {
    __builtin_amdgcn_sched_barrier(0);
    if (!BWD && kept != nullptr) __builtin_amdgcn_raw_buffer_store_b128(a[i], to_kept, at + i * kThreads * 16, 0, kAux);
    Pack<DT> y;
#pragma unroll
    for (int e = 0; e < V; ++e)
      y.v[e] = Elem<DT>::down(result(up_again<DT>(a[i][e / E], e % E), BWD ? up_again<DT>(b[i][e / E], e % E) : 0.0f));
    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, y), to, at + i * kThreads * 16, 0, kAux);
  }
  if (has_single) {
    if (!BWD && kept != nullptr) (kept + r.lo)[single] = (in + r.lo)[single];
    (out + r.lo)[single] = Elem<DT>::down(result(sa, sb));
  }
}

// Behind gn_resident_kernel: the parameter gradients of channel blockIdx.x from its rows' partials of every sample
// (backward, blocks [0, C) if they are wanted), and the chunks on the list, if there is one, one block after the other.
template <int DT, bool BWD>
__global__ __launch_bounds__(kThreads) void gn_resident_rest_kernel(ResidentArgs q, ApplyArgs p, void* gw, void* gb, int wdtype, long long N) {
  const int tid = threadIdx.x;
  if (BWD && (gw != nullptr || gb != nullptr) && blockIdx.x < p.C) {
    const int c = blockIdx.x;
    float s0 = 0.0f, s1 = 0.0f;
    for (long long i = tid; i < N * q.chunks; i += kThreads) {
      const long long n = i / q.chunks;
      const float2 v = pair_of(q.slot[(n * p.C + c) * q.chunks + (i - n * q.chunks)]);
      s0 += v.x;
      s1 += v.y;
    }
    const float2 sums = block_total2(s0, s1);
    if (tid == 0 && gb != nullptr) store_as(gb, c, sums.x, wdtype);
    if (tid == 0 && gw != nullptr) store_as(gw, c, sums.y, wdtype);
  }
  const unsigned left = q.left != nullptr ? *q.left : 0;
  for (unsigned i = blockIdx.x; i < left; i += gridDim.x) {
    const HeldRange r = held_range(q, p, q.list[i]);
    float m, rs, q1, q2;
    held_statistics<DT, BWD>(q, p, r.unit, 1, m, rs, q1, q2);
    if (!BWD && r.k == 0 && tid == 0) {
      q.mean[r.unit] = m;
      q.rstd[r.unit] = rs;
    }
    apply_range<DT, BWD, true>(p, r.c, m, rs, q1, q2, r.lo, r.hi, true);
    __syncthreads();
  }
}

int chunks_of(long long len) {
  long long c = (len + kChunk - 1) / kChunk;
  if (c < 1) c = 1;
  if (c > kMaxChunks) c = kMaxChunks;
  return (int)c;
}

// chunk length: a multiple of 8 elements, so that chunk starts keep the 16-byte alignment
long long chunk_len_of(long long len, int chunks) {
  long long l = (len + chunks - 1) / chunks;
  return (l + 7) / 8 * 8;
}

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

int check(const char* who, int64_t N, int64_t C, int64_t S, int64_t G, int dtype) {
  JG_REQUIRE(dtype == JG_F32 || dtype == JG_BF16 || dtype == JG_F16, "%s: unknown dtype %d", who, dtype);
  JG_REQUIRE(N >= 0 && C >= 1 && S >= 0 && G >= 1, "%s: bad shape", who);
  JG_REQUIRE(C % G == 0, "%s: %lld channels do not divide into %lld groups", who, (long long)C, (long long)G);
  JG_REQUIRE(N * C * (int64_t)kMaxChunks < (1ll << 31), "%s: too many rows", who);
  return JG_OK;
}

size_t ws_need(int64_t N, int64_t C, int64_t S) {
  // the larger of: per-row partials (backward), per-group partials (forward); and the two sums of every group
  const size_t rows = (size_t)N * (size_t)C;
  return (rows * (size_t)chunks_of(S) * 2 + rows * 2) * sizeof(float) + 256;
}

// What resident_launch wants: two words for every chunk and every unit, and the list of chunks
size_t resident_need(long long chunks, long long units) { return (size_t)(chunks * 3 + units * 2 + 1) * sizeof(float); }

// chunk partials of `units` spans of `len` elements into ws
template <int DT, int MODE>
int partials_launch(const void* x, const void* y, const float* mean, const float* rstd, int cpg, long long units,
                    long long len, float* ws, hipStream_t s, const char* who) {
  typedef typename Elem<DT>::T T;
  if (units == 0) return JG_OK;
  const int chunks = chunks_of(len);
  const bool vec_ok = aligned16(x) && (MODE < 2 || aligned16(y));
  gn_reduce_kernel<DT, MODE><<<(unsigned)(units * chunks), kThreads, 0, s>>>(
      ws, static_cast<const T*>(x), static_cast<const T*>(y), mean, rstd, cpg, len, chunks, chunk_len_of(len, chunks), vec_ok);
  JG_CHECK_LAUNCH(who);
  return JG_OK;
}

template <int DT, int MODE>
int reduce_launch(float* out, const void* x, const float* mean, long long units, long long len, float* ws, hipStream_t s,
                  const char* who) {
  if (units == 0) return JG_OK;
  int rc = partials_launch<DT, MODE>(x, nullptr, mean, nullptr, 1, units, len, ws, s, who);
  if (rc) return rc;
  gn_finish_kernel<<<(unsigned)((units + kThreads - 1) / kThreads), kThreads, 0, s>>>(out, nullptr, ws, units, chunks_of(len));
  JG_CHECK_LAUNCH(who);
  return JG_OK;
}

template <int DT>
int moments_launch(float* mean, float* sq, float* count_sum, float* rstd, const void* x, long long units, long long len,
                   float eps, float* ws, hipStream_t s, const char* who) {
  if (units == 0 || len == 0) return JG_OK;
  const int chunks = chunks_of(len);
  const long long cl = chunk_len_of(len, chunks);
  gn_moments_kernel<DT><<<(unsigned)(units * chunks), kThreads, 0, s>>>(ws, static_cast<const typename Elem<DT>::T*>(x), len,
                                                                       chunks, cl, aligned16(x));
  JG_CHECK_LAUNCH(who);
  gn_moments_finish_kernel<<<(unsigned)units, 64, 0, s>>>(mean, sq, count_sum, rstd, ws, len, chunks, cl, eps);
  JG_CHECK_LAUNCH(who);
  return JG_OK;
}

// The two sums of every (sample, group) and the parameter gradients; mean == NULL: `x` is x_norm.
template <int DT>
int bwd_sums_launch(float* sum0, float* sum1, int stride, void* gw, void* gb, int wdtype, const void* g, const void* x,
                    const float* mean, const float* rstd, const void* weight, long long N, long long C, long long S,
                    long long G, float* ws, hipStream_t s, const char* who) {
  if (N * C == 0 || S == 0) return JG_OK;
  const int cpg = (int)(C / G);
  const int rc = mean == nullptr ? partials_launch<DT, 2>(g, x, nullptr, nullptr, cpg, N * C, S, ws, s, who)
                                 : partials_launch<DT, 3>(g, x, mean, rstd, cpg, N * C, S, ws, s, who);
  if (rc) return rc;
  gn_bwd_finish_kernel<DT><<<(unsigned)(N * G + C), 64, 0, s>>>(sum0, sum1, stride, gw, gb, wdtype, ws,
                                                                static_cast<const typename Elem<DT>::T*>(weight), N, (int)C,
                                                                (int)G, chunks_of(S));
  JG_CHECK_LAUNCH(who);
  return JG_OK;
}

template <int DT, bool BWD, bool FROM_X>
int apply_launch(const ApplyArgs& a, long long N, long long S, hipStream_t s, const char* who) {
  const long long rows = N * a.C;
  if (rows == 0 || S == 0) return JG_OK;
  const int chunks = chunks_of(S);
  const bool vec_ok = aligned16(a.out) && aligned16(a.in) && aligned16(a.in2) && aligned16(a.out_norm) && aligned16(a.out_kept);
  gn_apply_kernel<DT, BWD, FROM_X><<<(unsigned)(rows * chunks), kThreads, 0, s>>>(a, S, chunks, chunk_len_of(S, chunks), vec_ok);
  JG_CHECK_LAUNCH(who);
  return JG_OK;
}

// gn_resident_kernel where a unit's chunks take at most half of the blocks that fit the chip (so that one unit loads while
// another one writes); false: the separate launches, which read a tensor twice.
template <int DT, bool BWD>
bool resident_launch(ResidentArgs q, const ApplyArgs& a, void* gw, void* gb, int wdtype, long long N, long long S, float* ws, size_t ws_bytes, hipStream_t s) {
  const long long units = N * a.G, cpg = a.C / a.G, rows = N * a.C, most = (long long)kThreads * Elem<DT>::VEC * kHeld<BWD>;
  if (rows == 0 || S == 0 || q.polls == 0) return false;
  const long long chunks = (S + most - 1) / most, fit = 4ll * jg::cu_count(), total = rows * chunks;
  const bool vec_ok = aligned16(a.out) && aligned16(a.in) && aligned16(a.in2) && aligned16(a.out_kept);
  if (!vec_ok || cpg * chunks > std::min<long long>(kMaxPartials, fit / 2) || total > 1ll << 23 || (reinterpret_cast<uintptr_t>(ws) & 7) != 0 ||
      ws_bytes < resident_need(total, units))
    return false;
  q.slot = reinterpret_cast<unsigned long long*>(ws);
  q.result = q.slot + total;
  q.left = reinterpret_cast<unsigned*>(q.result + units);
  q.list = q.left + 1;
  q.chunks = (unsigned)chunks;
  q.partials = (unsigned)(cpg * chunks);
  q.S = S;
  q.chunk_len = chunk_len_of(S, (int)chunks);
  const bool own_choice = q.polls == kOwnChoice;
  if (own_choice) q.polls = kPolls;
  const long long channels = gw != nullptr || gb != nullptr ? a.C : 0, bytes = rows * S * (long long)sizeof(typename Elem<DT>::T);
  // A unit of up to kWhole chunks is one block's.
  if (own_choice && q.partials <= kWhole && bytes < kStreamed) {
    gn_resident_kernel<DT, BWD, false, true><<<(unsigned)units, kThreads * q.partials, 0, s>>>(q, a);
    q.left = nullptr;
    if (channels > 0) gn_resident_rest_kernel<DT, BWD><<<(unsigned)channels, kThreads, 0, s>>>(q, a, gw, gb, wdtype, N);
    return true;
  }
  gn_resident_clear_kernel<<<(unsigned)((total + units + kThreads - 1) / kThreads), kThreads, 0, s>>>(q.slot, q.left, total + units);
  // Two tensors that fill the last-level cache (256 MB) go past it; smaller ones stay for whoever reads them next. Forward and
  // backward: 8 x 32 x 512^2 bf16 (134 MB) 155 us against 170, 8 x 64 x 1024^2 1159 against 1262; 4 x 64 x 300 x 311 fp32
  // (95 MB) 153 against 135.
  if (bytes >= kStreamed) gn_resident_kernel<DT, BWD, true, false><<<(unsigned)total, kThreads, 0, s>>>(q, a);
  else gn_resident_kernel<DT, BWD, false, false><<<(unsigned)total, kThreads, 0, s>>>(q, a);
  gn_resident_rest_kernel<DT, BWD><<<(unsigned)std::max(channels, std::min(total, fit)), kThreads, 0, s>>>(q, a, gw, gb, wdtype, N);
  return true;
}

int check_ws(const char* who, const void* ws, size_t bytes, int64_t batch, int64_t channels, int64_t spatial) {
  const size_t need = batch <= 0 || channels <= 0 || spatial <= 0 ? 256 : ws_need(batch, channels, spatial);
  if (ws == nullptr || bytes < need) JG_FAIL(JG_ERR_WORKSPACE, "%s: workspace %zu < %zu bytes", who, bytes, need);
  return JG_OK;
}

}  // namespace

extern "C" size_t jg_gn_workspace_bytes(int64_t batch, int64_t channels, int64_t spatial) {
  if (batch <= 0 || channels <= 0 || spatial <= 0) return 256;
  const long long least = (long long)kThreads * Elem<JG_F32>::VEC * kHeld<true>, rows = batch * channels;  // elements of the smallest chunk a block keeps
  return std::max(ws_need(batch, channels, spatial), resident_need(rows * std::min<long long>((spatial + least - 1) / least, kMaxPartials), rows));
}

#define JG_GN_DISPATCH(CALL)                    \
  switch (dtype) {                              \
    case JG_F32: return CALL(JG_F32);           \
    case JG_BF16: return CALL(JG_BF16);         \
    default: return CALL(JG_F16);               \
  }

extern "C" int jg_gn_partial_sum(float* sum, const void* x, int64_t batch, int64_t channels, int64_t spatial,
                                 int64_t groups, int dtype, void* workspace, size_t workspace_bytes,
                                 void* stream) {
  const char* who = "jg_gn_partial_sum";
  int rc = check(who, batch, channels, spatial, groups, dtype);
  if (rc) return rc;
  JG_REQUIRE(sum && x, "%s: NULL pointer", who);
  if ((rc = check_ws(who, workspace, workspace_bytes, batch, channels, spatial))) return rc;
  hipStream_t s = static_cast<hipStream_t>(stream);
  const long long units = batch * groups, len = channels / groups * spatial;
#define CALL(DT) reduce_launch<DT, 0>(sum, x, nullptr, units, len, static_cast<float*>(workspace), s, who)
  JG_GN_DISPATCH(CALL)
#undef CALL
}

extern "C" int jg_gn_partial_sqdev(float* sq, const void* x, const float* mean, int64_t batch, int64_t channels,
                                   int64_t spatial, int64_t groups, int dtype, void* workspace,
                                   size_t workspace_bytes, void* stream) {
  const char* who = "jg_gn_partial_sqdev";
  int rc = check(who, batch, channels, spatial, groups, dtype);
  if (rc) return rc;
  JG_REQUIRE(sq && x && mean, "%s: NULL pointer", who);
  if ((rc = check_ws(who, workspace, workspace_bytes, batch, channels, spatial))) return rc;
  hipStream_t s = static_cast<hipStream_t>(stream);
  const long long units = batch * groups, len = channels / groups * spatial;
#define CALL(DT) reduce_launch<DT, 1>(sq, x, mean, units, len, static_cast<float*>(workspace), s, who)
  JG_GN_DISPATCH(CALL)
#undef CALL
}

extern "C" int jg_gn_moments(float* mean, float* sq, float* count_sum, const void* x, int64_t batch, int64_t channels,
                             int64_t spatial, int64_t groups, int dtype, void* workspace, size_t workspace_bytes,
                             void* stream) {
  const char* who = "jg_gn_moments";
  int rc = check(who, batch, channels, spatial, groups, dtype);
  if (rc) return rc;
  JG_REQUIRE(mean && sq && count_sum && x, "%s: NULL pointer", who);
  if ((rc = check_ws(who, workspace, workspace_bytes, batch, channels, spatial))) return rc;
  hipStream_t s = static_cast<hipStream_t>(stream);
  const long long units = batch * groups, len = channels / groups * spatial;
#define CALL(DT) moments_launch<DT>(mean, sq, count_sum, nullptr, x, units, len, 0.0f, static_cast<float*>(workspace), s, who)
  JG_GN_DISPATCH(CALL)
#undef CALL
}

static int apply_forward(const char* who, void* y, void* x_norm, void* x_kept, const void* x, const float* mean, const float* rstd,
                         const void* weight, const void* bias, int64_t batch, int64_t channels, int64_t spatial,
                         int64_t groups, int dtype, void* stream) {
  int rc = check(who, batch, channels, spatial, groups, dtype);
  if (rc) return rc;
  JG_REQUIRE(y && x && mean && rstd, "%s: NULL pointer", who);
  hipStream_t s = static_cast<hipStream_t>(stream);
  ApplyArgs a = {};
  a.out = y; a.out_norm = x_norm; a.out_kept = x_kept; a.in = x; a.mean = mean; a.rstd = rstd; a.weight = weight; a.bias = bias;
  a.C = (int)channels; a.G = (int)groups;
#define CALL(DT) apply_launch<DT, false, true>(a, batch, spatial, s, who)
  JG_GN_DISPATCH(CALL)
#undef CALL
}

extern "C" int jg_gn_apply(void* y, void* x_norm, const void* x, const float* mean, const float* rstd,
                           const void* weight, const void* bias, int64_t batch, int64_t channels,
                           int64_t spatial, int64_t groups, int dtype, void* stream) {
  return apply_forward("jg_gn_apply", y, x_norm, nullptr, x, mean, rstd, weight, bias, batch, channels, spatial, groups, dtype, stream);
}

extern "C" int jg_gn_apply_keep(void* y, void* x_kept, const void* x, const float* mean, const float* rstd,
                                const void* weight, const void* bias, int64_t batch, int64_t channels,
                                int64_t spatial, int64_t groups, int dtype, void* stream) {
  return apply_forward("jg_gn_apply_keep", y, nullptr, x_kept, x, mean, rstd, weight, bias, batch, channels, spatial, groups, dtype, stream);
}

// Both passes of the forward / of the backward for a tensor that one rank holds whole.
namespace {
template <int DT>
int forward_all(void* y, void* x_kept, float* mean, float* rstd, const void* x, const void* weight, const void* bias, long long N,
                long long C, long long S, long long G, float eps, unsigned polls, float* ws, size_t ws_bytes, hipStream_t s, const char* who) {
  ApplyArgs a = {};
  a.out = y; a.out_kept = x_kept; a.in = x; a.mean = mean; a.rstd = rstd; a.weight = weight; a.bias = bias; a.C = (int)C; a.G = (int)G;
  a.count = (float)(C / G * S);
  ResidentArgs q = {};
  q.mean = mean; q.rstd = rstd; q.eps = eps; q.polls = polls;
  if (resident_launch<DT, false>(q, a, nullptr, nullptr, 0, N, S, ws, ws_bytes, s)) {
    JG_CHECK_LAUNCH(who);
    return JG_OK;
  }
  const int rc = moments_launch<DT>(mean, nullptr, nullptr, rstd, x, N * G, C / G * S, eps, ws, s, who);
  if (rc) return rc;
  return apply_launch<DT, false, true>(a, N, S, s, who);
}

template <int DT>
int backward_all(void* gx, void* gw, void* gb, int wdtype, const void* g, const void* x, const float* mean, const float* rstd,
                 const void* weight, long long N, long long C, long long S, long long G, unsigned polls, float* ws, size_t ws_bytes, hipStream_t s,
                 const char* who) {
  const long long rows = N * C;
  float* sums = ws + (size_t)rows * chunks_of(S) * 2;
  ApplyArgs a = {};
  a.out = gx; a.in = g; a.in2 = x; a.mean = mean; a.rstd = rstd; a.gsum = sums; a.gxsum = sums + 1; a.stride = 2;
  a.count = (float)(C / G * S);
  a.weight = weight; a.C = (int)C; a.G = (int)G;
  ResidentArgs q = {};
  q.mean = const_cast<float*>(mean); q.rstd = const_cast<float*>(rstd); q.polls = polls;
  if (gx != nullptr && resident_launch<DT, true>(q, a, gw, gb, wdtype, N, S, ws, ws_bytes, s)) {
    JG_CHECK_LAUNCH(who);
    return JG_OK;
  }
  int rc = bwd_sums_launch<DT>(sums, sums + 1, 2, gw, gb, wdtype, g, x, mean, rstd, weight, N, C, S, G, ws, s, who);
  if (rc || gx == nullptr) return rc;
  return apply_launch<DT, true, true>(a, N, S, s, who);
}
}  // namespace

// jg_gn_forward_keep and jg_gn_backward as they are but for `polls`: how often a block asks for the rest of its group before
// it leaves its chunk to the second launch (1: nearly always; 0: separate launches, which read the tensors twice; kOwnChoice). Not
// in the header: tests reach every launch through them.
extern "C" int jg_gn_forward_polls(void* y, void* x_kept, float* mean, float* rstd, const void* x, const void* weight,
                                   const void* bias, int64_t batch, int64_t channels, int64_t spatial, int64_t groups,
                                   float eps, int dtype, unsigned polls, void* workspace, size_t workspace_bytes, void* stream);
extern "C" int jg_gn_backward_polls(void* gx, void* gw, void* gb, const void* g, const void* x, const float* mean,
                                    const float* rstd, const void* weight, int64_t batch, int64_t channels, int64_t spatial,
                                    int64_t groups, int dtype, int grad_dtype, unsigned polls, void* workspace,
                                    size_t workspace_bytes, void* stream);

extern "C" int jg_gn_forward(void* y, float* mean, float* rstd, const void* x, const void* weight, const void* bias,
                             int64_t batch, int64_t channels, int64_t spatial, int64_t groups, float eps, int dtype,
                             void* workspace, size_t workspace_bytes, void* stream) {
  return jg_gn_forward_keep(y, nullptr, mean, rstd, x, weight, bias, batch, channels, spatial, groups, eps, dtype, workspace,
                            workspace_bytes, stream);
}

extern "C" int jg_gn_forward_keep(void* y, void* x_kept, float* mean, float* rstd, const void* x, const void* weight,
                                  const void* bias, int64_t batch, int64_t channels, int64_t spatial, int64_t groups,
                                  float eps, int dtype, void* workspace, size_t workspace_bytes, void* stream) {
  return jg_gn_forward_polls(y, x_kept, mean, rstd, x, weight, bias, batch, channels, spatial, groups, eps, dtype, kOwnChoice, workspace,
                             workspace_bytes, stream);
}

extern "C" int jg_gn_forward_polls(void* y, void* x_kept, float* mean, float* rstd, const void* x, const void* weight,
                                   const void* bias, int64_t batch, int64_t channels, int64_t spatial, int64_t groups,
                                   float eps, int dtype, unsigned polls, void* workspace, size_t workspace_bytes, void* stream) {
  const char* who = "jg_gn_forward";
  int rc = check(who, batch, channels, spatial, groups, dtype);
  if (rc) return rc;
  JG_REQUIRE(y && mean && rstd && x, "%s: NULL pointer", who);
  if ((rc = check_ws(who, workspace, workspace_bytes, batch, channels, spatial))) return rc;
  hipStream_t s = static_cast<hipStream_t>(stream);
#define CALL(DT)                                                                                                                 \
  forward_all<DT>(y, x_kept, mean, rstd, x, weight, bias, batch, channels, spatial, groups, eps, polls,                          \
                  static_cast<float*>(workspace), workspace_bytes, s, who)
  JG_GN_DISPATCH(CALL)
#undef CALL
}

extern "C" int jg_gn_backward(void* gx, void* gw, void* gb, const void* g, const void* x, const float* mean,
                              const float* rstd, const void* weight, int64_t batch, int64_t channels, int64_t spatial,
                              int64_t groups, int dtype, int grad_dtype, void* workspace, size_t workspace_bytes,
                              void* stream) {
  return jg_gn_backward_polls(gx, gw, gb, g, x, mean, rstd, weight, batch, channels, spatial, groups, dtype, grad_dtype, kOwnChoice,
                              workspace, workspace_bytes, stream);
}

extern "C" int jg_gn_backward_polls(void* gx, void* gw, void* gb, const void* g, const void* x, const float* mean,
                                    const float* rstd, const void* weight, int64_t batch, int64_t channels, int64_t spatial,
                                    int64_t groups, int dtype, int grad_dtype, unsigned polls, void* workspace,
                                    size_t workspace_bytes, void* stream) {
  const char* who = "jg_gn_backward";
  int rc = check(who, batch, channels, spatial, groups, dtype);
  if (rc) return rc;
  JG_REQUIRE(jg::dtype_size(grad_dtype) != 0, "%s: unknown gradient dtype %d", who, grad_dtype);
  JG_REQUIRE(g && x && mean && rstd, "%s: NULL pointer", who);
  if ((rc = check_ws(who, workspace, workspace_bytes, batch, channels, spatial))) return rc;
  hipStream_t s = static_cast<hipStream_t>(stream);
#define CALL(DT)                                                                                                                 \
  backward_all<DT>(gx, gw, gb, grad_dtype, g, x, mean, rstd, weight, batch, channels, spatial, groups, polls,                    \
                   static_cast<float*>(workspace), workspace_bytes, s, who)
  JG_GN_DISPATCH(CALL)
#undef CALL
}

// The pieces of the backward of a sharded tensor, from x_norm (mean NULL) or from x.
extern "C" int jg_gn_partial_bwd_x(float* sums, void* gw, void* gb, const void* g, const void* x, const float* mean,
                                   const float* rstd, const void* weight, int64_t batch, int64_t channels, int64_t spatial,
                                   int64_t groups, int dtype, int grad_dtype, void* workspace, size_t workspace_bytes,
                                   void* stream) {
  const char* who = "jg_gn_partial_bwd_x";
  int rc = check(who, batch, channels, spatial, groups, dtype);
  if (rc) return rc;
  JG_REQUIRE(jg::dtype_size(grad_dtype) != 0, "%s: unknown gradient dtype %d", who, grad_dtype);
  JG_REQUIRE(sums && g && x && mean && rstd, "%s: NULL pointer", who);
  if ((rc = check_ws(who, workspace, workspace_bytes, batch, channels, spatial))) return rc;
  hipStream_t s = static_cast<hipStream_t>(stream);
#define CALL(DT) bwd_sums_launch<DT>(sums, sums + 1, 2, gw, gb, grad_dtype, g, x, mean, rstd, weight, batch, channels, spatial, groups, static_cast<float*>(workspace), s, who)
  JG_GN_DISPATCH(CALL)
#undef CALL
}

extern "C" int jg_gn_bwd_apply_x(void* gx, const void* g, const void* x, const void* weight, const float* mean,
                                 const float* rstd, const float* sums, const float* count, int64_t batch, int64_t channels,
                                 int64_t spatial, int64_t groups, int dtype, void* stream) {
  const char* who = "jg_gn_bwd_apply_x";
  int rc = check(who, batch, channels, spatial, groups, dtype);
  if (rc) return rc;
  JG_REQUIRE(gx && g && x && mean && rstd && sums && count, "%s: NULL pointer", who);
  hipStream_t s = static_cast<hipStream_t>(stream);
  ApplyArgs a = {};
  a.out = gx; a.in = g; a.in2 = x; a.mean = mean; a.rstd = rstd; a.gsum = sums; a.gxsum = sums + 1; a.stride = 2;
  a.cnt = count; a.weight = weight; a.C = (int)channels; a.G = (int)groups;
#define CALL(DT) apply_launch<DT, true, true>(a, batch, spatial, s, who)
  JG_GN_DISPATCH(CALL)
#undef CALL
}

extern "C" int jg_gn_partial_bwd(float* gsum, float* gxsum, float* gw, float* gb, const void* g,
                                 const void* x_norm, const void* weight, int64_t batch, int64_t channels,
                                 int64_t spatial, int64_t groups, int dtype, void* workspace,
                                 size_t workspace_bytes, void* stream) {
  const char* who = "jg_gn_partial_bwd";
  int rc = check(who, batch, channels, spatial, groups, dtype);
  if (rc) return rc;
  JG_REQUIRE(gsum && gxsum && g && x_norm, "%s: NULL pointer", who);
  if ((rc = check_ws(who, workspace, workspace_bytes, batch, channels, spatial))) return rc;
  hipStream_t s = static_cast<hipStream_t>(stream);
#define CALL(DT) bwd_sums_launch<DT>(gsum, gxsum, 1, gw, gb, JG_F32, g, x_norm, nullptr, nullptr, weight, batch, channels, spatial, groups, static_cast<float*>(workspace), s, who)
  JG_GN_DISPATCH(CALL)
#undef CALL
}

extern "C" int jg_gn_bwd_apply(void* gx, const void* g, const void* x_norm, const void* weight, const float* rstd,
                               const float* gsum, const float* gxsum, const float* count, int64_t batch,
                               int64_t channels, int64_t spatial, int64_t groups, int dtype, void* stream) {
  const char* who = "jg_gn_bwd_apply";
  int rc = check(who, batch, channels, spatial, groups, dtype);
  if (rc) return rc;
  JG_REQUIRE(gx && g && x_norm && rstd && gsum && gxsum && count, "%s: NULL pointer", who);
  hipStream_t s = static_cast<hipStream_t>(stream);
  ApplyArgs a = {};
  a.out = gx; a.in = g; a.in2 = x_norm; a.rstd = rstd; a.gsum = gsum; a.gxsum = gxsum; a.stride = 1;
  a.cnt = count; a.weight = weight; a.C = (int)channels; a.G = (int)groups;
#define CALL(DT) apply_launch<DT, true, false>(a, batch, spatial, s, who)
  JG_GN_DISPATCH(CALL)
#undef CALL
}
