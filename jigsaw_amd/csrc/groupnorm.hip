// GroupNorm over a spatially sharded input: the per-(sample, group) partial sums that
// the ranks add up, the normalise + affine pass, and the backward partials and pass.
// x is (N, C, S) contiguous (S = product of the local spatial extents); a group is
// C / G consecutive channels, so the elements of one (sample, group) are one contiguous
// span. Everything is HBM-bound: 16-byte loads, fp32 accumulation, block partials that a
// second small kernel adds up in a fixed order (deterministic, no atomics).
//
// Passes over the tensor: forward two (the moments of every group from ONE pass, centred on a
// sample of the block's own elements; normalise + affine), backward two (the sums; the input
// gradient), both from x and the statistics, x_hat recomputed in fp32 on the way. x_hat itself
// is only written for a caller that asks for it (jg_gn_apply with x_norm, jg_gn_partial_bwd,
// jg_gn_bwd_apply): it is rounded, and the backward is less exact from it. A step whose backward takes x
// keeps a copy of it (jg_gn_apply_keep, jg_gn_forward_keep), which the second pass writes beside y: the caller
// may change x before the backward. On 8 x 64 x 1024^2 bf16, 8 groups (1.07 GB a tensor) forward +
// backward is 1.80 ms = 5.4 TB/s over nine tensors, what a copy reaches; 1.55 ms without the copy, 2.17 ms with
// three passes forward and x_hat stored. Both passes of a sample before the next one, to find its tensor in the
// last-level cache, were tried: 0.12 ms more (eight launches that are each too small to fill the memory system).
// Rows and spans start anywhere (S need not be a multiple of 8): a block takes the whole 16-byte
// words of its range as vectors and the elements before the first and behind the last one by one.
//
// Reference behaviour restated here:
//   jigsaw/modules/normalization/_functional.py:352-385 (forward: sum, centred squares, apply)
//   jigsaw/modules/normalization/_functional.py:431-468 (backward)
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
  __device__ static __forceinline__ uint16_t down(float v) { return jg::f32_to_bf16(v); }
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

// MODE 0: part[0] = sum x                      over a chunk of a (sample, group) span
// MODE 1: part[0] = sum (x - mean[unit])^2      "
// MODE 2: part[0] = sum g, part[1] = sum g * y  over a chunk of a (sample, channel) row
// MODE 3: part[0] = sum g, part[1] = sum g * (y - mean[seg]) * rstd[seg], seg the (sample, group) of the row
// Partials at part[blockIdx.x * 2 + {0, 1}].
template <int DT, int MODE>
__global__ __launch_bounds__(kThreads) void gn_reduce_kernel(float* __restrict__ part,
                                                             const typename Elem<DT>::T* __restrict__ x,
                                                             const typename Elem<DT>::T* __restrict__ y,
                                                             const float* __restrict__ mean, const float* __restrict__ rstd,
                                                             int channels_per_group, long long len,
                                                             int chunks, long long chunk_len, bool vec_ok) {
  constexpr int V = Elem<DT>::VEC;
  long long unit, lo, hi;
  chunk_range(blockIdx.x, len, chunks, chunk_len, &unit, &lo, &hi);
  const float m = MODE == 1 ? mean[unit] : MODE == 3 ? mean[unit / channels_per_group] : 0.0f;
  float a = 0.0f, b = 0.0f;
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
  if (threadIdx.x == 0) {
    part[(size_t)blockIdx.x * 2 + 0] = a;
    part[(size_t)blockIdx.x * 2 + 1] = MODE == 3 ? b * rstd[unit / channels_per_group] : b;
  }
}

// Moments of a chunk in one pass: part = (mean, sum of squares about it). The sums are centred on the mean of the
// chunk's first (up to) 256 elements, so that the square of the mean does not swamp the variance.
template <int DT>
__global__ __launch_bounds__(kThreads) void gn_moments_kernel(float* __restrict__ part, const typename Elem<DT>::T* __restrict__ x,
                                                              long long len, int chunks, long long chunk_len, bool vec_ok) {
  constexpr int V = Elem<DT>::VEC;
  __shared__ float centre_s;
  long long unit, lo, hi;
  chunk_range(blockIdx.x, len, chunks, chunk_len, &unit, &lo, &hi);
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
  if (threadIdx.x == 0) {
    const float shift = n > 0 ? a / (float)n : 0.0f;
    part[(size_t)blockIdx.x * 2 + 0] = centre + shift;
    part[(size_t)blockIdx.x * 2 + 1] = n > 0 ? fmaxf(b - a * shift, 0.0f) : 0.0f;
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

// Forward:  x_norm = (x - mean) * rstd, y = x_norm * w[c] + b[c]
// Backward: gx = rstd * (g * w[c] - gsum / cnt - x_norm * gxsum / cnt); FROM_X: x_norm from x as in the forward
template <int DT, bool BWD, bool FROM_X>
__global__ __launch_bounds__(kThreads) void gn_apply_kernel(ApplyArgs p, long long S, int chunks, long long chunk_len, bool vec_ok) {
  typedef typename Elem<DT>::T T;
  constexpr int V = Elem<DT>::VEC;
  long long row, lo, hi;
  // Last block first: the pass before read the tensors from front to back, so that their ends are what the last-level
  // cache still holds.
  chunk_range(gridDim.x - 1 - blockIdx.x, S, chunks, chunk_len, &row, &lo, &hi);
  const int c = (int)(row % p.C);
  const long long seg = row / p.C * p.G + c / (p.C / p.G);
  const float w = p.weight != nullptr ? Elem<DT>::up(static_cast<const T*>(p.weight)[c]) : 1.0f;
  const float bv = (!BWD && p.bias != nullptr) ? Elem<DT>::up(static_cast<const T*>(p.bias)[c]) : 0.0f;
  const float m = BWD && !FROM_X ? 0.0f : p.mean[seg], rs = p.rstd[seg];
  const float inv = BWD ? 1.0f / (p.cnt != nullptr ? p.cnt[seg] : p.count) : 0.0f;
  const float q1 = BWD ? p.gsum[seg * p.stride] * inv : 0.0f, q2 = BWD ? p.gxsum[seg * p.stride] * inv : 0.0f;
  const T* in = static_cast<const T*>(p.in);
  const T* in2 = static_cast<const T*>(p.in2);
  T* out = static_cast<T*>(p.out);
  T* norm = static_cast<T*>(p.out_norm);
  T* kept = static_cast<T*>(p.out_kept);
  // forward: (y, x_norm): x_norm is rounded to the compute dtype and y computed from the rounded value, as the
  // reference computes y from the x_norm tensor
  auto forward = [&](float v, float& xn) {
    xn = Elem<DT>::up(Elem<DT>::down((v - m) * rs));
    return xn * w + bv;
  };
  auto backward = [&](float g, float x) { return rs * (g * w - q1 - (FROM_X ? (x - m) * rs : x) * q2); };
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

int check_ws(const char* who, const void* ws, size_t bytes, int64_t batch, int64_t channels, int64_t spatial) {
  const size_t need = batch <= 0 || channels <= 0 || spatial <= 0 ? 256 : ws_need(batch, channels, spatial);
  if (ws == nullptr || bytes < need) JG_FAIL(JG_ERR_WORKSPACE, "%s: workspace %zu < %zu bytes", who, bytes, need);
  return JG_OK;
}

}  // namespace

extern "C" size_t jg_gn_workspace_bytes(int64_t batch, int64_t channels, int64_t spatial) {
  if (batch <= 0 || channels <= 0 || spatial <= 0) return 256;
  return ws_need(batch, channels, spatial);
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
                long long C, long long S, long long G, float eps, float* ws, hipStream_t s, const char* who) {
  int rc = moments_launch<DT>(mean, nullptr, nullptr, rstd, x, N * G, C / G * S, eps, ws, s, who);
  if (rc) return rc;
  ApplyArgs a = {};
  a.out = y; a.out_kept = x_kept; a.in = x; a.mean = mean; a.rstd = rstd; a.weight = weight; a.bias = bias; a.C = (int)C; a.G = (int)G;
  return apply_launch<DT, false, true>(a, N, S, s, who);
}

template <int DT>
int backward_all(void* gx, void* gw, void* gb, int wdtype, const void* g, const void* x, const float* mean, const float* rstd,
                 const void* weight, long long N, long long C, long long S, long long G, float* ws, hipStream_t s, const char* who) {
  const long long rows = N * C;
  float* sums = ws + (size_t)rows * chunks_of(S) * 2;
  int rc = bwd_sums_launch<DT>(sums, sums + 1, 2, gw, gb, wdtype, g, x, mean, rstd, weight, N, C, S, G, ws, s, who);
  if (rc || gx == nullptr) return rc;
  ApplyArgs a = {};
  a.out = gx; a.in = g; a.in2 = x; a.mean = mean; a.rstd = rstd; a.gsum = sums; a.gxsum = sums + 1; a.stride = 2;
  a.count = (float)(C / G * S);
  a.weight = weight; a.C = (int)C; a.G = (int)G;
  return apply_launch<DT, true, true>(a, N, S, s, who);
}
}  // namespace

extern "C" int jg_gn_forward(void* y, float* mean, float* rstd, const void* x, const void* weight, const void* bias,
                             int64_t batch, int64_t channels, int64_t spatial, int64_t groups, float eps, int dtype,
                             void* workspace, size_t workspace_bytes, void* stream) {
  return jg_gn_forward_keep(y, nullptr, mean, rstd, x, weight, bias, batch, channels, spatial, groups, eps, dtype, workspace,
                            workspace_bytes, stream);
}

extern "C" int jg_gn_forward_keep(void* y, void* x_kept, float* mean, float* rstd, const void* x, const void* weight,
                                  const void* bias, int64_t batch, int64_t channels, int64_t spatial, int64_t groups,
                                  float eps, int dtype, void* workspace, size_t workspace_bytes, void* stream) {
  const char* who = "jg_gn_forward";
  int rc = check(who, batch, channels, spatial, groups, dtype);
  if (rc) return rc;
  JG_REQUIRE(y && mean && rstd && x, "%s: NULL pointer", who);
  if ((rc = check_ws(who, workspace, workspace_bytes, batch, channels, spatial))) return rc;
  hipStream_t s = static_cast<hipStream_t>(stream);
#define CALL(DT) forward_all<DT>(y, x_kept, mean, rstd, x, weight, bias, batch, channels, spatial, groups, eps, static_cast<float*>(workspace), s, who)
  JG_GN_DISPATCH(CALL)
#undef CALL
}

extern "C" int jg_gn_backward(void* gx, void* gw, void* gb, const void* g, const void* x, const float* mean,
                              const float* rstd, const void* weight, int64_t batch, int64_t channels, int64_t spatial,
                              int64_t groups, int dtype, int grad_dtype, void* workspace, size_t workspace_bytes,
                              void* stream) {
  const char* who = "jg_gn_backward";
  int rc = check(who, batch, channels, spatial, groups, dtype);
  if (rc) return rc;
  JG_REQUIRE(jg::dtype_size(grad_dtype) != 0, "%s: unknown gradient dtype %d", who, grad_dtype);
  JG_REQUIRE(g && x && mean && rstd, "%s: NULL pointer", who);
  if ((rc = check_ws(who, workspace, workspace_bytes, batch, channels, spatial))) return rc;
  hipStream_t s = static_cast<hipStream_t>(stream);
#define CALL(DT) backward_all<DT>(gx, gw, gb, grad_dtype, g, x, mean, rstd, weight, batch, channels, spatial, groups, static_cast<float*>(workspace), s, who)
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
