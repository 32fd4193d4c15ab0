// Sums of partial results in fixed orders: the weight gradients of projections, the parameter gradients of a LayerNorm, the
// relative-position table of windowed attention. Each has a kernel of its own behind the one that writes the partials, and
// all of a backward's can be left for one launch at its end (jg_reduce_many): the same sums, whichever does them.
#pragma once
#include "jg_common.h"

namespace jg {

constexpr int RED_THREADS = 1024;
enum { RED_SLICES = 0, RED_COLUMNS = 1, RED_TABLE = 2 };

// Shared memory of a block of RED_THREADS.
union ReduceShared {
  float4 slices[16][64];
  float columns[2][16][16];
  float table[2][32][33];
};

// out[i] = sum over `parts` slices of part[k * count + i]. Group `sub` of W wavefronts (4, or 16 where there are many slices) takes
// outputs 256 block ..: a lane 4 values, wavefront w the slices w, w + W, ...; the W sums are added in order.
inline __host__ __device__ int slice_waves(int parts) { return parts >= 32 ? 16 : 4; }
template <int W, typename Store>
__device__ __forceinline__ void reduce_slices(float4 (*sm)[64], const float* part, size_t count, int parts, bool vec, size_t block, int grp, int q, Store store) {
  const size_t i0 = block * 256 + (size_t)q * 4;
  float acc[4] = {0.0f, 0.0f, 0.0f, 0.0f};
  if (i0 < count) {
    if (vec) {
#pragma unroll 4
      for (int k = grp; k < parts; k += W) {
        const float4 v = *reinterpret_cast<const float4*>(part + (size_t)k * count + i0);
        acc[0] += v.x;
        acc[1] += v.y;
        acc[2] += v.z;
        acc[3] += v.w;
      }
    } else {
      for (int k = grp; k < parts; k += W)
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (i0 + e < count) acc[e] += part[(size_t)k * count + i0 + e];
    }
  }
  sm[grp][q] = make_float4(acc[0], acc[1], acc[2], acc[3]);
  __syncthreads();
  if (grp != 0 || i0 >= count) return;
  float4 t = sm[0][q];
#pragma unroll
  for (int w = 1; w < W; ++w) {
    t.x += sm[w][q].x;
    t.y += sm[w][q].y;
    t.z += sm[w][q].z;
    t.w += sm[w][q].w;
  }
  store(i0, t);
}
__device__ __forceinline__ bool slices_vec(const float* part, const void* out, size_t count) {
  return (count & 3) == 0 && ((reinterpret_cast<uintptr_t>(part) | reinterpret_cast<uintptr_t>(out)) & 15) == 0;
}

// Column sums of partials part[k][which][col], k < n: a block of 1024 owns 16 consecutive columns, so that a wavefront reads 64 bytes
// of 4 partials at a time; its 16 wavefronts take the partials k = 4 w + lane / 16, ... + 64, ... in 4 independent chains
// each, and all chain sums are added in a fixed order. Bound by the latency of a chain: 1024 partials of
// 128 columns 7.2 us with 64 columns a block (two blocks), 4.9 us with 16.
constexpr int RED_COLS = 16, RED_WAVES = RED_THREADS / 64;
template <typename Store>
__device__ __forceinline__ void reduce_columns(float (*red)[RED_WAVES][RED_COLS], const float* part, int n, long long cols, unsigned block, Store store) {
  const int col = threadIdx.x % RED_COLS, first = threadIdx.x / RED_COLS;
  constexpr int STEP = 4 * RED_WAVES;  // partials the block reads at a time
  const long long c = (long long)block * RED_COLS + col;
  float a[4] = {0.f, 0.f, 0.f, 0.f}, b[4] = {0.f, 0.f, 0.f, 0.f};
  if (c < cols) {
    int k = first;
    for (; k + 3 * STEP < n; k += 4 * STEP) {
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        a[u] += part[((long long)(k + STEP * u) * 2 + 0) * cols + c];
        b[u] += part[((long long)(k + STEP * u) * 2 + 1) * cols + c];
      }
    }
    for (; k < n; k += STEP) {
      a[0] += part[((long long)k * 2 + 0) * cols + c];
      b[0] += part[((long long)k * 2 + 1) * cols + c];
    }
  }
  float sw = (a[0] + a[1]) + (a[2] + a[3]), sb = (b[0] + b[1]) + (b[2] + b[3]);
#pragma unroll
  for (int o = RED_COLS; o < 64; o <<= 1) {
    sw += __shfl_xor(sw, o, 64);
    sb += __shfl_xor(sb, o, 64);
  }
  if (first % 4 == 0) {
    red[0][first / 4][col] = sw;
    red[1][first / 4][col] = sb;
  }
  __syncthreads();
  if (first != 0 || c >= cols) return;
  sw = sb = 0.0f;
#pragma unroll
  for (int i = 0; i < RED_WAVES; ++i) {
    sw += red[0][i][col];
    sb += red[1][i][col];
  }
  store(c, sw, sb);
}

// Gradient of a (225, heads) table from the bins (workers, 2, 225) of the wavefronts that took windows of one head each, worker w of head
// w % heads. A block of 1024 takes 32 bins of one head: 32 lanes a bin pair each, 32 chunks of consecutive workers beside each other.
constexpr int RED_BINS = 225, RED_TABLE_BLOCKS = (RED_BINS + 31) / 32;  // of one head
__device__ __forceinline__ void reduce_table(float (*sm)[32][33], const float* bins, float* dtable, int workers, int heads, unsigned block) {
  const int head = block / RED_TABLE_BLOCKS, j = threadIdx.x & 31, chunk = threadIdx.x >> 5, i = (int)(block % RED_TABLE_BLOCKS) * 32 + j;
  const int mine = workers / heads, per = (mine + 31) / 32, g0 = chunk * per, g1 = min(g0 + per, mine);
  float lo = 0.0f, hi = 0.0f;
  if (i < RED_BINS) {
#pragma unroll 8
    for (int g = g0; g < g1; ++g) {
      const float* at = bins + ((size_t)g * heads + head) * (2 * RED_BINS) + i;
      lo += at[0];
      hi += at[RED_BINS];
    }
  }
  sm[0][chunk][j] = lo;
  sm[1][chunk][j] = hi;
  __syncthreads();
  if (chunk != 0 || i >= RED_BINS) return;
  float acc = 0.0f;
#pragma unroll
  for (int c = 0; c < 32; ++c) acc += sm[0][c][j] + sm[1][c][j];
  dtable[(size_t)i * heads + head] = acc;
}

inline unsigned reduction_blocks(const jg_reduction& r) {
  if (r.kind == RED_SLICES) return (unsigned)((r.count + (slice_waves(r.parts) == 16 ? 256 : 1024) - 1) / (slice_waves(r.parts) == 16 ? 256 : 1024));
  if (r.kind == RED_COLUMNS) return (unsigned)((r.count + RED_COLS - 1) / RED_COLS);
  return (unsigned)(r.count * RED_TABLE_BLOCKS);
}
// `later` with one more job, or JG_ERR_BAD_ARG where there is no room.
inline int add_reduction(jg_reductions* later, int kind, int parts, int64_t count, const float* part, float* out, float* out2) {
  JG_REQUIRE(later->n >= 0 && later->n < JG_MOST_REDUCTIONS, "reductions: more than %d left for later", JG_MOST_REDUCTIONS);
  jg_reduction& r = later->job[later->n++];
  r.kind = kind;
  r.parts = parts;
  r.count = count;
  r.part = part;
  r.out = out;
  r.out2 = out2;
  return JG_OK;
}

}  // namespace jg
