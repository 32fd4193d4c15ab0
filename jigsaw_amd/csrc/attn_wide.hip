// Blockwise (flash-style) attention over the K/V chunks of a ring on the bf16 / fp16 matrix cores for
// head sizes up to 128 (multiples of 8), any lengths, non-causal, no bias: forward (output +
// natural-log LSE) and backward from a given (global) output and LSE. Same arithmetic as the
// bf16 kernels of head size 64, written for clarity rather than hand-scheduled: tiles of 32 keys
// (forward, dQ) or 32 queries (dK/dV) pass through a double-buffered LDS stage, fetched to
// registers one tile ahead.
//
//   widths         kernels of 32, 64, 96 and 128 columns (D); a smaller head is staged with zeros in
//                  the columns it does not have. Rows past the end of a tensor are staged as zeros
//                  too; keys past the end get the score -inf, queries past the end the lse +inf.
//   groups         a workgroup is KS groups of W wavefronts. A group walks every KS-th tile of
//                  the streamed side with a stage of its own, and the groups' sums are combined
//                  through LDS at the end: where a launch has fewer workgroups than the chip has
//                  CUs, more wavefronts share the rows of one (see two_groups on the host side), and
//                  where it has fewer than half, workgroups have 64 or 32 rows (attn_width).
//
// Forward + backward of a ring, before (lengths and head size padded on the host, one launch and one merge per
// chunk) and in one launch each: 4 heads x 128 x 2 chunks of 128 keys, head size 32: 402 -> 48 us (host time); 12 heads x 869 x 869,
// head size 96, fp16: 528 -> 99 us; 16 heads x 2424 x 2424, head size 32, fp16: 568 -> 225 us.
//
//   forward / dQ   lane = query. S^T = K Q^T (A = K rows from LDS, B = Q rows kept in
//                  registers), so the running max / sum, lse and delta of a query are
//                  scalars of the two lanes that share it. P^T (or dS^T) leaves the
//                  accumulator already in B-fragment position for O^T += V^T P^T
//                  (dQ^T += K^T dS^T): the A operand comes from the same tile by LDS transpose
//                  reads, its 16 rows in the order the accumulator holds them.
//   dK / dV        lane = key. S = Q K^T and dP = dO V^T with K, V rows in registers;
//                  lse and delta of the tile's queries are read from LDS per accumulator
//                  row; dV^T += dO^T P and dK^T += Q^T dS by transpose reads of the dO
//                  and Q tiles.
//
// A transposed copy of the tile beside it, fetched and written a second time, had these kernels at (copy : transpose reads, with the loads
// above and two tiles a round; forward / dQ / dK and dV, us) 6 heads x 4050 x 4 chunks, head size 80 460 / 559 / 931 : 312 / 336 / 366; 24 x 1000 x 2, 128
// 65 / 83 / 125 : 57 / 61 / 106; 24 x 739 x 5, 32 54 / 62 / 52 : 45 / 43 / 30; 8 x 4096 x 2, fp16 64 193 / 240 / 195 : 165 / 156 / 161. What is
// left is one chain per wavefront, scores, exponentials, products, with two wavefronts a SIMD to fill its gaps, and, up to 64 columns where the
// chip is full, a second block of rows in each (launch_fwd, launch_dq).
//
// Reference behaviour restated here:
//   jigsaw/modules/attention/_functional/cores/math.py:69-78   (forward)
//   jigsaw/modules/attention/_functional/cores/math.py:125-149 (backward)
#include <algorithm>
#include <type_traits>

#include "attn_chunks.h"

namespace {

using jg::BlockOf;
using jg::ChunkTable;
using jg::block_of;
using jg::chunk_entry;
using jg::parts8;

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef short i16x4 __attribute__((ext_vector_type(4)));

// W: wavefronts of a group. A workgroup has 32 W rows (queries or keys), 32 per wavefront of a group, a group 64 W threads.
constexpr int BT = 32;          // rows of a streamed tile
constexpr float LOG2E = 1.4426950408889634f;
constexpr float NO_SCORE = -1.0e30f;  // running maximum before the first key: finite, so that a group without a key weighs 0

template <int D>
struct Geo {
  static constexpr int C16 = D / 16, NB = D / 32;
  static constexpr int RP = D * 2;  // bytes per row of a tile (32 rows of D)
  static constexpr int TILE = BT * RP;
  // Row r has its 16-byte pieces XOR-ed with swizzle(r). The 16 rows a row fragment's read takes at a time then meet all banks once, and so do
  // the 64 bytes of 4 rows of a transposed fragment. (Rows 16 bytes apart instead: two to a bank there; dQ of 8 heads x 4096 x 2 chunks at head
  // size 96 270 : 240 us, fp16 64 211 : 188.)
  __device__ static __forceinline__ int swizzle(int r) { return ((r >> 2) & 3) | (D == 64 ? ((r >> 1) & 1) << 2 : (D == 128 ? (r & 3) << 2 : 0)); }
  static constexpr int RV = D == 64 ? 4 : (D == 128 ? 8 : 2), TV = RV / 2;  // pieces, and blocks of 32 columns, whose swizzles differ
  static constexpr int CHUNKS = BT * D / 8;  // 16-byte pieces of a tile
  static constexpr int DOTS = D == 96 ? 3 : 1;  // sums that a row's dot product comes in (tile_row_dots)
};

template <int D, int W>
struct TileRegs {
  static constexpr int GROUP = W * 64, PER = (Geo<D>::CHUNKS + GROUP - 1) / GROUP;
  u32x4 v[PER];
  int rows;
};

// 32 rows of a row-major matrix of row length d <= D to registers; rows from `rows` on and columns from d on become zero on their way to LDS.
// (REPEAT: such rows are the last row there is.) They are read from the last row and piece there is: a load under a condition is waited for where the paths meet, on the spot (24 heads x
// 739 x 5 chunks, head size 32: forward 63 -> 48 us, dQ 54 -> 46). tid: thread of the group; at least one row lies before `rows`.
template <int D, int W>
__device__ __forceinline__ void tile_fetch(TileRegs<D, W>& r, const uint16_t* src, int tid, int rows, int d) {
  r.rows = rows;
#pragma unroll
  for (int i = 0; i < TileRegs<D, W>::PER; ++i) {
    const int c = min(tid + i * (W * 64), Geo<D>::CHUNKS - 1);
    r.v[i] = *reinterpret_cast<const u32x4*>(src + min(c / (D / 8), rows - 1) * d + min(c % (D / 8) * 8, d - 8));
  }
}
template <int D, int W, bool REPEAT = false>
__device__ __forceinline__ void tile_store(const TileRegs<D, W>& r, unsigned char* dst, int tid, int d) {
#pragma unroll
  for (int i = 0; i < TileRegs<D, W>::PER; ++i) {
    const int c = tid + i * (W * 64);
    if (c < Geo<D>::CHUNKS) {
      const int row = c / (D / 8), piece = c % (D / 8);
      const bool there = (REPEAT || row < r.rows) && piece * 8 < d;
      u32x4 v;
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = there ? r.v[i][e] : 0u;
      *reinterpret_cast<u32x4*>(dst + row * Geo<D>::RP + ((piece ^ Geo<D>::swizzle(row)) << 4)) = v;
    }
  }
}

// dots[row] = sum over the columns of a b for the rows of two fetched tiles, zero for rows and without columns that do not exist. The lanes of a
// row's pieces lie behind each other: a tree over them, or, 12 of them, over each four: three sums, dots[32 i + row].
template <int D, bool F16, int W>
__device__ __forceinline__ void tile_row_dots(const TileRegs<D, W>& a, const TileRegs<D, W>& b, float* dots, int tid, int d);

__device__ __forceinline__ f32x16 zero16() {
  f32x16 z;
#pragma unroll
  for (int i = 0; i < 16; ++i) z[i] = 0.0f;
  return z;
}
// The 16-bit element type of q, k, v: bf16 or fp16. Both have a 32x32x16 MFMA with the same operand
// layout; they differ in the conversions from and to fp32.
template <bool F16>
struct Half;
template <>
struct Half<false> {
  typedef bf16x8 x8;
  __device__ static __forceinline__ f32x16 mma(x8 a, x8 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
  }
  __device__ static __forceinline__ uint32_t pair(float a, float b) {
    const f32x2 v = {a, b};
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2));
  }
  __device__ static __forceinline__ void unpair(uint32_t w, float& a, float& b) {
    a = __uint_as_float(w << 16);
    b = __uint_as_float(w & 0xffff0000u);
  }
};
template <>
struct Half<true> {
  typedef f16x8 x8;
  __device__ static __forceinline__ f32x16 mma(x8 a, x8 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
  }
  __device__ static __forceinline__ uint32_t pair(float a, float b) {
    const f32x2 v = {a, b};
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, f16x2));
  }
  __device__ static __forceinline__ void unpair(uint32_t w, float& a, float& b) {
    const f32x2 v = __builtin_convertvector(__builtin_bit_cast(f16x2, w), f32x2);
    a = v.x;
    b = v.y;
  }
};
template <bool F16>
__device__ __forceinline__ typename Half<F16>::x8 frag(const unsigned char* at) {
  return __builtin_bit_cast(typename Half<F16>::x8, *reinterpret_cast<const u32x4*>(at));
}
template <int D, bool F16, int W>
__device__ __forceinline__ void tile_row_dots(const TileRegs<D, W>& a, const TileRegs<D, W>& b, float* dots, int tid, int d) {
  constexpr int PIECES = D / 8, TREE = PIECES / Geo<D>::DOTS;
  static_assert((TREE & (TREE - 1)) == 0, "a power of two");
#pragma unroll
  for (int i = 0; i < TileRegs<D, W>::PER; ++i) {
    const int c = tid + i * (W * 64), row = c / PIECES, piece = c % PIECES;
    float sum = 0.0f;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      float a0, a1, b0, b1;
      Half<F16>::unpair(a.v[i][e], a0, a1);
      Half<F16>::unpair(b.v[i][e], b0, b1);
      sum = __builtin_fmaf(a0, b0, sum);
      sum = __builtin_fmaf(a1, b1, sum);
    }
    sum = row < a.rows && piece * 8 < d ? sum : 0.0f;
#pragma unroll
    for (int o = 1; o < TREE; o <<= 1) sum += __shfl_xor(sum, o, 64);
    if (piece % TREE == 0 && c < Geo<D>::CHUNKS) dots[piece / TREE * BT + row] = sum;
  }
}
// Where a lane finds its parts of a tile: fragments of row ln (columns 16 c + 8 kg + 0..7), and transposed ones by LDS transpose reads (within
// 16 lanes, lane i receives element i % 4 of the 8 bytes that lanes i / 4 + 4 j point at, j = 0..3): lane (ln, kg) gets column ln of
// block nb and, of 16 rows, rows 4 kg + 0..3 and 8 + 4 kg + 0..3, the order in which an accumulator lane holds its rows.
template <int D, bool F16>
struct TileView {
  typedef Geo<D> G;
  typedef typename Half<F16>::x8 X8;
  int row[G::RV], lo[G::TV], hi[G::TV];
  __device__ __forceinline__ explicit TileView(int lane) {
    const int ln = lane & 31, kg = lane >> 5, p = lane & 15, r = 4 * kg + (p >> 2);
#pragma unroll
    for (int c = 0; c < G::RV; ++c) row[c] = ln * G::RP + (((2 * c + kg) ^ G::swizzle(ln)) << 4);
#pragma unroll
    for (int v = 0; v < G::TV; ++v) {
      const int piece = 4 * v + ((lane >> 4) & 1) * 2 + ((p >> 1) & 1);
      lo[v] = r * G::RP + ((piece ^ G::swizzle(r)) << 4) + 8 * (p & 1);
      hi[v] = (r + 8) * G::RP + ((piece ^ G::swizzle(r + 8)) << 4) + 8 * (p & 1);
    }
  }
  __device__ __forceinline__ X8 rows(const unsigned char* tile, int c) const { return frag<F16>(tile + row[c % G::RV] + c / G::RV * 64); }
  __device__ __forceinline__ X8 trans(const unsigned char* tile, int nb, int half) const {  // rows 16 half + ...
    typedef __attribute__((address_space(3))) i16x4* tr_ptr;
    const unsigned char* const at = tile + nb / G::TV * 64 + half * 16 * G::RP;
    const i16x4 l = __builtin_amdgcn_ds_read_tr16_b64_v4i16((tr_ptr)(at + lo[nb % G::TV])), h = __builtin_amdgcn_ds_read_tr16_b64_v4i16((tr_ptr)(at + hi[nb % G::TV]));
    u32x4 w;
    w.x = __builtin_bit_cast(u32x2, l).x;
    w.y = __builtin_bit_cast(u32x2, l).y;
    w.z = __builtin_bit_cast(u32x2, h).x;
    w.w = __builtin_bit_cast(u32x2, h).y;
    return __builtin_bit_cast(X8, w);
  }
};
template <bool F16>
__device__ __forceinline__ typename Half<F16>::x8 pack8(const float* v) {
  u32x4 r;
  r.x = Half<F16>::pair(v[0], v[1]);
  r.y = Half<F16>::pair(v[2], v[3]);
  r.z = Half<F16>::pair(v[4], v[5]);
  r.w = Half<F16>::pair(v[6], v[7]);
  return __builtin_bit_cast(typename Half<F16>::x8, r);
}
template <bool F16>
__device__ __forceinline__ u32x2 pack4(float a, float b, float c, float d) {
  u32x2 r;
  r.x = Half<F16>::pair(a, b);
  r.y = Half<F16>::pair(c, d);
  return r;
}

// c + a x v for eight fp32 values in B-fragment position, none of them rounded (see parts8). A bf16 fragment goes in
// as it is; an fp16 one as two bf16 parts, which hold its 11 bits and its whole range.
template <bool F16>
__device__ __forceinline__ f32x16 mma_exact(typename Half<F16>::x8 a, const bf16x8 (&part)[3], f32x16 c) {
  if constexpr (!F16) {
#pragma unroll
    for (int t = 2; t >= 0; --t) c = Half<false>::mma(a, part[t], c);
  } else {
    bf16x8 hi, lo;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float f = (float)a[e];
      hi[e] = (__bf16)f;
      const float h = (float)hi[e];
      lo[e] = (__bf16)(f == h ? 0.0f : f - h);
    }
#pragma unroll
    for (int t = 2; t >= 0; --t) {
      c = Half<false>::mma(lo, part[t], c);
      c = Half<false>::mma(hi, part[t], c);
    }
  }
  return c;
}

// 16-byte piece `col` / 8 of a row in memory, zero past the head's columns
template <int D, bool F16>
__device__ __forceinline__ typename Half<F16>::x8 row_frag(const uint16_t* row, int col, int d) {
  u32x4 v = {0u, 0u, 0u, 0u};
  if (col < d) v = *reinterpret_cast<const u32x4*>(row + col);
  return __builtin_bit_cast(typename Half<F16>::x8, v);
}

// Which tile of which chunk a group takes next: number ks, ks + KS, ... of the tiles of the rows lo .. hi - 1 of all chunks in their order. Every
// group makes `steps` steps; in a step past the last tile rows_left is <= 0. (Tiles ks, ks + KS, ... of each chunk by itself left most groups
// without one wherever a chunk has few, above all in the exact pass, whose chunks have one to four: forward of 7 heads x 387 x 6 chunks,
// bf16 64 32.8 -> 19.6 us, 36 x 69 x 7 at 64 19.1 -> 11.4, 8 x 397 x 7 at 64 37.8 -> 23.4, 12 x 131 x 5 at 96 19.7 -> 15.7; launches of one group as before.) ks: wave-uniform.
template <int KS>
struct Stream {
  int steps, lo, hi, per_chunk, chunks, tile, chunk;
  int by_chunks, by_tiles;  // KS tiles on are so many chunks and tiles: a step is a few selects and no branch, which the tile's instructions could not pass
  __device__ Stream(int lo_, int hi_, int chunks_, int ks) : lo(lo_), hi(hi_), per_chunk((hi_ - lo_ + BT - 1) / BT), chunks(chunks_) {
    steps = (per_chunk * chunks + KS - 1) / KS;
    by_chunks = KS / per_chunk;
    by_tiles = KS - by_chunks * per_chunk;
    chunk = ks / per_chunk;
    tile = ks - chunk * per_chunk;
    clamp();
  }
  __device__ __forceinline__ int first_row() const { return lo + tile * BT; }
  __device__ __forceinline__ int rows_left() const { return hi - first_row(); }
  __device__ __forceinline__ void clamp() {  // past the last tile: the one behind it, which has no row
    const bool past = chunk >= chunks;
    tile = past ? per_chunk : tile;
    chunk = past ? chunks - 1 : chunk;
  }
  __device__ __forceinline__ void next() {
    tile += KS == 1 ? 1 : by_tiles;
    chunk += KS == 1 ? 0 : by_chunks;
    const bool over = tile >= per_chunk;
    tile -= over ? per_chunk : 0;
    chunk += over ? 1 : 0;
    if (KS > 1) clamp();
  }
};

struct Args {
  const uint16_t* q;
  const uint16_t* out;   // backward: the global output
  const uint16_t* dout;  // backward
  const float* lse_in;   // backward: the global lse
  float* delta;          // backward workspace (batch, sq): written by the dQ kernel, read by the dK/dV kernel (not where they are one launch)
  uint16_t* o;           // forward output, or NULL when only the merge is wanted
  float* lse;            // forward output, or NULL
  float* out_acc;        // forward: fp32 (batch, sq, d) accumulator of the ring, merged in place, or NULL
  float* lse_acc;        // forward: fp32 (batch, sq), merged in place, or NULL
  uint16_t* dq;
  int sq, sk;            // sk: keys per chunk
  int d;                 // columns of a head, <= D and a multiple of 8
  int nchunks;
  int exact_from;        // forward: first key of a chunk whose probabilities are not rounded (see exact_from())
  float scale;
};

// The larger of a lane's value and that of lane ^ 32, by a swap of registers instead of a round trip through LDS.
__device__ __forceinline__ float pair_max(float v) {
  const uint32_t bits = __float_as_uint(v);
  const auto both = __builtin_amdgcn_permlane32_swap(bits, bits, false, false);
  return fmaxf(__uint_as_float(both[0]), __uint_as_float(both[1]));
}

// ------------------------------------------------------------------- forward
// EXACT: some keys' probabilities are not rounded (p.exact_from < p.sk). A second loop and kernels of their own: with the
// choice inside the one loop every tile took 4 to 10 % longer, with both loops in every kernel up to 7 % (head sizes 96
// and 128, lengths that are multiples of 128).
// What it costs, forward / backward of 64 heads x 100 queries x 8 chunks of 100 keys, rounded -> not: bf16, head size 64
// 33 / 52 -> 34 / 58 us, 96 34 / 62 -> 40 / 78, 128 (127 keys) 35 / 86 -> 49 / 102; fp16, whose operands go in as two parts, 64
// 34 / 52 -> 45 / 79. The one-thread-per-row kernels, which these chunks ran before, took 1107 / 2418 us at bf16 64, eight launches each way.
// QB: blocks of 32 queries a wavefront. With two, a fragment from LDS feeds two matrix instructions, and the scores and products of one block run
// under the exponentials of the other; one block leaves both to what other wavefronts the SIMD holds.
template <int D, bool F16, int W, int KS, bool EXACT, int QB>
__global__ __launch_bounds__(64 * W * KS) void attn_wide_fwd_kernel(ChunkTable, Args p) {
  typedef Geo<D> G;
  typedef typename Half<F16>::x8 X8;
  constexpr int BUF = 2 * G::TILE;  // K tile, V tile
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const int tid = threadIdx.x % (64 * W), ks = __builtin_amdgcn_readfirstlane(threadIdx.x / (64 * W));
  const int lane = tid & 63, wave = tid >> 6;
  const int ln = lane & 31, kg = lane >> 5;
  const BlockOf wg = block_of();
  const long long bh = wg.bh;
  const int q0 = wg.blk * (32 * W * QB) + wave * (32 * QB) + ln;  // and q0 + 32, ..
  const long long chunk_off = bh * p.sk * p.d;
  const float c2 = p.scale * LOG2E;
  unsigned char* lds = smem + ks * 2 * BUF;
  const TileView<D, F16> view(lane);

  X8 qf[QB][G::C16];
  f32x16 o[QB][G::NB];
  float m[QB], l[QB];
#pragma unroll
  for (int qb = 0; qb < QB; ++qb) {
    const uint16_t* qrow = p.q + (bh * p.sq + min(q0 + 32 * qb, p.sq - 1)) * p.d;
#pragma unroll
    for (int c = 0; c < G::C16; ++c) qf[qb][c] = row_frag<D, F16>(qrow, 16 * c + 8 * kg, p.d);
#pragma unroll
    for (int nb = 0; nb < G::NB; ++nb) o[qb][nb] = zero16();
    m[qb] = NO_SCORE;
    l[qb] = 0.0f;
  }

#pragma unroll
  for (int pass = 0; pass < (EXACT ? 2 : 1); ++pass) {
    // the keys lo .. hi - 1 of every chunk
    const bool exact = EXACT && pass == 1;
    const int lo = exact ? p.exact_from : 0, hi = EXACT && !exact ? p.exact_from : p.sk;
    if (EXACT && lo == hi) continue;
    TileRegs<D, W> rk, rv;
    Stream<KS> load(lo, hi, p.nchunks, ks), soft(lo, hi, p.nchunks, ks);
    const int ntiles = load.steps;
    auto fetch = [&]() {
      const uint16_t* kb = reinterpret_cast<const uint16_t*>(chunk_entry(0, load.chunk)) + chunk_off;
      const uint16_t* vb = reinterpret_cast<const uint16_t*>(chunk_entry(1, load.chunk)) + chunk_off;
      const long long at = (long long)load.first_row() * p.d;
      tile_fetch<D, W>(rk, kb + at, tid, load.rows_left(), p.d);
      tile_fetch<D, W>(rv, vb + at, tid, load.rows_left(), p.d);
      load.next();
    };
    auto store = [&](int buf) {
      tile_store<D, W>(rk, lds + buf * BUF, tid, p.d);
      tile_store<D, W>(rv, lds + buf * BUF + G::TILE, tid, p.d);
    };
    fetch();
    store(0);
    // The fragments that came straight from memory are waited for here, once. Left to the first matrix
    // instruction that reads them, the wait sits inside the loop, behind the tile loads every iteration has
    // just issued, and counts those too: each iteration then waited for its own prefetch.
#pragma unroll
    for (int qb = 0; qb < QB; ++qb)
#pragma unroll
      for (int c = 0; c < G::C16; ++c) asm volatile("" : "+v"(qf[qb][c]));
    __syncthreads();
    auto tile = [&](int t, int buf) __attribute__((always_inline)) {
      const unsigned char* kt = lds + buf * BUF;
      const unsigned char* vt = kt + G::TILE;
      if (t + 1 < ntiles) fetch();
      // S^T: lane = query ln, register i = key 8*(i/4) + 4*kg + i%4 of the tile
      f32x16 s[QB];
#pragma unroll
      for (int qb = 0; qb < QB; ++qb) s[qb] = zero16();
#pragma unroll
      for (int c = 0; c < G::C16; ++c) {
        const X8 kf = view.rows(kt, c);
#pragma unroll
        for (int qb = 0; qb < QB; ++qb) s[qb] = Half<F16>::mma(kf, qf[qb][c], s[qb]);
      }
      if (soft.rows_left() < BT) {  // wave-uniform
#pragma unroll
        for (int qb = 0; qb < QB; ++qb)
#pragma unroll
          for (int i = 0; i < 16; ++i)
            if (8 * (i >> 2) + 4 * kg + (i & 3) >= soft.rows_left()) s[qb][i] = -INFINITY;
      }
      soft.next();
#pragma unroll
      for (int qb = 0; qb < QB; ++qb) {
        const f32x16& sc = s[qb];
        // maxima of three: one instruction for two comparisons
        auto max3 = [](float a, float b, float c) { return fmaxf(fmaxf(a, b), c); };
        const float t0 = max3(sc[0], sc[1], sc[2]), t1 = max3(sc[3], sc[4], sc[5]), t2 = max3(sc[6], sc[7], sc[8]);
        const float t3 = max3(sc[9], sc[10], sc[11]), t4 = max3(sc[12], sc[13], sc[14]);
        const float mx = max3(max3(t0, t1, t2), max3(t3, t4, sc[15]), m[qb]);  // of the lane's own 16 keys and those before
        // the maximum settles after a few tiles: the other half's keys and a rescale only when some query of the wavefront saw a larger score
        if (__builtin_amdgcn_ballot_w64(mx > m[qb]) != 0) {
          const float mn = pair_max(mx);
          const float alpha = __builtin_amdgcn_exp2f((m[qb] - mn) * c2);  // first tile: 0
          l[qb] *= alpha;
#pragma unroll
          for (int nb = 0; nb < G::NB; ++nb)
#pragma unroll
            for (int i = 0; i < 16; ++i) o[qb][nb][i] *= alpha;
          m[qb] = mn;
        }
        const float off = m[qb] * c2;
        float pr[16], sum[2] = {0.0f, 0.0f};
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          pr[i] = __builtin_amdgcn_exp2f(sc[i] * c2 - off);
          sum[i & 1] += pr[i];
        }
        l[qb] += sum[0] + sum[1];
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
          if (exact) {
            bf16x8 part[3];
            parts8<true>(pr + 8 * ks, part);
#pragma unroll
            for (int nb = 0; nb < G::NB; ++nb) o[qb][nb] = mma_exact<F16>(view.trans(vt, nb, ks), part, o[qb][nb]);
          } else {
            const X8 pf = pack8<F16>(pr + 8 * ks);
#pragma unroll
            for (int nb = 0; nb < G::NB; ++nb) o[qb][nb] = Half<F16>::mma(view.trans(vt, nb, ks), pf, o[qb][nb]);
          }
        }
      }
      if (t + 1 < ntiles) store(buf ^ 1);
      __syncthreads();
    };
    int t = 0;
    for (; t + 1 < ntiles; t += 2) {  // a stage is then a constant offset of the LDS reads (8 heads x 4096 x 2 chunks, 128 287 -> 253 us, fp16 64 184 -> 165)
      tile(t, 0);
      tile(t + 1, 1);
    }
    if (t < ntiles) tile(t, 0);
  }
  // the two lanes of a query saw the same maxima; their sums cover disjoint keys
#pragma unroll
  for (int qb = 0; qb < QB; ++qb) l[qb] += __shfl_xor(l[qb], 32, 64);
  if constexpr (KS > 1) {
    // the groups hand over to the one below them, halving their number each time
    constexpr int XB = (16 * G::NB + 2) * 64, XO = QB * XB;  // floats of 32 queries and of a wavefront (in the stages' place, see launch_fwd)
    float* xo = reinterpret_cast<float*>(smem) + ((ks % (KS / 2)) * W + wave) * XO + lane;
#pragma unroll
    for (int half = KS / 2; half >= 1; half >>= 1) {
      if (ks >= half && ks < 2 * half) {
        float* to = reinterpret_cast<float*>(smem) + ((ks - half) * W + wave) * XO + lane;
#pragma unroll
        for (int qb = 0; qb < QB; ++qb) {
#pragma unroll
          for (int nb = 0; nb < G::NB; ++nb)
#pragma unroll
            for (int i = 0; i < 16; ++i) to[qb * XB + (nb * 16 + i) * 64] = o[qb][nb][i];
          to[qb * XB + 16 * G::NB * 64] = m[qb];
          to[qb * XB + (16 * G::NB + 1) * 64] = l[qb];
        }
      }
      __syncthreads();
      if (ks < half) {
#pragma unroll
        for (int qb = 0; qb < QB; ++qb) {
          const float m1 = xo[qb * XB + 16 * G::NB * 64], l1 = xo[qb * XB + (16 * G::NB + 1) * 64];
          const float mn = fmaxf(m[qb], m1);
          const float a0 = __builtin_amdgcn_exp2f((m[qb] - mn) * c2), a1 = __builtin_amdgcn_exp2f((m1 - mn) * c2);
          l[qb] = l[qb] * a0 + l1 * a1;
          m[qb] = mn;
#pragma unroll
          for (int nb = 0; nb < G::NB; ++nb)
#pragma unroll
            for (int i = 0; i < 16; ++i) o[qb][nb][i] = o[qb][nb][i] * a0 + xo[qb * XB + (nb * 16 + i) * 64] * a1;
        }
      }
      __syncthreads();
    }
    if (ks != 0) return;
  }
#pragma unroll
  for (int qb = 0; qb < QB; ++qb) {
    const int qi = q0 + 32 * qb;
    if (qi >= p.sq) return;
    const bool none = l[qb] == 0.0f;  // no finite score: out 0, lse -inf, no weight in a merge (a score that is NaN makes l NaN)
    const float inv = none ? 0.0f : 1.0f / l[qb];
    const float lse_j = none ? -INFINITY : m[qb] * p.scale + __logf(l[qb]);
    const long long row = bh * p.sq + qi;
    // Ring merge (the reference's _online_softmax_merge_): w = sigmoid(lse_j - lse), out += w (out_j - out),
    // lse = logaddexp(lse, lse_j), with out_j rounded to the core's output dtype first as the unfused path has it.
    float w = 0.0f;
    if (p.out_acc != nullptr && !none) {
      const float l_old = p.lse_acc[row];  // both lanes of the query read it before lane kg = 0 writes
      w = 1.0f / (1.0f + __expf(l_old - lse_j));  // l_old = -inf -> 1
      if (kg == 0) p.lse_acc[row] = fmaxf(l_old, lse_j) + log1pf(__expf(-fabsf(l_old - lse_j)));
    }
    if (p.lse != nullptr && kg == 0) p.lse[row] = lse_j;
    // register i of block nb: output column nb*32 + 8*(i/4) + 4*kg + i%4
#pragma unroll
    for (int nb = 0; nb < G::NB; ++nb)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int dv = nb * 32 + 8 * j + 4 * kg;
        if (dv >= p.d) continue;
        const f32x16& ov = o[qb][nb];
        const u32x2 h = pack4<F16>(ov[4 * j] * inv, ov[4 * j + 1] * inv, ov[4 * j + 2] * inv, ov[4 * j + 3] * inv);
        if (p.o != nullptr) *reinterpret_cast<u32x2*>(p.o + row * p.d + dv) = h;
        if (p.out_acc != nullptr) {
          f32x4* dst = reinterpret_cast<f32x4*>(p.out_acc + row * p.d + dv);
          f32x4 a = *dst;
          float h0, h1, h2, h3;
          Half<F16>::unpair(h.x, h0, h1);
          Half<F16>::unpair(h.y, h2, h3);
          a.x += w * (h0 - a.x);
          a.y += w * (h1 - a.y);
          a.z += w * (h2 - a.z);
          a.w += w * (h3 - a.w);
          *dst = a;
        }
      }
  }
}

// The groups' sums to group 0: each hands over to the one below it, halving their number each time (in the stages' place, which a
// barrier has closed).
template <int NB, int W, int KS>
__device__ __forceinline__ void hand_over(float* lds, int ks, int wave, int lane, f32x16 (&sum)[NB]) {
#pragma unroll
  for (int half = KS / 2; half >= 1; half >>= 1) {
    float* const at = lds + ((ks % half) * W + wave) * (16 * NB * 64) + lane;
    if (ks >= half && ks < 2 * half) {
#pragma unroll
      for (int nb = 0; nb < NB; ++nb)
#pragma unroll
        for (int i = 0; i < 16; ++i) at[(nb * 16 + i) * 64] = sum[nb][i];
    }
    __syncthreads();
    if (ks < half) {
#pragma unroll
      for (int nb = 0; nb < NB; ++nb)
#pragma unroll
        for (int i = 0; i < 16; ++i) sum[nb][i] += at[(nb * 16 + i) * 64];
    }
    __syncthreads();
  }
}

// ------------------------------------------------------------------- dQ (and delta)
// EXACT (here and in the dK/dV kernel): dS and the probabilities are not rounded (chunks of fewer than EXACT_KEYS keys).
// STORE: delta goes to the workspace for a dK/dV launch.
// QB: blocks of 32 queries a wavefront, see the forward kernel.
template <int D, bool F16, int W, int KS, bool EXACT, bool STORE, int QB = 1>
__device__ __forceinline__ void dq_block(const Args& p, const BlockOf& wg) {
  typedef Geo<D> G;
  typedef typename Half<F16>::x8 X8;
  constexpr int BUF = 2 * G::TILE;  // K tile, V tile
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const int tid = threadIdx.x % (64 * W), ks = __builtin_amdgcn_readfirstlane(threadIdx.x / (64 * W));
  const int lane = tid & 63, wave = tid >> 6;
  const int ln = lane & 31, kg = lane >> 5;
  const long long bh = wg.bh;
  const int q0 = wg.blk * (32 * W * QB) + wave * (32 * QB) + ln;  // and q0 + 32, ..
  const long long chunk_off = bh * p.sk * p.d;
  const float c2 = p.scale * LOG2E;
  unsigned char* lds = smem + ks * 2 * BUF;
  const TileView<D, F16> view(lane);

  X8 qf[QB][G::C16], dof[QB][G::C16];
  float delta[QB], lse2[QB];
  f32x16 dq[QB][G::NB];
#pragma unroll
  for (int qb = 0; qb < QB; ++qb) {
    const long long row = bh * p.sq + min(q0 + 32 * qb, p.sq - 1), qoff = row * p.d;
    float dl = 0.0f;
#pragma unroll
    for (int c = 0; c < G::C16; ++c) {
      qf[qb][c] = row_frag<D, F16>(p.q + qoff, 16 * c + 8 * kg, p.d);
      dof[qb][c] = row_frag<D, F16>(p.dout + qoff, 16 * c + 8 * kg, p.d);
      const X8 of = row_frag<D, F16>(p.out + qoff, 16 * c + 8 * kg, p.d);
#pragma unroll
      for (int j = 0; j < 8; ++j) dl += (float)dof[qb][c][j] * (float)of[j];
    }
    // delta = rowsum(dO o O): the two lanes of a query hold disjoint halves of the row
    delta[qb] = dl + __shfl_xor(dl, 32, 64);
    if (STORE && kg == 0 && ks == 0 && q0 + 32 * qb < p.sq) p.delta[row] = delta[qb];
    lse2[qb] = p.lse_in[row] * LOG2E;
#pragma unroll
    for (int nb = 0; nb < G::NB; ++nb) dq[qb][nb] = zero16();
  }

  TileRegs<D, W> rk, rv;
  Stream<KS> load(0, p.sk, p.nchunks, ks), soft(0, p.sk, p.nchunks, ks);
  const int ntiles = load.steps;
  auto fetch = [&]() {
    const long long at = chunk_off + (long long)load.first_row() * p.d;
    const uint16_t* kb = reinterpret_cast<const uint16_t*>(chunk_entry(0, load.chunk)) + at;
    const uint16_t* vb = reinterpret_cast<const uint16_t*>(chunk_entry(1, load.chunk)) + at;
    tile_fetch<D, W>(rk, kb, tid, load.rows_left(), p.d);
    tile_fetch<D, W>(rv, vb, tid, load.rows_left(), p.d);
    load.next();
  };
  auto store = [&](int buf) {
    unsigned char* at = lds + buf * BUF;
    tile_store<D, W>(rk, at, tid, p.d);
    tile_store<D, W>(rv, at + G::TILE, tid, p.d);
  };
  fetch();
  store(0);
  // waited for once, here (see the forward kernel)
#pragma unroll
  for (int qb = 0; qb < QB; ++qb)
#pragma unroll
    for (int c = 0; c < G::C16; ++c) asm volatile("" : "+v"(qf[qb][c]), "+v"(dof[qb][c]));
  __syncthreads();
  auto tile = [&](int t, int buf) __attribute__((always_inline)) {
    const unsigned char* kt = lds + buf * BUF;
    const unsigned char* vt = kt + G::TILE;
    if (t + 1 < ntiles) fetch();
    f32x16 s[QB], dp[QB];
#pragma unroll
    for (int qb = 0; qb < QB; ++qb) s[qb] = dp[qb] = zero16();
#pragma unroll
    for (int c = 0; c < G::C16; ++c) {
      const X8 kf = view.rows(kt, c);
#pragma unroll
      for (int qb = 0; qb < QB; ++qb) s[qb] = Half<F16>::mma(kf, qf[qb][c], s[qb]);
      const X8 vf = view.rows(vt, c);
#pragma unroll
      for (int qb = 0; qb < QB; ++qb) dp[qb] = Half<F16>::mma(vf, dof[qb][c], dp[qb]);
    }
    if (soft.rows_left() < BT) {  // wave-uniform
#pragma unroll
      for (int qb = 0; qb < QB; ++qb)
#pragma unroll
        for (int i = 0; i < 16; ++i)
          if (8 * (i >> 2) + 4 * kg + (i & 3) >= soft.rows_left()) s[qb][i] = -INFINITY;
    }
    soft.next();
#pragma unroll
    for (int qb = 0; qb < QB; ++qb) {
      float ds[16];
#pragma unroll
      for (int i = 0; i < 16; ++i) ds[i] = __builtin_amdgcn_exp2f(s[qb][i] * c2 - lse2[qb]) * (dp[qb][i] - delta[qb]);
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) {
        if constexpr (EXACT) {
          bf16x8 part[3];
          parts8<false>(ds + 8 * ks, part);
#pragma unroll
          for (int nb = 0; nb < G::NB; ++nb) dq[qb][nb] = mma_exact<F16>(view.trans(kt, nb, ks), part, dq[qb][nb]);
        } else {
          const X8 dsf = pack8<F16>(ds + 8 * ks);
#pragma unroll
          for (int nb = 0; nb < G::NB; ++nb) dq[qb][nb] = Half<F16>::mma(view.trans(kt, nb, ks), dsf, dq[qb][nb]);
        }
      }
    }
    if (t + 1 < ntiles) store(buf ^ 1);
    __syncthreads();
  };
  int t = 0;
  for (; t + 1 < ntiles; t += 2) {
    tile(t, 0);
    tile(t + 1, 1);
  }
  if (t < ntiles) tile(t, 0);
  if constexpr (KS > 1) {
#pragma unroll
    for (int qb = 0; qb < QB; ++qb) hand_over<G::NB, W, KS>(reinterpret_cast<float*>(smem), ks, wave, lane, dq[qb]);
    if (ks != 0) return;
  }
#pragma unroll
  for (int qb = 0; qb < QB; ++qb) {
    if (q0 + 32 * qb >= p.sq) return;
    uint16_t* row = p.dq + (bh * p.sq + q0 + 32 * qb) * p.d;
#pragma unroll
    for (int nb = 0; nb < G::NB; ++nb)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int col = nb * 32 + 8 * j + 4 * kg;
        const f32x16& sum = dq[qb][nb];
        if (col < p.d)
          *reinterpret_cast<u32x2*>(row + col) = pack4<F16>(sum[4 * j] * p.scale, sum[4 * j + 1] * p.scale, sum[4 * j + 2] * p.scale, sum[4 * j + 3] * p.scale);
      }
  }
}

// (Two blocks a wavefront: two wavefronts a SIMD are asked for, that is 256 registers. At 64 columns the kernel takes them all and spills four, in
// front of and behind the tile loop.)
template <int D, bool F16, int W, int KS, bool EXACT, int QB>
__global__ __launch_bounds__(64 * W * KS, QB) void attn_wide_dq_kernel(ChunkTable, Args p) {
  dq_block<D, F16, W, KS, EXACT, true, QB>(p, block_of());
}

// ------------------------------------------------------------------- dK, dV
// MODE 0 forms dK and dV in one pass (two d x 32 accumulators a wavefront). That fits two workgroups
// per CU in 256 registers a lane at head size 96 but not at 128 (it would spill, and ran 1.3x slower
// that way), so head sizes above 96 run the kernel twice: MODE 1 forms dV only (from P), MODE 2 dK only
// (from dS), each with one accumulator and two workgroups per CU; the scores are computed in both.
// A launch with no more workgroups than CUs gains nothing from that and keeps the single pass.
// OWN: delta of a tile's queries from its rows of O and dO, which are here for it, and not from a dQ launch before.
template <int D, bool F16, int MODE, int W, int KS, bool EXACT, bool OWN>
__device__ __forceinline__ void dkv_block(const Args& p, const BlockOf& wg) {
  typedef Geo<D> G;
  typedef typename Half<F16>::x8 X8;
  constexpr bool DV = MODE != 2, DK = MODE != 1;
  constexpr int STATS = (1 + (OWN ? G::DOTS : 1)) * BT * 4;   // lse * log2(e) and delta of the tile's queries
  constexpr int BUF = 2 * G::TILE + STATS;                    // Q tile, dO tile, stats
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const int tid = threadIdx.x % (64 * W), ks = __builtin_amdgcn_readfirstlane(threadIdx.x / (64 * W));
  const int lane = tid & 63, wave = tid >> 6;
  const int ln = lane & 31, kg = lane >> 5;
  const long long bh = wg.bh;
  const bool live = wg.blk * (32 * W) + wave * 32 + ln < p.sk;
  const long long koff = (bh * p.sk + (live ? wg.blk * (32 * W) + wave * 32 + ln : p.sk - 1)) * p.d;
  const uint16_t* qb = p.q + bh * p.sq * p.d;
  const uint16_t* gb = p.dout + bh * p.sq * p.d;
  const float* lb = p.lse_in + bh * p.sq;
  const float* db = OWN ? lb : p.delta + bh * p.sq;
  const uint16_t* ob = OWN ? p.out + bh * p.sq * p.d : nullptr;
  const float c2 = p.scale * LOG2E;
  unsigned char* lds = smem + ks * 2 * BUF;
  const TileView<D, F16> view(lane);

  X8 kf[G::C16], vf[DK ? G::C16 : 1];
  {
    const uint16_t* krow = reinterpret_cast<const uint16_t*>(chunk_entry(0, wg.chunk)) + koff;
    const uint16_t* vrow = reinterpret_cast<const uint16_t*>(chunk_entry(1, wg.chunk)) + koff;
#pragma unroll
    for (int c = 0; c < G::C16; ++c) {
      kf[c] = row_frag<D, F16>(krow, 16 * c + 8 * kg, p.d);
      if (DK) vf[c] = row_frag<D, F16>(vrow, 16 * c + 8 * kg, p.d);
    }
  }
  f32x16 dk[DK ? G::NB : 1], dv[DV ? G::NB : 1];
#pragma unroll
  for (int nb = 0; nb < G::NB; ++nb) {
    if (DK) dk[nb] = zero16();
    if (DV) dv[nb] = zero16();
  }

  TileRegs<D, W> rq, rg, ro;
  float st = 0.0f;  // one statistic per thread of the group's first wavefront: lse2 (lanes 0-31) or delta (32-63)
  int st_rows = 0;  // rows of the tile it belongs to
  Stream<KS> load(0, p.sq, 1, ks);
  const int ntiles = load.steps;
  auto fetch = [&]() {
    const long long at = (long long)load.first_row() * p.d;
    const int rows = load.rows_left();
    tile_fetch<D, W>(rq, qb + at, tid, rows, p.d);
    tile_fetch<D, W>(rg, gb + at, tid, rows, p.d);
    if (OWN) tile_fetch<D, W>(ro, ob + at, tid, rows, p.d);
    if (tid < 2 * BT) {
      const float* src = tid < BT ? lb : db;  // every lane loads; the factor is applied when stored
      st = src[min(load.first_row() + (tid & (BT - 1)), p.sq - 1)];
    }
    st_rows = rows;
    load.next();
  };
  auto store = [&](int buf) {
    unsigned char* base = lds + buf * BUF;
    // A query past the end is the last one once more, whose score less an lse of +inf is -inf: a row of zeros makes NaN of an infinite key, and
    // NaN no probability of 0. (dO's row is zeros: what a probability that parts8 keeps above 0 is multiplied by.)
    tile_store<D, W, true>(rq, base, tid, p.d);
    tile_store<D, W>(rg, base + G::TILE, tid, p.d);
    if (tid < 2 * BT) {
      float v = tid < BT ? st * LOG2E : st;
      if ((tid & (BT - 1)) >= st_rows) v = tid < BT ? INFINITY : 0.0f;  // a query past the end: probability 0
      if (!OWN || tid < BT) reinterpret_cast<float*>(base + 2 * G::TILE)[tid] = v;
    }
    if constexpr (OWN) tile_row_dots<D, F16, W>(rg, ro, reinterpret_cast<float*>(base + 2 * G::TILE) + BT, tid, p.d);
  };
  fetch();
  store(0);
  // waited for once, here (see the forward kernel)
#pragma unroll
  for (int c = 0; c < G::C16; ++c) {
    asm volatile("" : "+v"(kf[c]));
    if (DK) asm volatile("" : "+v"(vf[c]));
  }
  __syncthreads();
  auto tile = [&](int t, int buf) __attribute__((always_inline)) {
    const unsigned char* qt = lds + buf * BUF;
    const unsigned char* gt = qt + G::TILE;
    const float* stats = reinterpret_cast<const float*>(gt + G::TILE);
    if (t + 1 < ntiles) fetch();
    // S and dP: lane = key ln, register i = query 8*(i/4) + 4*kg + i%4 of the tile
    f32x16 s = zero16(), dp = zero16();
#pragma unroll
    for (int c = 0; c < G::C16; ++c) {
      s = Half<F16>::mma(view.rows(qt, c), kf[c], s);
      if (DK) dp = Half<F16>::mma(view.rows(gt, c), vf[c], dp);
    }
    float pr[16], ds[16];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const f32x4 l4 = *reinterpret_cast<const f32x4*>(stats + 8 * j + 4 * kg);
      f32x4 d4 = {0.0f, 0.0f, 0.0f, 0.0f};
      if (DK) {
        d4 = *reinterpret_cast<const f32x4*>(stats + BT + 8 * j + 4 * kg);
#pragma unroll
        for (int i = 1; i < (OWN ? G::DOTS : 1); ++i) d4 += *reinterpret_cast<const f32x4*>(stats + (1 + i) * BT + 8 * j + 4 * kg);
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int i = 4 * j + e;
        pr[i] = __builtin_amdgcn_exp2f(s[i] * c2 - l4[e]);
        ds[i] = pr[i] * (dp[i] - d4[e]);
      }
    }
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      if constexpr (EXACT) {
        bf16x8 part[3];
        if (DV) {
          parts8<true>(pr + 8 * ks, part);
#pragma unroll
          for (int nb = 0; nb < G::NB; ++nb) dv[nb] = mma_exact<F16>(view.trans(gt, nb, ks), part, dv[nb]);
        }
        if (DK) {
          parts8<false>(ds + 8 * ks, part);
#pragma unroll
          for (int nb = 0; nb < G::NB; ++nb) dk[nb] = mma_exact<F16>(view.trans(qt, nb, ks), part, dk[nb]);
        }
      } else {
        if (DV) {
          const X8 pf = pack8<F16>(pr + 8 * ks);
#pragma unroll
          for (int nb = 0; nb < G::NB; ++nb) dv[nb] = Half<F16>::mma(view.trans(gt, nb, ks), pf, dv[nb]);
        }
        if (DK) {
          const X8 dsf = pack8<F16>(ds + 8 * ks);
#pragma unroll
          for (int nb = 0; nb < G::NB; ++nb) dk[nb] = Half<F16>::mma(view.trans(qt, nb, ks), dsf, dk[nb]);
        }
      }
    }
    if (t + 1 < ntiles) store(buf ^ 1);
    __syncthreads();
  };
  int t = 0;
  if constexpr (D == 96 && MODE == 0) {  // (two tiles a round have no registers left there: 6 heads x 4050 x 4 chunks 366 -> 405 us)
    for (; t < ntiles; ++t) tile(t, t & 1);
  } else {
    for (; t + 1 < ntiles; t += 2) {
      tile(t, 0);
      tile(t + 1, 1);
    }
    if (t < ntiles) tile(t, 0);
  }
  if constexpr (KS > 1) {
    static_assert(MODE == 0, "hand-over of both sums");
    hand_over<G::NB, W, KS>(reinterpret_cast<float*>(smem), ks, wave, lane, dk);
    hand_over<G::NB, W, KS>(reinterpret_cast<float*>(smem), ks, wave, lane, dv);
    if (ks != 0) return;
  }
  if (!live) return;
  uint16_t* krow = reinterpret_cast<uint16_t*>(const_cast<char*>(chunk_entry(2, wg.chunk))) + koff;
  uint16_t* vrow = reinterpret_cast<uint16_t*>(const_cast<char*>(chunk_entry(3, wg.chunk))) + koff;
#pragma unroll
  for (int nb = 0; nb < G::NB; ++nb)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int col = nb * 32 + 8 * j + 4 * kg;
      if (col >= p.d) continue;
      if (DK)
        *reinterpret_cast<u32x2*>(krow + col) = pack4<F16>(dk[nb][4 * j] * p.scale, dk[nb][4 * j + 1] * p.scale,
                                                           dk[nb][4 * j + 2] * p.scale, dk[nb][4 * j + 3] * p.scale);
      if (DV)
        *reinterpret_cast<u32x2*>(vrow + col) =
            pack4<F16>(dv[nb][4 * j], dv[nb][4 * j + 1], dv[nb][4 * j + 2], dv[nb][4 * j + 3]);
    }
}

template <int D, bool F16, int MODE, int W, int KS, bool EXACT>
__global__ __launch_bounds__(64 * W * KS, KS == 1 && (D <= 96 || MODE != 0) ? 2 : 1) void attn_wide_dkv_kernel(ChunkTable, Args p) {
  dkv_block<D, F16, MODE, W, KS, EXACT, false>(p, block_of());
}

// ------------------------------------------------------------------- dQ, dK and dV in one launch
// The first dq_blocks workgroups form dQ, the others dK and dV, with delta of their own (see one_launch_width).
template <int D, bool F16, int W, bool EXACT>
__global__ __launch_bounds__(256, D <= 64 ? 2 : 1) void attn_wide_bwd_kernel(ChunkTable, Args p, unsigned dq_blocks, unsigned q_rows, unsigned k_rows) {
  const unsigned rest = gridDim.x - dq_blocks;
  if (blockIdx.x < dq_blocks) dq_block<D, F16, W, 4 / W, EXACT, false>(p, jg::block_at(blockIdx.x, dq_blocks, q_rows, 1));
  else dkv_block<D, F16, 0, W, 4 / W, EXACT, true>(p, jg::block_at(blockIdx.x - dq_blocks, rest, k_rows, p.nchunks));
}

// Workgroups of 128 rows (attn_width: half of the CUs and more have one; at head size 32 all of them): where some CU has none, two
// groups share the streamed side.
bool two_groups(long long workgroups) { return workgroups < jg::cu_count(); }
bool keys_from(const Args& a, long long n) { return (long long)a.sk * a.nchunks >= n; }

// `args` in a launch of `kernel` that needs more LDS than the default limit
template <typename K>
int launch(K kernel, dim3 grid, int threads, int lds, const ChunkTable& tab, const Args& a, hipStream_t s, const char* who) {
  if (lds > 64 * 1024 &&
      hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, lds) != hipSuccess)
    JG_FAIL(JG_ERR_LAUNCH, "%s: cannot reserve %d bytes of LDS", who, lds);
  kernel<<<grid, threads, lds, s>>>(tab, a);
  JG_CHECK_LAUNCH(who);
  return JG_OK;
}

typedef std::integral_constant<int, 1> One;
typedef std::integral_constant<int, 2> Two;
typedef std::integral_constant<int, 4> Four;
template <int D>
using Most = std::integral_constant<int, D <= 64 ? 8 : 4>;  // groups of one wavefront each whose stages LDS holds

// Wavefronts that share a tile and groups of them, by kernel
struct Shape {
  int w, ks;
};
template <int D>
Shape dq_shape(const Args& a, long long batch) {
  switch (jg::attn_width(a.sq, batch, D)) {
    case 1: return {1, Most<D>::value};
    case 2: return {2, 4};
  }
  return {4, D > 32 && two_groups(jg::cdiv(a.sq, 128) * batch) ? 2 : 1};
}
template <int D>
Shape dkv_shape(const Args& a, long long batch) {
  switch (jg::attn_width(a.sk, batch * a.nchunks, D)) {  // (four wavefronts: a head of 128 then has the registers for both sums)
    case 1: return {1, 4};
    case 2: return {2, 2};
  }
  return {4, D > 32 && D <= 96 && two_groups(jg::cdiv(a.sk, 128) * batch * a.nchunks) ? 2 : 1};
}

template <int D, bool F16, bool EXACT>
int launch_fwd(const ChunkTable& tab, const Args& a, long long batch, hipStream_t s) {
  typedef Geo<D> G;
  auto go = [&](auto w, auto k, auto qb) {
    constexpr int W = decltype(w)::value, KS = decltype(k)::value, QB = decltype(qb)::value;
    constexpr int STAGES = KS * 2 * 2 * G::TILE, SUMS = KS / 2 * W * QB * (16 * G::NB + 2) * 64 * 4;  // stages; what the groups hand over
    static_assert(STAGES <= 160 * 1024 && SUMS <= 160 * 1024, "fits LDS");
    return launch(&attn_wide_fwd_kernel<D, F16, W, KS, EXACT, QB>, dim3((unsigned)jg::cdiv(a.sq, 32 * W * QB), (unsigned)batch, 1), 64 * W * KS,
                  std::max(STAGES, SUMS), tab, a, s, "jg_attn_fwd(wide)");
  };
  switch (jg::attn_width(a.sq, batch, D)) {
    case 1: return go(One{}, Most<D>{}, One{});
    case 2:  // (not past two a compute unit for keys that four groups cannot share: 600 x 64 x 1 at 32 8.9 us, 6.8 with 128 rows)
      if (D > 32 || keys_from(a, 128) || jg::cdiv(a.sq, 64) * batch <= 2 * jg::cu_count()) return go(Two{}, Four{}, One{});
  }
  // 128 queries a workgroup, up to 64 columns: two blocks a wavefront in as many wavefronts, where the walk over the keys is long enough for the groups'
  // hand-over. One block : two, us, in four wavefronts: 48 x 1000 x 3 chunks, fp16 64 83 : 74, 28 x 1162 x 2, fp16 64 64 : 58, 16 x 2924 x 4 at 32
  // 242 : 191, 15 x 3241 x 6 at 32 398 : 309, 64 x 270 x 2 at 32 10.9 : 10.0; 300 x 96 x 3, fp16 64 24.6 : 27.9, 64 x 520 x 1, fp16 64 18.6 : 19.8, 600 x 64 x 1 at 32 6.7 :
  // 7.7. In eight: 24 x 1193 x 7, fp16 64 113 : 107, 8 x 2690 x 6 210 : 189; 24 x 1000 x 2 32.7 : 33.7, 32 x 754 x 2 25.2 : 25.6. Above 64 columns there are no registers for it.
  const bool two = two_groups(jg::cdiv(a.sq, 128) * batch);
  if constexpr (D > 64) return two ? go(Four{}, Two{}, One{}) : go(Four{}, One{}, One{});
  else if constexpr (D > 32) {
    if (two) return keys_from(a, 4096) ? go(Two{}, Four{}, Two{}) : go(Four{}, Two{}, One{});
  }
  if constexpr (D <= 64) return keys_from(a, D == 32 ? 512 : 1024) ? go(Two{}, Two{}, Two{}) : go(Four{}, One{}, One{});
}

template <int D, bool F16, bool EXACT>
int launch_dq(const ChunkTable& tab, const Args& a, long long batch, hipStream_t s) {
  typedef Geo<D> G;
  auto go = [&](auto w, auto k, auto qb) {
    constexpr int W = decltype(w)::value, KS = decltype(k)::value, QB = decltype(qb)::value;
    constexpr int STAGES = KS * 2 * 2 * G::TILE, SUMS = KS / 2 * W * 16 * G::NB * 64 * 4;
    static_assert(STAGES <= 160 * 1024 && SUMS <= 160 * 1024, "fits LDS");
    return launch(&attn_wide_dq_kernel<D, F16, W, KS, EXACT, QB>, dim3((unsigned)jg::cdiv(a.sq, 32 * W * QB), (unsigned)batch, 1), 64 * W * KS,
                  std::max(STAGES, SUMS), tab, a, s, "jg_attn_bwd(wide, dq)");
  };
  const Shape shape = dq_shape<D>(a, batch);
  if (shape.w == 1) return go(One{}, Most<D>{}, One{});
  if (shape.w == 2) return go(Two{}, Four{}, One{});
  // Two blocks a wavefront as in the forward, backward in all, one : two, us, four wavefronts: 14 x 3596 x 2 at 32 306 : 256, 16 x 2924 x 4 at 32 425 : 401,
  // 28 x 1162 x 2, fp16 64 135 : 121, 8 x 4096 x 2, fp16 64 306 : 293; 64 x 500 x 2 at 32 30.6 : 31.3, 150 x 256 x 3, fp16 64 61.4 : 62.6. Eight: 8 x 2690 x 6, fp16 64 451 : 437.
  if constexpr (D > 64) return shape.ks == 2 ? go(Four{}, Two{}, One{}) : go(Four{}, One{}, One{});
  else if constexpr (D > 32) {
    if (shape.ks == 2) return keys_from(a, 4096) ? go(Two{}, Four{}, Two{}) : go(Four{}, Two{}, One{});
  }
  if constexpr (D <= 64) return keys_from(a, 2048) ? go(Two{}, Two{}, Two{}) : go(Four{}, One{}, One{});
}

template <int D, bool F16, bool EXACT>
int launch_dkv(const ChunkTable& tab, const Args& a, long long batch, hipStream_t s) {
  typedef Geo<D> G;
  auto go = [&](auto mode, auto w, auto k) {
    constexpr int W = decltype(w)::value, KS = decltype(k)::value;
    constexpr int STAGES = KS * 2 * (2 * G::TILE + 2 * BT * 4), SUMS = KS / 2 * W * 16 * G::NB * 64 * 4;
    static_assert(STAGES <= 160 * 1024 && SUMS <= 160 * 1024, "fits LDS");
    return launch(&attn_wide_dkv_kernel<D, F16, decltype(mode)::value, W, KS, EXACT>,
                  dim3((unsigned)jg::cdiv(a.sk, 32 * W), (unsigned)batch, (unsigned)a.nchunks), 64 * W * KS, std::max(STAGES, SUMS), tab, a, s,
                  "jg_attn_bwd(wide, dkv)");
  };
  typedef std::integral_constant<int, 0> Both;
  const long long workgroups = jg::cdiv(a.sk, 128) * batch * a.nchunks;
  const Shape shape = dkv_shape<D>(a, batch);
  if (shape.w == 1) return go(Both{}, One{}, Four{});
  if (shape.w == 2) return go(Both{}, Two{}, Two{});
  // up to head size 96 (64 with EXACT): dK and dV in one pass; above: one pass each when the launch has more workgroups
  // than the chip has CUs, and with EXACT always (register budget, see the kernel)
  if constexpr (D <= (EXACT ? 64 : 96)) {
    if constexpr (D > 32)
      if (shape.ks == 2) return go(Both{}, Four{}, Two{});
  } else if (EXACT || workgroups > jg::cu_count()) {
    const int rc = go(One{}, Four{}, One{});
    return rc != JG_OK ? rc : go(Two{}, Four{}, One{});
  }
  if constexpr (D <= 64 || !EXACT) return go(Both{}, Four{}, One{});
  return JG_OK;
}

// ---- dQ, dK and dV in one launch, or in two. Two launches one after the other each leave the compute units idle that their own workgroups do
// not fill or that wait for the last of them, and a short step waits for the host's second launch; in one launch the two kinds fill the
// chip together, for delta computed again by every dK/dV workgroup.
// Up to 64 columns both ways are priced in steps of a workgroup of four wavefronts (about 0.45 us at 32 columns, 0.75 at 64): a compute unit makes
// one at a time, 1.1 of them where it has a workgroup alone, and one of eight wavefronts takes 1.8 and 2. In one launch a head of 64 columns takes 1.25 (its
// registers let two workgroups on a compute unit), and workgroups of 32 rows, which fetch a tile for one wavefront each, 1.2 and 1.7. A launch more is
// six steps. Taken where one launch is expected to need less than 0.8 of the two (0.72 up to 96 columns, 0.85 above: the rings below). Backward, two launches : one, us: 4 heads x 128 x 2 chunks at 32
// 11.3 : 7.7, 15 x 710 x 3 at 32 38.6 : 24.2, 3 x 1497 x 2 at 32 30.1 : 20.4, 16 x 802 x 3 at 32 41.7 : 31.6, 3 x 3000 x 4 at 32 140 : 100, 64 x 64 x 1 at 64
// 14.6 : 7.1, 48 x 69 x 3 at 64 22.0 : 14.2, 7 x 387 x 6, fp16 64 36.5 : 27.3. Where it says no: 8 x 1024 x 8 at 32
// 59.0 : 61.5, 24 x 1000 x 2, fp16 64 71.7 : 74.7 (but 15 x 313 x 7, fp16 64 37.0 : 31.6, which it prices at 34 steps and 38).
// Wider heads have one workgroup of the one launch on a compute unit: it is taken where all of them fit at once, priced in us by what a step took
// there, by rows, with nine for a launch and what surrounds it. 13 x 102 x 2 at 128 21.8 : 12.7, 7 x 265 x 1 at 128 26.5 : 19.7, 2 x 2000 x 2 at 128
// 119 : 93, 2 x 1000 x 3 at 96 52.3 : 33.0, 16 x 200 x 3 at 96 23.4 : 15.4, 40 x 90 x 4 at 80 27.4 : 19.2, 1 x 2500 x 2 at 96 92 : 66. Where it says no: 12 x 1180 x 1
// at 96 53.8 : 74.6, 12 x 503 x 2 at 80 30.9 : 34.3, 11 x 845 x 2 at 80 48 : 53, 8 x 512 x 4 at 128 56.8 : 61.5, 33 x 193 x 3 at 128 40.7 : 44.3 (but 30 x 140 x 4 at 128 40.8 : 34.7, more workgroups than fit).
double steps_alone(long long workgroups, long long steps, int wavefronts) {
  const long long each = jg::cdiv(workgroups, jg::cu_count());
  return (wavefronts == 8 ? (each == 1 ? 1.8 : 2.0 * each) : (each == 1 ? 1.1 : 1.0 * each)) * steps;
}
// Rows a workgroup / 32 of the one launch (0: two launches). Its workgroups lie in one dimension of the grid, which holds 2^32 threads: 2^24 workgroups of
// 256. (Two launches have three dimensions. Rings of very many short heads come that far: 65535 x 64 queries against 16 x 1024 keys.)
constexpr long long MOST_BLOCKS = (1ll << 24) - 1;
template <int D>
int one_launch_width(const Args& a, long long batch) {
  const int tq = jg::cdiv(a.sq, BT), tk = jg::cdiv(a.sk, BT);
  // workgroups and steps of either kind with w wavefronts to a tile and ks groups of them
  auto blocks_q = [&](int w) { return jg::cdiv(tq, w) * batch; };
  auto blocks_k = [&](int w) { return jg::cdiv(tk, w) * batch * a.nchunks; };
  auto steps_q = [&](int ks) { return (long long)jg::cdiv((long long)tk * a.nchunks, ks); };
  auto steps_k = [&](int ks) { return (long long)jg::cdiv(tq, ks); };
  auto fit = [&](int w) { return blocks_q(w) + blocks_k(w) <= MOST_BLOCKS; };
  const Shape q = dq_shape<D>(a, batch), k = dkv_shape<D>(a, batch);
  int width = 0;
  if (D <= 64) {
    double least = 0.8 * (steps_alone(blocks_q(q.w), steps_q(q.ks), q.w * q.ks) + steps_alone(blocks_k(k.w), steps_k(k.ks), k.w * k.ks) + 6.0);
    for (int w = 1; w <= 4; w *= 2) {
      const double load = double(blocks_q(w) * steps_q(4 / w) + blocks_k(w) * steps_k(4 / w)) / jg::cu_count();
      const double one = std::max(1.1 * std::max(steps_q(4 / w), steps_k(4 / w)), load * (w == 1 ? (D == 32 ? 1.2 : 1.7) : (D == 32 ? 1.0 : 1.25)));
      if (one < least && fit(w)) least = one, width = w;
    }
    return width;
  }
  auto us_q = [](int w) { return w == 1 ? 1.2 : w == 2 ? 0.9 : 0.77; };
  auto us_k = [](int w) { return w == 1 ? 3.0 : w == 2 ? 2.05 : 1.75; };
  auto alone = [&](long long workgroups, double us, int wavefronts) { return us * (wavefronts == 8 ? 1.5 : 1.0) * jg::cdiv(workgroups, jg::cu_count()) + 9.0; };
  double least = (D <= 96 ? 0.72 : 0.85) * (alone(blocks_q(q.w), us_q(q.w) * steps_q(q.ks), q.w * q.ks) + alone(blocks_k(k.w), us_k(k.w) * steps_k(k.ks), k.w * k.ks));
  for (int w = 1; w <= 4; w *= 2) {
    const double one = std::max(us_q(w) * steps_q(4 / w), us_k(w) * steps_k(4 / w)) + 9.0;
    if (blocks_q(w) + blocks_k(w) <= jg::cu_count() && one < least) least = one, width = w;
  }
  return width;
}
template <int D, bool F16, bool EXACT>
int launch_bwd(const ChunkTable& tab, const Args& a, long long batch, int width, hipStream_t s) {
  typedef Geo<D> G;
  const char* const who = "jg_attn_bwd(wide)";
  auto go = [&](auto w) {
    constexpr int W = decltype(w)::value, KS = 4 / W;
    constexpr int STAGES = KS * 2 * (2 * G::TILE + (1 + G::DOTS) * BT * 4), SUMS = KS / 2 * W * 16 * G::NB * 64 * 4, LDS = std::max(STAGES, SUMS);
    static_assert(LDS <= 160 * 1024, "fits LDS");
    const long long rq = jg::cdiv(a.sq, 32 * W), rk = jg::cdiv(a.sk, 32 * W), nq = rq * batch, nk = rk * batch * a.nchunks;
    constexpr auto kernel = &attn_wide_bwd_kernel<D, F16, W, EXACT>;
    if (LDS > 64 * 1024 && hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, LDS) != hipSuccess)
      JG_FAIL(JG_ERR_LAUNCH, "%s: cannot reserve %d bytes of LDS", who, LDS);
    kernel<<<(unsigned)(nq + nk), 256, LDS, s>>>(tab, a, (unsigned)nq, (unsigned)rq, (unsigned)rk);
    JG_CHECK_LAUNCH(who);
    return JG_OK;
  };
  return width == 1 ? go(One{}) : width == 2 ? go(Two{}) : go(Four{});
}

// f(D constant, F16 constant) for the narrowest kernel that holds the head. (attention.py brings long bf16 sequences of narrow heads with zero
// columns to the kernels of 64, by a line drawn before these had two blocks a wavefront.)
template <typename F>
int by_width(int d, int dtype, F f) {
  auto typed = [&](auto width) { return dtype == JG_F16 ? f(width, std::true_type{}) : f(width, std::false_type{}); };
  if (d <= 32) return typed(std::integral_constant<int, 32>{});
  if (d <= 64) return typed(std::integral_constant<int, 64>{});
  if (d <= 96) return typed(std::integral_constant<int, 96>{});
  return typed(std::integral_constant<int, 128>{});
}

}  // namespace

namespace jg {

int attn_wide_bwd_one_launch_width(long long batch, int sq, int sk, int d, int nchunks) {
  Args a{};
  a.sq = sq; a.sk = sk; a.nchunks = nchunks;
  return by_width(d, JG_BF16, [&](auto width, auto) { return one_launch_width<width()>(a, batch); });
}

bool attn_wide_supported(long long batch, int sq, int sk, int d, int dtype, bool has_bias) {
  return (dtype == JG_BF16 || dtype == JG_F16) && !has_bias && d > 0 && d <= 128 && d % 8 == 0 && sq > 0 && sk > 0 &&
         batch > 0 && batch <= 65535;
}

int attn_wide_fwd_chunks(void* out, float* lse, const void* q, const void* const* k, const void* const* v, int nchunks,
                         long long batch, int sq, int sk, int d, int dtype, float scale, float* out_acc, float* lse_acc,
                         hipStream_t s) {
  Args a{};
  a.q = static_cast<const uint16_t*>(q);
  a.o = static_cast<uint16_t*>(out);
  a.lse = lse;
  a.out_acc = out_acc;
  a.lse_acc = lse_acc;
  a.sq = sq; a.sk = sk; a.d = d; a.nchunks = nchunks; a.scale = scale;
  a.exact_from = exact_from(sk, d, dtype);
  const ChunkTable tab = chunk_table(k, v, nullptr, nullptr, nchunks);
  return by_width(d, dtype, [&](auto width, auto f16) {
    return a.exact_from < sk ? launch_fwd<width(), f16(), true>(tab, a, batch, s) : launch_fwd<width(), f16(), false>(tab, a, batch, s);
  });
}

// dk, dv NULL: dQ (and delta) only
int attn_wide_bwd_chunks(void* dq, void* const* dk, void* const* dv, const void* dout, const void* q, const void* const* k,
                         const void* const* v, int nchunks, const void* out, const float* lse, long long batch, int sq,
                         int sk, int d, int dtype, float scale, void* ws, hipStream_t s) {
  Args a{};
  a.q = static_cast<const uint16_t*>(q);
  a.out = static_cast<const uint16_t*>(out);
  a.dout = static_cast<const uint16_t*>(dout);
  a.lse_in = lse;
  a.delta = static_cast<float*>(ws);
  a.dq = static_cast<uint16_t*>(dq);
  a.sq = sq; a.sk = sk; a.d = d; a.nchunks = nchunks; a.scale = scale;
  const ChunkTable tab = chunk_table(k, v, dk, dv, nchunks);
  return by_width(d, dtype, [&](auto width, auto f16) {
    const bool exact = sk < EXACT_KEYS;
    const int rows = dk != nullptr ? one_launch_width<width()>(a, batch) : 0;
    if (rows != 0) return exact ? launch_bwd<width(), f16(), true>(tab, a, batch, rows, s) : launch_bwd<width(), f16(), false>(tab, a, batch, rows, s);
    const int rc = exact ? launch_dq<width(), f16(), true>(tab, a, batch, s) : launch_dq<width(), f16(), false>(tab, a, batch, s);
    if (rc != JG_OK || dk == nullptr) return rc;
    return exact ? launch_dkv<width(), f16(), true>(tab, a, batch, s) : launch_dkv<width(), f16(), false>(tab, a, batch, s);
  });
}

}  // namespace jg
