// K/V chunks of a ring in the 16-bit attention kernels, and the order of their workgroups.
#pragma once
#include "jg_common.h"

namespace jg {

constexpr int ATTN_MAX_CHUNKS = 16;
constexpr int ATTN_MAX_KEYS = 1 << 23;  // rows of a chunk: the clamped transfers address them by 32-bit byte offsets

// Chunk c: k[c], v[c] (batch, sk, d) and, in the backward, where its gradients go. FIRST kernel parameter:
// entry c is read from the kernel-argument segment by its offset (a by-value struct indexed with a run-time
// value would otherwise be copied to private memory lane by lane).
struct ChunkTable {
  const uint16_t* k[ATTN_MAX_CHUNKS];
  const uint16_t* v[ATTN_MAX_CHUNKS];
  uint16_t* dk[ATTN_MAX_CHUNKS];
  uint16_t* dv[ATTN_MAX_CHUNKS];
};
__device__ __forceinline__ const char* chunk_entry(int which, int c) {  // which: 0 k, 1 v, 2 dk, 3 dv; c wave-uniform
#if defined(__HIP_DEVICE_COMPILE__)
  const char* const* kt = (const char* const*)__builtin_amdgcn_kernarg_segment_ptr();
  return kt[which * ATTN_MAX_CHUNKS + c];
#else
  (void)which; (void)c;
  return nullptr;
#endif
}
// dk / dv: NULL in the forward
inline ChunkTable chunk_table(const void* const* k, const void* const* v, void* const* dk, void* const* dv, int n) {
  ChunkTable tab;
  for (int c = 0; c < ATTN_MAX_CHUNKS; ++c) {
    const int u = c < n ? c : 0;
    tab.k[c] = static_cast<const uint16_t*>(k[u]);
    tab.v[c] = static_cast<const uint16_t*>(v[u]);
    tab.dk[c] = dk == nullptr ? nullptr : static_cast<uint16_t*>(dk[u]);
    tab.dv[c] = dv == nullptr ? nullptr : static_cast<uint16_t*>(dv[u]);
  }
  return tab;
}

// Which keys keep their probabilities in fp32. The kernels round P (and dS) to the 16 bits of the operands before P V
// (dS K, dS^T Q, P^T dO) where a chunk is long. Of a chunk with fewer than EXACT_KEYS keys nothing is rounded, forward
// and backward, nor are, in the forward, the keys behind the last multiple of EXACT_KEYS where the head fills a
// kernel's width: there the values go into the matrix product as three bf16 parts (see parts8).
constexpr int EXACT_KEYS = 128;
inline int exact_from(int sk, int d, int dtype) {  // first key of a chunk whose probabilities the forward keeps in fp32
  if (sk < EXACT_KEYS) return 0;
  return d == 96 || d == 128 || (d == 64 && dtype == JG_BF16) ? sk / EXACT_KEYS * EXACT_KEYS : sk;
}

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));

// Eight fp32 values as three bf16 ones each that add up to them exactly: the upper 16 bits, those of the rest, and those
// of what is left then (24 bits of significand in three pieces of 8, cut and not rounded, so that all three have
// the value's sign). The products with bf16 operands are exact in the matrix cores' fp32 accumulators, so a
// contraction over the parts is as exact as one in fp32, at three times the instructions and a fifth of the time of
// the fp32 matrix instructions. An infinite value is its first part. POSITIVE (probabilities): the
// lower parts are never 0, so that a probability that is not 0 times an infinite operand stays infinite as it does in fp32.
template <bool POSITIVE>
__device__ __forceinline__ void parts8(const float* v, bf16x8_t (&part)[3]) {
  u32x4_t w[3];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    float a = v[2 * i], b = v[2 * i + 1];
#pragma unroll
    for (int t = 0; t < 3; ++t) {
      const uint32_t ua = __float_as_uint(a), ub = __float_as_uint(b);
      w[t][i] = __builtin_amdgcn_perm(ub, ua, 0x07060302u);
      const float ha = __uint_as_float(ua & 0xffff0000u), hb = __uint_as_float(ub & 0xffff0000u);
      a = a == ha ? 0.0f : a - ha;
      b = b == hb ? 0.0f : b - hb;
      if (POSITIVE) {
        a = fmaxf(a, 1.1754943508222875e-38f);
        b = fmaxf(b, 1.1754943508222875e-38f);
      }
    }
  }
#pragma unroll
  for (int t = 0; t < 3; ++t) part[t] = __builtin_bit_cast(bf16x8_t, w[t]);
}

// Wavefronts of 32 rows each that share a tile of the streamed side in the kernels of attn_wide.hip: four, or as many fewer as it takes
// to give every compute unit a workgroup. A tile takes 1.3 to 2.5 us of latency whatever else runs there (fetch, scores, exponentials,
// products, one after the other), so that 48 workgroups of 128 rows left the chip idle for as long as a full one; with 64 or 32 rows they
// are two or four times as many, and what their fewer rows leave free takes more tiles at once (four to eight groups a workgroup).
// Forward / backward, us, before -> with it: 8 heads x 512 x 4 chunks at 128 47 / 84 -> 31 / 59, x 8 chunks at 32 39 / 59 -> 19 / 29. Forced, where 128 rows
// have a workgroup for every second compute unit or more: 60 x 529 x 4, fp16 96 94 / 190 -> 125 / 209 (64 rows). At head size 32, whose workgroups
// fit a compute unit several times, up to two of 32 rows and three of 64 each still gain. Forward / backward of two launches, 64 : 32 rows: 44 x 322 x 8 28.3 / 54 : 21.0 / 47, 5 x 1734 x 6
// 60.6 / 107 : 55.8 / 103, 30 x 531 x 3 19.0 / 38 : 14.8 / 34; beyond, 14 x 1782 x 3 48.9 / 108 : 57.1 / 117. 128 : 64 rows: 24 x 1388 x 7 158 / 284 : 127 / 252, 44 x 983 x 3 54.5 / 114 : 45.4 / 106,
// 14 x 3095 x 7 340 / 678 : 269 / 605; beyond, 33 x 1497 x 5 128 / 262 : 127 / 262, 42 x 1968 x 8 337 / 828 : 375 / 822.
inline int attn_width(long long rows, long long batch, int columns) {
  if (cdiv(rows, 32) * batch <= (columns == 32 ? 2 : 1) * cu_count()) return 1;
  return cdiv(rows, 64) * batch <= (columns == 32 ? 3 : 1) * cu_count() ? 2 : 4;
}
// (attn_wide.hip; dk, dv NULL: dQ and delta only)
int attn_wide_fwd_chunks(void* out, float* lse, const void* q, const void* const* k, const void* const* v, int nchunks,
                         long long batch, int sq, int sk, int d, int dtype, float scale, float* out_acc, float* lse_acc, hipStream_t s);
int attn_wide_bwd_chunks(void* dq, void* const* dk, void* const* dv, const void* dout, const void* q, const void* const* k,
                         const void* const* v, int nchunks, const void* out, const float* lse, long long batch, int sq,
                         int sk, int d, int dtype, float scale, void* ws, hipStream_t s);
// Rows of a workgroup / 32 where that forms dQ, dK and dV in one launch, 0 where it takes two
int attn_wide_bwd_one_launch_width(long long batch, int sq, int sk, int d, int nchunks);

// Workgroup -> (batch entry, chunk, row block) of a grid (row blocks, batch entries, chunks). Consecutive
// workgroup ids go to the 8 XCDs in turn; each XCD is given a contiguous range of the flat order (batch entry,
// chunk, block), so the workgroups that stream the same K / V (or Q / dO) share one L2 instead of every L2
// holding every head. Falls back to the plain order when the count does not divide.
struct BlockOf {
  long long bh;
  int blk;
  int chunk;
};
__device__ __forceinline__ BlockOf block_at(unsigned id, unsigned total, unsigned nblk, unsigned nch) {
  if ((total & 7u) == 0) id = (id & 7u) * (total >> 3) + (id >> 3);
  BlockOf b;
  b.blk = (int)(id % nblk);
  id /= nblk;
  b.chunk = (int)(id % nch);
  b.bh = id / nch;
  return b;
}
__device__ __forceinline__ BlockOf block_of() {
  const unsigned nblk = gridDim.x, nch = gridDim.z;
  return block_at((blockIdx.y * nch + blockIdx.z) * nblk + blockIdx.x, gridDim.x * gridDim.y * gridDim.z, nblk, nch);
}

}  // namespace jg
