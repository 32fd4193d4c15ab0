// Backward of the blockwise attention core on the bf16 matrix cores, head size
// 64, from the ring's GLOBAL out / lse (p = exp(s - lse) is already globally
// normalised). Two kernels, no atomics, deterministic:
//
//   dQ kernel      lane = query (as in the forward kernel). Per 64-key tile:
//                    S^T  = K Q^T                 A = K rows,    B = Q (registers)
//                    dP^T = V dO^T                A = V rows,    B = dO (registers)
//                    dS^T = P^T o (dP^T - delta) * scale      (lane-local)
//                    dQ^T += K^T dS^T             A = K^T (LDS transpose reads),
//                                                 B = dS^T straight from registers
//                  It also computes delta = rowsum(dO o O) and leaves it in the
//                  workspace for the second kernel.
//   dK/dV kernel   lane = key. Per 64-query tile:
//                    S  = Q K^T                   A = Q rows,    B = K (registers)
//                    dP = dO V^T                  A = dO rows,   B = V (registers)
//                    P, dS from lse / delta of the tile (broadcast LDS reads)
//                    dV^T += dO^T P               A = dO^T (LDS transpose reads)
//                    dK^T += Q^T dS               A = Q^T  (LDS transpose reads)
//   The score tile is recomputed in each kernel (7 matrix products instead of the
//   5 of a one-kernel formulation) so that P / dS are always produced in the
//   register layout the next MFMA consumes and never travel through LDS.
//
//   Workgroup: 8 wavefronts (dQ: 4 in small launches; dK/dV: 4) = 4 or 2 blocks of 32 rows (queries
//   for dQ, keys for dK/dV) x 2 halves of the streamed side, combined through LDS.
//   Streamed tiles (64 rows x 128 bytes; 32 rows where dQ has 2 blocks) travel from memory straight into LDS, row-major
//   with the 16-byte chunks of a row XOR-swizzled by row / 2 % 8 (no registers, no vector
//   instructions, no second, transposed copy). LDS has 64 banks, two of these rows, so that the 16 rows a
//   row fragment's read takes at a time meet all of them once; with row % 8 rows r and r + 8 lay on the same
//   ones (reads of eight wavefronts 294 : 460 bytes per ns and compute unit, transposed reads 300 either way; traced, 8 heads x
//   4096 x 4 chunks: dQ 222 -> 213 us, dK/dV 327 -> 310). The transposed fragments come from
//   ds_read_b64_tr_b16 (within 16 lanes, lane i receives element i % 4 of the 8 bytes
//   that lanes i / 4 + 4 j point at, j = 0..3), two reads of 4 consecutive rows each.
//
//   Several resident chunks in one pass (the ring backward from saved chunks,
//   jigsaw/modules/attention/_functional/backward.py:176-277): the dQ kernel walks the key tiles of
//   every chunk in turn with dQ in its registers (one launch, one rounding), and the chunk is a
//   third grid dimension of the dK/dV kernel. The chunk pointers travel in the kernel-argument
//   segment (first parameter), where a wavefront reads entry c with scalar loads.
//
//   RAGGED (sq or sk no multiple of 128): rows of a transfer clamped to the tensor's last one, resident rows
//   clamped when read and dropped when written; keys past the end get the score -inf (dQ kernel), queries past
//   the end the lse +inf (dK/dV kernel), so that their probabilities are 0.
//
// Reference behaviour restated here:
//   jigsaw/modules/attention/_functional/cores/math.py:125-149
#include "attn_chunks.h"
#include "lds_transfer.h"

#include <type_traits>

namespace {

using jg::BlockOf;
using jg::ChunkTable;
using jg::block_of;
using jg::chunk_entry;

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef short i16x4 __attribute__((ext_vector_type(4)));

constexpr int D = 64;
constexpr int BT = 64;            // streamed rows per tile
constexpr int ROWB = D * 2;       // bytes per row of a tile in LDS (no padding)
constexpr int NAT = BT * ROWB;    // 8192: one 64 x 64 bf16 tile
constexpr float LOG2E = 1.4426950408889634f;

__device__ __forceinline__ bf16x8 lds_frag(const unsigned char* p) {
  return __builtin_bit_cast(bf16x8, *reinterpret_cast<const u32x4*>(p));
}

// Offsets of a lane in a transfer of 8 rows (jg::to_lds_1k): lane L sits at row L / 8, chunk position L % 8 and
// fetches chunk (L % 8) ^ (row / 2 % 8) of its row; `second`: rows 8 .. 15 of 16. First for rows first_row + 0..7 of a tensor of
// `rows` rows, clamped to its last one.
__device__ __forceinline__ uint32_t dma_clamped_offset(int lane, int first_row, int rows, int second) {
  return (uint32_t)min(first_row + (lane >> 3), rows - 1) * ROWB + (uint32_t)(((lane & 7) ^ (lane >> 4) ^ (4 * second)) << 4);
}
__device__ __forceinline__ uint32_t dma_lane_offset(int lane) {
  return (uint32_t)((lane >> 3) * ROWB + (((lane & 7) ^ (lane >> 4)) << 4));  // the second 8 rows of 16: ^ 64
}

// fragment of a row-major tile: row r (0..63), 16-byte chunk c (0..7)
__device__ __forceinline__ bf16x8 nat_frag(const unsigned char* nat, int r, int c) {
  return lds_frag(nat + r * ROWB + ((c ^ ((r >> 1) & 7)) << 4));
}

// Per-lane constant part of the address of a TRANSPOSED fragment (A operand: 32 columns of the
// tile x 16 of its rows): lane p of a group of 16 points at row +4 kg + p / 4, columns 32 nb +
// 16 (group % 2) + 4 (p % 4); the row's swizzle is (4 kg + p / 4) / 2 whatever multiple of 16 the
// fragment starts at, and 4 more eight rows further on: the place of the other block there.
__device__ __forceinline__ int tr_lane_offset(int lane, int nb) {
  const int pp = lane & 15, g1 = (lane >> 4) & 1, kg = lane >> 5;
  const int row = 4 * kg + (pp >> 2);
  return row * ROWB + (((4 * nb + 2 * g1 + ((pp & 3) >> 1)) ^ (row >> 1)) << 4) + 8 * (pp & 1);
}
// Transposed fragment whose 16 rows start at `row0` (a multiple of 16): slots 0..3 = rows
// row0 + 4 kg + 0..3, slots 4..7 = rows row0 + 8 + 4 kg + 0..3: the order an accumulator lane
// holds its rows in.
__device__ __forceinline__ bf16x8 tr_frag(const unsigned char* nat, const int (&lane_off)[2], int nb, int row0) {
  typedef __attribute__((address_space(3))) i16x4* tr_ptr;
  const i16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((tr_ptr)(nat + lane_off[nb] + row0 * ROWB));
  const i16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((tr_ptr)(nat + lane_off[nb ^ 1] + (row0 + 8) * ROWB));
  u32x4 w;
  w.x = __builtin_bit_cast(u32x2, lo).x;
  w.y = __builtin_bit_cast(u32x2, lo).y;
  w.z = __builtin_bit_cast(u32x2, hi).x;
  w.w = __builtin_bit_cast(u32x2, hi).y;
  return __builtin_bit_cast(bf16x8, w);
}

__device__ __forceinline__ bf16x8 pack8(const float* e) {
  bf16x8 pk;
#pragma unroll
  for (int i = 0; i < 8; i += 2) {
    f32x2 v2 = {e[i], e[i + 1]};
    const bf16x2 h2 = __builtin_convertvector(v2, bf16x2);
    pk[i] = h2.x;
    pk[i + 1] = h2.y;
  }
  return pk;
}

struct BwdArgs {
  const uint16_t* dout;
  const uint16_t* q;
  const uint16_t* out;
  const float* lse;
  float* delta;     // (batch, sq) workspace
  uint16_t* dq;
  int sq, sk;       // sk: keys per chunk
  int nchunks;
  long long batch;
  float scale;
};

// ------------------------------------------------------------------ dQ kernel
constexpr int NBUF = 4;                     // tiles of a half in LDS: read back, current, read ahead, landing
// QB: query blocks per workgroup, 4 or 2. A tile holds 16 keys a query block: every wavefront moves 16 rows of it.
template <int QB>
struct DqPlan {
  static constexpr int THREADS = 64 * 2 * QB;
  static constexpr int ROWS = 32 * QB;        // queries
  static constexpr int TILE = 16 * QB;        // keys
  static constexpr int BLOCKS = TILE / 32;    // blocks of the pipeline in a tile
  static constexpr int BYTES = TILE * ROWB;
  static constexpr int BUF = 2 * BYTES;       // K tile, V tile
  static constexpr int HALF = NBUF * BUF;
  static constexpr int LDS = 2 * HALF;        // 131072 or 65536
  static_assert(LDS >= QB * 32 * 64 * 4, "the hand-over of the partial dQ reuses the tile buffers");
};

// Scheduling classes of __builtin_amdgcn_sched_group_barrier
#define JG_GROUP_VALU 0x002
#define JG_GROUP_MFMA 0x008
#define JG_GROUP_DS_READ 0x100

template <bool RAGGED, int QB>
__global__ __launch_bounds__(DqPlan<QB>::THREADS, QB == 2 ? 2 : 1) void attn_bwd_dq_kernel(ChunkTable chunks, BwdArgs p) {
  constexpr int DQ_BT = DqPlan<QB>::TILE, DQ_NAT = DqPlan<QB>::BYTES, DQ_BUF = DqPlan<QB>::BUF, BLOCKS = DqPlan<QB>::BLOCKS;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6;
  const int ln = lane & 31, kg = lane >> 5;
  const int qb = wave % QB, ks = wave / QB;
  const BlockOf where = block_of();
  const long long b = where.bh;
  const int q0 = where.blk * DqPlan<QB>::ROWS + qb * 32;
  // every chunk is cut in two key halves (one per wavefront group); a half's tiles of all chunks
  // form one stream of ntiles tiles
  const int tiles_per_chunk = (p.sk + 2 * DQ_BT - 1) / (2 * DQ_BT);
  const int ntiles = tiles_per_chunk * p.nchunks;
  const float c2 = p.scale * LOG2E;
  const bool q_live = !RAGGED || q0 + ln < p.sq;
  const long long qi = b * p.sq + (q_live ? q0 + ln : p.sq - 1);

  unsigned char* lds = smem + ks * DqPlan<QB>::HALF;
  // this wavefront moves rows 16 qb .. 16 qb + 15 of the K tile and of the V tile of its half
  const int ks_u = __builtin_amdgcn_readfirstlane(ks), qb_u = __builtin_amdgcn_readfirstlane(qb);
  const long long chunk_off = 2 * (b * p.sk * (long long)D);  // bytes into a chunk
  const int row_first = ks_u * tiles_per_chunk * DQ_BT + 16 * qb_u;
  int ld_chunk = 0, ld_tile = 0;  // the load cursor: tiles are requested in stream order
  const char* kdma = chunk_entry(0, 0) + chunk_off;
  const char* vdma = chunk_entry(1, 0) + chunk_off;
  const uint32_t dma_off = dma_lane_offset(lane);
  const uint32_t lds_dma = jg::lds_address(smem) + (uint32_t)(ks_u * DqPlan<QB>::HALF + 16 * qb_u * ROWB);
  const int tr_off[2] = {tr_lane_offset(lane, 0), tr_lane_offset(lane, 1)};
  // row fragments: row ln of a 32-row block, chunk 2 c + kg
  int row_off[4];
#pragma unroll
  for (int c = 0; c < 4; ++c) row_off[c] = ln * ROWB + (((2 * c + kg) ^ ((ln >> 1) & 7)) << 4);

  // K and V of tile t straight into its buffer (free since the barrier that ended the tile before)
  auto issue_loads = [&](int slot) {  // called with slot = 0, 1, 2, 3, 0, ... in turn
    const uint32_t dst = lds_dma + (uint32_t)(slot * DQ_BUF);
    const int row = row_first + ld_tile * DQ_BT;
    if (RAGGED) {
      const uint32_t o0 = dma_clamped_offset(lane, row, p.sk, 0), o1 = dma_clamped_offset(lane, row + 8, p.sk, 1);
      jg::to_lds_1k(kdma, o0, dst);
      jg::to_lds_1k(kdma, o1, dst + 8 * ROWB);
      jg::to_lds_1k(vdma, o0, dst + DQ_NAT);
      jg::to_lds_1k(vdma, o1, dst + DQ_NAT + 8 * ROWB);
    } else {
      const long long off = (long long)row * ROWB;
      jg::to_lds_1k(kdma + off, dma_off, dst);
      jg::to_lds_1k(kdma + off + 8 * ROWB, dma_off ^ 64u, dst + 8 * ROWB);
      jg::to_lds_1k(vdma + off, dma_off, dst + DQ_NAT);
      jg::to_lds_1k(vdma + off + 8 * ROWB, dma_off ^ 64u, dst + DQ_NAT + 8 * ROWB);
    }
    if (++ld_tile == tiles_per_chunk && ld_chunk + 1 < p.nchunks) {
      ld_tile = 0;
      ++ld_chunk;
      kdma = chunk_entry(0, ld_chunk) + chunk_off;
      vdma = chunk_entry(1, ld_chunk) + chunk_off;
    }
  };

  // the first tiles are on their way while the wavefront fetches its own rows
  issue_loads(0);
  if (ntiles > 1) issue_loads(1);

  bf16x8 qf[4], dof[4];
  float delta;
  {
    const uint16_t* qrow = p.q + qi * D + 8 * kg;
    const uint16_t* drow = p.dout + qi * D + 8 * kg;
    const uint16_t* orow = p.out + qi * D + 8 * kg;
    float dl = 0.0f;
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      qf[c] = lds_frag(reinterpret_cast<const unsigned char*>(qrow + 16 * c));
      dof[c] = lds_frag(reinterpret_cast<const unsigned char*>(drow + 16 * c));
      const bf16x8 of = lds_frag(reinterpret_cast<const unsigned char*>(orow + 16 * c));
#pragma unroll
      for (int i = 0; i < 8; ++i) dl += (float)dof[c][i] * (float)of[i];
    }
    delta = dl + __shfl_xor(dl, 32, 64);
    if (ks == 0 && kg == 0 && q_live) p.delta[qi] = delta;
  }
  const float lse2 = p.lse[qi] * LOG2E;
  f32x16 minus_delta;
#pragma unroll
  for (int i = 0; i < 16; ++i) minus_delta[i] = -delta;

  f32x16 dq[2];
#pragma unroll
  for (int nb = 0; nb < 2; ++nb)
#pragma unroll
    for (int i = 0; i < 16; ++i) dq[nb][i] = 0.0f;

  // The stream of 32-key blocks is software pipelined three deep. While the vector unit turns the
  // scores and dP of block j into dS (B), the matrix core computes the scores and dP of block
  // j + 1 (A, 8 instructions) and adds block j - 1 to dQ (C, 4 instructions): the three are
  // independent, so every matrix instruction has about seven vector instructions to run
  // under it. dS is kept without the softmax scale, which multiplies dQ once at the end.
  f32x16 s_cur, dp_cur;
  bf16x8 ds_prev[2];
  auto scores = [&](const unsigned char* kn, int sb, f32x16& s, f32x16& dp) {
#pragma unroll
    for (int i = 0; i < 16; ++i) s[i] = 0.0f;
    // dP starts from -delta (a lane is one query): the product then leaves dP - delta behind
    dp = minus_delta;
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      s = __builtin_amdgcn_mfma_f32_32x32x16_bf16(lds_frag(kn + sb * 32 * ROWB + row_off[c]), qf[c], s, 0, 0, 0);
      dp = __builtin_amdgcn_mfma_f32_32x32x16_bf16(lds_frag(kn + DQ_NAT + sb * 32 * ROWB + row_off[c]), dof[c], dp, 0, 0, 0);
    }
  };
  auto ds_frag = [&](int t) {
    float e[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const float pr = __builtin_amdgcn_exp2f(s_cur[8 * t + i] * c2 - lse2);
      e[i] = pr * dp_cur[8 * t + i];
    }
    return pack8(e);
  };
  auto add_to_dq = [&](const unsigned char* kn, int sb) {
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int nb = 0; nb < 2; ++nb)
        dq[nb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(tr_frag(kn, tr_off, nb, sb * 32 + 16 * t), ds_prev[t], dq[nb], 0, 0, 0);
  };
  // one step of the pipeline: A of (k_next, sb_next), B of the current block, C of (k_prev, sb_prev)
  int keys_left = p.sk - ks_u * tiles_per_chunk * DQ_BT, tile_at = 0;  // RAGGED: keys from the current block's first one on
  auto step = [&](const unsigned char* k_next, int sb_next, const unsigned char* k_prev, int sb_prev, bool ahead) {
    if (RAGGED) {
      if (keys_left < 32) {
#pragma unroll
        for (int i = 0; i < 16; ++i)
          if (8 * (i >> 2) + 4 * kg + (i & 3) >= keys_left) s_cur[i] = -INFINITY;
      }
      keys_left -= 32;
      if (++tile_at == BLOCKS * tiles_per_chunk) {  // the next block opens the next chunk
        tile_at = 0;
        keys_left += tiles_per_chunk * DQ_BT;
      }
    }
    f32x16 s_n, dp_n;
    if (ahead) scores(k_next, sb_next, s_n, dp_n);
    bf16x8 ds_now[2];
    ds_now[0] = ds_frag(0);
    ds_now[1] = ds_frag(1);
    add_to_dq(k_prev, sb_prev);
    if (ahead) {
#define JG_SLOT(reads)                                               \
  __builtin_amdgcn_sched_group_barrier(JG_GROUP_MFMA, 1, 0);          \
  __builtin_amdgcn_sched_group_barrier(JG_GROUP_DS_READ, reads, 0);   \
  __builtin_amdgcn_sched_group_barrier(JG_GROUP_VALU, 7, 0);
      JG_SLOT(2) JG_SLOT(2) JG_SLOT(2) JG_SLOT(2) JG_SLOT(2) JG_SLOT(2) JG_SLOT(2) JG_SLOT(2)
      JG_SLOT(0) JG_SLOT(0) JG_SLOT(0) JG_SLOT(0)
#undef JG_SLOT
      s_cur = s_n;
      dp_cur = dp_n;
    }
    ds_prev[0] = ds_now[0];
    ds_prev[1] = ds_now[1];
  };

  __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): this wavefront's transfers have landed
  __syncthreads();
  scores(lds, 0, s_cur, dp_cur);
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    ds_prev[0][i] = (__bf16)0.0f;  // block -1 adds nothing (times the finite K of block 0)
    ds_prev[1][i] = (__bf16)0.0f;
  }
  // Four tiles a round: a tile's buffer is then a constant offset of the LDS reads (8 heads x 4096 queries x 4 chunks 212 -> 203 us).
  auto tile = [&](int slot) { return lds + slot * DQ_BUF; };
  // all blocks of tile t, in buffer `slot`: each with the scores of the block behind it and the block before it added
  auto advance = [&](int t, int slot, bool last) __attribute__((always_inline)) {
    const unsigned char* const kn = tile(slot);
    const unsigned char* const back = t == 0 ? lds : tile((slot + 3) % NBUF);
    if (BLOCKS == 2) {
      step(kn, 1, back, t == 0 ? 0 : 1, true);
      step(tile((slot + 1) % NBUF), 0, kn, 0, !last);
    } else {
      step(tile((slot + 1) % NBUF), 0, back, 0, !last);
    }
  };
  auto advance_more = [&](int t, int slot) __attribute__((always_inline)) {
    if (t + 2 < ntiles) issue_loads((slot + 2) % NBUF);
    advance(t, slot, false);
    __builtin_amdgcn_s_waitcnt(0x0F70);
    __syncthreads();
  };
  int t = 0;
  for (; t + NBUF < ntiles; t += NBUF) {
#pragma unroll
    for (int i = 0; i < NBUF; ++i) advance_more(t + i, i);
  }
#pragma unroll 1
  for (; t + 1 < ntiles; ++t) advance_more(t, t % NBUF);
  advance(t, t % NBUF, true);
  add_to_dq(tile(t % NBUF), BLOCKS - 1);
  __syncthreads();  // the hand-over below reuses the tile buffers

  // combine the two key halves, then write dQ (lane = query, 4 consecutive d per store)
  float* xo = reinterpret_cast<float*>(smem) + qb * (32 * 64);
  if (ks == 1) {
#pragma unroll
    for (int nb = 0; nb < 2; ++nb)
#pragma unroll
      for (int i = 0; i < 16; ++i) xo[(nb * 16 + i) * 64 + lane] = dq[nb][i];
  }
  __syncthreads();
  if (ks == 1 || !q_live) return;
#pragma unroll
  for (int nb = 0; nb < 2; ++nb)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      f32x4 val;
      val.x = (dq[nb][4 * j + 0] + xo[(nb * 16 + 4 * j + 0) * 64 + lane]) * p.scale;
      val.y = (dq[nb][4 * j + 1] + xo[(nb * 16 + 4 * j + 1) * 64 + lane]) * p.scale;
      val.z = (dq[nb][4 * j + 2] + xo[(nb * 16 + 4 * j + 2) * 64 + lane]) * p.scale;
      val.w = (dq[nb][4 * j + 3] + xo[(nb * 16 + 4 * j + 3) * 64 + lane]) * p.scale;
      *reinterpret_cast<bf16x4*>(p.dq + qi * D + nb * 32 + 8 * j + 4 * kg) =
          __builtin_convertvector(val, bf16x4);
    }
}

// -------------------------------------------------------------- dK/dV kernel
constexpr int DKV_STATS = 2 * BT * 4;                 // lse2[64], delta[64] as floats
constexpr int DKV_HALF = 2 * NAT + DKV_STATS;         // Q tile, dO tile + stats
constexpr int DKV_LDS = 4 * DKV_HALF;                 // 67584: two query halves, double buffered
// Key blocks per workgroup: 2 (4 wavefronts, 64 keys), so that two workgroups share a CU. The two wavefronts of a SIMD then belong to
// different workgroups and do not march in step (the barrier per tile keeps the wavefronts of ONE workgroup in the same phase: all
// in their matrix instructions, then all in their exponentials), and a small launch fills more of the chip. With 4 (8 wavefronts) : 2,
// us: 24 heads x 2 chunks of 1000 46 : 37, 8 x 4 of 4096 327 : 311, 64 x 1 of 4096 625 : 572, 3 x 2 of 1497 28 : 20, 4 x 2 of 128
// 8.2 : 5.7, 16 x 1 of 2048 45 : 43; nothing slower.
constexpr int DKV_KB = 2;
constexpr int DKV_THREADS = 64 * 2 * DKV_KB;
constexpr int DKV_ROWS = 32 * DKV_KB;                 // keys per workgroup
constexpr int DKV_SHARE = BT / DKV_KB;                // rows of a streamed tile each wavefront of a half moves
static_assert(DKV_LDS >= DKV_KB * 64 * 64 * 4, "the hand-over of the partial dK / dV reuses the tile buffers");
static_assert(64 * DKV_KB >= 2 * BT, "one thread of a half per statistic");

template <bool RAGGED>
__global__ __launch_bounds__(DKV_THREADS, 8 / (2 * DKV_KB) >= 2 ? 2 : 1) void attn_bwd_dkv_kernel(ChunkTable chunks, BwdArgs p) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6;
  const int ln = lane & 31, kg = lane >> 5;
  const int kb = wave % DKV_KB, qs = wave / DKV_KB;
  const int th = tid % (64 * DKV_KB);
  const BlockOf where = block_of();
  const long long b = where.bh;
  const int k0 = where.blk * DKV_ROWS + kb * 32;
  const int ntiles = (p.sq + 2 * BT - 1) / (2 * BT);
  const float c2 = p.scale * LOG2E;
  const bool k_live = !RAGGED || k0 + ln < p.sk;
  const long long ki = b * p.sk + (k_live ? k0 + ln : p.sk - 1);

  unsigned char* lds = smem + qs * (2 * DKV_HALF);  // two buffers: Q tile, dO tile, stats
  const int half_row = qs * ntiles * BT;  // first query of this half
  // this wavefront moves its share of the rows of the Q tile and of the dO tile of its half
  const int qs_u = __builtin_amdgcn_readfirstlane(qs), kb_u = __builtin_amdgcn_readfirstlane(kb);
  const int row_first = qs_u * ntiles * BT + DKV_SHARE * kb_u;
  const char* qdma = reinterpret_cast<const char*>(p.q + b * p.sq * D);
  const char* ddma = reinterpret_cast<const char*>(p.dout + b * p.sq * D);
  const uint32_t dma_off = dma_lane_offset(lane);
  const uint32_t lds_dma = jg::lds_address(smem) + (uint32_t)(qs_u * (2 * DKV_HALF) + DKV_SHARE * kb_u * ROWB);
  const int tr_off[2] = {tr_lane_offset(lane, 0), tr_lane_offset(lane, 1)};

  float st_reg = 0.0f;
  auto issue_loads = [&](int t, int buf) {
    const uint32_t dst = lds_dma + (uint32_t)(buf * DKV_HALF);
#pragma unroll
    for (int r = 0; r < DKV_SHARE; r += 8) {
      const int row = row_first + t * BT + r;
      const long long off = RAGGED ? 0 : (long long)row * ROWB;
      const uint32_t lane_off = RAGGED ? dma_clamped_offset(lane, row, p.sq, r >> 3 & 1) : dma_off ^ (8u * (uint32_t)(r & 8));
      jg::to_lds_1k(qdma + off, lane_off, dst + r * ROWB);
      jg::to_lds_1k(ddma + off, lane_off, dst + NAT + r * ROWB);
    }
    // One plain load for every lane, used only when the statistics go to LDS: a load under a
    // per-lane condition, or arithmetic on its result here, would make the wavefront wait
    // for it (and for the transfers issued before it) on the spot.
    const float* src = th < BT ? p.lse : p.delta;
    const int row = half_row + t * BT + (th & (BT - 1));
    st_reg = src[b * p.sq + (RAGGED ? min(row, p.sq - 1) : row)];
  };
  auto store_stats = [&](int t, int buf) {
    unsigned char* base = lds + buf * DKV_HALF;
    if (th < 2 * BT) {
      float v = th < BT ? st_reg * LOG2E : -st_reg;
      if (RAGGED && half_row + t * BT + (th & (BT - 1)) >= p.sq) v = th < BT ? INFINITY : 0.0f;
      reinterpret_cast<float*>(base + 2 * NAT)[th] = v;
    }
    __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): the transfers into this buffer have landed
  };

  // the first tile is on its way while the wavefront fetches its own rows
  issue_loads(0, 0);

  bf16x8 kf[4], vf[4];
  {
    const uint16_t* krow = reinterpret_cast<const uint16_t*>(chunk_entry(0, where.chunk)) + ki * D + 8 * kg;
    const uint16_t* vrow = reinterpret_cast<const uint16_t*>(chunk_entry(1, where.chunk)) + ki * D + 8 * kg;
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      kf[c] = lds_frag(reinterpret_cast<const unsigned char*>(krow + 16 * c));
      vf[c] = lds_frag(reinterpret_cast<const unsigned char*>(vrow + 16 * c));
    }
  }

  f32x16 dk[2], dv[2];
#pragma unroll
  for (int nb = 0; nb < 2; ++nb)
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      dk[nb][i] = 0.0f;
      dv[nb][i] = 0.0f;
    }

  // dS is kept without the softmax scale, which multiplies dK once at the end
  auto compute_tile = [&](int buf) {
    const unsigned char* qn = lds + buf * DKV_HALF;
    const unsigned char* dn = qn + NAT;
    const float* st = reinterpret_cast<const float*>(qn + 2 * NAT);  // lse2[64] then -delta[64]
    bf16x8 pf[2][2], dsf[2][2];
#pragma unroll
    for (int sb = 0; sb < 2; ++sb) {
      f32x16 s, dp;
#pragma unroll
      for (int i = 0; i < 16; ++i) s[i] = 0.0f;
      // dP starts from -delta of its queries (register i: query sb*32 + 8*(i/4) + 4*kg + i%4)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const f32x4 d4 = *reinterpret_cast<const f32x4*>(st + BT + sb * 32 + 8 * j + 4 * kg);
#pragma unroll
        for (int e = 0; e < 4; ++e) dp[4 * j + e] = d4[e];
      }
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        s = __builtin_amdgcn_mfma_f32_32x32x16_bf16(nat_frag(qn, sb * 32 + ln, 2 * c + kg), kf[c], s, 0, 0, 0);
        dp = __builtin_amdgcn_mfma_f32_32x32x16_bf16(nat_frag(dn, sb * 32 + ln, 2 * c + kg), vf[c], dp, 0, 0, 0);
      }
      // register i of this lane: query sb*32 + 8*(i/4) + 4*kg + i%4, key ln
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        float pe[8], de[8];
#pragma unroll
        for (int jj = 0; jj < 2; ++jj) {
          const int j = 2 * t + jj;
          const f32x4 l4 = *reinterpret_cast<const f32x4*>(st + sb * 32 + 8 * j + 4 * kg);
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const float pr = __builtin_amdgcn_exp2f(s[4 * j + e] * c2 - l4[e]);
            pe[4 * jj + e] = pr;
            de[4 * jj + e] = pr * dp[4 * j + e];
          }
        }
        pf[sb][t] = pack8(pe);
        dsf[sb][t] = pack8(de);
      }
    }
#pragma unroll
    for (int sb = 0; sb < 2; ++sb)
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int nb = 0; nb < 2; ++nb) {
          dv[nb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(tr_frag(dn, tr_off, nb, sb * 32 + 16 * t), pf[sb][t], dv[nb], 0, 0, 0);
          dk[nb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(tr_frag(qn, tr_off, nb, sb * 32 + 16 * t), dsf[sb][t], dk[nb], 0, 0, 0);
        }
  };

  store_stats(0, 0);
  // The K / V fragments came straight from memory: they are waited for here, once. Left
  // to the first MFMA that reads them, the wait would sit inside the loop, behind the
  // tile loads that every iteration has just issued.
#pragma unroll
  for (int c = 0; c < 4; ++c) asm volatile("" : "+v"(kf[c]), "+v"(vf[c]));
  __syncthreads();
  auto advance = [&](int t, int buf) __attribute__((always_inline)) {
    const bool has_next = t + 1 < ntiles;
    if (has_next) issue_loads(t + 1, buf ^ 1);
    compute_tile(buf);
    if (has_next) store_stats(t + 1, buf ^ 1);
    __syncthreads();
  };
  int t = 0;
  for (; t + 1 < ntiles; t += 2) {  // a buffer is then a constant offset of the LDS reads (8 heads x 4096 x 4 chunks 304 -> 297 us)
    advance(t, 0);
    advance(t + 1, 1);
  }
  if (t < ntiles) advance(t, 0);

  // combine the two query halves, then write dK / dV (lane = key)
  float* xo = reinterpret_cast<float*>(smem) + kb * (64 * 64);
  if (qs == 1) {
#pragma unroll
    for (int nb = 0; nb < 2; ++nb)
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        xo[(nb * 16 + i) * 64 + lane] = dk[nb][i];
        xo[(32 + nb * 16 + i) * 64 + lane] = dv[nb][i];
      }
  }
  __syncthreads();
  if (qs == 1 || !k_live) return;
  uint16_t* dk_out = reinterpret_cast<uint16_t*>(const_cast<char*>(chunk_entry(2, where.chunk)));
  uint16_t* dv_out = reinterpret_cast<uint16_t*>(const_cast<char*>(chunk_entry(3, where.chunk)));
#pragma unroll
  for (int nb = 0; nb < 2; ++nb)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      f32x4 a, c;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        a[e] = (dk[nb][4 * j + e] + xo[(nb * 16 + 4 * j + e) * 64 + lane]) * p.scale;
        c[e] = dv[nb][4 * j + e] + xo[(32 + nb * 16 + 4 * j + e) * 64 + lane];
      }
      const int col = nb * 32 + 8 * j + 4 * kg;
      *reinterpret_cast<bf16x4*>(dk_out + ki * D + col) = __builtin_convertvector(a, bf16x4);
      *reinterpret_cast<bf16x4*>(dv_out + ki * D + col) = __builtin_convertvector(c, bf16x4);
    }
}

}  // namespace

namespace jg {

// (shorter chunks keep P and dS in fp32: attn_wide.hip)
bool attn_mfma_bwd_supported(long long batch, int sq, int sk, int d, int dtype, bool has_bias) {
  return dtype == JG_BF16 && !has_bias && d == D && sq > 0 && sk >= EXACT_KEYS && sq <= ATTN_MAX_KEYS && sk <= ATTN_MAX_KEYS &&
         batch > 0 && batch <= 65535;
}

// The ring backward over `nchunks` resident chunks: k[c], v[c] in, dk[c], dv[c] out, dq = the sum over
// the chunks, rounded once. nchunks = 1 is the plain backward of one chunk.
// Where bf16 heads of 64 go to attn_wide.hip for dQ, dK and dV in one launch: its rows of a workgroup / 32, else 0
int attn_mfma_bwd_one_launch_width(long long batch, int sq, int sk, int nchunks) {
  const bool ragged = sq % EXACT_KEYS != 0 || sk % EXACT_KEYS != 0;
  return ragged && attn_width(sq, batch, D) == 1 ? attn_wide_bwd_one_launch_width(batch, sq, sk, D, nchunks) : 0;
}

int attn_mfma_bwd_chunks(void* dq, void* const* dk, void* const* dv, const void* dout, const void* q,
                         const void* const* k, const void* const* v, int nchunks, const void* out, const float* lse,
                         long long batch, int sq, int sk, float scale, void* ws, hipStream_t s) {
  const ChunkTable tab = chunk_table(k, v, dk, dv, nchunks);
  BwdArgs a;
  a.dout = static_cast<const uint16_t*>(dout);
  a.q = static_cast<const uint16_t*>(q);
  a.out = static_cast<const uint16_t*>(out);
  a.lse = lse;
  a.delta = static_cast<float*>(ws);
  a.dq = static_cast<uint16_t*>(dq);
  a.sq = sq;
  a.sk = sk;
  a.nchunks = nchunks;
  a.batch = batch;
  a.scale = scale;
  static bool attr_set = false;
  if (!attr_set) {
    auto reserve = [](const void* f, int bytes) {
      return hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, bytes) == hipSuccess;
    };
    if (!reserve(reinterpret_cast<const void*>(&attn_bwd_dq_kernel<false, 4>), DqPlan<4>::LDS) ||
        !reserve(reinterpret_cast<const void*>(&attn_bwd_dq_kernel<true, 4>), DqPlan<4>::LDS) ||
        !reserve(reinterpret_cast<const void*>(&attn_bwd_dq_kernel<false, 2>), DqPlan<2>::LDS) ||
        !reserve(reinterpret_cast<const void*>(&attn_bwd_dq_kernel<true, 2>), DqPlan<2>::LDS) ||
        !reserve(reinterpret_cast<const void*>(&attn_bwd_dkv_kernel<false>), DKV_LDS) ||
        !reserve(reinterpret_cast<const void*>(&attn_bwd_dkv_kernel<true>), DKV_LDS))
      JG_FAIL(JG_ERR_LAUNCH, "jg_attn_bwd: cannot reserve LDS");
    attr_set = true;
  }
  const bool ragged = sq % (2 * BT) != 0 || sk % (2 * BT) != 0;
  auto launch_dq = [&](auto qb_c) {
    constexpr int QB = decltype(qb_c)::value;
    typedef DqPlan<QB> Plan;
    const dim3 grid((unsigned)cdiv(sq, Plan::ROWS), (unsigned)batch, 1);
    if (ragged) attn_bwd_dq_kernel<true, QB><<<grid, Plan::THREADS, Plan::LDS, s>>>(tab, a);
    else attn_bwd_dq_kernel<false, QB><<<grid, Plan::THREADS, Plan::LDS, s>>>(tab, a);
  };
  const dim3 dkv_grid((unsigned)cdiv(sk, DKV_ROWS), (unsigned)batch, (unsigned)nchunks);
  // Where even those of 64 would leave half of them without one, 32 queries and eight key groups (attn_width; this kernel with 64 : that one, us):
  // 1 x 8 heads x 1024 x 8 chunks 73 : 52, 1 x 8 x 512 x 4 20.8 : 18.0, 2 x 4096 x 2 70 : 52, 4 x 1024 x 1 12.2 : 12.4.
  // Where workgroups of 128 queries would leave half of the compute units without one, those of 64 queries (128 : 64, us): 8 heads x
  // 2048 queries x 4 chunks 94 : 81, 3 x 4000 x 8 321 : 285, 18 x 700 x 3 32 : 26. Elsewhere twice the tile
  // traffic and a barrier for half the keys cost more than the waves' independence gives: 8 x 4096 x 4 203 : 223, 32 x 1024 x 1
  // 18.0 : 18.9, 24 x 1000 x 2 30.8 : 32.1.
  // And there dQ, dK and dV in one launch where attn_wide.hip takes that to be the shorter way (two launches : one, us; fp16 for the latter): 7 x 387 x 6 chunks
  // 35.2 : 27.3, 6 x 400 x 4 25.8 : 20.2. (Not for lengths in multiples of 128, where dK and dV of a chunk have the same bits in a ring
  // and by themselves: attention.backward_chunks.)
  // Those of 64 queries go there too where the keys are many (four groups take tiles of all chunks in turn; this kernel with 64 : that one, backward, us): 32 x 270 x 8
  // 55.8 : 51.1, 30 x 394 x 6 65.8 : 61.4, 48 x 237 x 6 41.9 : 40.2, 4 x 2700 x 5 217 : 202; 18 x 745 x 2 35.4 : 35.9, 27 x 296 x 2 21.4 : 21.9. (Lengths in multiples of 128: not by a rule on the
  // chunks' number, as above.)
  const int width = attn_width(sq, batch, D);
  if (width == 1 || (width == 2 && (sq % EXACT_KEYS != 0 || sk % EXACT_KEYS != 0) && (long long)sk * nchunks >= 2048)) {
    if (attn_mfma_bwd_one_launch_width(batch, sq, sk, nchunks) != 0)
      return attn_wide_bwd_chunks(dq, dk, dv, dout, q, k, v, nchunks, out, lse, batch, sq, sk, D, JG_BF16, scale, ws, s);
    const int rc = attn_wide_bwd_chunks(dq, nullptr, nullptr, dout, q, k, v, nchunks, out, lse, batch, sq, sk, D, JG_BF16, scale, ws, s);
    if (rc != JG_OK) return rc;
  } else if (2 * batch * cdiv(sq, DqPlan<4>::ROWS) <= cu_count()) launch_dq(std::integral_constant<int, 2>{});
  else launch_dq(std::integral_constant<int, 4>{});
  JG_CHECK_LAUNCH("jg_attn_bwd(dq)");
  if (ragged) attn_bwd_dkv_kernel<true><<<dkv_grid, DKV_THREADS, DKV_LDS, s>>>(tab, a);
  else attn_bwd_dkv_kernel<false><<<dkv_grid, DKV_THREADS, DKV_LDS, s>>>(tab, a);
  JG_CHECK_LAUNCH("jg_attn_bwd(dkv)");
  return JG_OK;
}

}  // namespace jg
