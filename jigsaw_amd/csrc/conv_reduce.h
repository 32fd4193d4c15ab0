// The sums over workgroups' partials that end a convolution's weight gradient (conv_wgrad_mfma.hip, conv_f32.hip): as launches of their
// own, or beside the border cells of the input gradient in one launch (halo.hip). The same sums in the same order, whichever does them.
#pragma once
#include "jg_common.h"

namespace jg {

enum { CONV_REDUCE_NONE = 0, CONV_REDUCE_TILES = 1, CONV_REDUCE_F32 = 2 };
constexpr int CONV_RED_WAVES = 8, CONV_RED_CHAINS = 16, CONV_BIAS_CHANNELS = 16, CONV_F32_VALUES = 16;

union ConvReduceShared {
  float tiles[CONV_RED_WAVES][64][4];
  double f32[CONV_RED_CHAINS][64];
};

inline unsigned conv_reduce_blocks(const jg_conv_reduction& p) {
  if (p.kind == CONV_REDUCE_F32) return (unsigned)p.runs;
  return ((unsigned)p.runs << p.sub) + (p.gb != nullptr ? (unsigned)(p.bias_cout + CONV_BIAS_CHANNELS - 1) / CONV_BIAS_CHANNELS : 0u);
}

template <int DT>
__device__ __forceinline__ void store_gradient(void* out, size_t at, float v) {
  if (DT == JG_F32) static_cast<float*>(out)[at] = v;
  else if (DT == JG_F16) static_cast<_Float16*>(out)[at] = (_Float16)v;
  else static_cast<uint16_t*>(out)[at] = f32_to_bf16(v);
}

// gw = sum over the partials of a block of channels (its workgroups, and in split mode its part pairs, which
// lie behind each other), and gb the same over the bias partials. A workgroup owns a run of 256 >> sub values of a
// block's partial (a tap, a pair, four registers and 64 >> sub lanes of the kernel that wrote it), a lane four of them; 8
// wavefronts take 8 << sub partials at a time in chains of their own and the sums are added in a fixed order
// (deterministic). What bounds it is the latency of the chains, 16-byte loads, eight in flight a lane. A block of 32 x 32 is 36 runs
// of 256 values, which left most of the chip idle: 6 x 26 -> 27 of 197 x 140 took 12.4 us, and takes 6.6 cut in four.
// The workgroups behind those of the last block add up bias partials, 16 channels each, four partials a wavefront at a time.
template <int DT>
__device__ __forceinline__ void reduce_conv_tiles(const jg_conv_reduction& p, unsigned block, ConvReduceShared& shared) {
  typedef float f32x4 __attribute__((ext_vector_type(4)));
  f32x4 (*const red)[64] = reinterpret_cast<f32x4(*)[64]>(shared.tiles);
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const unsigned weight_blocks = (unsigned)p.runs << p.sub;
  if (block >= weight_blocks) {
    // bias: a channel's block at x block 0 and x part 0 holds its sums
    constexpr int PER = 64 / CONV_BIAS_CHANNELS, STEP = CONV_RED_WAVES * PER;
    const int c = (int)(block - weight_blocks) * CONV_BIAS_CHANNELS + lane % CONV_BIAS_CHANNELS;
    float s = 0.0f;
    if (c < p.bias_cout) {
      for (int gp = p.bias_parts - 1; gp >= 0; --gp) {
        // plain: one pair per block. Part pairs: the pair (gp, 0) is pair kBias of the block
        const int pair_k = p.npairs == 6 ? (gp == 2 ? 2 : (gp == 1 ? 4 : 5)) : 0;
        const int row = p.npairs == 1 ? gp * p.bias_cout + c : c;  // all parts in one block: parts are channels of it
        const size_t slot0 = ((size_t)(row / p.rows) * p.ci_blocks * p.npairs + pair_k) * p.slots;
        const float* src = p.bias_part + slot0 * p.rows + row % p.rows;
        float c8[8] = {};
        for (int k = w * PER + lane / CONV_BIAS_CHANNELS; k < p.slots; k += 8 * STEP) {
#pragma unroll
          for (int u = 0; u < 8; ++u) {
            const int at = k + u * STEP;
            c8[u] += at < p.slots ? src[(size_t)at * p.rows] : 0.0f;
          }
        }
        s += ((c8[0] + c8[1]) + (c8[2] + c8[3])) + ((c8[4] + c8[5]) + (c8[6] + c8[7]));
      }
    }
#pragma unroll
    for (int o = CONV_BIAS_CHANNELS; o < 64; o <<= 1) s += __shfl_xor(s, o, 64);
    red[w][lane].x = s;
    __syncthreads();
    if (w != 0 || lane >= CONV_BIAS_CHANNELS || c >= p.bias_cout) return;
    s = 0.0f;
#pragma unroll
    for (int k = 0; k < CONV_RED_WAVES; ++k) s += red[k][lane].x;
    store_gradient<DT>(p.gb, c, s);
    return;
  }
  const int lanes = 64 >> p.sub, chains = CONV_RED_WAVES << p.sub;  // lanes of a run, chains of a workgroup
  const int runs = 9 * p.pairs * 4;                                  // runs of 256 values in a block's partial
  const int own = block >> p.sub, blk = own / runs, run = own - blk * runs;
  const int at = (int)(block & ((1u << p.sub) - 1)) * lanes + (lane & (lanes - 1));  // the lane of the writing kernel whose values these are
  const int slots = p.slots * p.npairs;
  const size_t stride = (size_t)runs * 256;
  const float* src = p.part + (size_t)blk * slots * stride + (size_t)run * 256 + at * 4;
  f32x4 c[8] = {};
  int k = (w << p.sub) + (lane >> (6 - p.sub));
  for (; k + 7 * chains < slots; k += 8 * chains) {
#pragma unroll
    for (int u = 0; u < 8; ++u) c[u] += *reinterpret_cast<const f32x4*>(src + (size_t)(k + u * chains) * stride);
  }
#pragma unroll
  for (int u = 0; u < 7; ++u)
    if (k + u * chains < slots) c[u] += *reinterpret_cast<const f32x4*>(src + (size_t)(k + u * chains) * stride);
  f32x4 sum = ((c[0] + c[1]) + (c[2] + c[3])) + ((c[4] + c[5]) + (c[6] + c[7]));
  for (int o = lanes; o < 64; o <<= 1)
#pragma unroll
    for (int u = 0; u < 4; ++u) sum[u] += __shfl_xor(sum[u], o, 64);
  red[w][lane] = sum;
  __syncthreads();
  if (w != 0 || lane >= lanes) return;
  sum = red[0][lane];
#pragma unroll
  for (int u = 1; u < CONV_RED_WAVES; ++u) sum += red[u][lane];
  const int j = run & 3, pair = (run >> 2) % p.pairs, tap = (run >> 2) / p.pairs;
  const int cb = pair / p.cols, ib = pair % p.cols;
  const int cx = ib * 32 + (at & 31), kd = cx / p.ci_step;
  const int ci = (blk % p.ci_blocks) * p.ci_step + cx % p.ci_step;
  if (ci >= p.cin) return;
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const int co = (blk / p.ci_blocks) * p.rows + cb * 32 + 8 * j + 4 * (at >> 5) + u;
    if (co < p.cout) store_gradient<DT>(p.gw, (((size_t)co * p.cin + ci) * p.KD + kd) * 9 + tap, sum[u]);
  }
}

// gw and gb of the fp32 kernels from the slots of every block: 16 neighbouring values a workgroup, four slots a wavefront at a time, in 64
// chains added in order (a workgroup of WAVES = 8 wavefronts walks those of two of the 16 in each). Bound by the latency of the
// chains: 64 values a workgroup in 16 chains left 8 workgroups with 1024 slots, 4 x 3 -> 16 of 256^2 7.2 us; so 4.6 with the border cells.
template <int WAVES>
__device__ __forceinline__ void reduce_conv_f32(const jg_conv_reduction& p, unsigned at_block, ConvReduceShared& shared) {
  constexpr int EACH = CONV_RED_CHAINS / WAVES, PER = 64 / CONV_F32_VALUES, STEP = CONV_RED_CHAINS * PER;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, per_block = p.rows * p.cols / CONV_F32_VALUES;
  const int block = at_block / per_block, at = (at_block - block * per_block) * CONV_F32_VALUES + lane % CONV_F32_VALUES;
  const size_t stride = (size_t)p.rows * p.cols;
  const float* src = p.part + (size_t)block * p.slots * stride + at;
  double s[EACH][4] = {};
  int k[EACH];
#pragma unroll
  for (int e = 0; e < EACH; ++e) k[e] = (wave + e * WAVES) * PER + lane / CONV_F32_VALUES;
  for (; k[EACH - 1] + 3 * STEP < p.slots;) {  // (the last chain is the first to run out of whole steps)
#pragma unroll
    for (int e = 0; e < EACH; ++e) {
#pragma unroll
      for (int u = 0; u < 4; ++u) s[e][u] += src[(size_t)(k[e] + u * STEP) * stride];
      k[e] += 4 * STEP;
    }
  }
#pragma unroll
  for (int e = 0; e < EACH; ++e) {
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (k[e] + u * STEP < p.slots) s[e][u] += src[(size_t)(k[e] + u * STEP) * stride];
    double sum = (s[e][0] + s[e][1]) + (s[e][2] + s[e][3]);
#pragma unroll
    for (int o = CONV_F32_VALUES; o < 64; o <<= 1) sum += __shfl_xor(sum, o, 64);
    shared.f32[wave + e * WAVES][lane] = sum;
  }
  __syncthreads();
  if (wave != 0 || lane >= CONV_F32_VALUES) return;
  double total = 0.0;
#pragma unroll
  for (int u = 0; u < CONV_RED_CHAINS; ++u) total += shared.f32[u][lane];
  const float sum = (float)total;
  const int co = block / p.ci_blocks * p.rows + at / p.cols, j = at % p.cols, ci = block % p.ci_blocks * p.ci_step + j / 9;
  if (co >= p.cout) return;
  if (j < p.ci_step * 9 && ci < p.cin) static_cast<float*>(p.gw)[((size_t)co * p.cin + ci) * 9 + j % 9] = sum;
  if (j == p.ci_step * 9 && block % p.ci_blocks == 0 && p.gb != nullptr) static_cast<float*>(p.gb)[co] = sum;
}

// Whether `later` is something that the weight gradient can have left: an error where it is not (conv_api.hip).
int check_conv_reduction(const jg_conv_reduction& later, const char* who);
// Does what `later`, so checked, holds, by itself.
int conv_reduce(const jg_conv_reduction& later, hipStream_t s);

}  // namespace jg
