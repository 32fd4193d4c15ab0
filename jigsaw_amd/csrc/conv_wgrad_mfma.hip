// Weight gradient of the 3x3 (2-D) and 3x3x3 (3-D) convolution on the bf16 matrix
// cores, stride 1 (2-D also stride 2), dilation 1, channels-first tensors; a workgroup covers a block of 32 or
// 64 channels a side, any other channel counts are more blocks of the same launch. Optionally the
// bias gradient from the same pass over g. fp16 tensors run the same kernel on the fp16
// MFMA instruction (the gradient is reduced in fp32 and rounded to fp16 once); fp32 tensors
// run as sums of three bf16 parts per operand ("split mode": the parts are extra channels,
// their products are added up in fp32).
//
//   gw[co][ci][kd][kh][kw] = sum_{n,d,h,w} g[n][co][d][h][w] * x[n][ci][d+kd-pd][h+kh-ph][w+kw-pw]
//   gb[co]                 = sum_{n,d,h,w} g[n][co][d][h][w]
//
//   GEMM view   M = output channels, N = input channels (x depth taps), K = pixels.
//               Both operands are pixel-contiguous in the channels-first tensors, so
//               the tiles go to LDS untransposed. A 3-D problem is the 2-D one with
//               the depth taps folded into the x "channels": channel kd*Cin + ci of a
//               stage at output depth d is the plane x[n][ci][d + kd - pd].
//   MFMA roles  A = g (32 channels x 16 pixels of a row), B = x (16 pixels x 32
//               channels) shifted by the tap. The kw shift is not 16-byte aligned in
//               LDS, so a lane reads 10 consecutive pixels once (b128 + b32) and
//               builds the three kw fragments with funnel shifts.
//   Workgroup   one wavefront per (g channel block, x channel block, part of the columns or rows of a stage);
//               it keeps its 9 taps x 32x32 fp32 accumulators in registers for the
//               whole kernel (144 VGPRs) and walks the pixels. 64->64 2-D: 2x2x2 = 8
//               wavefronts (two per SIMD, which is what hides the barrier and LDS
//               write phases); 32->32 3-D: 1x3x2 = 6, plus two that only prefetch.
//   Stage       2 output rows x 64 columns (32 at stride 2); consecutive stages of a workgroup walk
//               down one column strip, so two of the four x rows a stage reads are
//               the previous stage's last two. The x rows therefore live in a ring of
//               6 rows per channel in LDS and a stage fetches only its two new rows
//               (each x element is read from memory once per strip, apart from the
//               8 halo columns), plus its two g rows (double buffered). Loads go
//               through registers and are issued a whole stage ahead. The first stage
//               of a strip or of a workgroup fetches its other two rows on the spot.
//               Channel strides in LDS are odd multiples of 16 bytes so that the 32
//               channel-lanes of a fragment read hit distinct banks.
//   Bias grad   the lanes that carry the g chunks to LDS add them up on the way
//               (fp32), one partial per workgroup and channel.
//   Reduction   the parts of a pair are added in LDS, the workgroup's partial goes
//               to the workspace; a second kernel sums the partials in a fixed order
//               (deterministic) and writes gw in the weight layout and gb, in their own dtype.
#include <algorithm>
#include <cmath>

#include "conv_common.h"
#include "conv_reduce.h"

namespace {

using jg::ConvGeom;
using jg::mfma_frame_bands;

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4_a4 __attribute__((ext_vector_type(4), aligned(4)));

constexpr int SR = 2;                         // output rows per stage
constexpr int X_ROW = 144;                    // bytes of an x row in LDS: 66 pixels used
constexpr int X_CPR = 8;                      // 8-pixel chunks per x row; 2 more pixels follow as one dword
// By stride (1 or 2, the same along both axes). At stride 2 a stage of 2 x 32 output pixels reads 5 x 65 of x:
// the rows are as long as at stride 1. They go to LDS with their even columns in front and the odd ones behind
// (80 bytes on), so that the taps of a row are runs of consecutive pixels again: even[j], odd[j], even[j + 1].
// (The stride-1 kernel on a gradient with zeros between its pixels did four times the work, and the copies
// that made it: 64 -> 128 channels of 4 x 257 x 257 took 100 us.)
template <int ST>
struct Stage {
  static constexpr int SW = 64 / ST;              // output columns per stage
  static constexpr int XR = ST * (SR - 1) + 3;    // x rows a stage reads
  static constexpr int NEW = ST * SR;             // of which this many are new; the others are the stage above's last
  static constexpr int RING = XR + NEW;           // x rows resident per channel
  static constexpr int G_CH = SR * SW * 2 + 16;   // bytes per g channel
  static constexpr int X_CH = (RING * X_ROW) % 32 == 0 ? RING * X_ROW + 16 : RING * X_ROW + 32;  // per x channel: an odd multiple of 16
};
constexpr int X_ODD = 80;                         // stride 2: where the odd columns of a row start

struct WgradParams {
  const uint16_t* x;  // (N, Cin, Din, Hin, Win)
  const uint16_t* g;  // (N, Cout, Dout, Hout, Wout)
  const char* x_end;  // one past the last byte of x
  const char* g_end;  // one past the last byte of g
  float* part;        // [block][workgroup][tap9][32 x 32 pair][4][lane][4] (see the end of the kernel)
  float* bias_part;   // [block][workgroup][co], written by the blocks at the first x channel, or NULL
  // Framed input: xt (N, Cin, tn_d, tn_h, tn_w) is the own tile, at [tlo, tlo + tn) inside x.
  // A row pair whose window lies inside the tile is read from xt. NULL: all from x.
  const uint16_t* xt;
  int tlo_d, tlo_h, tlo_w, tn_d, tn_h, tn_w;
  // Blocks of channels, one per blockIdx.y: (block of g channels, block of x channels, part pair), the pair
  // fastest. cin, cout are the channels of one part (plain tensors have one), pair k multiplies part
  // (gparts >> 2 k) & 3 of g with part (xparts >> 2 k) & 3 of x. A channel past the last one repeats it and
  // is dropped where the partial sums are added up.
  int cin, cout, ci_blocks, npairs;
  uint32_t gparts, xparts;
  int cin_total, cout_total;  // channels of the tensors (parts * cin, parts * cout): batch strides
  int Din, Hin, Win, Dout, Hout, Wout;
  int pad_d, pad_h, pad_w;
  int row_pairs, col_tiles;
  long long total_stages;  // N * Dout * col_tiles * row_pairs
  long long per;           // of them a workgroup takes
  jg::Div by_rp, by_ct, by_od, by_pairs, by_ci;  // row_pairs, col_tiles, Dout, npairs, ci_blocks
};

// Wavefronts per workgroup: (g block, x block) pairs x parts of a stage's pixels. Blocks of 64 x 64 and those of a
// volume have two parts, the halves of the columns; a 6-wavefront shape gets two more wavefronts that only help with the prefetch.
// Blocks with one or two pairs have four, at stride 1 the quarters of the columns, at stride 2 halves of each row: with two
// parts there was one wavefront a SIMD, and what it did between its matrix instructions (loads, moves to LDS, the barrier)
// nothing ran beside; a part's fewer fragments leave room for two (200 to 256 registers; 302 to 320 before, 400 to 435 at stride 2).
// Partials and their reduction included: 2 x 40 -> 72 of 217 x 301 bf16 51 -> 44 us, 4 x 32 -> 64 of 512 x 512 80 -> 73, 7 x 5 -> 118
// of 229 x 380 92 -> 83, at stride 2 of 6 x 91 -> 23 of 244 x 446 76 -> 64 and of 2 x 77 -> 211 of 436 x 84 80 -> 57; the smallest
// layers (2 x 20 -> 33 of 100 x 150, 23 us) wait for the setup, the partials and the second launch, as before.
constexpr int wgrad_parts(int cgb, int cxb) { return cgb * cxb <= 2 ? 4 : 2; }
constexpr int wgrad_threads(int cgb, int cxb) {
  const int waves = cgb * cxb * wgrad_parts(cgb, cxb);
  return waves > 4 ? 512 : 64 * waves;
}
// LDS of a workgroup: two buffers of g and the ring of x, in whose place the parts meet at the end.
template <int CGB, int CXB, int ST>
constexpr size_t wgrad_lds() {
  const size_t stage = 2 * (size_t)(32 * CGB * Stage<ST>::G_CH) + (size_t)(32 * CXB * Stage<ST>::X_CH);
  const size_t waves = CGB * CXB * wgrad_parts(CGB, CXB), meet = waves * (12 - 12 / wgrad_parts(CGB, CXB)) * 1024;
  return stage > meet ? stage : meet;
}
// Workgroups of one pair fit a compute unit twice.
constexpr int wgrad_waves_per_simd(int cgb, int cxb) { return wgrad_parts(cgb, cxb) == 4 || wgrad_threads(cgb, cxb) == 512 ? 2 : 1; }

// sum of the 8 values of a chunk
template <bool F16>
__device__ __forceinline__ float sum_of_8(const u32x4& v) {
  if (F16) {
    const f16x8 h = __builtin_bit_cast(f16x8, v);
    float s = (float)h[0] + (float)h[1];
    s += (float)h[2] + (float)h[3];
    s += (float)h[4] + (float)h[5];
    s += (float)h[6] + (float)h[7];
    return s;
  }
  float s = __uint_as_float(v.x << 16) + __uint_as_float(v.x & 0xffff0000u);
  s += __uint_as_float(v.y << 16) + __uint_as_float(v.y & 0xffff0000u);
  s += __uint_as_float(v.z << 16) + __uint_as_float(v.z & 0xffff0000u);
  s += __uint_as_float(v.w << 16) + __uint_as_float(v.w & 0xffff0000u);
  return s;
}

// F16: x and g hold fp16 instead of bf16 (v_mfma_f32_32x32x16_f16); the partial sums are fp32 either way.
// EVEN: 0 = rows may start on odd pixels: a chunk is read from the dword below it, with the dword of its last
// pixel, and moved into place on its way to LDS (2-byte loads took 52 us where this takes 23: 40 x 72
// channels, 2 x 217 x 301), 1 = even row lengths,
// 4-byte aligned tensors and an even padding across W, so that a stage's windows start on dwords and
// the 16-byte vector loads apply, 2 = the same with an odd padding: the x window is staged from one
// pixel earlier, where it is dword aligned again, and the fragments are built one pixel further in.
// ALLIN: the host has checked that every window of every stage lies inside x and every stage's
// rows inside g (a convolution without padding over a tensor that holds its halo, tiles of whole
// stages): the kernel is built without the element-wise border path, and its stage loop loads and
// stores without conditions.
template <int CGB, int CXB, int EVEN, bool FRAMED, bool F16 = false, bool ALLIN = false, int ST = 1>
__global__ __launch_bounds__(wgrad_threads(CGB, CXB), wgrad_waves_per_simd(CGB, CXB)) void wgrad3x3_mfma_kernel(WgradParams p) {
  constexpr int THREADS = wgrad_threads(CGB, CXB);
  constexpr int LEAD = EVEN == 2 ? 1 : 0;
  static_assert(!(FRAMED && EVEN != 1), "the framed input is read with even windows only");
  static_assert(ST == 1 || (EVEN != 2 && !FRAMED && !ALLIN && CXB != 3), "stride 2 is built for plain 2-D tensors");
  constexpr int SW = Stage<ST>::SW, XR = Stage<ST>::XR, NEW = Stage<ST>::NEW, RING = Stage<ST>::RING;
  constexpr int G_CH = Stage<ST>::G_CH, X_CH = Stage<ST>::X_CH;
  constexpr int G_CPR = SW / 8;  // chunks per g row
  constexpr int PARTS = wgrad_parts(CGB, CXB);
  constexpr int COL_PARTS = ST == 1 ? PARTS : 2, ROW_PARTS = PARTS / COL_PARTS;
  constexpr int CWAVES = CGB * CXB * PARTS;  // wavefronts that own accumulators
  constexpr int GC = 32 * CGB, XC = 32 * CXB;
  constexpr int G_BYTES = GC * G_CH;          // one g buffer
  constexpr int G_CHUNKS = GC * SR * G_CPR;
  constexpr int XP_CHUNKS = XC * NEW * X_CPR;   // the new x rows of a stage
  // Rounds of loads, a chunk a thread: those of g first (the last of them may leave lanes over), then those of x
  constexpr int G_ROUNDS = (G_CHUNKS + THREADS - 1) / THREADS, X_FIRST = G_ROUNDS * THREADS;
  constexpr int CHUNKS = X_FIRST + XP_CHUNKS;
  constexpr int ROUNDS = (CHUNKS + THREADS - 1) / THREADS;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  unsigned char* const lds_x = smem + 2 * G_BYTES;
  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6;
  const int ln = lane & 31, kgp = lane >> 5;
  const int pair = wave % (CGB * CXB), part = (wave / (CGB * CXB)) % PARTS;
  const int cb = pair / CXB, ib = pair % CXB;

  // contiguous range of stages for this workgroup; stage -> (n, d, column tile, row pair),
  // row pair fastest, so consecutive stages walk down one column strip of one plane
  // Workgroups are dealt to the 8 XCDs round robin; the ranges are numbered so that one
  // XCD holds neighbouring column strips, whose x rows share cache lines in that XCD's L2.
  const unsigned wg_rank = gridDim.x % 8 == 0 ? (blockIdx.x % 8) * (gridDim.x / 8) + blockIdx.x / 8 : blockIdx.x;
  const long long s_begin = min(p.per * wg_rank, p.total_stages);
  const long long s_end = min(p.per * (wg_rank + 1), p.total_stages);

  // ---- the block of channels
  constexpr int KD = CXB == 3 ? 3 : 1, CIN_B = XC / KD;  // three x blocks are the depth taps of 32 channels
  int cin_valid, cout_valid;                             // channels of the block that exist
  const uint16_t *xb, *gb;                               // its first channel in batch entry 0
  const int block = blockIdx.y;
  bool first_x;
  {
    const int rest = jg::quotient(block, p.by_pairs), pair_k = block - rest * p.npairs, co_block = jg::quotient(rest, p.by_ci);
    const int ci0 = (rest - co_block * p.ci_blocks) * CIN_B, co0 = co_block * GC;
    const int gpart = (int)((p.gparts >> (2 * pair_k)) & 3u), xpart = (int)((p.xparts >> (2 * pair_k)) & 3u);
    cin_valid = min(CIN_B, p.cin - ci0);
    cout_valid = min(GC, p.cout - co0);
    xb = p.x + (size_t)(xpart * p.cin + ci0) * ((size_t)p.Hin * p.Win * p.Din);
    gb = p.g + (size_t)(gpart * p.cout + co0) * ((size_t)p.Hout * p.Wout * p.Dout);
    first_x = ci0 == 0 && xpart == 0;  // the bias sum of these g rows is this block's
  }
  float* const bias_part = p.bias_part != nullptr && first_x ? p.bias_part : nullptr;

  const size_t plane_x = (size_t)p.Hin * p.Win, plane_g = (size_t)p.Hout * p.Wout;
  const size_t x_cs = plane_x * p.Din, g_cs = plane_g * p.Dout;  // channel strides

  // ---- per-thread chunk bookkeeping, fixed for the whole kernel. Chunk q < G_CHUNKS
  // is 8 pixels of a g row, the others 8 pixels of one of the two x rows of a pair.
  uint32_t c_goff[ROUNDS];  // byte offset from the origin of its tensor window
  // byte offset inside the g buffer / inside the x ring, row slot 0 (stride 1: of the chunk's own row, the new rows being a pair that
  // never lies across the ring's end)
  uint32_t c_lds[ROUNDS];
  uint32_t x_row = 0;       // stride 2, two bits per round: the chunk's row among the new ones
  static_assert(ST == 2 || RING % NEW == 0, "pairs of rows stay together in the ring");
#pragma unroll
  for (int rd = 0; rd < ROUNDS; ++rd) {
    const int q = tid + rd * THREADS;
    if (q < G_CHUNKS) {
      const int c8 = q % G_CPR, r = (q / G_CPR) % SR, ch = q / (G_CPR * SR);
      const int che = ch < cout_valid ? ch : cout_valid - 1;  // a channel past the last one reads the last
      c_goff[rd] = (uint32_t)((che * g_cs + (size_t)r * p.Wout + c8 * 8) * 2);
      c_lds[rd] = (uint32_t)(ch * G_CH + r * (SW * 2) + c8 * 16);
    } else if (q >= X_FIRST && q < CHUNKS) {
      const int qx = q - X_FIRST;
      const int c8 = qx % X_CPR;
      const int rr = qx / X_CPR;
      const int r2 = rr % NEW, ch = rr / NEW;   // ch = kd * CIN_B + ci
      const int kd = ch / CIN_B, cib = ch - kd * CIN_B;
      const int ci = cib < cin_valid ? cib : cin_valid - 1;
      c_goff[rd] = (uint32_t)((ci * x_cs + kd * plane_x + (size_t)r2 * p.Win + c8 * 8) * 2);
      c_lds[rd] = (uint32_t)(ch * X_CH + c8 * (16 / ST) + (ST == 1 ? r2 * X_ROW : 0));
      if (ST == 2) x_row |= (uint32_t)r2 << (2 * rd);
    } else {
      c_goff[rd] = 0;
      c_lds[rd] = 0;
    }
  }
  // pixels 64, 65 of an x row (and 66, 67 of a window staged one pixel early): one or two dwords,
  // carried by the first NEW * XC threads
  static_assert(NEW * XC <= THREADS, "a thread carries one tail");
  const bool has_tail = tid < NEW * XC;
  uint32_t t_goff = 0, t_lds = 0;
  if (has_tail) {
    const int r2 = tid % NEW, ch = tid / NEW;
    const int kd = ch / CIN_B, cib = ch - kd * CIN_B;
    const int ci = cib < cin_valid ? cib : cin_valid - 1;
    t_goff = (uint32_t)((ci * x_cs + kd * plane_x + (size_t)r2 * p.Win + 64) * 2);
    t_lds = (uint32_t)(ch * X_CH + 128 / ST + (ST == 1 ? r2 * X_ROW : 0));
  }
  // the same x offsets inside the own tile (framed input)
  const size_t plane_t = (size_t)p.tn_h * p.tn_w, t_cs = plane_t * p.tn_d;
  uint32_t c_toff[ROUNDS];
  uint32_t t_toff = 0;
  uint32_t x_kd = 0;  // 2 bits per round: depth tap of the chunk; bits 30-31: of the tail
  if (FRAMED) {
#pragma unroll
    for (int rd = 0; rd < ROUNDS; ++rd) {
      const int q = tid + rd * THREADS;
      c_toff[rd] = 0;
      if (q >= X_FIRST && q < CHUNKS) {
        const int qx = q - X_FIRST;
        const int c8 = qx % X_CPR, rr = qx / X_CPR;
        const int r2 = rr & 1, ch = rr >> 1;
        const int kd = ch / CIN_B, ci = ch - kd * CIN_B;
        c_toff[rd] = (uint32_t)((ci * t_cs + kd * plane_t + (size_t)r2 * p.tn_w + c8 * 8) * 2);
        x_kd |= (uint32_t)kd << (2 * rd);
      }
    }
    if (has_tail) {
      const int r2 = tid & 1, ch = tid >> 1;
      const int kd = ch / CIN_B, ci = ch - kd * CIN_B;
      t_toff = (uint32_t)((ci * t_cs + kd * plane_t + (size_t)r2 * p.tn_w + SW) * 2);
      x_kd |= (uint32_t)kd << 30;
    }
  }

  struct Staged {
    u32x4 v[ROUNDS];
    uint32_t tail;
    uint32_t tail_b;       // LEAD; EVEN == 0: the dword of the tail's second pixel
    uint32_t next[ROUNDS];  // EVEN == 0: the dword of the chunk's last pixel
    uint32_t odd;           // EVEN == 0: one bit per round, the chunk starts on the upper half of a dword; bit 31: the tail
    // a stage whose windows stick out of the tensors: pixels of the chunks that exist (one bit each, a thread's
    // chunks all have the same columns), rounds whose row exists (one bit each), pixels of the tail
    bool masked;
    uint32_t g_cols, x_cols, rows, tail_cols;
    uint32_t over;  // rounds (bit 31: the tail) whose bytes reach over the tensor's ends and are not loaded yet
    const char *g_org, *x_org;
  };

  // Loads of one stage into `v`: its two g rows (want_g) and one pair of its x rows
  // (pair 0: the rows shared with the stage above, pair 1: the two new rows).
  // Position of a stage: row pair (fastest), column tile, output depth, batch entry, and the first bytes of its g rows and its new x
  // rows. Decoded once, then stepped: down a strip the two addresses move by a constant, and only a new strip works
  // them out. (From scratch in every stage they were most of its 120 to 170 scalar instructions: 2 x 40 -> 72 of 217 x 301 37.2 -> 34.6 us,
  // 2 x 48 -> 19 of 121 x 126 x 78 538 -> 509, 2 x 32 -> 32 of 128^3 284 -> 268; 64 x 64 blocks without edges do not wait for them, 617 -> 615.)
  struct Cursor {
    int hp, ct, od, n;
    const char *g, *x;
  };
  const uint32_t g_step = 2u * SR * (uint32_t)p.Wout, x_step = 2u * NEW * (uint32_t)p.Win;  // of one stage
  auto place = [&](Cursor& c) {
    c.g = reinterpret_cast<const char*>(gb) +
          2 * (((size_t)c.n * p.cout_total * p.Dout + c.od) * plane_g + (size_t)(c.hp * SR) * p.Wout + c.ct * SW);
    c.x = reinterpret_cast<const char*>(xb) +
          2 * ((ptrdiff_t)((size_t)c.n * p.cin_total * p.Din * plane_x) + (ptrdiff_t)(c.od - p.pad_d) * (ptrdiff_t)plane_x +
               (ptrdiff_t)(ST * c.hp * SR - p.pad_h + XR - NEW) * p.Win + (ST * c.ct * SW - p.pad_w - LEAD));
  };
  auto decode = [&](long long stage) {
    Cursor c;
    if (p.total_stages < (1ll << 31)) {
      const int col = jg::quotient((uint32_t)stage, p.by_rp), plane = jg::quotient(col, p.by_ct);
      c.hp = (int)stage - col * p.row_pairs;
      c.ct = col - plane * p.col_tiles;
      c.n = jg::quotient(plane, p.by_od);
      c.od = plane - c.n * p.Dout;
    } else {
      c.hp = (int)(stage % p.row_pairs);
      long long t = stage / p.row_pairs;
      c.ct = (int)(t % p.col_tiles);
      t /= p.col_tiles;
      c.od = (int)(t % p.Dout);
      c.n = (int)(t / p.Dout);
    }
    place(c);
    return c;
  };
  auto advance = [&](Cursor& c) {
    c.g += g_step;
    c.x += x_step;
    if (++c.hp == p.row_pairs) {
      c.hp = 0;
      if (++c.ct == p.col_tiles) {
        c.ct = 0;
        if (++c.od == p.Dout) {
          c.od = 0;
          ++c.n;
        }
      }
      place(c);
    }
  };

  auto issue_loads = [&](Staged& sg, const Cursor& cur, bool want_g, int xpair) {
    u32x4 (&v)[ROUNDS] = sg.v;
    const int hp = cur.hp, ct = cur.ct, od = cur.od, n = cur.n;
    const int oh0 = hp * SR, ow0 = ct * SW;
    // first of the rows: of the new ones, or (xpair 0) as many rows further up, the last of which a first stage lacks
    const int id0 = od - p.pad_d, ih0 = ST * oh0 - p.pad_h + XR - (xpair ? 1 : 2) * NEW, iw0 = ST * ow0 - p.pad_w - LEAD;
    const char* const g_org = cur.g;
    const char* const x_org = xpair ? cur.x : cur.x - x_step;
    // (with LEAD the window's last dword holds one pixel more than is used; it shares its dword with one that is)
    const bool rows_inside = oh0 + SR <= p.Hout && ih0 >= 0 && ih0 + NEW <= p.Hin && id0 >= 0 && id0 + KD <= p.Din;
    // All that a stage's loads of x and g reach lies inside the tensors, whatever columns the rows have
    constexpr bool kWhole = !FRAMED;  // (the framed kernels have no registers for it)
    auto whole = [&]() {
      const char* const x_last = x_org + 2 * ((size_t)(cin_valid - 1) * x_cs + (size_t)(KD - 1) * plane_x + (size_t)(NEW - 1) * p.Win) + 2 * 64 + 16;
      const char* const g_last = g_org + 2 * ((size_t)(cout_valid - 1) * g_cs + (size_t)(SR - 1) * p.Wout) + 2 * SW + 8;
      return kWhole && rows_inside && x_org >= reinterpret_cast<const char*>(p.x) && x_last <= p.x_end && g_last <= p.g_end;
    };
    // (at stride 2 the window's last pixel is read and not used: a tile that holds one halo column ends before it)
    const bool inside = ALLIN || (oh0 + SR <= p.Hout && ow0 + SW <= p.Wout && ih0 >= 0 &&
                        ih0 + NEW <= p.Hin && iw0 >= 0 && (iw0 + 66 + LEAD <= p.Win || (ST == 2 && iw0 + 65 <= p.Win && whole())) &&
                        id0 >= 0 && id0 + KD <= p.Din);
    sg.masked = !inside;
    sg.odd = 0;
    if (FRAMED && inside) {
      // Rows and columns of the pair's window inside the own tile (wave-uniform): a chunk
      // whose depth plane is a plane of the tile comes from the tile itself, at whatever
      // alignment its rows give the window; the planes outside the tile are halo planes,
      // which the frame holds whole.
      const int dt = id0 - p.tlo_d, ht = ih0 - p.tlo_h, wt = iw0 - p.tlo_w;
      if (ht >= 0 && ht + 2 <= p.tn_h && wt >= 0 && wt + SW + 2 <= p.tn_w) {
        const char* t_org = reinterpret_cast<const char*>(p.xt) +
                            2 * ((ptrdiff_t)((size_t)n * p.cin_total * t_cs) + (ptrdiff_t)dt * (ptrdiff_t)plane_t +
                                 (ptrdiff_t)ht * p.tn_w + wt);
        // 4-byte aligned accesses only (2-byte aligned vector loads run at a fraction of the
        // rate): a window that starts on an odd column is read one pixel early and shifted.
        // tn_w is even (checked on the host), so the parity is the same for every chunk.
        const bool odd = (reinterpret_cast<uintptr_t>(t_org) & 2) != 0;  // wave-uniform
        uint32_t lead[ROUNDS];
#pragma unroll
        for (int rd = 0; rd < ROUNDS; ++rd) {
          const int q = tid + rd * THREADS;
          lead[rd] = 0u;
          if (q < G_CHUNKS) {
            if (want_g) v[rd] = *reinterpret_cast<const u32x4_a4*>(g_org + c_goff[rd]);
          } else if (q < CHUNKS) {
            const int dd = dt + (int)((x_kd >> (2 * rd)) & 3u);
            if (dd >= 0 && dd < p.tn_d) {
              if (odd) {
                lead[rd] = *reinterpret_cast<const uint32_t*>(t_org + c_toff[rd] - 2);
                v[rd] = *reinterpret_cast<const u32x4_a4*>(t_org + c_toff[rd] + 2);
              } else {
                v[rd] = *reinterpret_cast<const u32x4_a4*>(t_org + c_toff[rd]);
              }
            } else {
              v[rd] = *reinterpret_cast<const u32x4_a4*>(x_org + c_goff[rd]);
            }
          }
        }
        uint32_t tail_lead = 0u;
        bool tail_shift = false;
        if (has_tail) {
          const int dd = dt + (int)(x_kd >> 30);
          if (dd >= 0 && dd < p.tn_d) {
            if (odd) {
              tail_lead = *reinterpret_cast<const uint32_t*>(t_org + t_toff - 2);
              sg.tail = *reinterpret_cast<const uint32_t*>(t_org + t_toff + 2);
              tail_shift = true;
            } else {
              sg.tail = *reinterpret_cast<const uint32_t*>(t_org + t_toff);
            }
          } else {
            sg.tail = *reinterpret_cast<const uint32_t*>(x_org + t_goff);
          }
        }
        if (odd) {
#pragma unroll
          for (int rd = 0; rd < ROUNDS; ++rd) {
            const int q = tid + rd * THREADS;
            if (q >= X_FIRST && q < CHUNKS) {
              const int dd = dt + (int)((x_kd >> (2 * rd)) & 3u);
              if (dd >= 0 && dd < p.tn_d) {
                const u32x4 t = v[rd];
                v[rd].x = __builtin_amdgcn_alignbit(t.x, lead[rd], 16);
                v[rd].y = __builtin_amdgcn_alignbit(t.y, t.x, 16);
                v[rd].z = __builtin_amdgcn_alignbit(t.z, t.y, 16);
                v[rd].w = __builtin_amdgcn_alignbit(t.w, t.z, 16);
              }
            }
          }
          if (tail_shift) sg.tail = __builtin_amdgcn_alignbit(sg.tail, tail_lead, 16);
        }
        return;
      }
    }
    // One set of loads for every stage, from addresses that differ: a load under a condition leaves its register with
    // two possible values where the paths meet, and the compiler then waits for it right there instead of where it
    // is stored, half a stage later. Every lane loads in every round it is asked for (the lanes past the last chunk
    // and those without a tail read offset 0 of the window, or the workspace).
    uintptr_t at[ROUNDS];
    uintptr_t t_at = reinterpret_cast<uintptr_t>(x_org) + t_goff;
#pragma unroll
    for (int rd = 0; rd < ROUNDS; ++rd) at[rd] = reinterpret_cast<uintptr_t>(rd < G_ROUNDS ? g_org : x_org) + c_goff[rd];
    if (!inside) {
      // A stage at an edge. A chunk is read wherever its bytes lie inside its tensor, also past the end of its
      // row; store_loads clears the pixels that are not the row's. A chunk without any pixel of the tensor reads
      // the workspace instead, and so do the few whose bytes reach over the tensor's own ends: store_loads
      // fetches these.
      auto columns = [](int col, int count, int cols) {  // of the pixels col .. col + count - 1, those in [0, cols)
        const int first = max(0, min(count, -col)), past = max(0, min(count, cols - col));
        return ((1u << past) - 1u) & ~((1u << first) - 1u);
      };
      const int c8 = tid & 7;  // a round is a multiple of 8 chunks: the same in all of them
      sg.g_cols = columns(ow0 + (tid % G_CPR) * 8, 8, p.Wout);
      sg.x_cols = columns(iw0 + c8 * 8, 8, p.Win);
      sg.rows = 0;
      sg.over = 0;
      sg.g_org = g_org;
      sg.x_org = x_org;
      // Where only the columns stick out and what is read past them is the tensors' all the same (every strip at the end of
      // the rows but for its ends), nothing but these masks differs from a stage inside. The workgroups on such a strip
      // are the last ones to end: 2 x 40 -> 72 channels of 216 x 318 41 -> 37.4 us, of
      // 217 x 301 48.3 -> 44.6; 4 x 64 -> 128 of 256 x 256 at stride 2, whose padded rows are 257 pixels, 48.6 -> 41.4.
      if (whole()) {
        sg.rows = ~0u;
        sg.tail_cols = has_tail ? columns(iw0 + 64, 2 + 2 * LEAD, p.Win) : 0u;
      } else {
        const uintptr_t safe = reinterpret_cast<uintptr_t>(p.part);
#pragma unroll
        for (int rd = 0; rd < ROUNDS; ++rd) {
          const bool g_round = rd < G_ROUNDS;
          const int q = tid + rd * THREADS;
          bool row_ok;
          if (g_round) {
            row_ok = oh0 + (q / G_CPR) % SR < p.Hout;
          } else {
            const int rr = (q - X_FIRST) / X_CPR;
            const int row = ih0 + rr % NEW, dd = id0 + (rr / NEW) / CIN_B;
            row_ok = q < CHUNKS && row >= 0 && row < p.Hin && dd >= 0 && dd < p.Din;
          }
          const bool need = row_ok && (g_round ? sg.g_cols : sg.x_cols) != 0u;
          const bool fits = at[rd] >= reinterpret_cast<uintptr_t>(g_round ? p.g : p.x) &&
                            at[rd] + 16 <= reinterpret_cast<uintptr_t>(g_round ? p.g_end : p.x_end);
          sg.rows |= (need ? 1u : 0u) << rd;
          sg.over |= (need && !fits ? 1u : 0u) << rd;
          at[rd] = need && fits ? at[rd] : safe;
        }
        const int row = ih0 + tid % NEW, dd = id0 + (tid / NEW) / CIN_B;
        const bool ok = has_tail && dd >= 0 && dd < p.Din && row >= 0 && row < p.Hin;
        sg.tail_cols = ok ? columns(iw0 + 64, 2 + 2 * LEAD, p.Win) : 0u;
        const bool fits = t_at >= reinterpret_cast<uintptr_t>(p.x) && t_at + 4 + 4 * LEAD <= reinterpret_cast<uintptr_t>(p.x_end);
        sg.over |= (sg.tail_cols != 0u && !fits ? 1u : 0u) << 31;
        t_at = sg.tail_cols != 0u && fits ? t_at : safe;
      }
    }
#pragma unroll
    for (int rd = 0; rd < ROUNDS; ++rd) {
      const bool g_round = rd < G_ROUNDS;
      if (!want_g && g_round) continue;
      v[rd] = jg::load_16_bytes_at(EVEN == 0 ? at[rd] & ~(uintptr_t)3 : at[rd]);
      if (EVEN == 0) {
        sg.next[rd] = jg::load_4_bytes_at((at[rd] + 14) & ~(uintptr_t)3);
        sg.odd |= (uint32_t)((at[rd] >> 1) & 1) << rd;
      }
    }
    sg.tail = jg::load_4_bytes_at(t_at & ~(uintptr_t)3);
    if (LEAD) sg.tail_b = jg::load_4_bytes_at(t_at + 4);
    if (EVEN == 0) {
      sg.tail_b = jg::load_4_bytes_at((t_at + 2) & ~(uintptr_t)3);
      sg.odd |= (uint32_t)((t_at >> 1) & 1) << 31;
    }
  };
  // The chunks of an edge stage whose bytes reach over the ends of their tensor: dword by dword, those that hold
  // a pixel of it.
  auto fetch_over = [&](Staged& sg, bool have_g) {
    auto dword_at = [](uintptr_t at, const void* begin, const char* end) {
      return at + 4 > reinterpret_cast<uintptr_t>(begin) && at < reinterpret_cast<uintptr_t>(end) ? jg::load_4_bytes_at(at) : 0u;
    };
#pragma unroll
    for (int rd = 0; rd < ROUNDS; ++rd) {
      const bool g_round = rd < G_ROUNDS;
      if ((!have_g && g_round) || ((sg.over >> rd) & 1u) == 0) continue;
      const void* begin = g_round ? p.g : p.x;
      const char* end = g_round ? p.g_end : p.x_end;
      const uintptr_t at = reinterpret_cast<uintptr_t>(g_round ? sg.g_org : sg.x_org) + c_goff[rd];
      const uintptr_t down = at & ~(uintptr_t)3;
#pragma unroll
      for (int j = 0; j < 4; ++j) sg.v[rd][j] = dword_at(down + 4 * j, begin, end);
      if (EVEN == 0) {
        sg.next[rd] = dword_at((at + 14) & ~(uintptr_t)3, begin, end);
        sg.odd = (sg.odd & ~(1u << rd)) | ((uint32_t)((at >> 1) & 1) << rd);
      }
    }
    if ((sg.over >> 31) != 0) {
      const uintptr_t at = reinterpret_cast<uintptr_t>(sg.x_org) + t_goff;
      sg.tail = dword_at(at & ~(uintptr_t)3, p.x, p.x_end);
      if (LEAD) sg.tail_b = dword_at(at + 4, p.x, p.x_end);
      if (EVEN == 0) {
        sg.tail_b = dword_at((at + 2) & ~(uintptr_t)3, p.x, p.x_end);
        sg.odd = (sg.odd & 0x7fffffffu) | ((uint32_t)((at >> 1) & 1) << 31);
      }
    }
  };

  // Registers of a stage to LDS: g rows into g buffer `gbuf`, the x rows into ring rows
  // slot0, slot0 + 1, ..; the g chunks are added into the bias partials on the way.
  float bsum[ROUNDS];
#pragma unroll
  for (int rd = 0; rd < ROUNDS; ++rd) bsum[rd] = 0.0f;
  auto store_loads = [&](Staged& sg, bool have_g, int gbuf, int slot0, bool counted = true) {
    uint32_t g_keep[4], x_keep[4];
    if (!ALLIN && sg.masked) {
      if (__builtin_amdgcn_ballot_w64(sg.over != 0u) != 0) fetch_over(sg, have_g);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        g_keep[j] = (((sg.g_cols >> (2 * j)) & 1u) * 0xffffu) | (((sg.g_cols >> (2 * j + 1)) & 1u) * 0xffff0000u);
        x_keep[j] = (((sg.x_cols >> (2 * j)) & 1u) * 0xffffu) | (((sg.x_cols >> (2 * j + 1)) & 1u) * 0xffff0000u);
      }
    }
#pragma unroll
    for (int rd = 0; rd < ROUNDS; ++rd) {
      const int q = tid + rd * THREADS;
      const bool g_round = rd < G_ROUNDS;
      if (g_round && !have_g) continue;
      u32x4 val = sg.v[rd];
      if (EVEN == 0) {
        const uint32_t shift = ((sg.odd >> rd) & 1u) << 4;
        val.x = __builtin_amdgcn_alignbit(val.y, val.x, shift);
        val.y = __builtin_amdgcn_alignbit(val.z, val.y, shift);
        val.z = __builtin_amdgcn_alignbit(val.w, val.z, shift);
        val.w = __builtin_amdgcn_alignbit(sg.next[rd], val.w, shift);
      }
      if (!ALLIN && sg.masked) {  // uniform
        const uint32_t row = 0u - ((sg.rows >> rd) & 1u);
        val.x &= (g_round ? g_keep[0] : x_keep[0]) & row;
        val.y &= (g_round ? g_keep[1] : x_keep[1]) & row;
        val.z &= (g_round ? g_keep[2] : x_keep[2]) & row;
        val.w &= (g_round ? g_keep[3] : x_keep[3]) & row;
      }
      if (g_round) {
        if (G_CHUNKS % THREADS == 0 || q < G_CHUNKS) *reinterpret_cast<u32x4*>(smem + gbuf * G_BYTES + c_lds[rd]) = val;
        if (bias_part != nullptr) bsum[rd] += counted ? sum_of_8<F16>(val) : 0.0f;
      } else if (q < CHUNKS) {
        int slot = slot0;
        if (ST == 2) {
          slot += (int)((x_row >> (2 * rd)) & 3u);
          if (slot >= RING) slot -= RING;
        }
        unsigned char* const at = lds_x + c_lds[rd] + slot * X_ROW;
        if (ST == 1) {
          *reinterpret_cast<u32x4*>(at) = val;
        } else {
          *reinterpret_cast<uint64_t*>(at) = (uint64_t)__builtin_amdgcn_perm(val.y, val.x, 0x05040100u) |
                                             (uint64_t)__builtin_amdgcn_perm(val.w, val.z, 0x05040100u) << 32;
          *reinterpret_cast<uint64_t*>(at + X_ODD) = (uint64_t)__builtin_amdgcn_perm(val.y, val.x, 0x07060302u) |
                                                     (uint64_t)__builtin_amdgcn_perm(val.w, val.z, 0x07060302u) << 32;
        }
      }
    }
    if (has_tail) {
      int slot = slot0;
      if (ST == 2) {
        slot += tid % NEW;
        if (slot >= RING) slot -= RING;
      }
      unsigned char* at = lds_x + t_lds + slot * X_ROW;
      uint32_t t = sg.tail, tb = sg.tail_b;
      if (EVEN == 0) t = __builtin_amdgcn_alignbit(tb, t, (sg.odd >> 31) << 4);
      if (!ALLIN && sg.masked) {
        t &= ((sg.tail_cols & 1u) * 0xffffu) | (((sg.tail_cols >> 1) & 1u) * 0xffff0000u);
        if (LEAD) tb &= (((sg.tail_cols >> 2) & 1u) * 0xffffu) | (((sg.tail_cols >> 3) & 1u) * 0xffff0000u);
      }
      *reinterpret_cast<uint32_t*>(at) = t;
      if (LEAD) *reinterpret_cast<uint32_t*>(at + 4) = tb;
    }
  };

  f32x16 acc[3][3];
#pragma unroll
  for (int a = 0; a < 3; ++a)
#pragma unroll
    for (int b = 0; b < 3; ++b)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[a][b][i] = 0.0f;

  // one 16-pixel column group (cgi = 0 or 1 of this wavefront's part) of a stage whose
  // x rows sit in ring rows base .. base + XR - 1 (mod RING): first all its LDS reads
  // (read_group), then its matrix instructions (mfma_group), so that a stage can ask for both
  // of its groups before the first matrix instruction and meets the LDS latency once.
  constexpr int GROUPS = SW / 16 / COL_PARTS;
  constexpr int PR = SR / ROW_PARTS, PXR = ST * (PR - 1) + 3;  // output rows of a part, x rows it reads
  struct Frags {
    u32x4 a[PR];
    u32x4 d[PXR];
    uint32_t d4[PXR], d5[PXR];
    u32x4 odd[PXR];  // stride 2
  };
  const int row0 = ROW_PARTS == 1 ? 0 : part / COL_PARTS;  // first output row of the part
  auto read_group = [&](Frags& f, int gbuf, int base, int cgi) __attribute__((always_inline)) {
    const unsigned char* gb = smem + gbuf * G_BYTES + (cb * 32 + ln) * G_CH + kgp * 16;
    const unsigned char* xb = lds_x + (ib * 32 + ln) * X_CH + kgp * 16;
    const int cg = part % COL_PARTS * GROUPS + cgi;  // 16-pixel column group of this wavefront
#pragma unroll
    for (int r = 0; r < PR; ++r) f.a[r] = *reinterpret_cast<const u32x4*>(gb + (row0 + r) * (SW * 2) + cg * 32);
#pragma unroll
    for (int rho = 0; rho < PXR; ++rho) {
      // (stride 1: two pairs of rows, each in one piece of the ring)
      int slot = base + ST * row0 + (ST == 1 ? rho / NEW * NEW : rho);
      if (slot >= RING) slot -= RING;
      if (ST == 1) slot += rho % NEW;
      f.d[rho] = *reinterpret_cast<const u32x4*>(xb + slot * X_ROW + cg * 32);
      f.d4[rho] = *reinterpret_cast<const uint32_t*>(xb + slot * X_ROW + cg * 32 + 16);
      f.d5[rho] = 0u;
      if (LEAD) f.d5[rho] = *reinterpret_cast<const uint32_t*>(xb + slot * X_ROW + cg * 32 + 20);
      if (ST == 2) f.odd[rho] = *reinterpret_cast<const u32x4*>(xb + slot * X_ROW + X_ODD + cg * 32);
    }
  };
  auto mfma_group = [&](Frags& f) __attribute__((always_inline)) {
    bf16x8 a[PR];
#pragma unroll
    for (int r = 0; r < PR; ++r) a[r] = __builtin_bit_cast(bf16x8, f.a[r]);
#pragma unroll
    for (int rho = 0; rho < PXR; ++rho) {
      u32x4 d = f.d[rho];
      uint32_t d4 = f.d4[rho], d5 = f.d5[rho];
      // The values are made opaque so that the kw = 2 fragment below is built with register
      // moves: left alone, the compiler reads it again from LDS at a 4-byte offset, as dword
      // pairs whose 880-byte lane stride runs into 4-way bank conflicts.
      asm("" : "+v"(d), "+v"(d4), "+v"(d5));
      u32x4 s1, s2;
      s1.x = __builtin_amdgcn_alignbit(d.y, d.x, 16);
      s1.y = __builtin_amdgcn_alignbit(d.z, d.y, 16);
      s1.z = __builtin_amdgcn_alignbit(d.w, d.z, 16);
      s1.w = __builtin_amdgcn_alignbit(d4, d.w, 16);
      s2.x = d.y; s2.y = d.z; s2.z = d.w; s2.w = d4;
      u32x4 s3;  // LEAD: the window was staged one pixel early, the taps sit one pixel further in
      s3.x = __builtin_amdgcn_alignbit(d.z, d.y, 16);
      s3.y = __builtin_amdgcn_alignbit(d.w, d.z, 16);
      s3.z = __builtin_amdgcn_alignbit(d4, d.w, 16);
      s3.w = __builtin_amdgcn_alignbit(d5, d4, 16);
      const bf16x8 b0 = __builtin_bit_cast(bf16x8, LEAD ? s1 : d);
      const bf16x8 b1 = __builtin_bit_cast(bf16x8, ST == 2 ? f.odd[rho] : LEAD ? s2 : s1);
      const bf16x8 b2 = __builtin_bit_cast(bf16x8, ST == 2 ? s1 : LEAD ? s3 : s2);
#pragma unroll
      for (int r = 0; r < PR; ++r) {
        const int kh = rho - ST * r;
        if (kh >= 0 && kh < 3) {
          if (F16) {
            const f16x8 ah = __builtin_bit_cast(f16x8, a[r]);
            acc[kh][0] = __builtin_amdgcn_mfma_f32_32x32x16_f16(ah, __builtin_bit_cast(f16x8, b0), acc[kh][0], 0, 0, 0);
            acc[kh][1] = __builtin_amdgcn_mfma_f32_32x32x16_f16(ah, __builtin_bit_cast(f16x8, b1), acc[kh][1], 0, 0, 0);
            acc[kh][2] = __builtin_amdgcn_mfma_f32_32x32x16_f16(ah, __builtin_bit_cast(f16x8, b2), acc[kh][2], 0, 0, 0);
          } else {
            acc[kh][0] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[r], b0, acc[kh][0], 0, 0, 0);
            acc[kh][1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[r], b1, acc[kh][1], 0, 0, 0);
            acc[kh][2] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[r], b2, acc[kh][2], 0, 0, 0);
          }
        }
      }
    }
  };
  // Stage k of this workgroup reads ring rows base_k .. base_k + XR - 1 with base_k = NEW k mod RING: its
  // first OLD rows are the last ones the stage before read, its new rows go behind them. A stage that does
  // not continue the strip of the stage before fetches the old rows itself, into those same ring rows (as
  // many rows as the new ones at stride 2, of which the last is the old one: the others go to ring rows
  // that nobody reads).
  static_assert(GROUPS == 2 || GROUPS == 1, "the stage loop is written for one or two column groups per wavefront");
  auto wrap = [](int v) { return v >= RING ? v - RING : v; };
  if (s_begin < s_end) {
    Staged stg;
    int gbuf = 0, base = 0;
    Cursor c_next = decode(s_begin);  // stage whose loads are issued next
    constexpr int OLD = XR - NEW;  // rows a stage shares with the one above
    {
      Staged top;  // both sets of loads under way at once
      issue_loads(stg, c_next, true, 1);
      issue_loads(top, c_next, false, 0);
      store_loads(stg, true, 0, OLD);
      store_loads(top, false, 0, (OLD - NEW + RING) % RING);
    }
    {
      // The loads of a stage are issued, and the registers of the stage before stored, in EVERY
      // stage: the cursor stops at the workgroup's last stage, which the last two stages fetch
      // again for nothing, and what the last stage stores nobody reads. A load or a store under
      // a condition leaves the staged registers with two possible states where the paths meet;
      // the compiler then waits for the loads at the end of the stage that issued them (to copy
      // the registers together) instead of where they are stored, half a stage later.
      if (s_begin + 1 < s_end) advance(c_next);
      Cursor c_store = c_next;  // stage whose registers are stored next
      const int stages = (int)(s_end - s_begin);
      issue_loads(stg, c_next, true, 1);
      if (s_begin + 2 < s_end) advance(c_next);
      __syncthreads();
      // Wavefronts w and w + 4 share a SIMD and would do everything at the same time: both issue
      // matrix instructions, then both store and load while the matrix core idles (measured with
      // the cycle counter: 1150 cycles of a 4400-cycle stage spent by the older wavefront of each
      // SIMD waiting at the barrier for the younger one). So the two take the stage's halves in
      // opposite order: w multiplies while w + 4 stores the registers of the next stage and
      // issues the loads of the one after, then the other way round. What is stored goes to the
      // g buffer and the ring rows that no wavefront reads in this stage.
      // (With six multiplying wavefronts, two SIMDs hold a wavefront that only stages; there the
      // split measured slower, and every wavefront stores and loads between its two groups.)
      const bool stage_first = CWAVES == 8 && (wave & 4) != 0;
      // Both groups' fragments before the first matrix instruction; not in the kernels of a volume that have edges, where the second
      // group's 28 registers between the two are what the test of `whole` takes (without it a volume whose rows end inside a strip paid for
      // every stage what the tensor's ends cost): 1 x 30 -> 9 of 38 x 66 x 15 45.1 -> 40.7 us, 2 x 64 -> 64 of 30 x 50 x 20 79.6 -> 74.1,
      // 2 x 48 -> 8 of 36 x 48 x 76 83.5 -> 80.0.
      constexpr bool kBothFirst = CWAVES == 8 || ALLIN || FRAMED;
      for (int st = 0; st < stages; ++st) {
        Frags f0, f1;
        (void)f1;
        if (stage_first) {
          store_loads(stg, true, gbuf ^ 1, wrap(base + XR), st + 1 < stages);
          issue_loads(stg, c_next, true, 1);
        }
        if (wave < CWAVES) {
          read_group(f0, gbuf, base, 0);
          if (GROUPS == 2 && kBothFirst) read_group(f1, gbuf, base, 1);
          mfma_group(f0);
          if (GROUPS == 2 && CWAVES == 8) mfma_group(f1);
        }
        if (!stage_first) {
          store_loads(stg, true, gbuf ^ 1, wrap(base + XR), st + 1 < stages);
          issue_loads(stg, c_next, true, 1);
        }
        if (GROUPS == 2 && CWAVES != 8 && wave < CWAVES) {
          if (!kBothFirst) read_group(f1, gbuf, base, 1);
          mfma_group(f1);
        }
        const Cursor c_issued = c_next;
        if (st + 3 < stages) advance(c_next);
        __syncthreads();
        if (st + 1 < stages && c_store.hp == 0) {
          // the next stage starts a new strip: its first two x rows, on the spot
          Staged top;
          issue_loads(top, c_store, false, 0);
          store_loads(top, false, 0, wrap(base + OLD));
          // These loads have all been stored, but the tail's under a per-lane condition: where
          // the compiler cannot see a load waited for on every path, it waits at the loop's end,
          // and that wait takes the stage's own loads with it. vmcnt(0), said once, here:
          __builtin_amdgcn_s_waitcnt(0x0F70);
          __syncthreads();
        }
        c_store = c_issued;
        base = wrap(base + NEW);
        gbuf ^= 1;
      }
    }
  }

  // bias partial of this workgroup: the lanes that carried a channel's chunks add up
  const size_t slot = (size_t)block * gridDim.x + blockIdx.x;
  if (bias_part != nullptr) {
#pragma unroll
    for (int rd = 0; rd < ROUNDS; ++rd) {
      const int q = tid + rd * THREADS;
      if (rd < G_ROUNDS) {
        float s = bsum[rd];
#pragma unroll
        for (int off = SR * G_CPR / 2; off > 0; off >>= 1) s += __shfl_xor(s, off, 64);
        if (q < G_CHUNKS && tid % (SR * G_CPR) == 0) bias_part[slot * GC + q / (SR * G_CPR)] = s;
      }
    }
  }

  // Partial of this workgroup. The parts of a pair meet in LDS (the stage buffers are free: a barrier closed the last stage), three taps
  // at a time: their twelve 16-byte pieces a lane are dealt to the parts, a part leaves the others' with them, adds up its own and
  // stores them, [tap9][pair][4][lane][4]. (Upper parts handing all of theirs to the lower ones, half of them at a time, kept most
  // wavefronts waiting at twelve barriers: 3.4 us of a 64 x 32 block, 3.1 of 32 x 32, where this takes 2.8 and 2.3.)
  constexpr int OWN = 12 / PARTS;  // pieces of three taps that a part adds up
  static_assert(CWAVES * (12 - OWN) * 1024 <= wgrad_lds<CGB, CXB, ST>(), "the pieces of three taps fit");
  float* const out = p.part + slot * (size_t)(9 * GC * XC) + pair * 1024 + lane * 4;
#pragma unroll
  for (int kh = 0; kh < 3; ++kh) {
    // [pair][part that owns][part that gives, without the owner][piece][lane][4]
    auto place = [&](int owner, int giver, int k) {
      return reinterpret_cast<float*>(smem) + (((pair * PARTS + owner) * (PARTS - 1) + (giver < owner ? giver : giver - 1)) * OWN + k) * 256 + lane * 4;
    };
    auto piece = [&](int q) { return f32x4{acc[kh][q / 4][4 * (q % 4)], acc[kh][q / 4][4 * (q % 4) + 1], acc[kh][q / 4][4 * (q % 4) + 2], acc[kh][q / 4][4 * (q % 4) + 3]}; };
    if (wave < CWAVES) {
#pragma unroll
      for (int owner = 0; owner < PARTS; ++owner)
        if (owner != part) {
#pragma unroll
          for (int k = 0; k < OWN; ++k) *reinterpret_cast<f32x4*>(place(owner, part, k)) = piece(owner * OWN + k);
        }
    }
    __syncthreads();
    if (wave < CWAVES) {
#pragma unroll
      for (int owner = 0; owner < PARTS; ++owner)
        if (owner == part) {
#pragma unroll
          for (int k = 0; k < OWN; ++k) {
            f32x4 v[PARTS];
#pragma unroll
            for (int g = 0; g < PARTS; ++g) v[g] = g == owner ? piece(owner * OWN + k) : *reinterpret_cast<const f32x4*>(place(owner, g, k));
            const int q = owner * OWN + k;
            const f32x4 sum = PARTS == 4 ? (v[0] + v[2]) + (v[1] + v[3]) : v[0] + v[1];
            *reinterpret_cast<f32x4*>(out + (size_t)(kh * 3 + q / 4) * (GC * XC) + q % 4 * 256) = sum;
          }
        }
    }
    __syncthreads();
  }
}

template <int DT>
__global__ __launch_bounds__(64 * jg::CONV_RED_WAVES) void wgrad_reduce_kernel(jg_conv_reduction p) {
  __shared__ jg::ConvReduceShared shared;
  jg::reduce_conv_tiles<DT>(p, blockIdx.x, shared);
}

// gw[co][ci][t] (fp32) = sum over the part pairs (i, j), i + j <= parts - 1, smallest first, of
// tmp[i * cout + co][j * cin + ci][t]: the part products of the split mode from one launch.
__global__ __launch_bounds__(256) void wgrad_combine_parts_kernel(float* __restrict__ gw, const float* __restrict__ tmp,
                                                                  int cout, int cin, int taps, int parts) {
  const int idx = blockIdx.x * 256 + threadIdx.x;
  if (idx >= cout * cin * taps) return;
  const int t = idx % taps, ci = (idx / taps) % cin, co = idx / (taps * cin);
  float sum = 0.0f;
  for (int order = parts - 1; order >= 0; --order)
    for (int i = 0; i <= order; ++i) {
      const int j = order - i;
      sum += tmp[((size_t)(i * cout + co) * (parts * cin) + (j * cin + ci)) * taps + t];
    }
  gw[idx] = sum;
}

int stage_columns(const ConvGeom& g) { return g.s[2] == 2 ? Stage<2>::SW : Stage<1>::SW; }
long long stage_count(const ConvGeom& g) {
  const int sw = stage_columns(g);
  return g.batch * g.out[0] * ((g.out[1] + SR - 1) / SR) * ((g.out[2] + sw - 1) / sw);
}

// Channel blocking. A workgroup accumulates a block of GC output x CIN_B input channels (32 or 64 each; with a
// depth kernel of 3 always 32 x 32, so that the x side spans 96); a block with fewer channels than its width
// re-reads its last channel and its extra rows and columns are dropped. All blocks of a problem run in one
// launch: one launch each (with its own reduction) took 269 us where this takes 97, 119 -> 191 channels of 4 x 74 x 88.
struct Plan {
  int cgb, cxb, KD;
  int co_blocks, ci_blocks, npairs;
  int parts_in_block;  // split mode: parts that are channels of the one block (1: the parts are block pairs)
  int wgs;             // workgroups per block
  size_t GC() const { return 32 * cgb; }
  size_t XC() const { return 32 * cxb; }
  size_t blocks() const { return (size_t)co_blocks * ci_blocks * npairs; }
  size_t partial() const { return 9 * GC() * XC(); }  // floats
  size_t bytes() const { return (blocks() * wgs * (partial() + GC()) * sizeof(float) + 255) / 256 * 256; }
};
bool covered(const ConvGeom& g) {
  if (g.groups != 1) return false;
  if (g.k[1] != 3 || g.k[2] != 3 || (g.k[0] != 1 && g.k[0] != 3)) return false;
  if (g.k[0] == 1 && g.in[0] != 1) return false;
  const bool strided = g.s[1] == 2 && g.s[2] == 2 && g.k[0] == 1;
  for (int a = 0; a < 3; ++a)
    if ((g.s[a] != 1 && !(strided && a > 0)) || g.d[a] != 1) return false;
  if (g.cin <= 0 || g.cout <= 0) return false;
  // per-lane byte offsets inside one batch entry are 32-bit
  const size_t xs = (size_t)g.cin * g.in[0] * g.in[1] * g.in[2] * 2;
  const size_t gs = (size_t)g.cout * g.out[0] * g.out[1] * g.out[2] * 2;
  return xs < (1ull << 31) && gs < (1ull << 31);
}
Plan plan_of(const ConvGeom& g, int parts) {
  Plan p;
  p.KD = g.k[0];
  const int widest = p.KD == 3 ? 32 : 64;
  p.parts_in_block = parts > 1 && parts * g.cout <= widest && parts * g.cin <= widest ? parts : 1;
  const int cout = p.parts_in_block * g.cout, cin = p.parts_in_block * g.cin;
  // 64 channels a side where that pads no further than 32 would: the wider block reads its operands for twice
  // the products
  auto width = [&](int c) { return widest == 64 && (c + 63) / 64 * 64 <= (c + 31) / 32 * 32 ? 64 : 32; };
  const int cob = width(cout), cib = width(cin);
  p.cgb = cob / 32;
  p.cxb = p.KD * cib / 32;
  p.co_blocks = (cout + cob - 1) / cob;
  p.ci_blocks = (cin + cib - 1) / cib;
  p.npairs = parts > 1 && p.parts_in_block == 1 ? 6 : 1;
  // Workgroups per block. More of them shorten the walk over the pixels and lengthen the reduction of their
  // partials: a walk of `stages` at about 2 us each (a 64 x 64 block; a smaller one waits as long for its loads)
  // against partials that are written and read at about 4 TB/s, W = sqrt(stages * 2 us * 4 TB/s / 2 / bytes)
  // workgroups in all; not more than the chip holds at once, and whole XCD rounds where there are that many.
  const long long stages = stage_count(g);
  const double blocks = (double)p.blocks(), bytes = (double)p.partial() * sizeof(float);
  const double best = sqrt((double)stages * blocks * 4.0e6 / bytes);
  const double most = jg::cu_count() * (p.cgb * p.cxb == 1 ? 2.0 : 1.0);
  long long n = (long long)((best < most ? best : most) / blocks);
  if (n >= 8) n = n / 8 * 8;
  if (n > stages) n = stages;
  if (n < 1) n = 1;
  // No more than the walks need, but for up to seven that make the number a multiple of the XCDs: 1080 stages in walks of four are 270
  // workgroups and 272 are launched, of the 336 that the rule asks for 66 wrote a partial of nothing.
  const long long walk = (stages + n - 1) / n, busy = (stages + walk - 1) / walk;
  if (n >= 8) n = std::min(n, (busy + 7) / 8 * 8);
  else n = busy;
  p.wgs = (int)n;
  return p;
}

// Pieces (their logarithm) that a run of 256 values is cut into: up to two workgroups a compute unit.
int reduce_sub(long long runs) {
  const long long most = 2ll * jg::cu_count();
  return 4 * runs <= most ? 2 : 2 * runs <= most ? 1 : 0;
}

template <int CGB, int CXB>
int launch(const WgradParams& p, int even, bool f16, bool all_inside, int stride, dim3 grid, hipStream_t s, const char* who) {
  constexpr int THREADS = wgrad_threads(CGB, CXB);
  const size_t lds = stride == 2 ? wgrad_lds<CGB, CXB, 2>() : wgrad_lds<CGB, CXB, 1>();
  void (*kern)(WgradParams) = nullptr;
  if (stride == 2) {
    if constexpr (CXB != 3) {
      if (f16) kern = even == 1 ? &wgrad3x3_mfma_kernel<CGB, CXB, 1, false, true, false, 2> : &wgrad3x3_mfma_kernel<CGB, CXB, 0, false, true, false, 2>;
      else kern = even == 1 ? &wgrad3x3_mfma_kernel<CGB, CXB, 1, false, false, false, 2> : &wgrad3x3_mfma_kernel<CGB, CXB, 0, false, false, false, 2>;
    }
  } else if (f16)  // never framed (checked by the caller)
    kern = even == 1 ? &wgrad3x3_mfma_kernel<CGB, CXB, 1, false, true>
                     : (even == 2 ? &wgrad3x3_mfma_kernel<CGB, CXB, 2, false, true> : &wgrad3x3_mfma_kernel<CGB, CXB, 0, false, true>);
  else if (p.xt != nullptr)
    kern = &wgrad3x3_mfma_kernel<CGB, CXB, 1, true>;  // the framed input needs the even layout (checked by the caller)
  else if (all_inside && even == 1)
    kern = &wgrad3x3_mfma_kernel<CGB, CXB, 1, false, false, true>;
  else
    kern = even == 1 ? &wgrad3x3_mfma_kernel<CGB, CXB, 1, false>
                     : (even == 2 ? &wgrad3x3_mfma_kernel<CGB, CXB, 2, false> : &wgrad3x3_mfma_kernel<CGB, CXB, 0, false>);
  hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                     hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  if (e != hipSuccess) JG_FAIL(JG_ERR_LAUNCH, "%s: cannot reserve %zu bytes of LDS", who, lds);
  kern<<<grid, THREADS, lds, s>>>(p);
  return JG_OK;
}

}  // namespace

namespace jg {

// fp32 is split into three bf16 parts per operand; fp16 has its own MFMA instruction and runs like bf16
static int parts_of(int dtype) { return dtype == JG_F32 ? 3 : 1; }
// fp32 runs in split mode: both operands are copied as three bf16 parts each (as extra channels) and
// the six part products whose indices add up to at most 2 are accumulated in fp32.
bool mfma_wgrad_supported(const ConvGeom& g, int dtype) {
  if ((dtype != JG_BF16 && dtype != JG_F32 && dtype != JG_F16) || g.batch <= 0) return false;
  return covered(g);
}

static size_t split_copy_bytes(size_t elements, int parts) { return (elements * parts * 2 + 255) / 256 * 256; }
// workspace: [partials | x parts | g parts (fp32 only) | part products of the one-block launch]
size_t mfma_wgrad_workspace(const ConvGeom& g, int dtype) {
  const int parts = parts_of(dtype);
  const Plan plan = plan_of(g, parts);
  size_t n = plan.bytes();
  if (parts > 1) {
    n += split_copy_bytes((size_t)g.batch * g.cin * g.in[0] * g.in[1] * g.in[2], parts);
    n += split_copy_bytes((size_t)g.batch * g.cout * g.out[0] * g.out[1] * g.out[2], parts);
    if (plan.parts_in_block > 1) n += ((size_t)parts * parts * g.cout * g.cin * plan.KD * 9 * sizeof(float) + 255) / 256 * 256;
  }
  return n;
}

// Whether the framed weight-gradient kernel covers a geometry: even row lengths (its
// vector loads), and every row pair / column tile whose window leaves the own tile lies
// inside the bands that the frame holds.
bool mfma_wgrad_frame_ok(const ConvGeom& g, const int tlo[3], const int tn[3]) {
  if (g.in[2] % 2 != 0 || g.p[2] % 2 != 0 || g.out[2] % 2 != 0 || tn[2] % 2 != 0) return false;
  if (!covered(g) || g.s[2] != 1) return false;
  constexpr int SW = Stage<1>::SW;
  const Plan plan = plan_of(g, 1);  // the framed input is read by a single block of exactly its width
  if (g.cin * plan.KD != (int)plan.XC() || g.cout != (int)plan.GC()) return false;
  int blo[3], bhi[3];
  mfma_frame_bands(g, tlo, tn, blo, bhi);
  const int row_pairs = (g.out[1] + SR - 1) / SR, col_tiles = (g.out[2] + SW - 1) / SW;
  for (int j = 0; j < row_pairs + 1; ++j) {  // x row pairs of all stages: [2j - pad, 2j - pad + 2)
    const int r = 2 * j - g.p[1];
    const bool in_tile = r >= tlo[1] && r + 2 <= tlo[1] + tn[1];
    const int r_end = r + 2 < g.in[1] ? r + 2 : g.in[1];  // what lies past the tensor is not read
    const bool in_band = r_end <= blo[1] || r >= g.in[1] - bhi[1];
    if (!in_tile && !in_band) return false;
  }
  for (int ct = 0; ct < col_tiles; ++ct) {
    const int c = ct * SW - g.p[2];
    const bool in_tile = c >= tlo[2] && c + SW + 2 <= tlo[2] + tn[2];
    const int c_end = c + SW + 2 < g.in[2] ? c + SW + 2 : g.in[2];
    const bool in_band = c_end <= blo[2] || c >= g.in[2] - bhi[2];
    if (!in_tile && !in_band) return false;
  }
  return true;
}

int tiles_reduce(const jg_conv_reduction& r, hipStream_t s) {
  const unsigned grid = conv_reduce_blocks(r);
  if (r.dtype == JG_F32) wgrad_reduce_kernel<JG_F32><<<grid, 64 * CONV_RED_WAVES, 0, s>>>(r);
  else if (r.dtype == JG_F16) wgrad_reduce_kernel<JG_F16><<<grid, 64 * CONV_RED_WAVES, 0, s>>>(r);
  else wgrad_reduce_kernel<JG_BF16><<<grid, 64 * CONV_RED_WAVES, 0, s>>>(r);
  JG_CHECK_LAUNCH("jg_conv_wgrad(reduce)");
  return JG_OK;
}

int mfma_wgrad(void* gw, void* gb, const void* x, const void* go, const ConvGeom& g, void* ws,
               size_t ws_bytes, hipStream_t s, const void* xt, const int* tlo, const int* tn, int dtype, jg_conv_reduction* later) {
  const char* who = "jg_conv_wgrad(mfma)";
  if (!covered(g)) JG_FAIL(JG_ERR_UNSUPPORTED, "%s: geometry not covered", who);
  if (ws == nullptr || ws_bytes < mfma_wgrad_workspace(g, dtype))
    JG_FAIL(JG_ERR_WORKSPACE, "%s: workspace %zu < %zu bytes", who, ws_bytes,
            mfma_wgrad_workspace(g, dtype));
  JG_REQUIRE((reinterpret_cast<uintptr_t>(ws) & 15) == 0, "%s: workspace must be 16-byte aligned",
             who);
  const size_t x_cs = (size_t)g.in[0] * g.in[1] * g.in[2], g_cs = (size_t)g.out[0] * g.out[1] * g.out[2];
  const int parts = parts_of(dtype);
  const Plan plan = plan_of(g, parts);
  const bool f16 = dtype == JG_F16;
  float* one_block_tmp = nullptr;
  if (dtype != JG_BF16 && xt != nullptr) JG_FAIL(JG_ERR_UNSUPPORTED, "%s: the framed input is bf16", who);
  if (parts > 1) {
    char* base = static_cast<char*>(ws) + plan.bytes();
    uint16_t* xs = reinterpret_cast<uint16_t*>(base);
    base += split_copy_bytes((size_t)g.batch * g.cin * x_cs, parts);
    uint16_t* gs = reinterpret_cast<uint16_t*>(base);
    base += split_copy_bytes((size_t)g.batch * g.cout * g_cs, parts);
    one_block_tmp = reinterpret_cast<float*>(base);
    int rc = split_parts_bf16(xs, x, dtype, (size_t)g.batch, (size_t)g.cin * x_cs, s);
    if (rc) return rc;
    rc = split_parts_bf16(gs, go, dtype, (size_t)g.batch, (size_t)g.cout * g_cs, s);
    if (rc) return rc;
    x = xs;
    go = gs;
  }
  // 0, 1 or 2: the EVEN mode of the kernel (2: odd padding across W, windows staged one pixel early)
  const bool even_rows = (g.in[2] % 2 == 0) && (g.out[2] % 2 == 0) && ((reinterpret_cast<uintptr_t>(x) & 3) == 0) &&
                         ((reinterpret_cast<uintptr_t>(go) & 3) == 0);
  const int even = !even_rows ? 0 : (g.p[2] % 2 == 0 ? 1 : 2);
  if (xt != nullptr && (even != 1 || !mfma_wgrad_frame_ok(g, tlo, tn)))
    JG_FAIL(JG_ERR_UNSUPPORTED, "%s: the framed input does not cover this geometry / alignment", who);
  WgradParams p;
  p.part = static_cast<float*>(ws);
  p.bias_part = gb != nullptr ? p.part + plan.blocks() * plan.wgs * plan.partial() : nullptr;
  p.x = static_cast<const uint16_t*>(x);
  p.g = static_cast<const uint16_t*>(go);
  p.x_end = static_cast<const char*>(x) + 2 * (size_t)g.batch * parts * g.cin * x_cs;
  p.g_end = static_cast<const char*>(go) + 2 * (size_t)g.batch * parts * g.cout * g_cs;
  p.cin = plan.parts_in_block * g.cin; p.cout = plan.parts_in_block * g.cout;
  p.cin_total = parts * g.cin; p.cout_total = parts * g.cout;
  p.ci_blocks = plan.ci_blocks; p.npairs = plan.npairs;
  // part products (g part, x part), smallest first; plain mode: the one product
  p.gparts = plan.npairs == 6 ? 0u | (1u << 2) | (2u << 4) | (0u << 6) | (1u << 8) | (0u << 10) : 0u;
  p.xparts = plan.npairs == 6 ? 2u | (1u << 2) | (0u << 4) | (1u << 6) | (0u << 8) | (0u << 10) : 0u;
  p.Din = g.in[0]; p.Hin = g.in[1]; p.Win = g.in[2];
  p.Dout = g.out[0]; p.Hout = g.out[1]; p.Wout = g.out[2];
  p.pad_d = g.p[0]; p.pad_h = g.p[1]; p.pad_w = g.p[2];
  p.row_pairs = (g.out[1] + SR - 1) / SR;
  p.col_tiles = (g.out[2] + stage_columns(g) - 1) / stage_columns(g);
  p.total_stages = stage_count(g);
  p.per = (p.total_stages + plan.wgs - 1) / plan.wgs;
  p.by_rp = jg::div_by(p.row_pairs);
  p.by_ct = jg::div_by(p.col_tiles);
  p.by_od = jg::div_by(p.Dout);
  p.by_pairs = jg::div_by(p.npairs);
  p.by_ci = jg::div_by(p.ci_blocks);
  // Every stage whole and every window inside x: the kernel without the border path (see ALLIN).
  constexpr int SW = Stage<1>::SW;
  const bool all_inside = g.s[2] == 1 && even == 1 && xt == nullptr && g.p[0] == 0 && g.p[1] == 0 && g.p[2] == 0 &&
                          g.out[1] % SR == 0 && g.out[2] % SW == 0 && g.out[1] + 2 <= g.in[1] &&
                          g.out[2] + 2 <= g.in[2] && g.out[0] - 1 + g.k[0] <= g.in[0];
  p.xt = static_cast<const uint16_t*>(xt);
  p.tlo_d = tlo ? tlo[0] : 0; p.tlo_h = tlo ? tlo[1] : 0; p.tlo_w = tlo ? tlo[2] : 0;
  p.tn_d = tn ? tn[0] : 0; p.tn_h = tn ? tn[1] : 0; p.tn_w = tn ? tn[2] : 0;
  JG_REQUIRE(plan.blocks() < 65536, "%s: too many channels", who);
  const dim3 grid((unsigned)plan.wgs, (unsigned)plan.blocks());
  int rc;
  if (plan.cgb == 2 && plan.cxb == 2) rc = launch<2, 2>(p, even, f16, all_inside, g.s[2], grid, s, who);
  else if (plan.cgb == 1 && plan.cxb == 3) rc = launch<1, 3>(p, even, f16, all_inside, g.s[2], grid, s, who);
  else if (plan.cgb == 1 && plan.cxb == 1) rc = launch<1, 1>(p, even, f16, all_inside, g.s[2], grid, s, who);
  else if (plan.cgb == 2 && plan.cxb == 1) rc = launch<2, 1>(p, even, f16, all_inside, g.s[2], grid, s, who);
  else rc = launch<1, 2>(p, even, f16, all_inside, g.s[2], grid, s, who);
  if (rc) return rc;
  JG_CHECK_LAUNCH(who);

  jg_conv_reduction r = {};
  r.kind = jg::CONV_REDUCE_TILES;
  r.dtype = dtype;
  r.part = p.part; r.bias_part = p.bias_part;
  r.gw = plan.parts_in_block > 1 ? one_block_tmp : gw;
  r.gb = gb;
  r.slots = plan.wgs; r.npairs = plan.npairs;
  r.pairs = plan.cgb * plan.cxb; r.rows = (int)plan.GC(); r.cols = plan.cxb; r.ci_step = (int)plan.XC() / plan.KD;
  r.KD = plan.KD; r.cin = p.cin; r.cout = p.cout; r.ci_blocks = plan.ci_blocks;
  r.bias_cout = g.cout; r.bias_parts = parts;
  r.runs = plan.co_blocks * plan.ci_blocks * 9 * r.pairs * 4;
  r.sub = reduce_sub(r.runs);
  if (later != nullptr && plan.parts_in_block == 1) {
    *later = r;
    return JG_OK;
  }
  rc = tiles_reduce(r, s);
  if (rc) return rc;
  if (plan.parts_in_block > 1) {
    // few channels: all part products came from one block (the parts are channels of it); the ones that count
    // are added up
    const int gw_count = g.cout * g.cin * g.k[0] * 9;
    wgrad_combine_parts_kernel<<<(gw_count + 255) / 256, 256, 0, s>>>(static_cast<float*>(gw), one_block_tmp, g.cout, g.cin,
                                                                      plan.KD * 9, parts);
    JG_CHECK_LAUNCH(who);
  }
  return JG_OK;
}

}  // namespace jg
