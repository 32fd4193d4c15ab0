// Implicit-GEMM convolution on the bf16 matrix cores (v_mfma_f32_32x32x16_bf16):
// 3x3 (2-D, stride 1 or 2) and 3x3x3 (3-D, stride 1), dilation 1, channels-first tensors in and
// out. One kernel serves the forward pass and the input gradient.
//
//   GEMM view   Y[m][pixel] = sum_{tap, k} Wt[tap][m][k] * X[k][pixel + tap]
//               A 3-D problem is the 2-D one with the depth taps folded into the
//               contraction channels: channel kd*C + c of a tile at output depth d
//               is the plane X[c][d + kd - pad_d].
//   MFMA roles  A = weights (M = 32 produced channels, K = 16 contraction channels),
//               B = input pixels (K = 16 channels, N = 32 consecutive pixels of a
//               row), so an accumulator lane owns one pixel and 16 produced channels
//               and the stores run along W of the channels-first output.
//   Workgroup   512 threads = 8 wavefronts; output tile 16 rows x 64 columns x MT
//               produced channels; wavefront w owns rows 4*((w + 2*(w/4))%4).., columns 32*(w/4)..
//   LDS         the whole prepared weight block of the workgroup's produced-channel
//               tile stays resident; the input tile is streamed in stages of 16
//               contraction channels, double buffered (2 x 40.5 KiB). Input pixels
//               are stored "8 channels per 16-byte slot" so that a B fragment is one
//               ds_read_b128 per lane; the channels-first global rows (8 channels x
//               8 pixels per lane, 16-byte loads) are transposed in registers on the
//               way in. Slots of a row are interleaved by pixel phase (col % 8) so
//               that both the transposing writes and the fragment reads spread over
//               the banks.
//   Schedule    persistent workgroups (one per CU) walk a contiguous, XCD-local
//               range of tiles; the global loads of stage s+1 are issued before the
//               MFMAs of stage s and written to LDS between its MFMA groups (one
//               barrier per stage). A cursor decodes a tile's coordinates once and steps
//               through its stages by additions; the weight fragments of a group of 24
//               MFMAs are fetched under the group before, into the registers it frees.
//   Tile grid   tile column tw covers produced columns [org_w + 64 tw, + 64). The host picks
//               org_w <= 0 so that the staged row segments (144 bytes from input column
//               org_w + 64 tw - pad_w) start on cache lines where that costs no extra
//               tile column, and stages a window from one pixel earlier (lead) when it
//               would otherwise start on an odd column (4-byte aligned loads throughout).
//   Epilogue    16-bit results with rows of whole 16-byte pieces pass through LDS and leave as
//               16-byte stores; everything else as 2- or 4-byte stores along W.
//   dgrad       the same kernel on the output gradient with virtual zero padding
//               k-1-p and the weights flipped and transposed by the preparation.
//   Channels    any counts: the contraction is padded to 16-channel steps per depth tap
//               (zero weights; the registers of channels that do not exist are zeroed on
//               their way to LDS), the weights stay in LDS in groups of steps when they
//               do not fit at once, produced channels are padded to 32 and a ragged last
//               tile predicates its stores.
//   fp16        the same kernel on v_mfma_f32_32x32x16_f16 (a template flag; the staging moves
//               16-bit values without looking at them).
//   fp32        "split mode": an operand is the exact sum of three bf16 parts, kept as extra
//               channel groups; the contraction runs over the six part products that matter
//               and the result is stored as fp32. (A two-part form of it for fp16 operands
//               remains in the split kernels and is not dispatched.)
#include <algorithm>
#include <type_traits>
#include <utility>

#include "conv_common.h"
#include "lds_transfer.h"

namespace {

using jg::ConvGeom;

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4_a4 __attribute__((ext_vector_type(4), aligned(4)));

constexpr int KH = 3, KW = 3, TAPS = KH * KW;  // taps inside a plane
constexpr int TILE_H = 16, TILE_W = 64;        // output tile of a workgroup (stride 2: half of it each way)
constexpr int WAVES = 8, THREADS = WAVES * 64;
constexpr int IN_ROWS = TILE_H + KH - 1;       // 18
constexpr int IN_COLS = TILE_W + KW - 1;       // 66
constexpr int OCTS = 9;                        // 9 octets of 8 pixels cover 66 (+6) columns
constexpr int ROW_SLOTS = 8 * OCTS;            // 16-byte slots per LDS row
constexpr int CK = 16;                         // contraction channels per stage
constexpr int STAGE_SLOTS = 2 * IN_ROWS * ROW_SLOTS;  // [kg][row][slot]
constexpr int STAGE_BYTES = STAGE_SLOTS * 16;         // 41472
constexpr int TASKS = 2 * IN_ROWS * OCTS;             // 324 tasks of 8 channels x 8 pixels
constexpr int LANES_ODD = 64 / OCTS * OCTS;           // lanes of a wavefront with a task where rows start anywhere
static_assert(2 * IN_ROWS <= WAVES * (LANES_ODD / OCTS), "every row of tasks has a wavefront");

__device__ __forceinline__ int in_slot(int col) { return (col & 7) * OCTS + (col >> 3); }

// A tile's place from its number: three to five divisions, twice a tile and all of it in front of a workgroup's first load. The compiler's
// own (and one more, and a remainder of ragged channels by two of them in every stage) were 1.5 to 2 us of a workgroup with a tile or two.
// Read from the kernel-argument segment where it is wanted (walk_of): held from the kernel's start on, it pushes the stage loop's
// scalar registers out. Forward / gradient with the fold: 2 x 40 -> 72 of 217 x 301 31.4 -> 29.6 us / the same, 4 x 7 -> 91 of 163 x 957
// 67.6 -> 62.7 / 64.4 -> 60.5, 1 x 17 -> 24 of 50 x 76 x 26 23.2 -> 21.7 / 41.8 -> 39.6, 2 x 32 -> 32 of 128^3 280 -> 277 / 378 -> 367.
struct TileWalk {
  jg::Div by_plane, by_tw, by_od, by_wgs;  // tiles of a plane, tile columns, produced planes, workgroups of an XCD
  int per_plane, tiles_w, Dout;
};

struct FwdParams {
  const uint16_t* x;    // (N, C, Din, Hin, Win) bf16: the tensor that is convolved
  const char* x_end;    // one past the last byte of x
  const u32x4* wprep;   // prepared weights, [m_tile][group][wc16][kg][tap9][MT][8]
  const uint16_t* wraw;  // the weights as they are, which each workgroup puts in order itself (arrange_weights); NULL: wprep
  int transposed;        // (with wraw) as in prep_weights_kernel
  const uint16_t* bias; // (M,) or NULL
  uint16_t* y;          // (N, M, Dout, Hout, Wout)
  int N, C, M;          // batch, channels of x, produced channels
  int Cp;               // C rounded up to a multiple of 16: contraction channels per depth tap
  // Split mode (fp32 / fp16 operands as sums of 3 / 2 bf16 parts): x holds Cx = parts * C channels per
  // batch entry (one channel group per part), the contraction runs over nblk = 6 / 3 blocks of KD * Cp
  // channels, block b reads part (xmap >> 2 b) & 3 of x against the weight part the
  // preparation put there. Plain mode: nblk = 1, xmap = 0, Cx = C.
  int nblk, Cx;
  uint32_t xmap;
  int out_kind;         // dtype of y and bias: 0 bf16, 1 fp32, 2 fp16
  int KD;               // depth taps (1 for 2-D); contraction channels K = KD * C
  int Din, Hin, Win, Dout, Hout, Wout;
  int pad_d, pad_h, pad_w;  // virtual zero padding of x
  int tiles_h, tiles_w;
  // Tile column tw covers produced columns [org_w + tw * TW, + TW), org_w <= 0: the host shifts the
  // grid to put the staged row segments on cache-line boundaries where that is free.
  // The staged window starts `lead` (0 / 1) pixels before the first one a tile needs, so that its
  // rows stay 4-byte aligned whatever the parity of pad_w - org_w.
  int org_w, lead;
  // The first extra_h produced rows and extra_w columns (0, or pad_h / pad_w; org_w is then the same) lie above and left of the
  // tile grid: the workgroups at tile row / column 0 make them beside their tile, see compute_left and compute_top.
  int extra_h, extra_w;
  TileWalk walk;
  int total_tiles;      // N * Dout * tiles_h * tiles_w
  int nc16;             // KD * Cp / 16
  int wc16;             // 16-channel steps whose weights sit in LDS at a time (a group)
  int ngroups;          // ceil(nc16 / wc16); > 1: the weights are reloaded group by group
  // Fold mode (input gradient written to its owners): y is the unpadded tile
  // (N, M, nD, nH, nW); produced cells outside [lo, lo + n) go to the strip of the
  // neighbour that owns them. fold = 0: y is the whole produced tensor.
  int fold;
  int lo_d, lo_h, lo_w, nD, nH, nW;
  // Framed input: xt (N, C, tn_d, tn_h, tn_w) is the own tile, which sits at [tlo, tlo + tn)
  // inside x. A stage whose window lies inside the tile reads xt, so that only a frame of
  // x near the edges has to hold data. NULL: everything comes from x.
  const uint16_t* xt;
  int tlo_d, tlo_h, tlo_w, tn_d, tn_h, tn_w;
  // MODE 2: extent of the produced tensor and the layer's padding; Hout, Wout count positions (i, j), pad_h = pad_w = 1
  int Hx, Wx, px_h, px_w;
};

// Strips of the 26 neighbours, slot (dd+1)*9 + (dh+1)*3 + (dw+1); first kernel
// parameter, so that a lane can index it in the kernel-argument segment.
struct StripTable {
  void* p[27];
};

__device__ __forceinline__ void* strip_entry(int idx) {
#if defined(__HIP_DEVICE_COMPILE__)
  void* const* kt = (void* const*)__builtin_amdgcn_kernarg_segment_ptr();
  return kt[idx];
#else
  (void)idx;
  return nullptr;
#endif
}

__device__ __forceinline__ TileWalk walk_of() {
  typedef const __attribute__((address_space(4))) TileWalk* Arg;
  Arg arg = nullptr;
#if defined(__HIP_DEVICE_COMPILE__)
  arg = reinterpret_cast<Arg>(reinterpret_cast<uintptr_t>((void*)__builtin_amdgcn_kernarg_segment_ptr()) + sizeof(StripTable) + offsetof(FwdParams, walk));
  asm volatile("" : "+s"(arg));
#endif
  return {{arg->by_plane.m, arg->by_plane.s}, {arg->by_tw.m, arg->by_tw.s}, {arg->by_od.m, arg->by_od.s}, {arg->by_wgs.m, arg->by_wgs.s}, arg->per_plane, arg->tiles_w, arg->Dout};
}

// ---------------------------------------------------------------- weight prep
// dst[(((mt*ngroups + group)*wc16 + c16 in group)*2 + kg)*9 + tap9][m_local][8 k] (bf16), contraction channel
// k = kd*Cp + c (channels C..Cp-1 are zero padding). transposed = 0: A[m][k] = w[m][c][kd][kh][kw] (forward, w is
// (M, C, KD, 3, 3)); transposed = 1: A[m][k] = w[c][m][KD-1-kd][2-kh][2-kw] (input
// gradient, w is (C, M, KD, 3, 3)); transposed = 2: the six taps of a phase row of the strided input gradient
// (see compute_phases), mt = 2 * channel tile + pa, w is (C, M, 3, 3).
__device__ __forceinline__ bool phase_has(int pa, int tap) { return pa == 0 || tap >= 3; }
__device__ __forceinline__ int phase_tap(int pa, int tap) {
  const int kh = pa == 0 ? (tap < 3 ? 2 : 0) : 1, t = tap % 3;
  return kh * KW + (t == 0 ? 2 : t == 1 ? 0 : 1);
}
__global__ __launch_bounds__(256) void prep_weights_kernel(uint16_t* __restrict__ dst,
                                                           const uint16_t* __restrict__ w,
                                                           int M, int C, int Cp, int KD, int MT, int mtiles,
                                                           int wc16, int ngroups, int transposed) {
  const int K = KD * Cp;
  const int taps = transposed == 2 ? 6 : TAPS;
  const int total = mtiles * ngroups * taps * wc16 * 2 * MT * 8;
  for (int i = blockIdx.x * 256 + threadIdx.x; i < total; i += gridDim.x * 256) {
    int e = i & 7;
    int r = i >> 3;
    int ml = r % MT; r /= MT;
    int tap = r % taps; r /= taps;
    int kg = r & 1; r >>= 1;
    int c16l = r % wc16; r /= wc16;
    int grp = r % ngroups;
    int mt = r / ngroups;
    const int m = (transposed == 2 ? mt >> 1 : mt) * MT + ml;
    const int k = (grp * wc16 + c16l) * CK + kg * 8 + e;
    uint16_t v = 0;  // rows past M and steps past K are padding
    const int kd = k / Cp, c = k - kd * Cp;
    if (m < M && k < K && c < C) {
      const int kh = tap / KW, kw = tap % KW;
      if (transposed == 2) v = phase_has(mt & 1, tap) ? w[((size_t)c * M + m) * TAPS + phase_tap(mt & 1, tap)] : 0;
      else if (!transposed)
        v = w[((((size_t)m * C + c) * KD + kd) * KH + kh) * KW + kw];
      else
        v = w[((((size_t)c * M + m) * KD + (KD - 1 - kd)) * KH + (KH - 1 - kh)) * KW + (KW - 1 - kw)];
    }
    dst[i] = v;
  }
}

// ---------------------------------------------------------------- split mode
// An fp32 value is the sum of three bf16 parts (8 + 8 + 8 significand bits): high = bf16(v),
// middle = bf16(v - high), low = bf16(v - high - middle); the subtractions are exact. A
// product of two fp32 values is then, to 2^-24 relative, the sum of the six part products
// whose indices add up to at most 2, each of which the bf16 matrix cores form exactly and
// add in fp32. An fp16 value (11 significand bits) is the sum of two parts, and the three
// products (0,0), (0,1), (1,0) carry it to 2^-16 relative, far below fp16's own rounding.
__device__ __forceinline__ uint16_t split_part(float v, int part) {
  const uint16_t hi = jg::f32_to_bf16(v);
  if (part == 0) return hi;
  const float hf = jg::bf16_to_f32(hi);
  const float r1 = (hf - hf == 0.0f) ? v - hf : 0.0f;  // an infinite (or NaN) high part carries everything
  const uint16_t mid = jg::f32_to_bf16(r1);
  if (part == 1) return mid;
  return jg::f32_to_bf16(r1 - jg::bf16_to_f32(mid));
}
// Contraction blocks of a split mode: block b multiplies input part x[b] with weight part w[b]
// (two bits each, block 0 in the lowest bits).
struct SplitSpec {
  int parts, nblk;
  uint32_t xparts, wparts;
};
constexpr uint32_t pack_parts(int a, int b, int c, int d, int e, int f) {
  return (uint32_t)a | ((uint32_t)b << 2) | ((uint32_t)c << 4) | ((uint32_t)d << 6) | ((uint32_t)e << 8) | ((uint32_t)f << 10);
}
inline SplitSpec split_spec(int mode) {
  if (mode == 1) return SplitSpec{3, 6, pack_parts(0, 0, 1, 0, 1, 2), pack_parts(0, 1, 0, 2, 1, 0)};  // fp32
  if (mode == 2) return SplitSpec{2, 3, pack_parts(0, 0, 1, 0, 0, 0), pack_parts(0, 1, 0, 0, 0, 0)};  // fp16
  return SplitSpec{1, 1, 0u, 0u};
}
// Whether the blocks of a layer with few input channels C are joined: their channels are counted through and padded to a
// multiple of 16 once, not block by block, and x holds a copy of a part for every block that reads it. 3 channels of
// fp32 are 2 contraction steps instead of 6: 3 -> 16 of 4 x 512 x 512 forward 111 -> 67 us, 4 -> 8 of 32 x 64 x 64 73 -> 33 us,
// 20 -> 33 of 128 x 128 58 -> 45 us; the error against fp64 goes down with it (1.7e-7 -> 1.1e-7, 3.0e-7 -> 1.7e-7). Taken where the steps saved, about 19 ps a pixel each,
// are worth more than the 3 C more 16-bit copies that are written, about 1.5 C ps a pixel.
inline bool joined_blocks(int mode, int KD, int C) {
  const int saved = 6 * ((C + CK - 1) / CK) - (6 * C + CK - 1) / CK;
  return mode == 1 && 12 * saved * KD > C;
}
template <typename SRC>
__device__ __forceinline__ float to_float(SRC v) { return (float)v; }

// dst (batch, copies, per_batch) bf16 = parts of src (batch, per_batch), fp32 or fp16: copy b is part (map >> 2 b) & 3.
// V consecutive elements a thread (1 where per_batch or an address is no multiple of 4 elements): bound by memory, and with
// 2-byte stores by their number. 16 channels of 4 x 512 x 512 fp32 (168 MB): 39 us element by element, 27 us
// four at a time (6.1 TB/s).
template <typename SRC, int V>
__global__ __launch_bounds__(256) void split_kernel(uint16_t* __restrict__ dst, const SRC* __restrict__ src,
                                                    size_t per_batch, size_t total, int copies, uint32_t map) {
  typedef SRC in_v __attribute__((ext_vector_type(V)));
  typedef uint16_t out_v __attribute__((ext_vector_type(V)));
  for (size_t i = ((size_t)blockIdx.x * 256 + threadIdx.x) * V; i < total; i += (size_t)gridDim.x * 256 * V) {
    const size_t n = i / per_batch, r = i - n * per_batch;
    const in_v v = *reinterpret_cast<const in_v*>(src + i);
    out_v part[3];
#pragma unroll
    for (int e = 0; e < V; ++e)
#pragma unroll
      for (int q = 0; q < 3; ++q) part[q][e] = split_part(to_float(v[e]), q);
    uint16_t* d = dst + n * copies * per_batch + r;
#pragma unroll
    for (int b = 0; b < 6; ++b) {
      if (b == copies) break;
      const uint32_t q = (map >> (2 * b)) & 3u;
      *reinterpret_cast<out_v*>(d + b * per_batch) = q == 0 ? part[0] : (q == 1 ? part[1] : part[2]);
    }
  }
}

// prep_weights_kernel for a split mode: w is fp32 or fp16, the contraction has nblk blocks of
// KD * Cp channels, block b holds part (wparts >> 2 b) & 3 of the weights. joined: one block of KD * Cp channels,
// channel b * C + c of a depth tap is channel c of what would be block b.
template <typename SRC>
__global__ __launch_bounds__(256) void prep_weights_split_kernel(uint16_t* __restrict__ dst,
                                                                 const SRC* __restrict__ w, int M, int C, int Cp,
                                                                 int KD, int MT, int mtiles, int wc16, int ngroups,
                                                                 int transposed, int nblk, uint32_t wparts, bool joined) {
  const int KB = KD * Cp, K = joined ? KB : nblk * KB;
  const int taps = transposed == 2 ? 6 : TAPS;
  const int total = mtiles * ngroups * taps * wc16 * 2 * MT * 8;
  for (int i = blockIdx.x * 256 + threadIdx.x; i < total; i += gridDim.x * 256) {
    int e = i & 7;
    int r = i >> 3;
    int ml = r % MT; r /= MT;
    int tap = r % taps; r /= taps;
    int kg = r & 1; r >>= 1;
    int c16l = r % wc16; r /= wc16;
    int grp = r % ngroups;
    int mt = r / ngroups;
    const int m = (transposed == 2 ? mt >> 1 : mt) * MT + ml;
    const int k = (grp * wc16 + c16l) * CK + kg * 8 + e;
    int blk = k / KB;
    const int kin = k - blk * KB, kd = kin / Cp;
    int c = kin - kd * Cp;
    if (joined) {
      blk = c / C;
      c -= blk * C;
    }
    uint16_t v = 0;
    if (m < M && k < K && c < C && blk < nblk && (transposed != 2 || phase_has(mt & 1, tap))) {
      const int kh = tap / KW, kw = tap % KW;
      const float f = to_float(transposed == 2 ? w[((size_t)c * M + m) * TAPS + phase_tap(mt & 1, tap)] : !transposed ? w[((((size_t)m * C + c) * KD + kd) * KH + kh) * KW + kw]
                                           : w[((((size_t)c * M + m) * KD + (KD - 1 - kd)) * KH + (KH - 1 - kh)) * KW + (KW - 1 - kw)]);
      v = split_part(f, (int)((wparts >> (2 * blk)) & 3u));
    }
    dst[i] = v;
  }
}

// ------------------------------------------------------------ forward kernel
// EVEN: Win is even and x is 4-byte aligned, so that the 16 bytes of a task start on a dword. Otherwise
// rows and channel planes start on odd pixels as often as not. 2-byte loads (64 of them per task) took
// 68 us for 2 x 40 -> 72 channels of 217 x 301, where the kernel had to wait for nothing else; vector
// loads at 2-byte aligned addresses run at a fraction of the rate. Such a task reads the 16 bytes from the
// dword below its first pixel, and on their way to LDS the values move up by the odd pixel; the dword that
// comes in at the end is the first one of the next task of the row, in the next lane (a wavefront therefore
// holds 7 whole rows of 9 tasks).
// 2-byte stores with a scalar base and a 32-bit lane offset. The epilogue issues 128 of
// them per lane and tile; with the 64-bit lane addresses the compiler builds for plain
// pointer code each one moves 512 bytes of addresses to the memory pipeline, which is what
// the epilogue then waits on. `base` must be wave-uniform.
__device__ inline void store_bf16_lo(const void* base, uint32_t lane_off, uint32_t pair) {
  asm volatile("global_store_short %0, %1, %2" : : "v"(lane_off), "v"(pair), "s"(base) : "memory");
}
__device__ inline void store_bf16_hi(const void* base, uint32_t lane_off, uint32_t pair) {
  asm volatile("global_store_short_d16_hi %0, %1, %2" : : "v"(lane_off), "v"(pair), "s"(base) : "memory");
}
__device__ inline void store_16_bytes(const void* base, uint32_t lane_off, u32x4 v) {
  // The store reads its 16 bytes of data from the registers a little after it issues; a vector
  // instruction that overwrites them within two wait states would be stored instead. The
  // compiler pads that for its own stores but does not look inside an asm statement.
  asm volatile("global_store_dwordx4 %0, %1, %2\n\ts_nop 1" : : "v"(lane_off), "v"(v), "s"(base) : "memory");
}
__device__ inline void store_4_bytes(const void* base, uint32_t lane_off, uint32_t v) {
  asm volatile("global_store_dword %0, %1, %2" : : "v"(lane_off), "v"(v), "s"(base) : "memory");
}
__device__ inline void store_f32(const void* base, uint32_t lane_off, float v) {
  asm volatile("global_store_dword %0, %1, %2" : : "v"(lane_off), "v"(v), "s"(base) : "memory");
}

// F16: the 16-bit tensors hold fp16 instead of bf16 (v_mfma_f32_32x32x16_f16; everything else moves
// 16-bit values without looking at them, the epilogue converts by out_kind).
// PX: the MFMA operands are exchanged, D[pixel][channel] instead of D[channel][pixel]: an accumulator lane
// then owns ONE produced channel and 16 pixels, 8 consecutive ones per lane half and register octet, so that
// a lane's results are whole 16-byte pieces of an output row and leave straight from the registers. The rows
// of the pixel operand are dealt to the pixels with bits 2 and 3 of the row number exchanged (row 8j + 4h + t
// of the result lies in lane half h, register 4j + t; pixel 16 (j / 2) + 8 h + 4 (j % 2) + t goes there).
// Used where every row segment of the result is made of whole, aligned 16-byte pieces.
__device__ __forceinline__ int px_of_row(int m) { return (m & 0x13) | ((m & 4) << 1) | ((m & 8) >> 1); }

// MODE 1: the forward pass at stride 2 along both axes. A tile is 8 x 32 produced pixels, whose window is the
// same 18 x 72 pixels; the fragments of a tap take every second slot of a row, and with 64 produced channels a
// wavefront owns 2 rows x 32 pixels of 32 channels.
// MODE 2: the input gradient at stride 2. With ih + pad_h = 2 i + pa and iw + pad_w = 2 j + pb, a produced cell
// sums the taps kh = pa + 2 a, kw = pb + 2 b over g[i - a][j - b]: each of the four phases (pa, pb) is a stride-1
// convolution of g with 4, 2, 2 or 1 taps. A workgroup makes both pb of one pa (blockIdx.y = 2 * channel tile
// + pa) for 16 x 64 positions (i, j) and 32 channels, so that a lane holds two neighbouring pixels of a row.
// (The stride-1 kernels on every pixel, with a copy of every second one, took 66 + 16 us forward and 66 + 29 us
// backward for 64 -> 128 channels of 4 x 257 x 257.)
enum Mode { PLAIN = 0, STRIDED = 1, STRIDED_DGRAD = 2 };

// FOLD: the input gradient goes to its owners (see FwdParams::fold). FOLD_WHOLE: bf16, whole tiles of produced channels,
// stride 1; FOLD_ANY: any type, any number of channels, also the strided gradient.
enum Fold { FOLD_NONE = 0, FOLD_WHOLE = 1, FOLD_ANY = 2 };

template <int MT, bool EVEN, int FOLD, bool FRAMED, bool F16 = false, bool PX = false, int MODE = PLAIN, bool RIM = false>  // MT = produced channels per workgroup: 32 or 64
__global__ __launch_bounds__(THREADS) void conv3x3_mfma_kernel(StripTable strips, FwdParams p) {
  static_assert(MODE == PLAIN || (FOLD != FOLD_WHOLE && !FRAMED), "strided layers have neither that fold epilogue nor the framed input");
  static_assert(MODE != STRIDED || !FOLD, "the forward pass has nothing to fold");
  static_assert(MODE != STRIDED_DGRAD || (MT == 32 && !PX), "32 channels of two phases");
  constexpr int ST = MODE == STRIDED ? 2 : 1;
  constexpr int TH = TILE_H / ST, TW = TILE_W / ST;
  constexpr int WROWS = MODE != STRIDED ? 4 : MT / 32;                     // produced rows per wavefront
  constexpr int CB = MODE == STRIDED ? 1 : MODE == STRIDED_DGRAD ? 2 : MT / 32;  // blocks of 32 channels (or phases) per wavefront
  constexpr int WTAPS = MODE == STRIDED_DGRAD ? 6 : TAPS;                  // taps of prepared weights
  static_assert(!RIM || (FOLD && EVEN && !PX && !FRAMED), "built for the input gradient that goes to its owners");
  constexpr bool LEFT = RIM, TOP = RIM && MT == 32;  // see compute_left, compute_top
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const int w_slots = WTAPS * p.wc16 * 2 * MT;  // 16-byte slots of one group of weights
  u32x4* lds_w = reinterpret_cast<u32x4*>(smem);
  u32x4* lds_in = lds_w + w_slots;  // two stages
  float* lds_bias = reinterpret_cast<float*>(lds_in + 2 * STAGE_SLOTS);

  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // (scalar: what follows from it branches without masks)
  const int ln = lane & 31, kg = lane >> 5;
  // Wavefronts w and w + 4 share a SIMD. They hold different column halves, so when a tile's second
  // half lies past the row end every SIMD drops half of that tile's MFMAs, and row groups two apart,
  // so a tile with few valid rows keeps two SIMDs busy instead of one.
  const int wrow0 = MODE != STRIDED ? ((wave + 2 * (wave >> 2)) & 3) * WROWS : (wave % (TH / WROWS)) * WROWS;
  const int wcol0 = MODE != STRIDED ? (wave >> 2) * 32 : 0;
  const int mt = MODE == STRIDED_DGRAD ? blockIdx.y >> 1 : blockIdx.y;
  const int ch0 = MODE == STRIDED ? __builtin_amdgcn_readfirstlane(wave / (TH / WROWS)) * 32 : 0;  // the wavefront's first channel inside the tile

  // ---- tile schedule: XCD x (= blockIdx.x % 8) owns a contiguous range of tiles and
  // walks it cyclically from a start that differs per XCD. Without the stagger, ranges
  // that coincide with whole images make the 8 XCDs stream addresses that differ by a
  // multiple of the image size in lockstep, which piles them onto the same memory channels.
  const int G = gridDim.x;
  const int xcd = blockIdx.x & 7, slot_in_xcd = blockIdx.x >> 3;
  const int wg_per_xcd = (G + 7) >> 3;
  const int per_xcd = (p.total_tiles + 7) >> 3;
  const int t_begin = xcd * per_xcd;
  int t_end = t_begin + per_xcd;
  if (t_end > p.total_tiles) t_end = p.total_tiles;
  const int t_len = t_end - t_begin;
  if (slot_in_xcd >= t_len) return;
  const int t_rot = (int)(((long long)xcd * t_len) >> 3);
  const int my_tiles = jg::quotient(t_len - slot_in_xcd + wg_per_xcd - 1, p.walk.by_wgs);
  auto tile_of = [&](int ti) {  // ti-th tile of this workgroup
    int i = slot_in_xcd + ti * wg_per_xcd + t_rot;
    if (i >= t_len) i -= t_len;
    return t_begin + i;
  };

  // ---- weights and bias. With one group the weights stay in LDS for the life of the
  // workgroup; with more (many input channels) group g is loaded before the stages that
  // contract its channels. They go to LDS without passing through registers, all of a wavefront's transfers under way at once
  // and, at the start, beside the first stage's loads: 28 to 74 KB a workgroup register by register, and the stage behind them,
  // were 4 to 6 us before the first product, 2 to 4 now. 4 x 48 -> 48 of 256 x 256 forward 27.4 -> 25.3 us, 2 x 40 -> 72 of
  // 217 x 301 input gradient 37.3 -> 34.4, 1 x 70 -> 55 of 69 x 38 forward (two groups) 32.4 -> 28.5. (The second stage's loads there too,
  // in registers of their own: no faster, and spills.) transfers_landed() before the barrier behind which they are read.
  auto load_weights = [&](int grp) {
    const char* const src = reinterpret_cast<const char*>(p.wprep + ((size_t)blockIdx.y * p.ngroups + grp) * w_slots);
    const uint32_t lds_at = jg::lds_address(smem);
    for (int i = __builtin_amdgcn_readfirstlane(wave * 64); i < w_slots; i += THREADS)  // (64 divides the slots)
      jg::to_lds_1k(src, (uint32_t)(i + lane) * 16u, lds_at + (uint32_t)i * 16u);
  };
  // The same from the weights as they are. raw_weights() puts the workgroup's share into the stage buffers (one run of memory
  // forward, a run for each contraction channel in the input gradient) and arrange_weights() deals it out from there, a slot of eight
  // channels and nine taps at a time (72 reads of two bytes and nine stores of sixteen a thread for 64 x 64 channels, 1.5 to 2 us). The
  // preparation is a launch of 4.7 us less, twice a step, and the host's time for it: 64 -> 128 at stride 2 of 4 x 256 x 256, the step
  // 144.6 -> 141 us; 2 x 31 -> 39 of 52 x 40 at stride 2 forward 11.7 -> 10.7, 4 x 32 -> 32 of 256 x 256 input gradient 22.3 -> 20.9; with
  // 64 x 64 channels and one tile a workgroup the kernel's share of it is about what the launch took.
  const int left_m = min(MT, p.M - mt * MT);     // produced channels of the tile that exist
  const int taps_m = p.KD * TAPS;                // weights of a pair of channels
  const int run = p.transposed ? left_m * taps_m : left_m * p.C * taps_m, runs = p.transposed && left_m != p.M ? p.C : 1;
  const int raw_len = p.transposed && runs == 1 ? p.C * run : run;  // elements of a run of memory
  auto raw_weights = [&]() {
    const uint16_t* const src = p.wraw + (size_t)mt * MT * taps_m * (p.transposed ? 1 : p.C);
    const uint32_t lds_at = jg::lds_address(lds_in);
    const int per = raw_len / 8, pieces = runs * per;  // whole 16-byte pieces (with several runs a run is whole pieces: see the host)
    for (int i = __builtin_amdgcn_readfirstlane(wave * 64); i < pieces; i += THREADS) {
      const int at = min(i + lane, pieces - 1), r = runs == 1 ? 0 : at / per;
      const uint32_t off = 2u * (uint32_t)r * (uint32_t)(p.M * taps_m) + 16u * (uint32_t)(at - r * per);
      jg::to_lds_1k(src, off, lds_at + (uint32_t)i * 16u);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (raw_len % 8 != 0) {  // the last few elements, which share their piece with what lies behind the tensor
      if (tid < raw_len % 8) reinterpret_cast<uint16_t*>(lds_in)[per * 8 + tid] = src[per * 8 + tid];
      __syncthreads();
    }
  };
  auto arrange_weights = [&]() {
    const uint16_t* const raw = reinterpret_cast<const uint16_t*>(lds_in);
    const int octs = p.wc16 * 2;
    // Whole octets of channels forward, one depth tap: a slot's 72 elements lie behind each other from a 16-byte boundary on, nine reads
    // and 36 permutations: as many lanes hit a bank, with an eighth of the reads. Forward of 2 x 64 -> 64, 128^2 16.2 -> 14.9 us,
    // 64 -> 128 of 4 x 256^2 at stride 2 27.7 -> 26.3, 1 x 48 -> 48, 64^2 12.9 -> 12.1.
    if (FOLD == FOLD_NONE && MODE != STRIDED_DGRAD && !p.transposed && p.KD == 1 && p.C % 8 == 0) {  // wave-uniform
      const int have = p.C >> 3;  // octets that exist (the last one of a step of 16 may not)
      for (int q = tid; q < octs * MT; q += THREADS) {
        const int hi = (q >> 3) / octs, m = hi * 8 + (q & 7), o = (q >> 3) - hi * octs;
        const u32x4* const at = reinterpret_cast<const u32x4*>(lds_in) + (min(m, left_m - 1) * have + min(o, have - 1)) * 9;
        const uint32_t keep = m < left_m && o < have ? 0xffffffffu : 0u;
        uint32_t d[36];
#pragma unroll
        for (int i = 0; i < 9; ++i) {
          const u32x4 v = at[i];
          d[4 * i] = v.x; d[4 * i + 1] = v.y; d[4 * i + 2] = v.z; d[4 * i + 3] = v.w;
        }
#pragma unroll
        for (int t = 0; t < TAPS; ++t) {
          u32x4 v;
#pragma unroll
          for (int j = 0; j < 4; ++j) {  // channels 2 j (low half) and 2 j + 1: elements 18 j + t and 18 j + 9 + t
            const int a = 18 * j + t, b = a + 9;
            v[j] = __builtin_amdgcn_perm(d[b / 2], d[a / 2], (a & 1 ? 0x0302u : 0x0100u) | (b & 1 ? 0x07060000u : 0x05040000u)) & keep;
          }
          lds_w[(o * TAPS + t) * MT + m] = v;
        }
      }
      __syncthreads();
      return;
    }
    for (int q = tid; q < octs * MT; q += THREADS) {
      // Lanes next to each other read from different banks: forward a channel's weights may lie a multiple of the banks apart, so
      // that eight of them and eight octets go together
      const int hi = p.transposed ? q / MT : (q >> 3) / octs;
      const int m = p.transposed ? q % MT : hi * 8 + (q & 7), o = p.transposed ? hi : (q >> 3) - hi * octs;
      const int kd = o * 8 / p.Cp, c0 = o * 8 - kd * p.Cp;
      const int first = p.transposed ? (c0 * left_m + m) * taps_m + (p.KD - 1 - kd) * TAPS : (m * p.C + c0) * taps_m + kd * TAPS;
      const int step = p.transposed ? left_m * taps_m : taps_m;
      const int have = m < left_m ? min(p.C - c0, 8) : 0;  // channels of the octet that exist
      u32x4 v[WTAPS];
#pragma unroll
      for (int t = 0; t < WTAPS; ++t) v[t] = u32x4{0u, 0u, 0u, 0u};
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const uint16_t* const w = raw + (j < have ? first + j * step : 0);
        const uint32_t keep = j < have ? 0xffffu : 0u;
#pragma unroll
        for (int t = 0; t < WTAPS; ++t) {
          uint32_t bits;
          if (MODE == STRIDED_DGRAD) bits = phase_has(blockIdx.y & 1, t) ? w[phase_tap(blockIdx.y & 1, t)] : 0u;
          else bits = w[t];
          v[t][j / 2] |= (bits & keep) << (16 * (j & 1));
        }
      }
#pragma unroll
      for (int t = 0; t < WTAPS; ++t) {
        const int tap = MODE != STRIDED_DGRAD && p.transposed ? TAPS - 1 - t : t;
        lds_w[(o * WTAPS + tap) * MT + m] = v[t];
      }
    }
    __syncthreads();
  };
  auto transfers_landed = [&]() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); };
  if (tid < MT)
    lds_bias[tid] = (p.bias == nullptr || mt * MT + tid >= p.M) ? 0.0f
                    : p.out_kind == 1 ? reinterpret_cast<const float*>(p.bias)[mt * MT + tid]
                    : p.out_kind == 2 ? (float)reinterpret_cast<const _Float16*>(p.bias)[mt * MT + tid]
                                      : jg::bf16_to_f32(p.bias[mt * MT + tid]);

  // ---- prefetch bookkeeping. A task = 8 channels x 8 pixels of one input row.
  const size_t plane = (size_t)p.Hin * p.Win;
  const size_t chan_stride = plane * p.Din;            // elements between channels
  const uint32_t chan_b = (uint32_t)(chan_stride * 2);  // bytes
  const bool has_task = EVEN ? tid < TASKS : lane < LANES_ODD && wave * (LANES_ODD / OCTS) + lane / OCTS < 2 * IN_ROWS;
  const int oct = EVEN ? tid % OCTS : lane % OCTS;
  const int rr = EVEN ? tid / OCTS : wave * (LANES_ODD / OCTS) + lane / OCTS;  // = g8 * IN_ROWS + row
  const int t_row = rr % IN_ROWS;
  const int t_col = oct * 8;
  const int g8 = rr / IN_ROWS;
  const uint32_t t_off = (uint32_t)(((size_t)g8 * 8 * chan_stride + (size_t)t_row * p.Win + t_col) * 2);
  const int t_lds = rr * ROW_SLOTS + oct;
  const size_t plane_t = (size_t)p.tn_h * p.tn_w;
  const size_t chan_stride_t = plane_t * p.tn_d;
  const uint32_t chan_bt = (uint32_t)(chan_stride_t * 2);
  const uint32_t t_off_t = (uint32_t)(((size_t)g8 * 8 * chan_stride_t + (size_t)t_row * p.tn_w + t_col) * 2);
  uint32_t stg[8][4];
  bool stg_masked = false;    // wave-uniform: the staged window sticks out of the tensor
  const char* stg_origin = nullptr;  // its origin (wave-uniform)
  uint32_t stg_mask = 0xffu;  // this task's pixels inside the tensor (one bit each), where stg_masked; bit 8: not loaded yet
  uint32_t stg_odd = 0;       // not EVEN: one bit per channel, the task starts on the upper half of a dword
  int stg_left = 0;           // channels from the staged step's first one to the end (wave-uniform)

  struct TileCoord {
    int n, od, th, tw;
  };
  auto coord = [&](int tile) {
    TileCoord c;
    const TileWalk w = walk_of();
    const int tq = jg::quotient(tile, w.by_plane);
    int j = tile - tq * w.per_plane;
    // With columns or rows beside the grid the tiles at its edge have more to do. The tiles of a plane are turned by one from plane to
    // plane and its columns from row to row: a workgroup, whose steps are whole rows or whole planes, would else stay at one
    // place of every plane for its life (2 x 32 -> 32 of 128^3 384 -> 339 us), and in one column, where the rows of a power of two
    // alias in L2 (8 x 64 -> 64 of 1024 x 1024 931 -> 829 us).
    if (RIM) j += tq - jg::quotient(tq, w.by_plane) * w.per_plane;
    if (RIM && j >= w.per_plane) j -= w.per_plane;
    c.th = jg::quotient(j, w.by_tw);
    c.tw = j - c.th * w.tiles_w;
    if (RIM) {
      c.tw += c.th - jg::quotient(c.th, w.by_tw) * w.tiles_w;
      if (c.tw >= w.tiles_w) c.tw -= w.tiles_w;
    }
    c.n = jg::quotient(tq, w.by_od);
    c.od = tq - c.n * w.Dout;
    return c;
  };

  // ---- load cursor: the (tile, 16-channel step) whose loads are issued next; it runs two stages
  // ahead of the MFMAs. Everything that takes a division (the tile's coordinates) is done when
  // the cursor enters a tile; inside a tile the step moves by additions.
  struct Cursor {
    int ti;          // index into this workgroup's tiles
    int blk;         // contraction block
    int kd, c0;      // depth tap and first channel of the step
    int od;          // produced depth plane of the tile
    int ih0, iw0;    // window origin in the input plane
    bool window_in;  // rows and columns of the window lie inside the plane
    bool window_in_t;  // ... inside the rank's own tile (framed input)
    bool depth_ok;   // the depth tap's plane exists
    const char* base;    // window origin in channel 0 of the batch entry, depth plane 0
    const char* base_t;  // the same in the rank's own tile (framed input)
    const char* at;      // window origin in the step's first channel and plane (before the tensor where padded)
  } cur;
  const uint32_t step_b = CK * chan_b;  // bytes between the steps of a depth tap
  // The origin is worked out for a depth tap and moves by additions inside it. From scratch in every stage, with 64-bit products and
  // comparisons, 64-bit lane addresses for each load, a product for each weight fragment's place and execution masks around what a whole
  // wavefront skips, a stage had 160 scalar and 140 vector instructions beside 36 or 72 matrix instructions, which the SIMD's other wavefront
  // hides only in part. Forward / gradient with the fold: 2 x 32 -> 32 of 128^3 285 -> 272 us / 387 -> 356, 2 x 48 -> 19 of
  // 121 x 126 x 78 365 -> 350 / 454 -> 429, 1 x 54 -> 84 of 105 x 65 19.3 -> 17.5 / 24.5 -> 22.5, 4 x 64 -> 128 of 256^2 at stride 2 30.5 -> 28.7
  // / 35.5 -> 32.9; 8 x 64 -> 64 of 1024^2 665 -> 667 / 792 -> 782 (matrix instructions and the fragments' reads).
  auto cursor_tap = [&]() __attribute__((always_inline)) {
    const int id = cur.od + cur.kd - p.pad_d;
    cur.c0 = 0;
    cur.depth_ok = id >= 0 && id < p.Din;
    cur.at = cur.base + 2 * ((ptrdiff_t)((size_t)((int)((p.xmap >> (2 * cur.blk)) & 3u) * p.C) * chan_stride) + (ptrdiff_t)id * (ptrdiff_t)plane);
  };
  auto cursor_enter = [&](int ti) __attribute__((always_inline)) {
    cur.ti = ti;
    cur.blk = 0; cur.kd = 0; cur.c0 = 0;
    if (ti >= my_tiles) return;
    const TileCoord tc = coord(tile_of(ti));
    cur.od = tc.od;
    cur.ih0 = ST * (tc.th * TH) + (TOP ? p.extra_h : 0) - p.pad_h;
    cur.iw0 = ST * (tc.tw * TW) + p.org_w - p.pad_w - p.lead;  // (org_w is 0 in the strided forward)
    cur.window_in = cur.ih0 >= 0 && cur.ih0 + IN_ROWS <= p.Hin && cur.iw0 >= 0 && cur.iw0 + p.lead + IN_COLS <= p.Win;
    cur.base = reinterpret_cast<const char*>(p.x) +
               2 * ((ptrdiff_t)((size_t)tc.n * p.Cx * chan_stride) + (ptrdiff_t)cur.ih0 * p.Win + cur.iw0);
    if (FRAMED) {
      const int ht = cur.ih0 - p.tlo_h, wt = cur.iw0 - p.tlo_w;
      cur.window_in_t = ht >= 0 && ht + IN_ROWS <= p.tn_h && wt >= 0 && wt + p.lead + IN_COLS <= p.tn_w;
      cur.base_t = reinterpret_cast<const char*>(p.xt) +
                   2 * ((ptrdiff_t)((size_t)tc.n * p.Cx * chan_stride_t) + (ptrdiff_t)ht * p.tn_w + wt);
    }
    cursor_tap();
  };
  auto cursor_advance = [&]() __attribute__((always_inline)) {
    cur.c0 += CK;
    cur.at += step_b;
    if (cur.c0 < p.Cp) return;
    if (++cur.kd == p.KD) {
      cur.kd = 0;
      if (++cur.blk == p.nblk) {
        cursor_enter(cur.ti + 1);
        return;
      }
    }
    cursor_tap();
  };

  // Loads of the stage under the cursor.
  auto issue_loads = [&]() __attribute__((always_inline)) {
    // Channels of this task that exist (all 8 unless C is not a multiple of 16). The vector
    // path below reads the others anyway (they lie inside the tensor: the interior test covers
    // all 16 channel planes) and store_stage zeroes them; the guarded paths skip them.
    stg_left = p.C - cur.c0;
    const int cvalid = stg_left - g8 * 8;
    const char* const origin = cur.at;  // wave-uniform
    // The last octet of a row holds 2 pixels that are used and 6 that no fragment
    // reads, so it may run past the row end as long as it stays inside the tensor.
    const uint32_t span = (CK - 1) * chan_b + 2u * ((IN_ROWS - 1) * (uint32_t)p.Win + OCTS * 8);
    const bool interior = cur.depth_ok && cur.window_in && __builtin_amdgcn_readfirstlane((int)((p.x_end - origin - span) >> 32)) >= 0;
    if (FRAMED) {
      // window inside the own tile (wave-uniform): read the tile itself, at whatever
      // alignment its rows give the window
      const int dt = cur.od + cur.kd - p.pad_d - p.tlo_d;
      const int cx0 = (int)((p.xmap >> (2 * cur.blk)) & 3u) * p.C + cur.c0;  // first channel of the step in x
      const char* origin_t = cur.base_t + 2 * ((ptrdiff_t)((size_t)cx0 * chan_stride_t) + (ptrdiff_t)dt * (ptrdiff_t)plane_t);
      if (dt >= 0 && dt < p.tn_d && cur.window_in_t) {
        stg_masked = false;
        stg_odd = 0;
        if (!has_task) return;
        // 4-byte aligned accesses only (2-byte aligned vector loads run at a fraction of the
        // rate): a window that starts on an odd column is read one pixel early and shifted.
        const bool odd = ((reinterpret_cast<uintptr_t>(origin_t) + t_off_t) & 2) != 0;  // wave-uniform
        const char* at = origin_t + t_off_t;
        if (!odd) {
          if (oct == OCTS - 1) {
            // the last octet holds the window's last 2 pixels; the other 6 may lie past the row
            // (and the tensor), so only one dword is read
#pragma unroll
            for (int c = 0; c < 8; ++c) {
              stg[c][0] = *reinterpret_cast<const uint32_t*>(at + (size_t)c * chan_bt);
              stg[c][1] = 0u; stg[c][2] = 0u; stg[c][3] = 0u;
            }
          } else {
#pragma unroll
            for (int c = 0; c < 8; ++c) {
              const u32x4_a4 v = *reinterpret_cast<const u32x4_a4*>(at + (size_t)c * chan_bt);
              stg[c][0] = v.x; stg[c][1] = v.y; stg[c][2] = v.z; stg[c][3] = v.w;
            }
          }
        } else {
          uint32_t d0[8];
#pragma unroll
          for (int c = 0; c < 8; ++c) d0[c] = *reinterpret_cast<const uint32_t*>(at - 2 + (size_t)c * chan_bt);
          if (oct == OCTS - 1) {
#pragma unroll
            for (int c = 0; c < 8; ++c) {
              const uint32_t d1 = *reinterpret_cast<const uint32_t*>(at + 2 + (size_t)c * chan_bt);
              stg[c][0] = __builtin_amdgcn_alignbit(d1, d0[c], 16);
              stg[c][1] = 0u; stg[c][2] = 0u; stg[c][3] = 0u;
            }
          } else {
#pragma unroll
            for (int c = 0; c < 8; ++c) {
              const u32x4_a4 v = *reinterpret_cast<const u32x4_a4*>(at + 2 + (size_t)c * chan_bt);
              stg[c][0] = __builtin_amdgcn_alignbit(v.x, d0[c], 16);
              stg[c][1] = __builtin_amdgcn_alignbit(v.y, v.x, 16);
              stg[c][2] = __builtin_amdgcn_alignbit(v.z, v.y, 16);
              stg[c][3] = __builtin_amdgcn_alignbit(v.w, v.z, 16);
            }
          }
        }
        return;
      }
    }
    stg_masked = !interior;
    stg_origin = origin;
    if (!has_task) return;
    // One set of loads for every window, from addresses that differ: a load under a condition leaves its register
    // with two possible values where the paths meet, and the compiler then waits for it right there, half a stage
    // before it is wanted (a border window took the whole latency of memory that way).
    // A wave-uniform base and a 32-bit lane offset that walks the channels.
    const char* from = origin;
    uint32_t off = t_off;
    uint32_t step = chan_b;
    int steps = 8;
    if (!interior) {
      // A window that sticks out of the tensor, or whose 16 channels do (a ragged last step). A task reads
      // its 16 bytes wherever they lie inside the tensor, also past the end of its row; store_stage clears
      // the pixels that are not the row's. Tasks without any pixel of the tensor read the first bytes of the window instead (of the
      // tensor, where the window starts outside of it; the prepared weights where there are no 16 bytes), and so do those whose bytes
      // reach over the tensor's own ends: store_stage fetches these.
      const int ih = cur.ih0 + t_row, iw = cur.iw0 + t_col;
      const bool row_ok = cur.depth_ok && ih >= 0 && ih < p.Hin && cvalid > 0;
      const int first = max(0, min(8, -iw)), past = max(0, min(8, p.Win - iw));
      stg_mask = row_ok ? ((1u << past) - 1u) & ~((1u << first) - 1u) : 0u;
      // (not EVEN: the task before takes its last pixel from this one's first dword)
      const bool need = EVEN ? stg_mask != 0u : row_ok && iw - 1 < p.Win && iw + 8 > 0;
      const char* const x0 = reinterpret_cast<const char*>(p.x);
      const char* a = origin + t_off;
      const uint32_t span_here = (uint32_t)(min(cvalid, 8) - 1) * chan_b;
      const bool fits = a >= x0 && a + (size_t)span_here + 16 <= p.x_end;
      if (need && !fits) stg_mask |= 0x100u;
      if (origin < x0 || origin + 16 > p.x_end) from = x0 + 16 <= p.x_end ? x0 : reinterpret_cast<const char*>(p.wprep);
      off = need && fits ? (uint32_t)(a - from) : 0u;
      step = need && fits ? chan_b : 0u;
      steps = cvalid;
    }
    if (!EVEN) {
      off += (uint32_t)reinterpret_cast<uintptr_t>(from) & 3u;
      from -= reinterpret_cast<uintptr_t>(from) & 3;
      // every second channel starts on the other half of a dword where a channel has an odd number of pixels
      stg_odd = ((off & 2u) != 0u ? 0xffu : 0u) ^ ((step & 2u) != 0u ? 0xaau : 0u);
    }
    uint32_t offs[8];
    offs[0] = off;
    if (stg_left >= CK) {  // wave-uniform: every channel of the step exists
#pragma unroll
      for (int c = 1; c < 8; ++c) offs[c] = offs[c - 1] + step;
    } else {
#pragma unroll
      for (int c = 1; c < 8; ++c) offs[c] = offs[c - 1] + (c < steps ? step : 0u);
    }
#pragma unroll
    for (int c = 0; c < 8; ++c) {
      const u32x4_a4 v = jg::load_16_bytes_at(reinterpret_cast<uintptr_t>(from) + (EVEN ? offs[c] : offs[c] & ~3u));
      stg[c][0] = v.x; stg[c][1] = v.y; stg[c][2] = v.z; stg[c][3] = v.w;
    }
  };

  auto store_stage = [&](int buf) {
    if (!has_task) return;
    if (stg_masked && __builtin_amdgcn_ballot_w64((stg_mask & 0x100u) != 0) != 0) {
      // a task whose bytes reach over the tensor's ends (the first and last rows of the first and last channel):
      // dword by dword, those that hold a pixel of the tensor
      if ((stg_mask & 0x100u) != 0) {
        const int cvalid = stg_left - g8 * 8;
        const char* a = stg_origin + t_off;
        stg_odd = 0;
#pragma unroll
        for (int c = 0; c < 8; ++c) {
          const uintptr_t at = reinterpret_cast<uintptr_t>(a) + (uint32_t)min(c, cvalid - 1) * (size_t)chan_b;
          const uintptr_t d = at & ~(uintptr_t)3;
          stg_odd |= (uint32_t)((at >> 1) & 1) << c;
#pragma unroll
          for (int j = 0; j < 4; ++j)
            stg[c][j] = d + 4 * j + 3 >= reinterpret_cast<uintptr_t>(p.x) && d + 4 * j < reinterpret_cast<uintptr_t>(p.x_end) ? jg::load_4_bytes_at(d + 4 * j) : 0u;
        }
      }
    }
    if (p.Cp != p.C) {  // uniform: zero the channels of this step that do not exist
      const int cvalid = stg_left - g8 * 8;
#pragma unroll
      for (int c = 0; c < 8; ++c)
        if (c >= cvalid) {
          stg[c][0] = 0u; stg[c][1] = 0u; stg[c][2] = 0u; stg[c][3] = 0u;
        }
    }
    if (!EVEN) {
#pragma unroll
      for (int c = 0; c < 8; ++c) {
        const uint32_t shift = ((stg_odd >> c) & 1u) << 4;
        // the first dword of the next lane (wavefront shift left by one)
        const uint32_t next = __builtin_amdgcn_update_dpp(0, stg[c][0], 0x130, 0xf, 0xf, false);
        stg[c][0] = __builtin_amdgcn_alignbit(stg[c][1], stg[c][0], shift);
        stg[c][1] = __builtin_amdgcn_alignbit(stg[c][2], stg[c][1], shift);
        stg[c][2] = __builtin_amdgcn_alignbit(stg[c][3], stg[c][2], shift);
        stg[c][3] = __builtin_amdgcn_alignbit(next, stg[c][3], shift);
      }
    }
    if (stg_masked) {  // uniform
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const uint32_t keep = (((stg_mask >> (2 * j)) & 1u) * 0xffffu) | (((stg_mask >> (2 * j + 1)) & 1u) * 0xffff0000u);
#pragma unroll
        for (int c = 0; c < 8; ++c) stg[c][j] &= keep;
      }
    }
    u32x4* row_base = lds_in + buf * STAGE_SLOTS + t_lds;
#pragma unroll
    for (int px = 0; px < 8; ++px) {
      // pixel px of the octet: low (px even) or high (px odd) half of dword px/2
      const uint32_t sel = (px & 1) ? 0x07060302u : 0x05040100u;
      u32x4 v;
      v.x = __builtin_amdgcn_perm(stg[1][px >> 1], stg[0][px >> 1], sel);
      v.y = __builtin_amdgcn_perm(stg[3][px >> 1], stg[2][px >> 1], sel);
      v.z = __builtin_amdgcn_perm(stg[5][px >> 1], stg[4][px >> 1], sel);
      v.w = __builtin_amdgcn_perm(stg[7][px >> 1], stg[6][px >> 1], sel);
      row_base[px * OCTS] = v;
    }
  };

  f32x16 acc[CB][WROWS];

  // One third (one kw) of a stage's MFMAs. The fragments roll through the stage: the weight
  // fragments of tap row kh are last used by input row kh + ST * (WROWS - 1) of the group, and the
  // same registers are refilled right there with the next group's fragments (the next kw, or
  // after the last kw the first group of the next stage: the weights do not change at the
  // barrier), and the group's last step requests the first input fragment of the next kw. So
  // only the first input fragment of a stage is waited for with nothing else to issue.
  bf16x8 a[KH][CB];
  u32x4 bnext;
  int a_step = -1;  // the step inside the weight group whose kw = 0 fragments `a` holds
  auto weight_frag = [&](int wstep, int kh, int kw, int cb) {
    const u32x4* wt = lds_w + kg * (WTAPS * MT) + ln + (wstep * (2 * WTAPS * MT) + ch0);  // a tap's distance is an immediate offset of the read
    return __builtin_bit_cast(bf16x8, wt[(kh * KW + kw) * MT + cb * 32]);
  };
  auto compute_kw = [&](int buf, int wstep, int kw, int wstep_next) {  // wstep: the stage's step inside its weight group
    const u32x4* in = lds_in + buf * STAGE_SLOTS + kg * (IN_ROWS * ROW_SLOTS) + ST * wrow0 * ROW_SLOTS;
    const int col0 = wcol0 + ST * (PX ? px_of_row(ln) : ln) + p.lead;  // the tile's pixel 0 sits `lead` slots into the staged row
    const u32x4* inb = in + in_slot(col0 + kw);
    if (kw == 0) {
      if (a_step != wstep) {  // wave-uniform: the first stage, after a tile without work, after a weight reload
#pragma unroll
        for (int kh = 0; kh < KH; ++kh)
#pragma unroll
          for (int cb = 0; cb < CB; ++cb) a[kh][cb] = weight_frag(wstep, kh, 0, cb);
      }
      bnext = inb[0];
    }
    // software pipeline over the input rows: the fragment of row rho+1 is requested
    // before the MFMAs of row rho are issued, so its LDS latency hides behind them
#pragma unroll
    for (int rho = 0; rho < ST * (WROWS - 1) + KH; ++rho) {
      const bf16x8 b = __builtin_bit_cast(bf16x8, bnext);
      if (rho + 1 < ST * (WROWS - 1) + KH) bnext = inb[(rho + 1) * ROW_SLOTS];
      else if (kw + 1 < KW) bnext = in[in_slot(col0 + kw + 1)];
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int kh = 0; kh < KH; ++kh) {
        const int r = (rho - kh) / ST;
        if (rho >= kh && (rho - kh) % ST == 0 && r < WROWS) {
#pragma unroll
          for (int cb = 0; cb < CB; ++cb)
            if (F16 && PX)
              acc[cb][r] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, b),
                                                                  __builtin_bit_cast(f16x8, a[kh][cb]), acc[cb][r], 0, 0, 0);
            else if (F16)
              acc[cb][r] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a[kh][cb]),
                                                                  __builtin_bit_cast(f16x8, b), acc[cb][r], 0, 0, 0);
            else if (PX)
              acc[cb][r] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(b, a[kh][cb], acc[cb][r], 0, 0, 0);
            else
              acc[cb][r] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[kh][cb], b, acc[cb][r], 0, 0, 0);
        }
      }
      __builtin_amdgcn_sched_barrier(0);
      const int kh_done = rho - ST * (WROWS - 1);  // this tap row's weights are not read again in this group
      if (kh_done >= 0) {
        if (kw + 1 < KW) {
#pragma unroll
          for (int cb = 0; cb < CB; ++cb) a[kh_done][cb] = weight_frag(wstep, kh_done, kw + 1, cb);
        } else if (p.ngroups == 1) {
#pragma unroll
          for (int cb = 0; cb < CB; ++cb) a[kh_done][cb] = weight_frag(wstep_next, kh_done, 0, cb);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    if (kw == KW - 1) a_step = p.ngroups == 1 ? wstep_next : -1;
  };

  // MODE 2: the products of one column offset of g. Prepared taps: 3 kh' + t, row offset kh' (kh = 2, 0 of phase
  // row 0 or none, 1 of phase row 1), t = 0: kw 2, read at column offset 0; 1: kw 0 and 2: kw 1, at offset 1. The
  // accumulators are [pb][row].
  auto compute_phases = [&](int buf, int wstep, int kw) __attribute__((always_inline)) {
    const bool upper = (blockIdx.y & 1) == 0;  // pa = 0: both row offsets have taps
    const u32x4* in = lds_in + buf * STAGE_SLOTS + kg * (IN_ROWS * ROW_SLOTS) + wrow0 * ROW_SLOTS + in_slot(wcol0 + ln + p.lead + kw);
    const u32x4* wt = lds_w + kg * (WTAPS * MT) + ln + wstep * (2 * WTAPS * MT);
    auto frag = [&](int tap) { return __builtin_bit_cast(bf16x8, wt[tap * MT]); };
    auto mfma = [&](const bf16x8& w, const bf16x8& b, f32x16& to) __attribute__((always_inline)) {
      to = F16 ? __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, w), __builtin_bit_cast(f16x8, b), to, 0, 0, 0)
               : __builtin_amdgcn_mfma_f32_32x32x16_bf16(w, b, to, 0, 0, 0);
    };
    bf16x8 w0[2], w1[2];
    u32x4 next = in[0];
#pragma unroll
    for (int kh = 0; kh < 2; ++kh) {
      w0[kh] = frag(3 * kh + (kw == 0 ? 0 : 1));
      if (kw == 1) w1[kh] = frag(3 * kh + 2);
    }
#pragma unroll
    for (int rho = 0; rho < WROWS + 1; ++rho) {
      const bf16x8 b = __builtin_bit_cast(bf16x8, next);
      if (rho < WROWS) next = in[(rho + 1) * ROW_SLOTS];
      __builtin_amdgcn_sched_barrier(0);
      if (rho < WROWS && upper) {
        mfma(w0[0], b, acc[0][rho]);
        if (kw == 1) mfma(w1[0], b, acc[CB - 1][rho]);
      }
      if (rho > 0) {
        mfma(w0[1], b, acc[0][rho - 1]);
        if (kw == 1) mfma(w1[1], b, acc[CB - 1][rho - 1]);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };

  // The produced columns left of the tile grid (FwdParams::extra_w): their windows lie in the first columns of the staged rows,
  // and what lies before these is padding, so that column c has the taps kw >= extra_w - c only. A wavefront takes 16 channels of
  // one column (or one phase of the strided gradient's first position) of the tile's 16 rows, on 16 x 16 x 16 products:
  // 3 to 6 a stage, 4 accumulators.
  f32x4 left;
  constexpr int LBLOCKS = MT / 16;  // blocks of 16 channels
  const int lcol = __builtin_amdgcn_readfirstlane(wave / LBLOCKS), lch = __builtin_amdgcn_readfirstlane(wave % LBLOCKS) * 16;
  auto has_left = [&](const TileCoord& tc) { return LEFT && tc.tw == 0 && lcol < (MODE == STRIDED_DGRAD ? 2 * p.extra_w : p.extra_w); };
  auto compute_left = [&](int buf, int wstep) __attribute__((always_inline)) {
    typedef short s16x4 __attribute__((ext_vector_type(4)));
    typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
    const int n = lane & 15, quad = (lane >> 4) & 1;  // pixel row / channel, half of the eight channels of a slot
    const u32x2* in = reinterpret_cast<const u32x2*>(lds_in + buf * STAGE_SLOTS + kg * (IN_ROWS * ROW_SLOTS) + n * ROW_SLOTS) + quad;
    const u32x2* wt = reinterpret_cast<const u32x2*>(lds_w + kg * (WTAPS * MT) + n + (wstep * (2 * WTAPS * MT) + lch)) + quad;
    auto product = [&](int tap, int row, int col) __attribute__((always_inline)) {
      const u32x2 a = wt[2 * tap * MT], b = in[2 * (row * ROW_SLOTS + in_slot(col))];
      left = F16 ? __builtin_amdgcn_mfma_f32_16x16x16f16(__builtin_bit_cast(f16x4, a), __builtin_bit_cast(f16x4, b), left, 0, 0, 0)
                 : __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(__builtin_bit_cast(s16x4, a), __builtin_bit_cast(s16x4, b), left, 0, 0, 0);
    };
    if (MODE == STRIDED_DGRAD) {  // position 0 reads column 0 only (taps t = 1 and 2 of compute_phases, by phase)
      if ((blockIdx.y & 1) == 0) product(1 + lcol, 0, 0);
      product(4 + lcol, 1, 0);
      return;
    }
#pragma unroll
    for (int kw = 0; kw < KW; ++kw)
      if (lcol + kw >= p.extra_w) {
#pragma unroll
        for (int kh = 0; kh < KH; ++kh) product(kh * KW + kw, kh, lcol + kw - p.extra_w);
      }
  };
  // The produced rows above it (FwdParams::extra_h), the same way: row r has the taps kh >= extra_h - r. Wavefronts 0 to 3 take a row
  // (or phase) and a half of the tile's columns each, 4 and 5 the corner, on the products of the tile itself: 3 or 6 a stage
  // (strided: 2 or 1), 16 accumulators, for which there are registers with 32 produced channels.
  f32x16 top;
  const int trow = __builtin_amdgcn_readfirstlane(wave & 1), tpart = __builtin_amdgcn_readfirstlane(wave >> 1);
  auto has_top = [&](const TileCoord& tc) {
    return TOP && tc.th == 0 && p.extra_h != 0 && (MODE == STRIDED_DGRAD || trow < p.extra_h) && (tpart < 2 || (tpart == 2 && tc.tw == 0 && p.extra_w != 0));
  };
  auto compute_top = [&](int buf, int wstep) __attribute__((always_inline)) {
    const u32x4* in = lds_in + buf * STAGE_SLOTS + kg * (IN_ROWS * ROW_SLOTS);
    const u32x4* wt = lds_w + kg * (WTAPS * MT) + ln + wstep * (2 * WTAPS * MT);
    const int col = tpart < 2 ? 32 * tpart + ln + p.lead : ln - p.extra_w;
    auto product = [&](int tap, int row, int kw) __attribute__((always_inline)) {
      const u32x4 a = wt[tap * MT], v = in[row * ROW_SLOTS + in_slot(max(col + kw, 0))];
      const u32x4 b = col + kw < 0 ? u32x4{0u, 0u, 0u, 0u} : v;
      top = F16 ? __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), top, 0, 0, 0)
                : __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), top, 0, 0, 0);
    };
    if (MODE == STRIDED_DGRAD) {
      if (trow == 0) product(3, 0, 0);
      product(4 + trow, 0, 1);
      return;
    }
#pragma unroll
    for (int kw = 0; kw < KW; ++kw)
#pragma unroll
      for (int kh = 0; kh < KH; ++kh)
        if (trow + kh >= p.extra_h) product(kh * KW + kw, trow + kh - p.extra_h, kw);
  };

  // Accumulator lane (ln, kg), register i of block cb: produced channel
  // cb*32 + 8*(i/4) + 4*kg + i%4, pixel column wcol0 + ln.
  auto init_acc = [&]() {
    if (PX) {  // a lane owns one channel per block
#pragma unroll
      for (int cb = 0; cb < CB; ++cb) {
        const float bv = lds_bias[ch0 + cb * 32 + ln];
#pragma unroll
        for (int r = 0; r < WROWS; ++r)
#pragma unroll
          for (int i = 0; i < 16; ++i) acc[cb][r][i] = bv;
      }
      return;
    }
#pragma unroll
    for (int cb = 0; cb < CB; ++cb)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const f32x4 bv = *reinterpret_cast<const f32x4*>(lds_bias + ch0 + (MODE == STRIDED_DGRAD ? 0 : cb * 32) + 8 * j + 4 * kg);
#pragma unroll
        for (int r = 0; r < WROWS; ++r) {
          acc[cb][r][4 * j + 0] = bv.x;
          acc[cb][r][4 * j + 1] = bv.y;
          acc[cb][r][4 * j + 2] = bv.z;
          acc[cb][r][4 * j + 3] = bv.w;
        }
      }
  };

  const int org_h = TOP ? p.extra_h : 0;  // first produced row of the tile grid
  const size_t plane_o = (size_t)p.Hout * p.Wout;
  const size_t ochan = plane_o * p.Dout;  // elements between produced channels
  // RAGGED: the last tile of produced channels when M is not a multiple of MT (its weight
  // rows past M are zero padding); a lane then stores only the channels that exist.
  // Rows of a wavefront through LDS: the accumulator holds one pixel and 32 channels per lane,
  // memory wants runs of pixels. A row of the wavefront (32 pixels x MT channels) is written to
  // LDS as 16-bit values, 64 bytes per channel, and read back as 16-byte pieces that go out as
  // 16-byte stores: 4 store instructions per row instead of 32 (MT = 64). The two channels a
  // lane pair (kg = 0, 1) writes at once, m and m + 4, sit in neighbouring 64-byte rows of the
  // scratch, so that the halves of the wavefront use different banks. `scratch`: 64 * MT bytes of
  // LDS of this wavefront. Needs 16-byte aligned row segments in y (checked by the caller).
  // `ytile` is wave-uniform (a scalar base), `row_off` the byte offset of the wavefront's row segment from it.
  // `pair(cb, i)`: the 16-bit values of accumulator registers i (low half) and i + 1 of block cb.
  auto row_through_lds = [&](unsigned char* scratch, auto pair, char* ytile, uint32_t row_off, size_t chan_bytes) {
    // lane's part of the write address: pixel ln of LDS row kg
    unsigned char* wr = scratch + kg * 64 + ln * 2;
#pragma unroll
    for (int cb = 0; cb < CB; ++cb)
#pragma unroll
      for (int i = 0; i < 16; i += 2) {
        const uint32_t h2 = pair(cb, i);
        // channel cb*32 + 8*(i/4) + i%4 (+ 4 kg): LDS row (that & ~7) + 2*(i%4) (+ kg); i + 1: two rows on
        const int row = cb * 32 + 8 * (i >> 2) + 2 * (i & 3);
        *reinterpret_cast<uint16_t*>(wr + row * 64) = (uint16_t)(h2 & 0xffffu);
        *reinterpret_cast<uint16_t*>(wr + (row + 2) * 64) = (uint16_t)(h2 >> 16);
      }
    // piece g = 64 q + lane: LDS row g / 4 = 16 q + lane / 4, pixels 8 (lane % 4) ..; its channel is
    // 16 q + (lane/4 & 8) + (lane/4 >> 1 & 3) + 4 (lane/4 & 1)
    const int l4 = lane >> 2;
    const int m_lane = (l4 & 8) + ((l4 >> 1) & 3) + ((l4 & 1) << 2);
    const uint32_t voff = (uint32_t)(m_lane * chan_bytes) + 16u * (lane & 3) + row_off;
    // all the row's pieces are requested before the first is stored: one LDS latency per row
    u32x4 piece[2 * CB];
#pragma unroll
    for (int q = 0; q < 2 * CB; ++q) piece[q] = *reinterpret_cast<const u32x4*>(scratch + (q * 64 + lane) * 16);
#pragma unroll
    for (int q = 0; q < 2 * CB; ++q) store_16_bytes(ytile + (size_t)q * 16 * chan_bytes, voff, piece[q]);
  };

  // PX layout: lane (ln, kg) holds channel cb * 32 + ln; registers 8 J .. 8 J + 7 hold the pixels
  // wcol0 + 16 J + 8 kg + (0 .. 7) of the wavefront's row: one 16-byte piece of 16-bit results.
  auto piece_16bit = [&](int cb, int r, int J) {
    u32x4 v;
#pragma unroll
    for (int d = 0; d < 4; ++d) {
      f32x2 v2 = {acc[cb][r][8 * J + 2 * d], acc[cb][r][8 * J + 2 * d + 1]};
      v[d] = F16 ? __builtin_bit_cast(uint32_t, __builtin_convertvector(v2, f16x2))
                 : __builtin_bit_cast(uint32_t, __builtin_convertvector(v2, bf16x2));
    }
    return v;
  };
  // A row of the wavefront (32 pixels x MT channels of 16-bit results) goes through LDS once, as 16-byte
  // pieces both ways: lane (channel ln, half kg) writes its pieces 2 J + kg of channels cb * 32 + ln, then
  // lane l reads piece l % 4 of channel 16 q + l / 4, so that four neighbouring lanes store 64 contiguous
  // bytes of one channel row. A channel's four pieces sit in one 64-byte LDS row, at slot piece ^ (channel / 4 % 4):
  // the 16 lanes of a write (consecutive channels, one piece) and of a read (four channels, all pieces)
  // then each cover all 64 banks once. `scratch`: 64 * MT bytes of LDS of this wavefront.
  auto epilogue_px = [&](const TileCoord& tc, int free_buf) {
    const int tw0 = tc.tw * TW + p.org_w;
    const size_t chan_bytes = 2 * ochan;
    unsigned char* scratch = reinterpret_cast<unsigned char*>(lds_in + free_buf * STAGE_SLOTS) + wave * (STAGE_BYTES / WAVES);
    // wave-uniform base: the tile's first column in produced channel mt * MT, row 0 (it may lie before
    // the row where the tile grid starts left of the tensor; such pieces are not stored)
    char* ytile = reinterpret_cast<char*>(p.y) +
                  2 * ((ptrdiff_t)(((size_t)tc.n * p.M + (size_t)mt * MT + ch0) * ochan + (size_t)tc.od * plane_o) + (ptrdiff_t)tw0);
    const int m_left = p.M - mt * MT - ch0;
    const int l4 = lane >> 2, pc = lane & 3;  // reading side: channel 16 q + l4, piece pc
    const int px = tw0 + wcol0 + 8 * pc;
    const bool px_ok = px >= 0 && px + 8 <= p.Wout;
    const uint32_t lane_off = (uint32_t)(l4 * chan_bytes) + 2u * (uint32_t)(wcol0 + 8 * pc);
    unsigned char* wr = scratch + ln * 64;
    const unsigned char* rd = scratch + l4 * 64 + ((pc ^ ((l4 >> 2) & 3)) << 4);
    const int wsw = (ln >> 2) & 3;
#pragma unroll
    for (int r = 0; r < WROWS; ++r) {
      const int oh = tc.th * TH + org_h + wrow0 + r;
#pragma unroll
      for (int cb = 0; cb < CB; ++cb)
#pragma unroll
        for (int J = 0; J < 2; ++J)
          *reinterpret_cast<u32x4*>(wr + cb * 32 * 64 + (((2 * J + kg) ^ wsw) << 4)) = piece_16bit(cb, r, J);
      u32x4 piece[2 * CB];
#pragma unroll
      for (int q = 0; q < 2 * CB; ++q) piece[q] = *reinterpret_cast<const u32x4*>(rd + q * 16 * 64);
      if (oh < p.Hout) {
        const uint32_t row_off = lane_off + 2u * (uint32_t)oh * (uint32_t)p.Wout;
#pragma unroll
        for (int q = 0; q < 2 * CB; ++q)
          if (px_ok && q * 16 + l4 < m_left) store_16_bytes(ytile + (size_t)q * 16 * chan_bytes, row_off, piece[q]);
      }
    }
  };

  // store(cb, i, vo) for every channel of the lane that exists, `vo` the byte offset of the channel: it starts at the
  // lane's first channel and walks by additions (a product per store costs a multiply, a 64-bit add and, with the scalar
  // registers this kernel has left, a spill reload). Groups of eight channels that do not exist are left out.
  const int m_here = p.M - mt * MT - ch0;  // channels from the wavefront's first one to the end
  auto walk_channels = [&](int blocks, uint32_t vo, uint32_t st, auto store) __attribute__((always_inline)) {
    const uint32_t st8 = 8u * st;
#pragma unroll
    for (int cb = 0; cb < CB; ++cb) {
      if (cb >= blocks) break;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int have = m_here - cb * 32 - 8 * j;
        uint32_t v = vo;
        if (have > 0) {
#pragma unroll
          for (int k = 0; k < 4; ++k) {
            if (4 * kg + k < have) store(cb, 4 * j + k, v);
            v += st;
          }
        }
        vo += st8;
      }
    }
  };

  auto epilogue_rows = [&](const TileCoord& tc, auto ragged, int free_buf) {
    constexpr bool RAGGED = decltype(ragged)::value;
    const int tw0 = tc.tw * TW + p.org_w;  // first produced column of the tile
    const int ow = tw0 + wcol0 + ln;
    if (!RAGGED && p.out_kind != 1 && (p.Wout & 7) == 0 && (tw0 & 7) == 0 && (reinterpret_cast<uintptr_t>(p.y) & 15) == 0 &&
        tw0 + wcol0 >= 0 && tw0 + wcol0 + 32 <= p.Wout) {  // wave-uniform
      unsigned char* scratch = reinterpret_cast<unsigned char*>(lds_in + free_buf * STAGE_SLOTS) + wave * (STAGE_BYTES / WAVES);
      char* ytile = reinterpret_cast<char*>(p.y) +
                    2 * (((size_t)tc.n * p.M + (size_t)mt * MT + ch0) * (plane_o * p.Dout) + (size_t)tc.od * plane_o +
                         (size_t)tw0);
#pragma unroll
      for (int r = 0; r < WROWS; ++r) {
        const int oh = tc.th * TH + org_h + wrow0 + r;
        auto pair = [&](int cb, int i) {
          f32x2 v2 = {acc[cb][r][i], acc[cb][r][i + 1]};
          return F16 ? __builtin_bit_cast(uint32_t, __builtin_convertvector(v2, f16x2))
                                 : __builtin_bit_cast(uint32_t, __builtin_convertvector(v2, bf16x2));
        };
        if (oh < p.Hout)
          row_through_lds(scratch, pair, ytile, (uint32_t)(2 * ((size_t)oh * p.Wout + wcol0)), 2 * plane_o * p.Dout);
      }
      return;
    }
    char* ybase = reinterpret_cast<char*>(p.y) +
                  2 * (((size_t)tc.n * p.M + (size_t)mt * MT + ch0) * ochan + (size_t)tc.od * plane_o);
    const int m_left = p.M - mt * MT - ch0 - 4 * kg;  // channels from this lane's first one to the end
    if (p.out_kind == 1) {  // uniform: the same walk with 4-byte stores
      char* ybase32 = reinterpret_cast<char*>(p.y) +
                      4 * (((size_t)tc.n * p.M + (size_t)mt * MT + ch0) * ochan + (size_t)tc.od * plane_o);
#pragma unroll
      for (int r = 0; r < WROWS; ++r) {
        const int oh = tc.th * TH + org_h + wrow0 + r;
        if (oh < p.Hout && ow >= 0 && ow < p.Wout) {
          const uint32_t voff = (uint32_t)(4 * ((size_t)(4 * kg) * ochan + (size_t)oh * p.Wout + ow));
          // the channel's base walks by additions (a product per store costs a scalar multiply, a 64-bit add
          // and, with the scalar registers this kernel has left, a spill reload)
          const char* yc = ybase32;
          const size_t cs = ochan * 4;
#pragma unroll
          for (int cb = 0; cb < CB; ++cb)
#pragma unroll
            for (int i = 0; i < 16; ++i) {
              const int m0 = cb * 32 + 8 * (i >> 2) + (i & 3);
              if (!RAGGED || m0 < m_left) store_f32(yc, voff, acc[cb][r][i]);
              yc += (i & 3) == 3 ? 5 * cs : cs;
            }
        }
      }
      return;
    }
#pragma unroll
    for (int r = 0; r < WROWS; ++r) {
      const int oh = tc.th * TH + org_h + wrow0 + r;
      if (oh < p.Hout && ow >= 0 && ow < p.Wout) {
        const uint32_t voff = (uint32_t)(2 * ((size_t)(4 * kg) * ochan + (size_t)oh * p.Wout + ow));
        const char* yc = ybase;  // walks by additions, as above
        const size_t cs = ochan * 2;
#pragma unroll
        for (int cb = 0; cb < CB; ++cb)
#pragma unroll
          for (int i = 0; i < 16; i += 2) {
            f32x2 v2 = {acc[cb][r][i], acc[cb][r][i + 1]};
            const uint32_t h2 = F16 ? __builtin_bit_cast(uint32_t, __builtin_convertvector(v2, f16x2))
                                                : __builtin_bit_cast(uint32_t, __builtin_convertvector(v2, bf16x2));
            const int m0 = cb * 32 + 8 * (i >> 2) + (i & 3);
            if (!RAGGED || m0 < m_left) store_bf16_lo(yc, voff, h2);
            yc += cs;
            if (!RAGGED || m0 + 1 < m_left) store_bf16_hi(yc, voff, h2);
            yc += (i & 2) ? 5 * cs : cs;
          }
      }
    }
  };
  // MODE 2: a lane's two phases are neighbouring pixels of a row and leave together, at whatever alignment the
  // row has (4-byte stores at 2-byte aligned addresses run at the rate of aligned ones).
  auto epilogue_phases = [&](const TileCoord& tc) {
    const int pa = blockIdx.y & 1;
    const int iw = 2 * (tc.tw * TW + p.org_w + wcol0 + ln) - p.px_w;
    const bool ok0 = iw >= 0 && iw < p.Wx, ok1 = iw + 1 >= 0 && iw + 1 < p.Wx;
    const size_t plane_x = (size_t)p.Hx * p.Wx;
    const int m_left = p.M - mt * MT - 4 * kg;
    // a wave-uniform base and a 32-bit lane offset that walks the channels by additions
    const uint32_t es = p.out_kind == 1 ? 4u : 2u;
    const char* const base = reinterpret_cast<const char*>(p.y) + es * (((size_t)tc.n * p.M + (size_t)mt * MT) * plane_x);
    const uint32_t st = es * (uint32_t)plane_x;
#pragma unroll
    for (int r = 0; r < WROWS; ++r) {
      const int ih = 2 * (tc.th * TH + org_h + wrow0 + r) + pa - p.px_h;
      if (ih < 0 || ih >= p.Hx) continue;
      const uint32_t row = 4 * kg * st + es * (uint32_t)(ih * p.Wx + iw);
      auto walk = [&](auto store) __attribute__((always_inline)) {
        uint32_t vo = row;
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          if (8 * (i >> 2) + (i & 3) < m_left) store(i, vo);
          vo += (i & 3) == 3 ? 5 * st : st;
        }
      };
      if (p.out_kind == 1) {
        if (ok0) walk([&](int i, uint32_t vo) { store_f32(base, vo, acc[0][r][i]); });
        if (ok1) walk([&](int i, uint32_t vo) { store_f32(base, vo + 4, acc[CB - 1][r][i]); });
        continue;
      }
      auto pair = [&](int i) {
        f32x2 v2 = {acc[0][r][i], acc[CB - 1][r][i]};
        return F16 ? __builtin_bit_cast(uint32_t, __builtin_convertvector(v2, f16x2))
                   : __builtin_bit_cast(uint32_t, __builtin_convertvector(v2, bf16x2));
      };
      if (ok0 && ok1) walk([&](int i, uint32_t vo) { store_4_bytes(base, vo, pair(i)); });
      else if (ok0) walk([&](int i, uint32_t vo) { store_bf16_lo(base, vo, pair(i)); });
      else if (ok1) walk([&](int i, uint32_t vo) { store_bf16_hi(base, vo + 2, pair(i)); });
    }
  };
  auto epilogue = [&](const TileCoord& tc, int free_buf) {
    if constexpr (MODE == STRIDED_DGRAD) epilogue_phases(tc);
    else if (PX) epilogue_px(tc, free_buf);
    else if ((mt + 1) * MT <= p.M) epilogue_rows(tc, std::false_type{}, free_buf);
    else epilogue_rows(tc, std::true_type{}, free_buf);
  };

  // Fold-mode epilogue: a produced cell goes to the unpadded tile when it lies inside
  // [lo, lo + n) on every axis, else to the strip of the neighbour that owns it (dropped
  // when that neighbour does not exist). Values pass through `0 + v`: the sign of a
  // zero is cleared, as the reference's scatter-add does for every cell.
  auto epilogue_fold = [&](const TileCoord& tc, int free_buf) {
    // bf16 pairs of the whole accumulator first (the fp32 registers are dead after this).
    // The sign of a zero only matters where a value is zero or rounds to zero, which is
    // rare: one min3 per two values finds out, and only then the bits are patched.
    uint32_t pk[CB][WROWS][8];
    float small = 3.0e38f;
#pragma unroll
    for (int cb = 0; cb < CB; ++cb)
#pragma unroll
      for (int r = 0; r < WROWS; ++r)
#pragma unroll
        for (int i = 0; i < 16; i += 2) {
          small = __builtin_fminf(small, __builtin_fminf(__builtin_fabsf(acc[cb][r][i]), __builtin_fabsf(acc[cb][r][i + 1])));
          f32x2 v2 = {acc[cb][r][i], acc[cb][r][i + 1]};
          pk[cb][r][i >> 1] = __builtin_bit_cast(uint32_t, __builtin_convertvector(v2, bf16x2));
        }
    if (__builtin_amdgcn_ballot_w64(!(small >= 1.0e-39f)) != 0) {  // bf16 rounds |v| <= 2^-134 to zero
#pragma unroll
      for (int cb = 0; cb < CB; ++cb)
#pragma unroll
        for (int r = 0; r < WROWS; ++r)
#pragma unroll
          for (int j = 0; j < 8; ++j) {
            uint32_t bits = pk[cb][r][j];
            if ((bits & 0x00007fffu) == 0) bits &= 0xffff0000u;
            if ((bits & 0x7fff0000u) == 0) bits &= 0x0000ffffu;
            pk[cb][r][j] = bits;
          }
    }
    const int ow = tc.tw * TW + p.org_w + wcol0 + ln;
    const int hi_d = p.Dout - p.lo_d - p.nD, hi_h = p.Hout - p.lo_h - p.nH, hi_w = p.Wout - p.lo_w - p.nW;
    const int od = tc.od;
    const int rd = od < p.lo_d ? 0 : (od < p.lo_d + p.nD ? 1 : 2);
    const int cd = od - (rd == 0 ? 0 : (rd == 1 ? p.lo_d : p.lo_d + p.nD));
    const int ed = rd == 0 ? p.lo_d : (rd == 1 ? p.nD : hi_d);
    const size_t plane0 = (size_t)tc.n * p.M + (size_t)mt * MT;
    const int th0 = tc.th * TH + org_h, tw0 = tc.tw * TW + p.org_w;
    // A tile that lies wholly inside the own extent (wave-uniform test): plain rows of
    // the unpadded tile, no per-cell routing.
    if (rd == 1 && th0 >= p.lo_h && th0 + TH <= p.lo_h + p.nH && tw0 >= p.lo_w && tw0 + TW <= p.lo_w + p.nW) {
      const size_t ps = (size_t)p.nD * p.nH * p.nW;
      char* ybase = reinterpret_cast<char*>(p.y) + 2 * (plane0 * ps + (size_t)cd * p.nH * p.nW);
      if (((tw0 - p.lo_w) & 7) == 0 && (p.nW & 7) == 0 && (reinterpret_cast<uintptr_t>(p.y) & 15) == 0) {  // uniform
        // the tile's rows start on the 16-byte grid of the unpadded tile (the host shifts the tile
        // grid to make it so): 16-byte stores through this wavefront's slice of the free stage buffer
        unsigned char* scratch =
            reinterpret_cast<unsigned char*>(lds_in + free_buf * STAGE_SLOTS) + wave * (STAGE_BYTES / WAVES);
        char* ytile = ybase + 2 * (ptrdiff_t)(tw0 - p.lo_w);
#pragma unroll
        for (int r = 0; r < WROWS; ++r) {
          const int oh = th0 + wrow0 + r - p.lo_h;
          auto pair = [&](int cb, int i) { return pk[cb][r][i >> 1]; };
          row_through_lds(scratch, pair, ytile, (uint32_t)(2 * ((size_t)oh * p.nW + wcol0)), 2 * ps);
        }
        return;
      }
      // One scalar base for the tile; the channel walks in the 32-bit lane offset (the host checks that MT
      // planes fit it): one vector add per store. A scalar base per channel cost a multiply, a 64-bit add and
      // the reload of a spilled scalar per store, three to four instructions for each 2-byte store.
      const uint32_t st = (uint32_t)(2 * ps), st5 = 5u * st;
#pragma unroll
      for (int r = 0; r < WROWS; ++r) {
        const int oh = th0 + wrow0 + r - p.lo_h;
        uint32_t vo = (uint32_t)(2 * ((size_t)(4 * kg) * ps + (size_t)oh * p.nW + (ow - p.lo_w)));
#pragma unroll
        for (int cb = 0; cb < CB; ++cb)
#pragma unroll
          for (int j = 0; j < 8; ++j) {  // channels cb * 32 + 8 * (j / 2) + 2 * (j % 2) and the one after (+ 4 kg, in vo)
            const uint32_t bits = pk[cb][r][j];
            store_bf16_lo(ybase, vo, bits);
            vo += st;
            store_bf16_hi(ybase, vo, bits);
            vo += (j & 1) ? st5 : st;
          }
      }
      return;
    }
    // Otherwise a cell goes to the unpadded tile when it lies inside [lo, lo + n) on every
    // axis, else to the strip of the neighbour that owns it (dropped when that neighbour
    // does not exist).
    const int rw = ow < p.lo_w ? 0 : (ow < p.lo_w + p.nW ? 1 : 2);
    const int cw = ow - (rw == 0 ? 0 : (rw == 1 ? p.lo_w : p.lo_w + p.nW));
    const int ew = rw == 0 ? p.lo_w : (rw == 1 ? p.nW : hi_w);
#pragma unroll
    for (int r = 0; r < WROWS; ++r) {
      const int oh = th0 + wrow0 + r;
      if (oh >= p.Hout || ow >= p.Wout || ow < 0) continue;
      const int rh = oh < p.lo_h ? 0 : (oh < p.lo_h + p.nH ? 1 : 2);
      const int ch = oh - (rh == 0 ? 0 : (rh == 1 ? p.lo_h : p.lo_h + p.nH));
      const int eh = rh == 0 ? p.lo_h : (rh == 1 ? p.nH : hi_h);
      // The row's three possible destinations (one per region across W) are read with wave-uniform indices,
      // i.e. through the scalar cache, and chosen per lane: a per-lane index into the table is a vector load,
      // and waiting for it also waits for every store the row before has just issued.
      const int slot0 = __builtin_amdgcn_readfirstlane(rd * 9 + rh * 3);
      char* const b_lo = static_cast<char*>(strip_entry(slot0));
      char* const b_mid = slot0 + 1 == 13 ? reinterpret_cast<char*>(p.y) : static_cast<char*>(strip_entry(slot0 + 1));
      char* const b_hi = static_cast<char*>(strip_entry(slot0 + 2));
      char* base = rw == 0 ? b_lo : (rw == 1 ? b_mid : b_hi);
      if (base == nullptr) continue;
      const uint32_t ps = (uint32_t)ed * (uint32_t)eh * (uint32_t)ew;  // elements per plane of that destination
      char* dst = base + 2 * ((plane0 + 4 * kg) * (size_t)ps + ((size_t)cd * eh + ch) * ew + cw);
      // bytes between produced channels (checked on the host to fit); the destination's plane size differs
      // from lane to lane, so the pointer walks by additions: a product per store is a quarter-rate
      // vector multiply
      const uint32_t step = 2u * ps, step5 = 5u * step;
#pragma unroll
      for (int cb = 0; cb < CB; ++cb)
#pragma unroll
        for (int j = 0; j < 8; ++j) {  // channels cb * 32 + 8 * (j / 2) + 2 * (j % 2) and the one after (+ 4 kg, in dst)
          const uint32_t bits = pk[cb][r][j];
          *reinterpret_cast<uint16_t*>(dst) = (uint16_t)(bits & 0xffffu);
          dst += step;
          *reinterpret_cast<uint16_t*>(dst) = (uint16_t)(bits >> 16);
          dst += (j & 1) ? step5 : step;
        }
    }
  };

  // The same for any type and number of channels, and for the strided gradient (a lane's two phases are the pixels ow and
  // ow + 1). One store a pixel (two neighbours of the strided gradient together) and channel, as the epilogues for such
  // rows have it; bound by the latency of a workgroup's few stages and these stores. It takes 2 to 20 us more than the plain
  // epilogue at the sizes below, and saves writing the padded gradient, its pack and its fold: gradient to finished fold of
  // 2 x 72 -> 40 channels of 217 x 301 bf16 56 -> 47 us, at stride 2 of 4 x 128 -> 64 of 256 x 256 72 -> 59 us and of
  // 8 x 99 -> 123 of 218 x 162 143 -> 122 us, of 2 x 79 -> 53 of 212 x 41 fp32 128 -> 127 us, each with one launch less.
  auto epilogue_fold_any = [&](const TileCoord& tc, int free_buf) {
    // The parameters as they are in the kernel-argument segment, read here: held in scalar registers from the kernel's
    // start on they push the stage loop's own out of them.
    typedef const __attribute__((address_space(4))) FwdParams* Args;
    Args args = nullptr;
#if defined(__HIP_DEVICE_COMPILE__)
    args = reinterpret_cast<Args>(reinterpret_cast<uintptr_t>((void*)__builtin_amdgcn_kernarg_segment_ptr()) + sizeof(StripTable));
    asm volatile("" : "+s"(args));
#endif
    const __attribute__((address_space(4))) FwdParams& p = *args;
    constexpr bool PHASES = MODE == STRIDED_DGRAD;
    const int pa = PHASES ? blockIdx.y & 1 : 0;
    const int Hp = PHASES ? p.Hx : p.Hout, Wp = PHASES ? p.Wx : p.Wout;  // the produced tensor
    const int ow = PHASES ? 2 * (tc.tw * TW + p.org_w + wcol0 + ln) - p.px_w : tc.tw * TW + p.org_w + wcol0 + ln;
    const int od = tc.od;
    const int rd = od < p.lo_d ? 0 : (od < p.lo_d + p.nD ? 1 : 2);
    const int cd = od - (rd == 0 ? 0 : (rd == 1 ? p.lo_d : p.lo_d + p.nD));
    const int ed = rd == 0 ? p.lo_d : (rd == 1 ? p.nD : p.Dout - p.lo_d - p.nD);
    const size_t plane0 = (size_t)tc.n * p.M + (size_t)mt * MT;
    const uint32_t es = p.out_kind == 1 ? 4u : 2u;
    auto region = [](int at, int lo, int n) { return at < lo ? 0 : (at < lo + n ? 1 : 2); };
    const int hi_h = Hp - p.lo_h - p.nH, hi_w = Wp - p.lo_w - p.nW;
    const int rw0 = region(ow, p.lo_w, p.nW), rw1 = region(ow + 1, p.lo_w, p.nW);
    const bool in0 = ow >= 0 && ow < Wp, in1 = PHASES && ow + 1 >= 0 && ow + 1 < Wp;
    auto pair16 = [&](float lo, float hi) {
      f32x2 v2 = {lo, hi};
      return F16 ? __builtin_bit_cast(uint32_t, __builtin_convertvector(v2, f16x2)) : __builtin_bit_cast(uint32_t, __builtin_convertvector(v2, bf16x2));
    };
    // The sign of a zero, and of what rounds to one, is cleared, as in epilogue_fold. Such values are rare; as integers they are the
    // least, so that one min3 per two values finds out (the zeros of channels that do not exist are none of them).
    const int least_zero = p.out_kind == 1 ? (int)0x80000000u : (F16 ? (int)0xb3000000u : (int)0x80008000u);  // -0, -2^-25, -2^-134
    int least = 0x7fffffff;
#pragma unroll
    for (int cb = 0; cb < CB; ++cb)
#pragma unroll
      for (int r = 0; r < WROWS; ++r)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const float v = acc[cb][r][i];  // (a bit cast of the element itself reads element 0)
          least = min(least, __builtin_bit_cast(int, v));
        }
    if (__builtin_amdgcn_ballot_w64(least <= least_zero) != 0) {
#pragma unroll
      for (int cb = 0; cb < CB; ++cb)
#pragma unroll
        for (int r = 0; r < WROWS; ++r)
#pragma unroll
          for (int i = 0; i < 16; ++i) {
            const float v = acc[cb][r][i];
            acc[cb][r][i] = __builtin_bit_cast(int, v) <= least_zero ? 0.0f : v;
          }
    }
    unsigned char* const scratch = reinterpret_cast<unsigned char*>(lds_in + free_buf * STAGE_SLOTS) + wave * (STAGE_BYTES / WAVES);
    const int blocks = PHASES ? 1 : CB;
#pragma unroll
    for (int r = 0; r < WROWS; ++r) {
      const int oh = __builtin_amdgcn_readfirstlane(PHASES ? 2 * (tc.th * TH + org_h + wrow0 + r) + pa - p.px_h : tc.th * TH + org_h + wrow0 + r);
      if (oh < 0 || oh >= Hp) continue;
      const int rh = region(oh, p.lo_h, p.nH);
      const int ch = oh - (rh == 0 ? 0 : (rh == 1 ? p.lo_h : p.lo_h + p.nH));
      const int eh = rh == 0 ? p.lo_h : (rh == 1 ? p.nH : hi_h);
      // (the table's entries by wave-uniform indices: see epilogue_fold)
      const int slot0 = __builtin_amdgcn_readfirstlane(rd * 9 + rh * 3);
      // The row's pixels between the edges: a wave-uniform base and a 32-bit lane offset that walks the channels
      char* const mid = slot0 + 1 == 13 ? reinterpret_cast<char*>(p.y) : static_cast<char*>(strip_entry(slot0 + 1));
      const uint32_t ps = (uint32_t)ed * (uint32_t)eh * (uint32_t)p.nW, st = es * ps;
      if (mid != nullptr) {
        char* const base = mid + es * (plane0 * (size_t)ps + (size_t)((cd * eh + ch) * p.nW));
        const uint32_t first = 4 * kg * st + es * (uint32_t)(ow - p.lo_w);
        const bool m0 = in0 && rw0 == 1, m1 = in1 && rw1 == 1;
        if (p.out_kind == 1) {
          if (m0) walk_channels(blocks, first, st, [&](int cb, int i, uint32_t vo) { store_f32(base, vo, acc[cb][r][i]); });
          if (m1) walk_channels(blocks, first + 4, st, [&](int, int i, uint32_t vo) { store_f32(base, vo, acc[CB - 1][r][i]); });
        } else if (!PHASES) {
          if (m0)
            walk_channels(blocks, first, st, [&](int cb, int i, uint32_t vo) {
              const uint32_t h2 = pair16(acc[cb][r][i & ~1], acc[cb][r][i | 1]);
              if (i & 1) store_bf16_hi(base, vo, h2);
              else store_bf16_lo(base, vo, h2);
            });
        } else {
          auto both = [&](int i) { return pair16(acc[0][r][i], acc[CB - 1][r][i]); };
          if (m0 && m1) walk_channels(blocks, first, st, [&](int, int i, uint32_t vo) { store_4_bytes(base, vo, both(i)); });
          if (m0 != m1)
            walk_channels(blocks, m0 ? first : first + 2, st, [&](int, int i, uint32_t vo) { store_bf16_lo(base, vo, m0 ? both(i) : both(i) >> 16); });
        }
      }
      // The few pixels at the edges, one after the other: its two lanes lay the channels into LDS, and each lane stores one
      // (a store per channel with one lane of 64 at work took 17 % of the kernel where half of the tiles have an edge)
      auto edge = [&](bool mine, int at, auto value) __attribute__((always_inline)) {
        for (uint32_t todo = (uint32_t)__builtin_amdgcn_ballot_w64(mine); todo != 0; todo &= todo - 1) {
          const int src = __builtin_ctz(todo), col = __builtin_amdgcn_readlane(at, src);
          const bool low = col < p.lo_w;
          char* const to = static_cast<char*>(strip_entry(slot0 + (low ? 0 : 2)));
          if (to == nullptr) continue;
          if (ln == src) {
#pragma unroll
            for (int cb = 0; cb < CB; ++cb) {
              if (cb >= blocks) break;
              unsigned char* const to4 = scratch + es * (cb * 32 + 4 * kg);  // channels cb * 32 + 2 i + 4 kg + 0..3
              if (p.out_kind == 1) {
#pragma unroll
                for (int i = 0; i < 16; i += 4)
                  *reinterpret_cast<f32x4*>(to4 + 8 * i) = f32x4{value(cb, i), value(cb, i + 1), value(cb, i + 2), value(cb, i + 3)};
              } else {
#pragma unroll
                for (int i = 0; i < 16; i += 4)
                  *reinterpret_cast<u32x2*>(to4 + 4 * i) = u32x2{pair16(value(cb, i), value(cb, i + 1)), pair16(value(cb, i + 2), value(cb, i + 3))};
              }
            }
          }
          asm volatile("" ::: "memory");  // (a wavefront's own reads and writes of LDS are done in order)
          const uint32_t ew = (uint32_t)(low ? p.lo_w : hi_w), pe = (uint32_t)ed * (uint32_t)eh * ew;
          const int cw = low ? col : col - p.lo_w - p.nW;
          const uintptr_t d = reinterpret_cast<uintptr_t>(to) + es * ((plane0 + lane) * (size_t)pe + (size_t)(cd * eh + ch) * ew + cw);
          if (lane < min(m_here, 32 * blocks)) {
            if (p.out_kind == 1)
              *reinterpret_cast<__attribute__((address_space(1))) uint32_t*>(d) = *reinterpret_cast<const uint32_t*>(scratch + 4 * lane);
            else
              *reinterpret_cast<__attribute__((address_space(1))) uint16_t*>(d) = *reinterpret_cast<const uint16_t*>(scratch + 2 * lane);
          }
          asm volatile("" ::: "memory");
        }
      };
      edge(in0 && rw0 != 1, ow, [&](int cb, int i) { return acc[cb][r][i]; });
      if (PHASES) edge(in1 && rw1 != 1, ow + 1, [&](int, int i) { return acc[CB - 1][r][i]; });
    }
  };

  // The columns left of the tile grid and the rows above it: pixel (oh, ow) and, count of them, channels m0 + step(i) of a lane. One of
  // oh and ow differs from lane to lane: ALONG_H says which.
  auto place = [&](const TileCoord& tc, int oh, int ow, auto along_h, int m0, int count, auto channel, auto value) __attribute__((always_inline)) {
    constexpr bool ALONG_H = decltype(along_h)::value;
    // (the parameters from the kernel-argument segment: see epilogue_fold_any)
    typedef const __attribute__((address_space(4))) FwdParams* Args;
    Args args = nullptr;
#if defined(__HIP_DEVICE_COMPILE__)
    args = reinterpret_cast<Args>(reinterpret_cast<uintptr_t>((void*)__builtin_amdgcn_kernarg_segment_ptr()) + sizeof(StripTable));
    asm volatile("" : "+s"(args));
#endif
    const __attribute__((address_space(4))) FwdParams& p = *args;
    const int Hp = MODE == STRIDED_DGRAD ? p.Hx : p.Hout, Wp = MODE == STRIDED_DGRAD ? p.Wx : p.Wout;  // the produced tensor
    if (oh < 0 || oh >= Hp || ow < 0 || ow >= Wp) return;
    const uint32_t es = p.out_kind == 1 ? 4u : 2u;
    auto region = [](int v, int lo, int n) { return v < lo ? 0 : (v < lo + n ? 1 : 2); };
    auto within = [](int v, int r, int lo, int n) { return v - (r == 0 ? 0 : (r == 1 ? lo : lo + n)); };
    auto extent = [](int r, int lo, int n, int all) { return r == 0 ? lo : (r == 1 ? n : all - lo - n); };
    const int rd = region(tc.od, p.lo_d, p.nD), rh = region(oh, p.lo_h, p.nH), rw = region(ow, p.lo_w, p.nW);
    // (wave-uniform indices into the table: see epilogue_fold)
    constexpr int STEP = ALONG_H ? 3 : 1;
    const int slot = __builtin_amdgcn_readfirstlane(rd * 9 + (ALONG_H ? rw : 3 * rh)), r = ALONG_H ? rh : rw;
    char* const low = static_cast<char*>(strip_entry(slot));
    char* const mid = slot + STEP == 13 ? reinterpret_cast<char*>(p.y) : static_cast<char*>(strip_entry(slot + STEP));
    char* const high = static_cast<char*>(strip_entry(slot + 2 * STEP));
    char* const base = r == 0 ? low : (r == 1 ? mid : high);
    const int eh = extent(rh, p.lo_h, p.nH, Hp), ew = extent(rw, p.lo_w, p.nW, Wp);
    const size_t ps = (size_t)extent(rd, p.lo_d, p.nD, p.Dout) * eh * ew;  // elements between channels of the destination
    const size_t at = ((size_t)within(tc.od, rd, p.lo_d, p.nD) * eh + within(oh, rh, p.lo_h, p.nH)) * ew + within(ow, rw, p.lo_w, p.nW);
    if (base == nullptr) return;
    const uintptr_t to = reinterpret_cast<uintptr_t>(base) + es * (((size_t)tc.n * p.M + m0) * ps + at);
#pragma unroll
    for (int i = 0; i < count; ++i) {
      if (m0 + channel(i) >= p.M) continue;
      const uintptr_t d = to + es * ps * channel(i);
      const float v = value(i);
      if (p.out_kind == 1) {
        *reinterpret_cast<JG_GLOBAL float*>(d) = 0.0f + v;  // (a sum with zero clears a zero's sign)
      } else {
        uint16_t bits = F16 ? __builtin_bit_cast(uint16_t, (_Float16)v) : __builtin_bit_cast(uint16_t, (__bf16)v);
        if ((bits & 0x7fffu) == 0) bits = 0;
        *reinterpret_cast<JG_GLOBAL uint16_t*>(d) = bits;
      }
    }
  };
  auto epilogue_left = [&](const TileCoord& tc) {  // a lane holds four neighbouring channels of the pixel in row lane % 16
    const int row = tc.th * TH + org_h + (lane & 15);
    place(tc, MODE == STRIDED_DGRAD ? 2 * row + (blockIdx.y & 1) - p.px_h : row, MODE == STRIDED_DGRAD ? lcol - p.px_w : lcol, std::true_type{},
          mt * MT + lch + 4 * (lane >> 4), 4, [](int i) { return i; }, [&](int i) { return left[i]; });
  };
  auto epilogue_top = [&](const TileCoord& tc) {
    const int pos = tpart < 2 ? tc.tw * TW + p.org_w + 32 * tpart + ln : ln;
    if (tpart == 2 && ln >= p.extra_w) return;
    place(tc, MODE == STRIDED_DGRAD ? (int)(blockIdx.y & 1) - p.px_h : trow, MODE == STRIDED_DGRAD ? 2 * pos + trow - p.px_w : pos, std::false_type{},
          mt * MT + 4 * kg, 16, [](int i) { return 8 * (i >> 2) + (i & 3); }, [&](int i) { return top[i]; });
  };

  // ---- main loop over the stages (tile, 16-channel step) of this workgroup. The
  // global loads of a stage are issued a whole stage ahead: right after the previous
  // stage's registers were written to LDS, in the middle of the stage before.
  const int stages = my_tiles * p.nc16;
  auto issue_stage = [&]() __attribute__((always_inline)) {
    issue_loads();
    cursor_advance();
  };
  // Which two stage at the head of a stage (see the stage loop) was tried all ways round, in engine cycles of
  // configuration 2: forward 4 and 5: 1.18 M, 0 and 1: 1.12 M, 2 and 3: 1.14 M, 0 to 3: 1.15 M, 2 to 5: 1.17 M;
  // dgrad with the fold epilogue 4 and 5: 1.455 M, 0 and 1: 1.47 M, 0 to 3: 1.48 M, nobody or 2 to 5: 1.49 M,
  // all six: 1.59 M. (In the fold's epilogue the older wavefronts of a SIMD get their stores out first and are
  // back in the stage loop while 4 to 7 still store.)
  const int wave_u = __builtin_amdgcn_readfirstlane(wave);
  const bool stage_early = FOLD == FOLD_WHOLE ? (wave_u == 4 || wave_u == 5) : (wave_u == 0 || wave_u == 1);
  // Does the epilogue put anything into the free stage buffer? Every epilogue but the fold's does (rows go
  // through LDS to leave as 16-byte pieces), and the fold's does where the tile grid lies on the 16-byte grid
  // of the unpadded gradient (the same test as in epilogue_fold; it is the same for every tile of a launch).
  const bool epilogue_uses_lds =
      FOLD == FOLD_ANY ? true : MODE == STRIDED_DGRAD ? false : !FOLD || ((((p.org_w - p.lo_w) & 7) == 0) && (p.nW & 7) == 0 && (reinterpret_cast<uintptr_t>(p.y) & 15) == 0);
  int buf = 0;
  cursor_enter(0);
  issue_stage();
  if (p.wraw != nullptr) {
    raw_weights();
    arrange_weights();
  } else if (p.ngroups == 1) {
    load_weights(0);
  }
  store_stage(0);
  transfers_landed();
  if (stages > 1) issue_stage();
  __syncthreads();
  int q = 0;
  for (int ti = 0; ti < my_tiles; ++ti) {
    init_acc();
    // a wavefront whose 4 x 32 pixels all lie outside the produced tensor (ragged last tiles) only
    // takes part in the staging and the barriers
    const TileCoord tcur = coord(tile_of(ti));
    const bool left_too = has_left(tcur), top_too = has_top(tcur);
    if (left_too) left = *reinterpret_cast<const f32x4*>(lds_bias + lch + 4 * (lane >> 4));
    if (top_too) {
#pragma unroll
      for (int i = 0; i < 16; ++i) top[i] = lds_bias[8 * (i >> 2) + 4 * kg + (i & 3)];
    }
    const int wave_col = tcur.tw * TW + p.org_w + wcol0;
    const bool live = wave_col < p.Wout && wave_col + 32 > 0 && tcur.th * TH + org_h + wrow0 < p.Hout;
    int wstep = 0, wgroup = 0;
    for (int c16 = 0; c16 < p.nc16; ++c16, ++q) {
      if (p.ngroups > 1 && wstep == 0) {
        // every wavefront is past the barrier that closed the last stage of the group before
        load_weights(wgroup);
        transfers_landed();
        __syncthreads();
      }
      const int wstep_next = wstep + 1 == p.wc16 ? 0 : wstep + 1;
      // Wavefronts 4 and 5 hold staging tasks like wavefronts 0..3 and share SIMD 0 and 1 with 0 and 1.
      // One of each pair stages at the head of the stage, while its SIMD's other wavefront multiplies, and that
      // one stages later, while the first multiplies; done at the same point, the two leave the matrix core idle.
      // (Not in a tile's first stage where the buffer is the last epilogue's scratch until the barrier below.)
      const bool after_epilogue = epilogue_uses_lds && c16 == 0 && ti > 0;
      const bool stage_now = stage_early && !after_epilogue;
      if (stage_now) {
        if (q + 1 < stages) store_stage(buf ^ 1);
        if (q + 2 < stages) issue_stage();
      }
      if (live) {
        if constexpr (MODE == STRIDED_DGRAD) {
          compute_phases(buf, wstep, 0);
        } else {
          compute_kw(buf, wstep, 0, wstep_next);
          compute_kw(buf, wstep, 1, wstep_next);
        }
      }
      // the buffer written next was the last epilogue's scratch (the fold's 2-byte stores leave from the registers:
      // nothing to wait for, and the wavefronts that are through with their stores do not wait for the others here)
      if (after_epilogue) __syncthreads();
      if (!stage_now) {
        if (q + 1 < stages) store_stage(buf ^ 1);  // other buffer: no hazard with this stage's reads
        if (q + 2 < stages) issue_stage();
      }
      if (live) {
        if constexpr (MODE == STRIDED_DGRAD) {
          compute_phases(buf, wstep, 1);
        } else {
          compute_kw(buf, wstep, 2, wstep_next);
        }
      }
      if (left_too) compute_left(buf, wstep);
      if (top_too) compute_top(buf, wstep);
      __syncthreads();
      buf ^= 1;
      if (++wstep == p.wc16) {
        wstep = 0;
        ++wgroup;
      }
    }
    // The epilogue stages its rows in the stage buffer the last stage was computed from, which is
    // free until the next stage is stored into it. That store waits (barrier above, in the first
    // stage of the next tile) until every wavefront has left this epilogue; until then a
    // wavefront that is done early already runs the next tile's MFMAs.
    if constexpr (FOLD == FOLD_ANY) epilogue_fold_any(tcur, buf ^ 1);
    else if constexpr (FOLD == FOLD_WHOLE) epilogue_fold(tcur, buf ^ 1);
    else epilogue(tcur, buf ^ 1);
    if (left_too) epilogue_left(tcur);
    if (top_too) epilogue_top(tcur);
  }
}

// ----------------------------------------------------------------- host side
// How a problem maps onto the kernel: produced channels in tiles of MT (M padded up to a
// multiple of 32 with zero weight rows), contraction steps of 16 channels in groups of wc16
// steps whose weights fit LDS beside the two input stages.
struct Layout {
  int MT, mtiles, nc16, wc16, ngroups;
  size_t prep_bytes, lds_bytes;
};

int pad16(int c) { return (c + CK - 1) / CK * CK; }

// Whether tiles of 64 produced channels pad no further than those of 32 do; the strided input gradient has tiles of 32 only.
bool may_take_64(int M, bool phases) { return (M + 31) / 32 * 32 % 64 == 0 && !phases; }

// K: contraction length with the channels padded to a multiple of 16 per depth tap. phases: the strided
// input gradient, tiles of 32 channels twice (one for each phase row), six taps each.
Layout layout_of(int K, int M, bool phases, int MT) {
  Layout L;
  const int taps = phases ? 6 : TAPS;
  const int mpad = (M + 31) / 32 * 32;
  L.MT = MT;
  L.mtiles = mpad / L.MT * (phases ? 2 : 1);
  L.nc16 = K / CK;
  const size_t budget = 160 * 1024 - 2 * (size_t)STAGE_BYTES - L.MT * 4;
  int cap = (int)(budget / ((size_t)taps * 2 * L.MT * 16));
  if (cap < 1) cap = 1;
  L.ngroups = (L.nc16 + cap - 1) / cap;
  if (L.ngroups < 1) L.ngroups = 1;
  L.wc16 = (L.nc16 + L.ngroups - 1) / L.ngroups;
  if (L.wc16 < 1) L.wc16 = 1;
  const size_t slots = (size_t)taps * L.wc16 * 2 * L.MT;
  L.prep_bytes = (size_t)L.mtiles * L.ngroups * slots * 16;
  L.lds_bytes = slots * 16 + 2 * (size_t)STAGE_BYTES + L.MT * 4;
  return L;
}

// C = channels of the convolved tensor, M = produced channels
bool shape_ok(int C, int M, const ConvGeom& g) {
  if (g.k[1] != KH || g.k[2] != KW) return false;
  if (g.k[0] != 1 && g.k[0] != 3) return false;
  if (g.k[0] == 1 && (g.in[0] != 1 || g.p[0] != 0)) return false;
  const bool strided = g.s[1] == 2 && g.s[2] == 2 && g.k[0] == 1;
  for (int a = 0; a < 3; ++a)
    if ((g.s[a] != 1 && !(strided && a > 0)) || g.d[a] != 1) return false;
  if (C <= 0 || M <= 0) return false;
  // per-lane byte offsets inside one batch entry are 32-bit
  const size_t in_sz = (size_t)g.in[0] * g.in[1] * g.in[2], out_sz = (size_t)g.out[0] * g.out[1] * g.out[2];
  const size_t big = in_sz > out_sz ? in_sz : out_sz;
  return big * 2 * 72 < (1ull << 31);
}


struct Launch {
  const void* x;
  const void* w;
  const void* bias;
  void* y;
  int split;                // split mode: 0 16-bit tensors as they are, 1 fp32 (six bf16 products), 2 fp16 (three)
  int f16;                  // the 16-bit tensors are fp16 (split 0 only)
  int N, C, M, KD;
  int Din, Hin, Win, Dout, Hout, Wout;
  int pad_d, pad_h, pad_w;
  int mode;                 // Mode of the kernel
  int px_h, px_w;           // STRIDED_DGRAD: the layer's padding
  int transposed;
  int fold;                 // fold mode: y is the unpadded tile, strips receive the halo cells
  int lo[3], n[3];          // own extent inside the produced tensor (fold mode)
  void* const* strips;      // 27 slots (fold mode)
  const uint16_t* xt;       // own tile for the framed input, or NULL (bf16 only)
  int tlo[3], tn[3];
};

// Bytes of the split copy of an input (its bf16 parts), rounded to 256
size_t split_bytes(size_t elements, int parts) { return (elements * parts * 2 + 255) / 256 * 256; }
size_t conv_ws_bytes(int split, int KD, int C, int M, size_t x_elements, bool phases) {
  const SplitSpec sp = split_spec(split);
  const bool joined = joined_blocks(split, KD, C);
  const int K = joined ? KD * pad16(sp.nblk * C) : sp.nblk * KD * pad16(C);
  size_t prep = layout_of(K, M, phases, 32).prep_bytes;
  if (may_take_64(M, phases)) prep = std::max(prep, layout_of(K, M, phases, 64).prep_bytes);
  return split ? (prep + 255) / 256 * 256 + split_bytes(x_elements, joined ? sp.nblk : sp.parts) : prep;
}

// Workgroups (a multiple of 8, one share per XCD) that walk the pixel tiles of one tile of produced channels; one
// workgroup fits a compute unit. With several channel tiles the chip is divided between them where that takes no
// more rounds of tiles: a chip full of workgroups for each was as many starts (weights, bias, the first stage's
// latency) on every compute unit, one after the other. 64 -> 128 channels of 4 x 256 x 256 at stride 2 forward 32.7 -> 27.2 us;
// 96 -> 96 of 4 x 128 x 256 input gradient 62 -> 54 us, 64 -> 128 of 8 x 512 x 512 forward 320 -> 305 us.
long long cus_per_xcd() { return jg::cu_count() / 8 > 0 ? jg::cu_count() / 8 : 1; }
int workgroups_for(long long tiles, int mtiles) {
  const long long cus = cus_per_xcd();
  const long long share = (tiles + 7) / 8;                        // tiles of an XCD
  const long long all = share < cus ? share : cus;
  if (mtiles > 1 && mtiles <= cus) {
    const long long walk = (share + cus / mtiles - 1) / (cus / mtiles);  // tiles of a workgroup
    if (walk <= (all * mtiles + cus - 1) / cus * ((share + all - 1) / all)) return 8 * (int)((share + walk - 1) / walk);
  }
  return 8 * (int)all;
}

template <typename SRC>
int split_launch(uint16_t* dst, const SRC* src, size_t batch, size_t per_batch, int copies, uint32_t map, hipStream_t s) {
  const size_t total = batch * per_batch;
  if (total == 0) return JG_OK;
  const bool wide = per_batch % 4 == 0 && ((reinterpret_cast<uintptr_t>(dst) | reinterpret_cast<uintptr_t>(src)) & 15) == 0;
  size_t blocks = (total + 255) / 256;
  if (wide) blocks = (blocks + 3) / 4;
  if (blocks > 65536) blocks = 65536;
  if (wide) split_kernel<SRC, 4><<<(unsigned)blocks, 256, 0, s>>>(dst, src, per_batch, total, copies, map);
  else split_kernel<SRC, 1><<<(unsigned)blocks, 256, 0, s>>>(dst, src, per_batch, total, copies, map);
  JG_CHECK_LAUNCH("split_parts_bf16");
  return JG_OK;
}

// The tile grid of a launch: produced channels a tile, origin and what lies beside it (FwdParams::org_w, extra_h, extra_w).
struct Tiling {
  int MT, org_w, extra_h, extra_w;
};

// Hout, Wout: produced cells, or positions of the strided input gradient. wide_rows: 16-bit rows of whole 16-byte pieces.
Tiling tiling_of(const Launch& L, int Hout, int Wout, bool wide_rows, bool even, bool on_lines) {
  const int TH = L.mode == STRIDED ? TILE_H / 2 : TILE_H, TW = L.mode == STRIDED ? TILE_W / 2 : TILE_W;
  const bool phases = L.mode == STRIDED_DGRAD;
  // Where to put the tile grid. A tile's staged rows start at input column org_w + TW * tw - pad_w.
  // When the rows of x are a multiple of 128 bytes apart, an origin that makes this a multiple of
  // TW puts every staged row segment on a cache-line boundary (144 bytes: two lines instead of
  // three); it is taken when it costs no extra tile column.
  int org_w = 0;
  // (not where it would take the 16-byte store path away: a plain 16-bit result with rows of whole pieces)
  if (!wide_rows && L.mode == PLAIN && L.pad_w % TW != 0 && L.Win % 64 == 0 && on_lines) {
    const int org = L.pad_w % TW - TW;
    if ((L.Wout - org + TW - 1) / TW <= (L.Wout + TW - 1) / TW) org_w = org;
  }
  // The first pad_w columns beside the first tile column and the first pad_h rows beside the first tile row, where that saves a
  // workgroup a tile: a power of two and its halo are 64 t + 1 or 2 columns wide and 16 u + 1 or 2 rows high, and the last
  // of their t + 1 tile columns and u + 1 rows cost as much as a whole one (staged rows, barriers) for what little they hold.
  // Rows of x then start at the first staged column, on cache lines where they are whole lines themselves. Gradient with the fold
  // of 2 x 32 -> 32 channels of 128^3 429 -> 338 us (16 tiles a plane for 27), at stride 2 of 4 x 64 -> 128 of 256 x 256 53.5 -> 34.8 (one
  // tile a workgroup for two).
  auto spare = [](int extent, int pad, int tile) {
    return (pad == 1 || pad == 2) && extent > pad && (extent - pad + tile - 1) / tile < (extent + tile - 1) / tile ? pad : 0;
  };
  auto walk = [&](int MT, int eh, int ew) {  // tiles a compute unit goes through
    const long long n = (long long)L.N * L.Dout * ((Hout - eh + TH - 1) / TH) * ((Wout - (ew ? ew : org_w) + TW - 1) / TW), share = (n + 7) / 8;
    const int mtiles = (L.M + MT - 1) / MT * (phases ? 2 : 1);
    const long long per = std::max(1, workgroups_for(n, mtiles) / 8);
    return (share + per - 1) / per * ((per * mtiles + cus_per_xcd() - 1) / cus_per_xcd());
  };
  // 64 produced channels a tile where they pad no further than 32 and the tiles go round: a tile of 32 takes 0.55 to 0.65 of the time of
  // one of 64 (the same rows staged, half of the products; 0.8 in the strided forward, whose tiles hold fewer), and where the chip is not
  // full twice as many of them run beside each other. Forward of 2 x 64 -> 64 of 128 x 128 24.2 -> 17.0 us, gradient with the fold of
  // 4 x 64 -> 64 of 256 x 256 (512 tiles of 32 with the rows and columns beside them for 340 of 64) 50 -> 42; forced, where the chip is
  // full, 5 x 49 -> 59 of 586 x 314 forward 105 -> 120. Tiles at the edge take about a tenth longer for rows above them.
  Tiling best{};
  double least = 0.0;
  for (const int MT : {64, 32}) {
    if (MT == 64 && !may_take_64(L.M, phases)) continue;
    if (MT == 32 && L.xt != nullptr && least > 0.0) continue;
    const int eh = L.fold && even && MT == 32 ? spare(Hout, L.pad_h, TH) : 0, ew = L.fold && even ? spare(Wout, L.pad_w, TW) : 0;
    const double tile = MT == 64 ? 1.0 : L.mode == STRIDED ? 0.8 : 0.65;
    bool taken = least == 0.0;
    for (const auto& e : {std::make_pair(0, 0), std::make_pair(0, ew), std::make_pair(eh, 0), std::make_pair(eh, ew)}) {
      const double cost = (double)walk(MT, e.first, e.second) * tile * (e.first ? 1.1 : 1.0);
      if (least == 0.0 || cost < (taken ? least : 0.9 * least)) {
        least = cost;
        best = Tiling{MT, e.second ? e.second : org_w, e.first, e.second};
        taken = true;
      }
    }
  }
  return best;
}

// Whether a workgroup's share of the weights can be fetched in whole 16-byte pieces (all but the last few elements of a tensor)
// and fits the stage buffers, filled 64 pieces at a time.
bool raw_weights_fit(const Launch& L, int MT) {
  if ((reinterpret_cast<uintptr_t>(L.w) & 15) != 0) return false;
  const long long taps_m = (long long)L.KD * TAPS, tile = std::min(MT, L.M);
  if (L.transposed && L.M > MT && L.M % 8 != 0) return false;  // runs of a tile's channels, one for each contraction channel
  return (tile * L.C * taps_m + 511) / 512 * 1024 <= 2 * (long long)STAGE_BYTES;
}

int launch_conv(const Launch& L, void* ws, size_t ws_bytes, hipStream_t s, const char* who) {
  const SplitSpec sp = split_spec(L.split);
  const bool joined = joined_blocks(L.split, L.KD, L.C);
  const int nblk = joined ? 1 : sp.nblk;
  const int C = joined ? sp.nblk * L.C : L.C;         // channels of a block
  const int copies = joined ? sp.nblk : sp.parts;     // of x
  const uint32_t copy_map = joined ? sp.xparts : pack_parts(0, 1, 2, 0, 0, 0);
  const int K = nblk * L.KD * pad16(C);
  const size_t x_elements = (size_t)L.N * L.C * L.Din * L.Hin * L.Win;
  const bool phases = L.mode == STRIDED_DGRAD;
  const size_t need = conv_ws_bytes(L.split, L.KD, L.C, L.M, x_elements, phases);
  if (ws == nullptr || ws_bytes < need)
    JG_FAIL(JG_ERR_WORKSPACE, "%s: workspace %zu < %zu bytes", who, ws_bytes, need);
  JG_REQUIRE((reinterpret_cast<uintptr_t>(ws) & 15) == 0, "%s: workspace must be 16-byte aligned",
             who);
  // the produced cells, or the positions (i, j) of the strided input gradient
  const int Hout = phases ? (L.Hout - 1 + L.px_h) / 2 + 1 : L.Hout, Wout = phases ? (L.Wout - 1 + L.px_w) / 2 + 1 : L.Wout;
  const bool wide_rows = !L.fold && L.split != 1 && L.Wout % 8 == 0 && !phases;
  const uintptr_t x_at = reinterpret_cast<uintptr_t>(L.split ? ws : L.x);  // (the parts of a split x lie a multiple of 256 bytes behind ws)
  // rows of the staged windows start at even columns where `lead` can see to it: 4-byte aligned loads
  const bool even = L.Win % 2 == 0 && (x_at & 3) == 0;
  const Tiling til = tiling_of(L, Hout, Wout, wide_rows, even, (x_at & 127) == 0);
  const int MT = til.MT;
  const Layout lay = layout_of(K, L.M, phases, MT);
  uint16_t* wprep = static_cast<uint16_t*>(ws);
  const size_t total_w = lay.prep_bytes / 2;
  JG_REQUIRE(total_w < (1ull << 31), "%s: weight tensor too large", who);
  const uint16_t* x16 = static_cast<const uint16_t*>(L.x);
  // Each workgroup puts its weights in order itself where they are 16-bit, stay in LDS and pass through the stage buffers: see arrange_weights
  const bool arranged = !L.split && lay.ngroups == 1 && raw_weights_fit(L, MT);
  if (L.split) {
    const unsigned wblocks = (unsigned)((total_w + 255) / 256);
    uint16_t* xs = reinterpret_cast<uint16_t*>(static_cast<char*>(ws) + (lay.prep_bytes + 255) / 256 * 256);
    int rc;
    if (L.split == 1) {
      prep_weights_split_kernel<float><<<wblocks, 256, 0, s>>>(wprep, static_cast<const float*>(L.w), L.M, L.C,
                                                                pad16(C), L.KD, MT, lay.mtiles, lay.wc16, lay.ngroups,
                                                                L.transposed, sp.nblk, sp.wparts, joined);
      rc = split_launch(xs, static_cast<const float*>(L.x), (size_t)L.N, x_elements / L.N, copies, copy_map, s);
    } else {
      prep_weights_split_kernel<_Float16><<<wblocks, 256, 0, s>>>(wprep, static_cast<const _Float16*>(L.w), L.M, L.C,
                                                                   pad16(C), L.KD, MT, lay.mtiles, lay.wc16,
                                                                   lay.ngroups, L.transposed, sp.nblk, sp.wparts, joined);
      rc = split_launch(xs, static_cast<const _Float16*>(L.x), (size_t)L.N, x_elements / L.N, copies, copy_map, s);
    }
    JG_CHECK_LAUNCH(who);
    if (rc) return rc;
    x16 = xs;
  } else if (!arranged) {
    prep_weights_kernel<<<(unsigned)((total_w + 255) / 256), 256, 0, s>>>(wprep, static_cast<const uint16_t*>(L.w), L.M,
                                                                           L.C, pad16(L.C), L.KD, MT, lay.mtiles,
                                                                           lay.wc16, lay.ngroups, L.transposed);
    JG_CHECK_LAUNCH(who);
  }

  FwdParams p;
  p.x_end = reinterpret_cast<const char*>(x16) + 2 * x_elements * copies;
  p.x = x16; p.wprep = reinterpret_cast<const u32x4*>(wprep);
  p.wraw = arranged ? static_cast<const uint16_t*>(L.w) : nullptr;
  p.transposed = L.transposed;
  p.bias = static_cast<const uint16_t*>(L.bias); p.y = static_cast<uint16_t*>(L.y);
  p.N = L.N; p.C = C; p.M = L.M; p.KD = L.KD;
  p.Cp = pad16(C);
  p.nblk = nblk; p.Cx = copies * L.C; p.xmap = joined ? 0u : sp.xparts; p.out_kind = L.f16 ? 2 : L.split;
  p.Din = L.Din; p.Hin = L.Hin; p.Win = L.Win;
  p.Dout = L.Dout; p.Hout = L.Hout; p.Wout = L.Wout;
  p.pad_d = L.pad_d; p.pad_h = L.pad_h; p.pad_w = L.pad_w;
  p.Hx = p.Wx = p.px_h = p.px_w = 0;
  if (phases) {  // the kernel's grid runs over the positions
    p.Hx = L.Hout; p.Wx = L.Wout;
    p.px_h = L.px_h; p.px_w = L.px_w;
    p.Hout = Hout;
    p.Wout = Wout;
  }
  const int TH = L.mode == STRIDED ? TILE_H / 2 : TILE_H, TW = L.mode == STRIDED ? TILE_W / 2 : TILE_W;
  p.org_w = til.org_w;
  p.extra_h = til.extra_h;
  p.extra_w = til.extra_w;
  p.lead = even ? (L.pad_w - p.org_w) & 1 : 0;
  p.tiles_h = (p.Hout - p.extra_h + TH - 1) / TH;
  p.tiles_w = (p.Wout - p.org_w + TW - 1) / TW;
  const long long tiles = (long long)L.N * L.Dout * p.tiles_h * p.tiles_w;
  JG_REQUIRE(tiles < (1ll << 30), "%s: too many tiles", who);
  p.total_tiles = (int)tiles;
  p.nc16 = lay.nc16;
  p.wc16 = lay.wc16;
  p.ngroups = lay.ngroups;
  p.fold = L.fold;
  p.lo_d = L.lo[0]; p.lo_h = L.lo[1]; p.lo_w = L.lo[2];
  p.nD = L.n[0]; p.nH = L.n[1]; p.nW = L.n[2];
  p.xt = L.xt;
  p.tlo_d = L.tlo[0]; p.tlo_h = L.tlo[1]; p.tlo_w = L.tlo[2];
  p.tn_d = L.tn[0]; p.tn_h = L.tn[1]; p.tn_w = L.tn[2];
  StripTable tab;
  for (int i = 0; i < 27; ++i) tab.p[i] = (L.fold && L.strips != nullptr) ? L.strips[i] : nullptr;
  if (tiles == 0) return JG_OK;
  const size_t lds = lay.lds_bytes;
  int wgs = workgroups_for(tiles, lay.mtiles);
  p.walk = TileWalk{jg::div_by(p.tiles_h * p.tiles_w), jg::div_by(p.tiles_w), jg::div_by(p.Dout), jg::div_by((wgs + 7) / 8), p.tiles_h * p.tiles_w, p.tiles_w, p.Dout};
  dim3 grid((unsigned)wgs, (unsigned)lay.mtiles, 1);
  void (*kern)(StripTable, FwdParams) = nullptr;
  if (L.f16 && L.xt != nullptr)
    JG_FAIL(JG_ERR_UNSUPPORTED, "%s: the framed input is built for bf16 only", who);
  const bool rim = p.extra_h != 0 || p.extra_w != 0;
  if (L.fold && (L.split || L.f16 || phases || lay.mtiles * MT != L.M)) {
    auto any = [&](auto f16) {
      constexpr bool F = decltype(f16)::value;
      if (phases)
        kern = rim    ? &conv3x3_mfma_kernel<32, true, FOLD_ANY, false, F, false, STRIDED_DGRAD, true>
               : even ? &conv3x3_mfma_kernel<32, true, FOLD_ANY, false, F, false, STRIDED_DGRAD>
                      : &conv3x3_mfma_kernel<32, false, FOLD_ANY, false, F, false, STRIDED_DGRAD>;
      else if (MT == 64)
        kern = rim    ? &conv3x3_mfma_kernel<64, true, FOLD_ANY, false, F, false, PLAIN, true>
               : even ? &conv3x3_mfma_kernel<64, true, FOLD_ANY, false, F>
                      : &conv3x3_mfma_kernel<64, false, FOLD_ANY, false, F>;
      else
        kern = rim    ? &conv3x3_mfma_kernel<32, true, FOLD_ANY, false, F, false, PLAIN, true>
               : even ? &conv3x3_mfma_kernel<32, true, FOLD_ANY, false, F>
                      : &conv3x3_mfma_kernel<32, false, FOLD_ANY, false, F>;
    };
    if (L.f16) any(std::true_type{});
    else any(std::false_type{});
  } else if (L.mode != PLAIN) {
    const bool wide = wide_rows && (reinterpret_cast<uintptr_t>(L.y) & 15) == 0;
    auto strided = [&](auto f16, auto px) {
      constexpr bool F = decltype(f16)::value, X = decltype(px)::value;
      if (MT == 64) kern = even ? &conv3x3_mfma_kernel<64, true, false, false, F, X, STRIDED> : &conv3x3_mfma_kernel<64, false, false, false, F, X, STRIDED>;
      else kern = even ? &conv3x3_mfma_kernel<32, true, false, false, F, X, STRIDED> : &conv3x3_mfma_kernel<32, false, false, false, F, X, STRIDED>;
    };
    if (phases) {
      if (L.f16) kern = even ? &conv3x3_mfma_kernel<32, true, false, false, true, false, STRIDED_DGRAD> : &conv3x3_mfma_kernel<32, false, false, false, true, false, STRIDED_DGRAD>;
      else kern = even ? &conv3x3_mfma_kernel<32, true, false, false, false, false, STRIDED_DGRAD> : &conv3x3_mfma_kernel<32, false, false, false, false, false, STRIDED_DGRAD>;
    } else if (L.f16) {
      if (wide) strided(std::true_type{}, std::true_type{});
      else strided(std::true_type{}, std::false_type{});
    } else {
      if (wide) strided(std::false_type{}, std::true_type{});
      else strided(std::false_type{}, std::false_type{});
    }
  } else if (L.fold) {
    if (MT == 64)
      kern = rim    ? &conv3x3_mfma_kernel<64, true, FOLD_WHOLE, false, false, false, PLAIN, true>
             : even ? &conv3x3_mfma_kernel<64, true, FOLD_WHOLE, false>
                    : &conv3x3_mfma_kernel<64, false, FOLD_WHOLE, false>;
    else
      kern = rim    ? &conv3x3_mfma_kernel<32, true, FOLD_WHOLE, false, false, false, PLAIN, true>
             : even ? &conv3x3_mfma_kernel<32, true, FOLD_WHOLE, false>
                    : &conv3x3_mfma_kernel<32, false, FOLD_WHOLE, false>;
  } else if (L.xt != nullptr) {
    if (MT == 64) kern = even ? &conv3x3_mfma_kernel<64, true, false, true> : &conv3x3_mfma_kernel<64, false, false, true>;
    else kern = even ? &conv3x3_mfma_kernel<32, true, false, true> : &conv3x3_mfma_kernel<32, false, false, true>;
  } else if (wide_rows && (reinterpret_cast<uintptr_t>(L.y) & 15) == 0) {
    // every row segment of the result is whole, aligned 16-byte pieces: results leave from the registers
    if (L.f16) {
      if (MT == 64)
        kern = even ? &conv3x3_mfma_kernel<64, true, false, false, true, true> : &conv3x3_mfma_kernel<64, false, false, false, true, true>;
      else
        kern = even ? &conv3x3_mfma_kernel<32, true, false, false, true, true> : &conv3x3_mfma_kernel<32, false, false, false, true, true>;
    } else {
      if (MT == 64)
        kern = even ? &conv3x3_mfma_kernel<64, true, false, false, false, true> : &conv3x3_mfma_kernel<64, false, false, false, false, true>;
      else
        kern = even ? &conv3x3_mfma_kernel<32, true, false, false, false, true> : &conv3x3_mfma_kernel<32, false, false, false, false, true>;
    }
  } else if (L.f16) {
    if (MT == 64)
      kern = even ? &conv3x3_mfma_kernel<64, true, false, false, true> : &conv3x3_mfma_kernel<64, false, false, false, true>;
    else
      kern = even ? &conv3x3_mfma_kernel<32, true, false, false, true> : &conv3x3_mfma_kernel<32, false, false, false, true>;
  } else {
    if (MT == 64) kern = even ? &conv3x3_mfma_kernel<64, true, false, false> : &conv3x3_mfma_kernel<64, false, false, false>;
    else kern = even ? &conv3x3_mfma_kernel<32, true, false, false> : &conv3x3_mfma_kernel<32, false, false, false>;
  }
  hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                     hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  if (e != hipSuccess) JG_FAIL(JG_ERR_LAUNCH, "%s: cannot reserve %zu bytes of LDS", who, lds);
  kern<<<grid, THREADS, lds, s>>>(tab, p);
  JG_CHECK_LAUNCH(who);
  return JG_OK;
}

}  // namespace

namespace jg {

// fp32 runs in split mode (three bf16 parts per operand, fp32 result); its 4-byte stores halve
// the extent the 32-bit lane offsets reach.
// fp32 runs in split mode; fp16 has its own MFMA instruction and runs like bf16
static int split_mode(int dtype) { return dtype == JG_F32 ? 1 : 0; }
static bool dtype_ok(const ConvGeom& g, int dtype) {
  if (g.groups != 1) return false;  // grouped layers run the direct kernels
  if (dtype == JG_BF16 || dtype == JG_F16) return true;
  if (dtype != JG_F32) return false;
  const size_t in_sz = (size_t)g.in[0] * g.in[1] * g.in[2], out_sz = (size_t)g.out[0] * g.out[1] * g.out[2];
  const size_t big = in_sz > out_sz ? in_sz : out_sz;
  return big * 4 * 72 < (1ull << 31);
}
int split_parts_bf16(uint16_t* dst, const void* src, int src_dtype, size_t batch, size_t per_batch, hipStream_t s) {
  if (src_dtype == JG_F32) return split_launch(dst, static_cast<const float*>(src), batch, per_batch, 3, pack_parts(0, 1, 2, 0, 0, 0), s);
  return split_launch(dst, static_cast<const _Float16*>(src), batch, per_batch, 2, pack_parts(0, 1, 0, 0, 0, 0), s);
}

bool mfma_fwd_supported(const ConvGeom& g, int dtype) {
  return dtype_ok(g, dtype) && shape_ok(g.cin, g.cout, g) && g.batch > 0;
}
bool mfma_dgrad_supported(const ConvGeom& g, int dtype) {
  if (!dtype_ok(g, dtype) || g.batch <= 0) return false;
  for (int a = 0; a < 3; ++a)
    if (g.p[a] > g.k[a] - 1) return false;
  return shape_ok(g.cout, g.cin, g);  // (strides 1 and 2)
}

size_t mfma_fwd_workspace(const ConvGeom& g, int dtype) {
  return conv_ws_bytes(split_mode(dtype), g.k[0], g.cin, g.cout, (size_t)g.batch * g.cin * g.in[0] * g.in[1] * g.in[2], false);
}
size_t mfma_dgrad_workspace(const ConvGeom& g, int dtype) {
  return conv_ws_bytes(split_mode(dtype), g.k[0], g.cout, g.cin, (size_t)g.batch * g.cout * g.out[0] * g.out[1] * g.out[2], g.s[2] == 2);
}

static int fwd_launch(void* y, const void* x, const void* xt, const int* tlo, const int* tn, const void* w,
                      const void* bias, const ConvGeom& g, void* ws, size_t ws_bytes, hipStream_t s,
                      const char* who, int dtype = JG_BF16) {
  Launch L;
  L.x = x; L.w = w; L.bias = bias; L.y = y;
  L.split = split_mode(dtype);
  L.f16 = dtype == JG_F16 ? 1 : 0;
  L.N = (int)g.batch; L.C = g.cin; L.M = g.cout; L.KD = g.k[0];
  L.Din = g.in[0]; L.Hin = g.in[1]; L.Win = g.in[2];
  L.Dout = g.out[0]; L.Hout = g.out[1]; L.Wout = g.out[2];
  L.pad_d = g.p[0]; L.pad_h = g.p[1]; L.pad_w = g.p[2];
  L.mode = g.s[2] == 2 ? STRIDED : PLAIN;
  L.px_h = L.px_w = 0;
  L.transposed = 0;
  L.fold = 0;
  L.strips = nullptr;
  L.xt = static_cast<const uint16_t*>(xt);
  for (int a = 0; a < 3; ++a) {
    L.lo[a] = L.n[a] = 0;
    L.tlo[a] = tlo ? tlo[a] : 0;
    L.tn[a] = tn ? tn[a] : 0;
  }
  return launch_conv(L, ws, ws_bytes, s, who);
}

int mfma_fwd(void* y, const void* x, const void* w, const void* bias, const ConvGeom& g, void* ws,
             size_t ws_bytes, hipStream_t s, int dtype) {
  return fwd_launch(y, x, nullptr, nullptr, nullptr, w, bias, g, ws, ws_bytes, s, "jg_conv_fwd(mfma)", dtype);
}

int mfma_fwd_framed(void* y, const void* x_frame, const void* xt, const int tlo[3], const int tn[3],
                    const void* w, const void* bias, const ConvGeom& g, void* ws, size_t ws_bytes,
                    hipStream_t s) {
  return fwd_launch(y, x_frame, xt, tlo, tn, w, bias, g, ws, ws_bytes, s, "jg_conv_fwd_framed(mfma)");
}

// Bands of the padded tile that the framed kernels read from x_frame: everything a
// 16 x 64 output tile window (18 x 72 cells) touches when it does not lie inside the tile.
void mfma_frame_bands(const ConvGeom& g, const int tlo[3], const int tn[3], int band_lo[3], int band_hi[3]) {
  // depth: a stage reads one plane; planes outside the tile are read whole
  band_lo[0] = tlo[0];
  band_hi[0] = g.in[0] - tlo[0] - tn[0];
  const int tile[3] = {1, TILE_H, TILE_W};
  const int reach[3] = {1, IN_ROWS, OCTS * 8};  // cells a window may touch (the last octet in full)
  const int need[3] = {1, IN_ROWS, IN_COLS};
  for (int a = 1; a < 3; ++a) {
    const int ntiles = (g.out[a] + tile[a] - 1) / tile[a];
    int first_in = -1, last_in = -1;  // tiles whose window lies inside [tlo, tlo + tn)
    for (int t = 0; t < ntiles; ++t) {
      const int w0 = t * tile[a] - g.p[a];
      if (w0 >= tlo[a] && w0 + need[a] <= tlo[a] + tn[a]) {
        if (first_in < 0) first_in = t;
        last_in = t;
      }
    }
    if (first_in < 0) {  // no tile reads the own tile along this axis: everything from the frame
      band_lo[a] = g.in[a];
      band_hi[a] = 0;
      continue;
    }
    int lo_end = (first_in - 1) * tile[a] - g.p[a] + reach[a];  // end of the last window before
    if (first_in == 0 || lo_end < 0) lo_end = 0;
    if (lo_end > g.in[a]) lo_end = g.in[a];
    int hi_begin = (last_in + 1) * tile[a] - g.p[a];             // start of the first window after
    if (last_in == ntiles - 1 || hi_begin > g.in[a]) hi_begin = g.in[a];
    if (hi_begin < 0) hi_begin = 0;
    band_lo[a] = lo_end;
    band_hi[a] = g.in[a] - hi_begin;
  }
}

// gx = conv(go zero-padded by k-1-p, flipped / transposed weights). With `own` given,
// the produced tensor is split between the unpadded tile gx and the neighbours' strips.
static int dgrad_launch(void* gx, void* const* strips, const int* lo, const int* n, const void* w,
                        const void* go, const ConvGeom& g, void* ws, size_t ws_bytes, hipStream_t s,
                        const char* who, int dtype = JG_BF16) {
  Launch L;
  L.x = go; L.w = w; L.bias = nullptr; L.y = gx;
  L.split = split_mode(dtype);
  L.f16 = dtype == JG_F16 ? 1 : 0;
  L.N = (int)g.batch; L.C = g.cout; L.M = g.cin; L.KD = g.k[0];
  L.Din = g.out[0]; L.Hin = g.out[1]; L.Win = g.out[2];
  L.Dout = g.in[0]; L.Hout = g.in[1]; L.Wout = g.in[2];
  L.pad_d = g.k[0] - 1 - g.p[0]; L.pad_h = KH - 1 - g.p[1]; L.pad_w = KW - 1 - g.p[2];
  L.mode = PLAIN;
  L.px_h = g.p[1]; L.px_w = g.p[2];
  L.transposed = 1;
  if (g.s[2] == 2) {
    L.mode = STRIDED_DGRAD;
    L.transposed = 2;
    L.pad_h = L.pad_w = 1;
  }
  L.fold = lo != nullptr;
  L.strips = strips;
  L.xt = nullptr;
  for (int a = 0; a < 3; ++a) {
    L.lo[a] = lo ? lo[a] : 0;
    L.n[a] = n ? n[a] : 0;
    L.tlo[a] = L.tn[a] = 0;
  }
  return launch_conv(L, ws, ws_bytes, s, who);
}

int mfma_dgrad(void* gx, const void* w, const void* go, const ConvGeom& g, void* ws,
               size_t ws_bytes, hipStream_t s, int dtype) {
  return dgrad_launch(gx, nullptr, nullptr, nullptr, w, go, g, ws, ws_bytes, s, "jg_conv_dgrad(mfma)", dtype);
}

int mfma_dgrad_fold(void* gx, void* const strips[27], const int lo[3], const int n[3], const void* w,
                    const void* go, const ConvGeom& g, void* ws, size_t ws_bytes, hipStream_t s, int dtype) {
  // the epilogues address the MT channel planes of a tile through a 32-bit byte offset
  const int MT = may_take_64(g.cin, g.s[2] == 2) ? 64 : 32, es = dtype == JG_F32 ? 4 : 2;
  if ((long long)n[0] * n[1] * n[2] * es * MT >= (1ll << 32) || (long long)g.in[0] * g.in[1] * g.in[2] * es * MT >= (1ll << 32))
    JG_FAIL(JG_ERR_UNSUPPORTED, "jg_conv_dgrad_fold(mfma): %d planes of the tile do not fit a 32-bit offset", MT);
  return dgrad_launch(gx, strips, lo, n, w, go, g, ws, ws_bytes, s, "jg_conv_dgrad_fold(mfma)", dtype);
}

}  // namespace jg
