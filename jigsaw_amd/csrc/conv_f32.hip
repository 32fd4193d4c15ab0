// 3 x 3 convolution of fp32 tensors (2-D, stride 1, dilation 1) on the fp32 matrix instruction, v_mfma_f32_16x16x4_f32:
// forward, input gradient (also split between the tile and the neighbours' strips) and weight gradient, channels-first
// tensors in and out, products and sums in fp32.
//
//   Forward     a workgroup of four wavefronts makes 8 rows x 64 columns of 16 MT produced channels, a wavefront two of the
//               rows. Eight channels of the 10 x 66 window and their weights sit in LDS at a time; the next eight channels'
//               window is on its way in registers meanwhile. A step is one tap of four channels: lane (n, q) holds channel
//               q of pixel n of a block of 16 pixels, straight from LDS at a constant offset from the lane's base. The planes are
//               720 floats apart, 16 beyond a multiple of 64, so that the four channels of a read lie on different banks.
//   Input grad. the same on the output gradient, weights transposed and reversed, padding 2 - p.
//   Weight grad the pixels are the contraction: g (16 MT channels) against 16 columns of (input channel, tap) a block, the
//               column behind the last tap is ones and gives the bias gradient. Lane (j, q) reads pixel q of its column at
//               the column's own offset into the window. Partials of every workgroup, added up by a second kernel in a
//               fixed order.
//
// Beside it, fp32 layers run as sums of three bf16 parts (conv_mfma.hip): a sixth of the bf16 rate, 0.4 PFLOP/s on paper against
// the 0.16 PFLOP/s of this instruction, but the parts are written and read, in launches of their own, and a step there is 16 channels of
// six products whatever the layer has. Batch 4, 3 -> 16 channels, 256^2 (that : this): forward 28 : 9.5 us, gradients of the
// weight and bias 46 : 10.5 and their sums beside the border cells, input gradient 55 : 13, 14 launches : 6. What bounds it there: latency, at one or two stages a workgroup;
// with many channels the instruction's rate: forward, 105 of 157 TFLOP/s at 8 x 64 -> 64, 512^2 (58 at 8 x 20 -> 20, 500^2, where 12 of a
// block's 32 produced channels do not exist). f32_conv_supported has the line
// between the two. Against float64 no result is further off than the three parts' (relative, 16 channels: y 1.9e-7 : 2.5e-7).
#include "conv_common.h"
#include "conv_reduce.h"

#include <algorithm>
#include <type_traits>

namespace {

using jg::ConvGeom;
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int THREADS = 256, WAVES = 4;
constexpr int TH = 8, TW = 64;                         // produced pixels of a workgroup
constexpr int IN_ROWS = TH + 2, IN_COLS = TW + 2;
constexpr int PITCH = 68, PLANE = 720;                 // floats of a row and of a channel's window in LDS
constexpr int CK = 8;                                  // channels of a stage
constexpr int X_ROWS = CK * IN_ROWS;                   // 80
constexpr int CH_PER_WAVE = CK / WAVES;                // 2
static_assert(IN_ROWS * PITCH <= PLANE && PLANE % 64 == 16 && CK % WAVES == 0 && X_ROWS * 2 <= THREADS, "staging layout");

struct Strips {
  void* p[27];
};

struct Params {
  const float* x;  // (N, C, H, W)
  const float* w;
  const float* bias;
  float* y;        // (N, M, Ho, Wo), or with a fold the tile (N, M, nH, nW)
  int N, C, M, H, W, Ho, Wo, pad_h, pad_w, tiles_h, tiles_w;
  jg::Div by_image, by_tw;  // tiles of an image, tile columns
  int transposed;
  int lo_h, lo_w, nH, nW;
};

// OUT_ROWS: one tensor. OUT_STREAM: one tensor whose rows are whole cache lines, stored past the L2 (a write stream of 537 MB:
// 221 -> 177 us; lines written by two rows lose by it, 250 -> 618 us). OUT_FOLD: each point to its owner.
enum Out { OUT_ROWS, OUT_STREAM, OUT_FOLD };

// SUMS: more than one stage; what a stage adds up goes to a second set of accumulators, so that no sum is longer than a stage's 72
// products and the number of stages.
// MT == 0: four produced channels, on v_mfma_f32_4x4x1_16b_f32, whose sixteen blocks are 64 pixels of a row times one channel of one tap: the
// 16 x 16 products waste the rows of the channels that do not exist, and with 3 of 16 they were 11 of the kernel's 28 us. A
// lane owns a pixel; the three tap rows have chains of their own (24 products each; relative error of 16 -> 3 channels 1.9e-7 -> 1.2e-7).
// Input gradient of 4 x 3 -> 16, 256^2 31.6 -> 13.4 us (with the staging below), forward of 2 x 60 -> 4, 200 x 100 46.0 -> 20.4.
template <int MT, Out OUT, bool SUMS>
__global__ __launch_bounds__(THREADS, MT == 2 ? 2 : (SUMS && MT != 0 ? 3 : 4)) void conv_f32_kernel(Strips strips, Params p) {
  constexpr bool FEW = MT == 0;
  constexpr int MC = FEW ? 4 : MT * 16;  // produced channels of a workgroup
  constexpr int W_FLOATS = CK * 9 * MC;
  __shared__ float lds_x[CK * PLANE];
  __shared__ float lds_w[W_FLOATS];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n16 = lane & 15, kq = lane >> 4;
  const int per_image = p.tiles_h * p.tiles_w;
  const int n = jg::quotient(blockIdx.x, p.by_image), t = blockIdx.x - n * per_image;
  const int th = jg::quotient(t, p.by_tw), tw = t - th * p.tiles_w;
  const int m0 = blockIdx.y * MC;
  const int y0 = th * TH - p.pad_h, x0 = tw * TW - p.pad_w;  // window origin
  const size_t plane = (size_t)p.H * p.W;
  const float* image = p.x + (size_t)n * p.C * plane;

  // Loads never stand under a condition (the compiler would wait for them where the paths meet): rows and columns outside are
  // read from the nearest place inside and cleared on their way to LDS.
  const int gx = x0 + lane, gxc = min(max(gx, 0), p.W - 1);
  const bool col_ok = gx >= 0 && gx < p.W;
  const int tail_row = min(tid >> 1, X_ROWS - 1), tail_col = TW + (tid & 1);
  const int tx = x0 + tail_col, txc = min(max(tx, 0), p.W - 1), ty = y0 + tail_row % IN_ROWS;
  const bool tail_ok = tid < 2 * X_ROWS && tx >= 0 && tx < p.W && ty >= 0 && ty < p.H;
  // A wavefront's rows are those of two channels of the stage: the places in LDS are constants, the two channels share their rows' offsets and
  // masks. (Rows dealt to the wavefronts in turn took a product and a test for each of twenty, twice a stage, and over 150 scalar
  // registers in spills: 3 -> 16 of 4 x 256^2 forward 12.3 -> 9.6 us, 16 -> 16 of 8 x 256^2 48.6 -> 40.6 and 58.8 -> 48.5 its gradient, 80 -> 6
  // of 2 x 256^2 86 -> 65.)
  float xr[CH_PER_WAVE][IN_ROWS], xt = 0.0f;
  auto issue = [&](int c0) {
    const float* chan[CH_PER_WAVE];
#pragma unroll
    for (int j = 0; j < CH_PER_WAVE; ++j) chan[j] = image + (size_t)min(c0 + wave * CH_PER_WAVE + j, p.C - 1) * plane;
#pragma unroll
    for (int r = 0; r < IN_ROWS; ++r) {
      const uint32_t off = (uint32_t)(min(max(y0 + r, 0), p.H - 1) * p.W + gxc);
#pragma unroll
      for (int j = 0; j < CH_PER_WAVE; ++j) xr[j][r] = chan[j][off];
    }
    const int c = c0 + tail_row / IN_ROWS;
    xt = image[(tail_ok && c < p.C ? (size_t)c * plane + (size_t)ty * p.W : 0) + txc];
  };
  auto store = [&](int c0) {
    float* const to = lds_x + wave * (CH_PER_WAVE * PLANE) + lane;
#pragma unroll
    for (int r = 0; r < IN_ROWS; ++r) {
      const bool row_ok = col_ok && y0 + r >= 0 && y0 + r < p.H;
#pragma unroll
      for (int j = 0; j < CH_PER_WAVE; ++j) to[j * PLANE + r * PITCH] = row_ok && c0 + wave * CH_PER_WAVE + j < p.C ? xr[j][r] : 0.0f;
    }
    if (tid < 2 * X_ROWS)
      lds_x[tail_row / IN_ROWS * PLANE + tail_row % IN_ROWS * PITCH + tail_col] = tail_ok && c0 + tail_row / IN_ROWS < p.C ? xt : 0.0f;
  };
  // Weights of a stage, [tap][channel][produced channels] in LDS. Fetched where they are stored; with 32 produced channels and several
  // stages on their way in registers beside the window's rows (14 -> 45 of 7 x 70 x 313 54.4 -> 51.5 us, 40 -> 24 of 2 x 100^2 37.1 -> 33.9): the others
  // spill or lose a wavefront's registers by it (3 -> 16 of 4 x 256^2 9.6 -> 12.3, 6 -> 80 of 2 x 256^2 26.5 -> 32.1).
  constexpr bool AHEAD = MT == 2 && SUMS;
  constexpr int W_ROUNDS = (W_FLOATS + THREADS - 1) / THREADS;
  float wr[W_ROUNDS];
  auto issue_weights = [&](int c0) {  // what does not exist is read from the last that does
#pragma unroll
    for (int e = 0; e < W_ROUNDS; ++e) {
      const int i = min(tid + e * THREADS, W_FLOATS - 1), m = min(m0 + i % MC, p.M - 1), k = i / MC, tap = k >> 3, c = min(c0 + (k & 7), p.C - 1);
      wr[e] = p.w[p.transposed ? ((size_t)c * p.M + m) * 9 + 8 - tap : ((size_t)m * p.C + c) * 9 + tap];
    }
  };
  auto store_weights = [&](int c0) {
#pragma unroll
    for (int e = 0; e < W_ROUNDS; ++e) {
      const int i = tid + e * THREADS;
      if (W_FLOATS % THREADS == 0 || i < W_FLOATS) lds_w[i] = m0 + i % MC < p.M && c0 + (i / MC & 7) < p.C ? wr[e] : 0.0f;
    }
  };
  auto weights = [&](int c0) {
    for (int i = tid; i < W_FLOATS; i += THREADS) {
      const int m = m0 + i % MC, k = i / MC, tap = k >> 3, c = c0 + (k & 7);
      float v = 0.0f;
      if (m < p.M && c < p.C) v = p.transposed ? p.w[((size_t)c * p.M + m) * 9 + 8 - tap] : p.w[((size_t)m * p.C + c) * 9 + tap];
      lds_w[i] = v;
    }
  };

  f32x4 acc[FEW ? 1 : MT][8], sum[SUMS && !FEW ? MT : 1][8];  // FEW: [row of the wavefront * 3 + tap row], sum [row]
#pragma unroll
  for (int mt = 0; mt < (FEW ? 1 : MT); ++mt) {
    f32x4 b = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int m = m0 + (FEW ? 0 : mt * 16 + 4 * kq) + i;
      if (p.bias != nullptr && m < p.M) b[i] = p.bias[m];
    }
#pragma unroll
    for (int nb = 0; nb < 8; ++nb) {
      acc[mt][nb] = FEW && nb % 3 != 0 ? f32x4{0.0f, 0.0f, 0.0f, 0.0f} : b;
      if (SUMS) sum[mt][nb] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    }
  }
  const bool live = th * TH + wave * 2 < p.Ho;
  const float* const xb = FEW ? lds_x + wave * 2 * PITCH + lane : lds_x + kq * PLANE + wave * 2 * PITCH + n16;
  const float* const wb = FEW ? lds_w + (lane & 3) : lds_w + kq * MC + n16;
  issue(0);
  if (AHEAD) issue_weights(0);
  for (int c0 = 0; c0 < p.C; c0 += CK) {
    if (c0 > 0) __syncthreads();
    store(c0);
    if (AHEAD) store_weights(c0);
    else weights(c0);
    __syncthreads();
    if (c0 + CK < p.C) {
      issue(c0 + CK);
      if (AHEAD) issue_weights(c0 + CK);
    }
    if (!live) continue;
    if constexpr (FEW) {
#pragma unroll 2
      for (int c = 0; c < CK && c0 + c < p.C; ++c) {
        float a[9], b[4][3];
#pragma unroll
        for (int tap = 0; tap < 9; ++tap) a[tap] = wb[(tap * CK + c) * MC];
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
          for (int kw = 0; kw < 3; ++kw) b[r][kw] = xb[c * PLANE + r * PITCH + kw];
#pragma unroll
        for (int kw = 0; kw < 3; ++kw)
#pragma unroll
          for (int q = 0; q < 6; ++q)
            acc[0][q] = __builtin_amdgcn_mfma_f32_4x4x1f32(a[q % 3 * 3 + kw], b[q / 3 + q % 3][kw], acc[0][q], 0, 0, 0);
      }
      if (SUMS) {
#pragma unroll
        for (int r = 0; r < 2; ++r) sum[0][r] += (acc[0][3 * r] + acc[0][3 * r + 1]) + acc[0][3 * r + 2];
#pragma unroll
        for (int q = 0; q < 6; ++q) acc[0][q] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
      }
      continue;
    }
    for (int cg = 0; cg < 2 && c0 + cg * 4 < p.C; ++cg) {
      const float* const xg = xb + cg * 4 * PLANE;
      const float* const wg = wb + cg * 4 * MC;
#pragma unroll
      for (int tap = 0; tap < 9; ++tap) {
        float a[FEW ? 1 : MT];
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) a[mt] = wg[tap * 8 * MC + mt * 16];
#pragma unroll
        for (int nb = 0; nb < 8; ++nb) {
          const float b = xg[(nb / 4 + tap / 3) * PITCH + nb % 4 * 16 + tap % 3];
#pragma unroll
          for (int mt = 0; mt < MT; ++mt) acc[mt][nb] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[mt], b, acc[mt][nb], 0, 0, 0);
        }
      }
    }
    if (SUMS) {
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int nb = 0; nb < 8; ++nb) {
          sum[mt][nb] += acc[mt][nb];
          acc[mt][nb] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        }
    }
  }
  if (!live) return;

  // lane (n16, kq), register i of block (mt, nb): channel m0 + 16 mt + 4 kq + i, pixel 16 (nb % 4) + n16 of row nb / 4. FEW: register i of
  // row nb is channel m0 + i of pixel `lane`
  auto region = [](int at, int lo, int size) { return at < lo ? 0 : (at < lo + size ? 1 : 2); };
#pragma unroll
  for (int nb = 0; nb < (FEW ? 2 : 8); ++nb) {
    const int oh = th * TH + wave * 2 + (FEW ? nb : nb / 4), ow = tw * TW + (FEW ? lane : nb % 4 * 16 + n16);
    if (oh >= p.Ho || ow >= p.Wo) continue;
    float* to = p.y;
    int eh = p.Ho, ew = p.Wo, ch = oh, cw = ow;
    if (OUT == OUT_FOLD) {  // to its owner (nowhere, if there is none)
      const int rh = region(oh, p.lo_h, p.nH), rw = region(ow, p.lo_w, p.nW);
      eh = rh == 0 ? p.lo_h : (rh == 1 ? p.nH : p.Ho - p.lo_h - p.nH);
      ew = rw == 0 ? p.lo_w : (rw == 1 ? p.nW : p.Wo - p.lo_w - p.nW);
      ch = oh - (rh == 0 ? 0 : (rh == 1 ? p.lo_h : p.lo_h + p.nH));
      cw = ow - (rw == 0 ? 0 : (rw == 1 ? p.lo_w : p.lo_w + p.nW));
      if (rh != 1 || rw != 1) {
#pragma unroll
        for (int s = 0; s < 9; ++s)
          if (s == rh * 3 + rw) to = static_cast<float*>(strips.p[9 + s]);
      }
      if (to == nullptr) continue;
    }
    const size_t step = (size_t)eh * ew;
    const int mq = FEW ? m0 : m0 + 4 * kq;
    float* at = to + ((size_t)n * p.M + mq) * step + (size_t)ch * ew + cw;
#pragma unroll
    for (int mt = 0; mt < (FEW ? 1 : MT); ++mt)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        if (mq + mt * 16 + i >= p.M) continue;
        // (`0 + v`: with a fold the sign of a zero is cleared, as the reference's scatter-add does)
        const float v = SUMS ? sum[mt][nb][i] : FEW ? (acc[0][3 * nb % 8][i] + acc[0][(3 * nb + 1) % 8][i]) + acc[0][(3 * nb + 2) % 8][i] : acc[mt][nb][i];
        if (OUT == OUT_STREAM) __builtin_nontemporal_store(v, at + (mt * 16 + i) * step);
        else at[(mt * 16 + i) * step] = OUT == OUT_FOLD ? v + 0.0f : v;
      }
  }
}

// ---- weight gradient
constexpr int FLUSH = 2;                    // see wgrad_f32_kernel
constexpr int GR = 4;                       // output rows of a tile
constexpr int GX_ROWS = GR + 2, GX_PLANE = GX_ROWS * PITCH;
constexpr int G_PLANE = GR * TW + 4;        // 4 beyond a multiple of 64: sixteen channels' four pixels on all banks

struct WgradParams {
  const float* x;
  const float* g;
  float* part;  // [block][slot][16 MT][columns]
  int N, C, M, H, W, Ho, Wo, pad_h, pad_w, tiles_h, tiles_w, ci_blocks;
  int total, per;  // tiles, and how many a workgroup takes
  jg::Div by_image, by_tw, by_ci;  // tiles of an image, tile columns, blocks of input channels
};

// NB blocks of 16 columns a wavefront, the rows of a tile split over RS groups of wavefronts. CI input channels: as many as
// the columns hold with one left for the bias.
template <int MT, int NB, int RS>
__global__ __launch_bounds__(THREADS) void wgrad_f32_kernel(WgradParams p) {
  constexpr int NW = WAVES / RS, COLS = NW * NB * 16, CI = (COLS - 1) / 9;
  constexpr int XROWS = CI * GX_ROWS, GPW = MT * 16, TAILS = (2 * XROWS + THREADS - 1) / THREADS;
  constexpr int CPW = (CI + WAVES - 1) / WAVES;  // input channels of a wavefront
  static_assert(GR == WAVES, "a wavefront takes one row of every g channel");
  __shared__ float lds_x[CI * GX_PLANE];
  __shared__ float lds_g[MT * 16 * G_PLANE];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n16 = lane & 15, kq = lane >> 4, wn = wave % NW, rs = wave / NW;
  const int co_block = jg::quotient(blockIdx.y, p.by_ci);
  const int ci0 = ((int)blockIdx.y - co_block * p.ci_blocks) * CI, co0 = co_block * (MT * 16);
  const size_t plane_x = (size_t)p.H * p.W, plane_g = (size_t)p.Ho * p.Wo;
  const int begin = min((int)blockIdx.x * p.per, p.total), end = min(begin + p.per, p.total);

  // A wavefront fetches the six rows of every fourth input channel and one row of every output channel: its rows' offsets and masks are
  // shared by the channels, whose addresses walk. (Rows dealt to the wavefronts in turn took a 64-bit product, two clamps and a test each,
  // 35 to 55 of them twice a tile: 85 to 433 scalar registers in spills. 4 x 3 -> 16, 256^2 13.4 -> 10.5 us, 8 x 16 -> 16, 256^2 89.9 -> 77.4,
  // 7 x 14 -> 45, 70 x 313 63.4 -> 55.0, 6 x 68 -> 13, 39 x 57 18.0 -> 13.0.)
  float xr[CPW][GX_ROWS], gr[GPW], xt[TAILS];
  struct At {
    int n, y0, x0, oh0, ow0;
  };
  auto where = [&](int tile) {
    const int per_image = p.tiles_h * p.tiles_w, n = jg::quotient(tile, p.by_image), t = tile - n * per_image;
    const int th = jg::quotient(t, p.by_tw), tw = t - th * p.tiles_w;
    return At{n, th * GR - p.pad_h, tw * TW - p.pad_w, th * GR, tw * TW};
  };
  auto issue = [&](const At& a) {
    const float* xi = p.x + (size_t)a.n * p.C * plane_x;
    const float* gi = p.g + (size_t)a.n * p.M * plane_g;
    const int gxc = min(max(a.x0 + lane, 0), p.W - 1), owc = min(a.ow0 + lane, p.Wo - 1);
    uint32_t off[GX_ROWS];
#pragma unroll
    for (int r = 0; r < GX_ROWS; ++r) off[r] = (uint32_t)(min(max(a.y0 + r, 0), p.H - 1) * p.W + gxc);
#pragma unroll
    for (int j = 0; j < CPW; ++j) {
      const float* const chan = xi + (size_t)min(ci0 + min(j * WAVES + wave, CI - 1), p.C - 1) * plane_x;
#pragma unroll
      for (int r = 0; r < GX_ROWS; ++r) xr[j][r] = chan[off[r]];
    }
    const float* chan = gi + (size_t)co0 * plane_g;
    const uint32_t at = (uint32_t)(min(a.oh0 + wave, p.Ho - 1) * p.Wo + owc);
#pragma unroll
    for (int i = 0; i < GPW; ++i) {
      gr[i] = chan[at];
      chan += co0 + i + 1 < p.M ? plane_g : 0;
    }
#pragma unroll
    for (int i = 0; i < TAILS; ++i) {
      const int e = min(i * THREADS + tid, 2 * XROWS - 1), r = e >> 1, c = min(ci0 + r / GX_ROWS, p.C - 1);
      const int y = min(max(a.y0 + r % GX_ROWS, 0), p.H - 1), x = min(max(a.x0 + TW + (e & 1), 0), p.W - 1);
      xt[i] = xi[(size_t)c * plane_x + (size_t)y * p.W + x];
    }
  };
  auto store = [&](const At& a) {
    const bool x_ok = a.x0 + lane >= 0 && a.x0 + lane < p.W, g_ok = a.ow0 + lane < p.Wo;
    float* const to = lds_x + wave * GX_PLANE + lane;
#pragma unroll
    for (int j = 0; j < CPW; ++j)
      if (CI % WAVES == 0 || j + 1 < CPW || j * WAVES + wave < CI) {
#pragma unroll
        for (int r = 0; r < GX_ROWS; ++r) to[j * (WAVES * GX_PLANE) + r * PITCH] = x_ok && a.y0 + r >= 0 && a.y0 + r < p.H ? xr[j][r] : 0.0f;
      }
    const bool row_ok = g_ok && a.oh0 + wave < p.Ho;
#pragma unroll
    for (int i = 0; i < GPW; ++i) lds_g[i * G_PLANE + wave * TW + lane] = row_ok ? gr[i] : 0.0f;
#pragma unroll
    for (int i = 0; i < TAILS; ++i) {
      const int e = i * THREADS + tid, r = e >> 1, y = a.y0 + r % GX_ROWS, x = a.x0 + TW + (e & 1);
      if (e < 2 * XROWS) lds_x[r / GX_ROWS * GX_PLANE + r % GX_ROWS * PITCH + TW + (e & 1)] = y >= 0 && y < p.H && x >= 0 && x < p.W ? xt[i] : 0.0f;
    }
  };

  // column j = 9 (input channel) + tap; the last one is ones
  const float* xb[NB];
  bool ones[NB];
#pragma unroll
  for (int nb = 0; nb < NB; ++nb) {
    const int j = (wn * NB + nb) * 16 + n16, c = min(j / 9, CI - 1), tap = j - j / 9 * 9;
    ones[nb] = j == CI * 9;
    xb[nb] = lds_x + c * GX_PLANE + (tap / 3) * PITCH + tap % 3 + kq + rs * (GR / RS) * PITCH;
  }
  const float* const gb = lds_g + n16 * G_PLANE + kq + rs * (GR / RS) * TW;
  // FLUSH products of the matrix instruction (four pixels each) are added up in fp32, those sums in double: the error stays that of
  // 4 FLUSH additions however many pixels there are.
  double total[MT][NB][4] = {};
  At now = where(min(begin, p.total - 1));
  issue(now);
  for (int tile = begin; tile < end; ++tile) {
    if (tile > begin) __syncthreads();
    store(now);
    __syncthreads();
    now = where(min(tile + 1, p.total - 1));
    issue(now);
#pragma unroll
    for (int r = 0; r < GR / RS; ++r)
#pragma unroll
      for (int s0 = 0; s0 < TW / 4; s0 += FLUSH) {
        f32x4 acc[MT][NB];
#pragma unroll
        for (int s = s0; s < s0 + FLUSH; ++s) {
          float a[MT], b[NB];
#pragma unroll
          for (int mt = 0; mt < MT; ++mt) a[mt] = gb[mt * 16 * G_PLANE + r * TW + 4 * s];
#pragma unroll
          for (int nb = 0; nb < NB; ++nb) {
            b[nb] = xb[nb][r * PITCH + 4 * s];
            b[nb] = ones[nb] ? 1.0f : b[nb];
          }
#pragma unroll
          for (int mt = 0; mt < MT; ++mt)
#pragma unroll
            for (int nb = 0; nb < NB; ++nb)
              acc[mt][nb] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[mt], b[nb], s == s0 ? f32x4{0.0f, 0.0f, 0.0f, 0.0f} : acc[mt][nb], 0, 0, 0);
        }
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
          for (int nb = 0; nb < NB; ++nb)
#pragma unroll
            for (int i = 0; i < 4; ++i) total[mt][nb][i] += (double)acc[mt][nb][i];
      }
  }
  const size_t slot = ((size_t)blockIdx.y * gridDim.x + blockIdx.x) * RS + rs;
  float* const out = p.part + slot * (MT * 16 * COLS) + 4 * kq * COLS + wn * NB * 16 + n16;
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
#pragma unroll
      for (int i = 0; i < 4; ++i) out[(mt * 16 + i) * COLS + nb * 16] = (float)total[mt][nb][i];
}

constexpr int REDUCE_THREADS = 64 * jg::CONV_RED_CHAINS;
__global__ __launch_bounds__(REDUCE_THREADS) void wgrad_f32_reduce_kernel(jg_conv_reduction p) {
  __shared__ jg::ConvReduceShared shared;
  jg::reduce_conv_f32<jg::CONV_RED_CHAINS>(p, blockIdx.x, shared);
}

// The weight gradient's blocks: input channels of a block, 16 MT output channels, workgroups of a block
struct Plan {
  int nb, rs, CI, MT, ci_blocks, co_blocks, cols, wgs, per, total, tiles_h, tiles_w;
  size_t bytes() const { return (size_t)ci_blocks * co_blocks * wgs * rs * MT * 16 * cols * sizeof(float); }
};
Plan plan_of(const ConvGeom& g) {
  Plan q;
  q.nb = g.cin > 7 ? 2 : 1;
  q.rs = g.cin > 3 ? 1 : (g.cin > 1 ? 2 : 4);
  q.cols = WAVES / q.rs * q.nb * 16;
  q.CI = (q.cols - 1) / 9;
  q.MT = g.cout > 16 ? 2 : 1;
  q.ci_blocks = (g.cin + q.CI - 1) / q.CI;
  q.co_blocks = (g.cout + q.MT * 16 - 1) / (q.MT * 16);
  q.tiles_h = (g.out[1] + GR - 1) / GR;
  q.tiles_w = (g.out[2] + TW - 1) / TW;
  q.total = (int)(g.batch * q.tiles_h * q.tiles_w);
  const int blocks = q.ci_blocks * q.co_blocks, want = std::max(1, 2 * jg::cu_count() / blocks);
  q.per = (q.total + want - 1) / want;
  q.wgs = (q.total + q.per - 1) / q.per;
  return q;
}

bool aligned4(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 3) == 0; }

int launch(Params p, const Strips& strips, bool fold, hipStream_t s, const char* who) {
  p.tiles_h = (p.Ho + TH - 1) / TH;
  p.tiles_w = (p.Wo + TW - 1) / TW;
  p.by_image = jg::div_by(p.tiles_h * p.tiles_w);
  p.by_tw = jg::div_by(p.tiles_w);
  const int MT = p.M > 16 ? 2 : p.M > 4 ? 1 : 0, MC = MT == 0 ? 4 : MT * 16;
  const dim3 grid((unsigned)(p.N * p.tiles_h * p.tiles_w), (unsigned)((p.M + MC - 1) / MC));
  auto pick = [&](auto out_c) -> void (*)(Strips, Params) {
    constexpr Out O = decltype(out_c)::value;
    if (p.C > CK) return MT == 2 ? &conv_f32_kernel<2, O, true> : MT == 1 ? &conv_f32_kernel<1, O, true> : &conv_f32_kernel<0, O, true>;
    return MT == 2 ? &conv_f32_kernel<2, O, false> : MT == 1 ? &conv_f32_kernel<1, O, false> : &conv_f32_kernel<0, O, false>;
  };
  void (*kern)(Strips, Params) = nullptr;
  if (fold) kern = pick(std::integral_constant<Out, OUT_FOLD>{});
  else if (p.Wo % 32 == 0) kern = pick(std::integral_constant<Out, OUT_STREAM>{});
  else kern = pick(std::integral_constant<Out, OUT_ROWS>{});
  kern<<<grid, THREADS, 0, s>>>(strips, p);
  JG_CHECK_LAUNCH(who);
  return JG_OK;
}

}  // namespace

namespace jg {

// Every direction of a layer has the same answer, so that none is less exact than the others.
bool f32_conv_supported(const ConvGeom& g, int dtype) {
  if (dtype != JG_F32 || g.groups != 1 || g.batch <= 0 || g.k[0] != 1 || g.in[0] != 1 || g.k[1] != 3 || g.k[2] != 3) return false;
  for (int a = 0; a < 3; ++a)
    if (g.s[a] != 1 || g.d[a] != 1 || g.p[a] > g.k[a] - 1 || g.out[a] < 1) return false;
  const long long tiles = g.batch * ((std::max(g.in[1], g.out[1]) + GR - 1) / GR) * ((std::max(g.in[2], g.out[2]) + TW - 1) / TW);
  if (tiles >= (1ll << 22) || (g.cin + 13) / 14 * ((g.cout + 15) / 16) >= 65536) return false;
  // Against sums of bf16 parts: the traced kernels of forward, weight and bias gradient and input gradient at padding 1, us (this : that).
  // Up to 16 channels on one side:
  //   4 x 3 -> 16, 256^2 36 : 122     8 x 16 -> 16, 512^2 547 : 780   2 x 12 -> 100, 150^2 120 : 219  8 x 3 -> 64, 512^2 534 : 1687
  //   8 x 16 -> 128, 256^2 918 : 956  8 x 128 -> 16, 256^2 772 : 972  but 4 x 15 -> 18, 512^2 418 : 396
  // and a layer whose workgroups are fewer than the compute units is bound by its launches, 6 here and 12 there, and by stages of which
  // a compute unit has one at a time. With 65 to 128 channels on one side (more have not been
  // measured) and up to 64 on the other that holds up to three workgroups for four compute units:
  //   2 x 24 -> 24, 200^2 100 : 137   1 x 64 -> 64, 100^2 132 : 159   1 x 64 -> 64, 180^2 168 : 183   2 x 48 -> 48, 150^2 158 : 174
  //   1 x 17 -> 65, 40^2 87 : 125     8 x 17 -> 80, 64^2 121 : 156    2 x 20 -> 70, 128^2 116 : 162   1 x 40 -> 80, 256 x 128 152 : 206
  //   2 x 127 -> 40, 48^2 160 : 201   2 x 48 -> 100, 64^2 147 : 192   4 x 40 -> 66, 48 x 90 130 : 195 1 x 64 -> 80, 128^2 157 : 184
  //   1 x 32 -> 128, 128^2 165 : 183
  // Beyond, their rate wins the more the larger the layer is; next to the line the two are within 14 % of each other:
  //   8 x 64 -> 64, 512^2 5308 : 3687 2 x 64 -> 64, 180^2 280 : 216   8 x 20 -> 20, 500^2 986 : 895   4 x 32 -> 32, 256^2 222 : 213
  //   4 x 20 -> 20, 300^2 218 : 222   8 x 28 -> 31, 300^2 455 : 477   4 x 17 -> 64, 256^2 279 : 299   1 x 96 -> 96, 128^2 207 : 223
  //   3 x 80 -> 128, 64^2 220 : 233   1 x 128 -> 17, 128 x 256 (256 workgroups) 175 : 198
  // Within the line the parts are faster in one direction or other: where 16 channels go into many more (they fill the parts' step; this
  // has two stages of 8), and in weight gradients that need a second block of columns here, 15 input channels and more (y, gw, gx):
  //   8 x 16 -> 128, 256^2 209 : 143, 485 : 482, 224 : 331            8 x 128 -> 16, 256^2 219 : 335, 352 : 497, 201 : 140
  //   4 x 15 -> 18, 512^2 99 : 102, 242 : 151, 78 : 143               2 x 48 -> 48, 150^2 42 : 58, 75 : 58, 41 : 58
  //   but 8 x 16 -> 16, 256^2 39 : 61, 74 : 87, 37 : 62               8 x 17 -> 80, 64^2 20 : 32, 42 : 45, 59 : 79
  // Those directions stay here too: the parts are less exact in all of them. Relative error against float64, 16 -> 128: y 1.6e-7 :
  // 2.5e-7, gw 6.4e-8 : 2.0e-7, input gradient of 128 from 16 1.6e-7 : 2.5e-7 (3 channels 0.94e-7 : 1.13e-7).
  const int few = std::min(g.cin, g.cout), many = std::max(g.cin, g.cout);
  const long long workgroups = g.batch * ((g.out[1] + TH - 1) / TH) * ((g.out[2] + TW - 1) / TW) * ((many + 31) / 32);
  return few <= 16 || (many <= 64 && workgroups <= cu_count()) || (few <= 64 && many <= 128 && 4 * workgroups <= 3ll * cu_count());
}

int f32_fwd(void* y, const void* x, const void* w, const void* bias, const ConvGeom& g, hipStream_t s) {
  Params p = {};
  p.x = static_cast<const float*>(x); p.w = static_cast<const float*>(w); p.bias = static_cast<const float*>(bias); p.y = static_cast<float*>(y);
  p.N = (int)g.batch; p.C = g.cin; p.M = g.cout; p.H = g.in[1]; p.W = g.in[2]; p.Ho = g.out[1]; p.Wo = g.out[2];
  p.pad_h = g.p[1]; p.pad_w = g.p[2];
  return launch(p, Strips{}, false, s, "jg_conv_fwd(fp32)");
}

int f32_dgrad(void* gx, void* const* strips, const int* lo, const int* n, const void* w, const void* go, const ConvGeom& g, hipStream_t s) {
  Params p = {};
  p.x = static_cast<const float*>(go); p.w = static_cast<const float*>(w); p.y = static_cast<float*>(gx);
  p.N = (int)g.batch; p.C = g.cout; p.M = g.cin; p.H = g.out[1]; p.W = g.out[2]; p.Ho = g.in[1]; p.Wo = g.in[2];
  p.pad_h = 2 - g.p[1]; p.pad_w = 2 - g.p[2];
  p.transposed = 1;
  Strips tab = {};
  if (lo != nullptr) {
    for (int i = 0; i < 27; ++i) tab.p[i] = strips[i];
    p.lo_h = lo[1]; p.lo_w = lo[2]; p.nH = n[1]; p.nW = n[2];
  }
  return launch(p, tab, lo != nullptr, s, "jg_conv_dgrad(fp32)");
}

size_t f32_wgrad_workspace(const ConvGeom& g) { return plan_of(g).bytes(); }

int f32_wgrad(void* gw, void* gb, const void* x, const void* go, const ConvGeom& g, void* ws, size_t ws_bytes, hipStream_t s,
              jg_conv_reduction* later) {
  const char* who = "jg_conv_wgrad(fp32)";
  const Plan q = plan_of(g);
  if (ws == nullptr || ws_bytes < q.bytes()) JG_FAIL(JG_ERR_WORKSPACE, "%s: workspace %zu < %zu bytes", who, ws_bytes, q.bytes());
  JG_REQUIRE(aligned4(ws), "%s: workspace must be 4-byte aligned", who);
  WgradParams p = {};
  p.x = static_cast<const float*>(x); p.g = static_cast<const float*>(go); p.part = static_cast<float*>(ws);
  p.N = (int)g.batch; p.C = g.cin; p.M = g.cout; p.H = g.in[1]; p.W = g.in[2]; p.Ho = g.out[1]; p.Wo = g.out[2];
  p.pad_h = g.p[1]; p.pad_w = g.p[2]; p.tiles_h = q.tiles_h; p.tiles_w = q.tiles_w; p.ci_blocks = q.ci_blocks;
  p.total = q.total; p.per = q.per;
  p.by_image = div_by(q.tiles_h * q.tiles_w);
  p.by_tw = div_by(q.tiles_w);
  p.by_ci = div_by(q.ci_blocks);
  const int blocks = q.ci_blocks * q.co_blocks;
  const dim3 grid((unsigned)q.wgs, (unsigned)blocks);
  void (*kern)(WgradParams) = nullptr;
  if (q.nb == 2) kern = q.MT == 2 ? &wgrad_f32_kernel<2, 2, 1> : &wgrad_f32_kernel<1, 2, 1>;
  else if (q.rs == 1) kern = q.MT == 2 ? &wgrad_f32_kernel<2, 1, 1> : &wgrad_f32_kernel<1, 1, 1>;
  else if (q.rs == 2) kern = q.MT == 2 ? &wgrad_f32_kernel<2, 1, 2> : &wgrad_f32_kernel<1, 1, 2>;
  else kern = q.MT == 2 ? &wgrad_f32_kernel<2, 1, 4> : &wgrad_f32_kernel<1, 1, 4>;
  kern<<<grid, THREADS, 0, s>>>(p);
  JG_CHECK_LAUNCH(who);
  jg_conv_reduction r = {};
  r.kind = CONV_REDUCE_F32;
  r.dtype = JG_F32;
  r.part = p.part; r.gw = gw; r.gb = gb;
  r.slots = q.wgs * q.rs; r.rows = q.MT * 16; r.cols = q.cols; r.ci_step = q.CI; r.ci_blocks = q.ci_blocks;
  r.cin = g.cin; r.cout = g.cout;
  r.runs = blocks * (r.rows * q.cols / CONV_F32_VALUES);
  if (later == nullptr) return f32_reduce(r, s);
  *later = r;
  return JG_OK;
}

int f32_reduce(const jg_conv_reduction& r, hipStream_t s) {
  wgrad_f32_reduce_kernel<<<conv_reduce_blocks(r), REDUCE_THREADS, 0, s>>>(r);
  JG_CHECK_LAUNCH("jg_conv_wgrad(fp32 reduce)");
  return JG_OK;
}

}  // namespace jg
