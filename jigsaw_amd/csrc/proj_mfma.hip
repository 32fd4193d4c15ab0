// Token projections around the attention core, with the head split / head merge done
// by the addressing of the GEMM instead of by a copy.
//
// Reference behaviour restated here (jigsaw/modules/attention/_attention.py:881-918):
//   qkv = self.qkv(x)                                   (rows, C) x (3 h d, C)^T + bias
//   rearrange(qkv, "... n s (three h d) -> three ... n h s d")
//   out = attn_core(q, k, v)                            (..., h, s, d)
//   rearrange(out, "... n h s d -> ... n s (h d)").contiguous(); self.head_concat(out)
//
// A matrix operand or result with rows = tokens and columns = features is addressed
// through a Map: either row-major (row * ld + feature), or "heads": the tensor is
// (t, B, H, S, D), token = b * S + s, feature = (t * H + h) * D + d. In both cases
// the element offset is row_part(token) + feat_part(feature), and 8 consecutive
// features starting at a multiple of 8 are contiguous (D % 8 == 0).
//
//   proj_nt_kernel   out(r, n) = sum_k a(r, k) * w[n][k] + bias[n]      (forward, and the
//                    input gradients with the transposed weight)
//   proj_tn_kernel   part[split](n, c) = sum_{r in split} g(r, n) * x(r, c)   (weight gradient;
//                    bias gradient sum_r g(r, n) on the way), then proj_reduce_kernel
//
// bf16 on v_mfma_f32_32x32x16_bf16 with fp32 accumulation. Workgroup tiles of 256 x 256 and 128 x 128 (eight wavefronts)
// and, NT, 64 x 64 (four); the operands travel from memory straight into LDS, 64 contraction elements a stage, one
// stage ahead of the MFMAs.
// proj_generic_kernel covers the other dtypes and unaligned shapes with plain FMAs.
#include <algorithm>
#include <type_traits>

#include "lds_transfer.h"
#include "reductions.h"

namespace {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));

using jg::Div;
using jg::div_by;
using jg::quotient;

struct Map {
  int heads;     // 0: row-major with leading dimension ld; 1: (t, B, H, S, D)
  long long ld;
  int B, H, S, D;
  Div by_S, by_D, by_H;
};

__device__ __forceinline__ long long row_part(const Map& m, long long r) {
  if (!m.heads) return r * m.ld;
  const long long b = r / m.S, s = r - b * m.S;
  return (b * m.H * m.S + s) * m.D;
}
__device__ __forceinline__ long long feat_part(const Map& m, int j) {
  if (!m.heads) return j;
  const int hd = j / m.D, d = j - hd * m.D;
  const int t = hd / m.H, h = hd - t * m.H;
  return ((long long)t * m.B * m.H + h) * m.S * m.D + d;
}

// The same as byte offsets, of tokens and features below 2^31. OFF: uint32_t where the tensor has fewer than 2^32 bytes.
template <typename OFF>
__device__ __forceinline__ OFF row_bytes(const Map& m, uint32_t r) {
  if (!m.heads) return (OFF)r * (OFF)m.ld * 2u;
  const uint32_t b = quotient(r, m.by_S), s = r - b * (uint32_t)m.S;
  return ((OFF)b * (OFF)m.H * (OFF)m.S + s) * (OFF)m.D * 2u;
}
template <typename OFF>
__device__ __forceinline__ OFF feat_bytes(const Map& m, uint32_t j) {
  if (!m.heads) return (OFF)j * 2u;
  const uint32_t hd = quotient(j, m.by_D), t = quotient(hd, m.by_H), d = j - hd * (uint32_t)m.D, h = hd - t * (uint32_t)m.H;
  return (((OFF)t * (OFF)m.B * (OFF)m.H + h) * (OFF)m.S * (OFF)m.D + d) * 2u;
}

// Tokens r, r + step, ... of a tensor as byte offsets; heads: (b * H * S + s) * D, row-major: r * ld.
template <typename OFF>
struct TokenWalk {
  OFF off;         // bytes
  int s, S;        // position in the batch entry and its length
  OFF row, jump;   // bytes between tokens of an entry; extra bytes from the end of an entry to the next one
  __device__ __forceinline__ void start(const Map& m, long long r) {
    row = (OFF)(m.heads ? m.D : m.ld) * 2u;
    S = m.heads ? m.S : 0x7fffffff;
    jump = m.heads ? (OFF)(m.H - 1) * (OFF)m.S * row : 0u;
    const long long b = !m.heads ? 0 : r < (1ll << 31) ? (long long)quotient((uint32_t)r, m.by_S) : r / m.S;
    s = m.heads ? (int)(r - b * m.S) : 0;
    off = m.heads ? ((OFF)b * (OFF)m.H * (OFF)m.S + (OFF)s) * row : (OFF)r * row;
  }
  __device__ __forceinline__ void advance(int by) {
    s += by;
    off += (OFF)by * row;
    if (S >= by) {  // wave-uniform: one entry further at most
      const bool over = s >= S;
      s -= over ? S : 0;
      off += over ? jump : (OFF)0;
    } else {
      while (s >= S) {
        s -= S;
        off += jump;
      }
    }
  }
};


// ------------------------------------------------------------------------ NT
constexpr int BK = 64;  // contraction elements per stage

struct NtParams {
  const uint16_t* a;
  const uint16_t* w;     // (N, K) row-major
  const uint16_t* bias;  // (N,) or NULL
  uint16_t* out;
  Map am, om;
  long long rows;
  int N, K;
  int tiles_n, tiles;
  Div by_tiles_n;
  // What happens to a result on its way out (the values are the bf16-rounded acc + bias, as a
  // separate elementwise pass over the stored tensor would see them; arithmetic in fp32):
  //   EPI_NONE  out = y
  //   EPI_GELU  out = y, aux = gelu(y)                (aux is written)
  //   EPI_DGELU out = y * gelu'(aux)                  (aux is read: the saved pre-activation)
  //   EPI_ADD   out = y + aux                         (aux is read: the residual)
  // aux has the layout of out.
  int epi;
  uint16_t* aux;
};
constexpr int EPI_NONE = 0, EPI_GELU = 1, EPI_DGELU = 2, EPI_ADD = 3;

// GELU in its erf form (torch.nn.GELU's default) and its derivative. (1 + erf(z)) / 2 with z = h / sqrt 2 from
// the rational approximation 7.1.26 of Abramowitz & Stegun, erfc |z| = p(t) exp(-z^2), t = 1 / (1 + 0.3275911 |z|),
// absolute error below 1.5e-7 (the results are rounded to 16 bits): one reciprocal, one exponential and
// five multiply-adds where the library's erff took the epilogue of the MLP's two fused GEMMs most of
// their time. Negative z takes erfc |z| / 2 directly, so the small values there keep their relative accuracy;
// exp(-z^2) = exp(-h^2 / 2) is also what the derivative's density term needs.
__device__ __forceinline__ float half_one_plus_erf(float h, float* density_exp) {
  const float az = __builtin_fabsf(h) * 0.70710678118654752f;
  const float t = __builtin_amdgcn_rcpf(__builtin_fmaf(0.3275911f, az, 1.0f));
  float poly = __builtin_fmaf(1.061405429f, t, -1.453152027f);
  poly = __builtin_fmaf(poly, t, 1.421413741f);
  poly = __builtin_fmaf(poly, t, -0.284496736f);
  poly = __builtin_fmaf(poly, t, 0.254829592f);
  const float e = __expf(-az * az);
  const float half_erfc = 0.5f * poly * t * e;
  *density_exp = e;
  return h >= 0.0f ? 1.0f - half_erfc : half_erfc;
}
__device__ __forceinline__ float gelu_f(float h) {
  float e;
  return h * half_one_plus_erf(h, &e);
}
__device__ __forceinline__ float dgelu_f(float h) {
  float e;
  const float cdf = half_one_plus_erf(h, &e);
  return __builtin_fmaf(h * 0.3989422804014327f, e, cdf);
}
// op on 8 bf16 values packed in 16 bytes (second operand optional)
template <typename F>
__device__ __forceinline__ u32x4 map8(u32x4 y, u32x4 r, F f) {
  uint32_t yy[4] = {y.x, y.y, y.z, y.w}, rr[4] = {r.x, r.y, r.z, r.w}, oo[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const f32x2 v = {f(__uint_as_float(yy[i] << 16), __uint_as_float(rr[i] << 16)),
                     f(__uint_as_float(yy[i] & 0xffff0000u), __uint_as_float(rr[i] & 0xffff0000u))};
    oo[i] = __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2));
  }
  return u32x4{oo[0], oo[1], oo[2], oo[3]};
}

// ------------------------------------------------- memory -> LDS, both GEMMs
// jg::to_lds_1k: 32-bit offsets where the host's check of the tensor sizes allows them, else 64-bit ones. One wait and one barrier per stage.
__device__ __forceinline__ void transfers_landed() { __builtin_amdgcn_s_waitcnt(0x0F70); }  // vmcnt(0)

// Shape of a workgroup: WM x WN wavefronts, each with IM x JN blocks of 32 tokens x 32 features.
template <int IM, int JN, int WM, int WN>
struct NtShape {
  static constexpr int TM = 32 * IM * WM, TNF = 32 * JN * WN;  // tokens, features of a tile
  static constexpr int WAVES = WM * WN, THREADS = 64 * WAVES;
  static constexpr int ROWB = BK * 2;                          // bytes of a row of a stage: 8 chunks of 8 k, chunk c at c ^ (row / 2 % 8)
  static constexpr int OP_A = TM * ROWB, OP_W = TNF * ROWB, STAGE = OP_A + OP_W;
  static constexpr int LDS = 2 * STAGE + 2 * TNF * 4;          // two stages, then the bias of two tiles as floats
  static constexpr int DMA_A = TM / 8 / WAVES, DMA_W = TNF / 8 / WAVES;  // 1 KB transfers (8 rows) of a wavefront per stage
  static constexpr int OUT_PITCH = 32 * JN * 2 + 16;           // bytes per token of a wavefront's block in LDS
  static_assert(TM % (8 * WAVES) == 0 && TNF % (8 * WAVES) == 0, "whole transfers");
  static_assert(WAVES % 2 == 0, "a wavefront's transfers start at the same row % 16");
  static_assert(32 * OUT_PITCH * WAVES <= STAGE, "the results pass through the stage just computed");
};

// Persistent workgroups walk the tiles of one XCD's contiguous range (consecutive tiles share a panel of `a`, which
// meets in one L2). The transfers of a stage are issued a stage ahead, across tile borders too, so that the first
// stage of a tile arrives under the last one of the tile before and under its epilogue: with K = 512 a tile is only
// eight stages long. A stage of the 256 x 256 tile is 2048 cycles of matrix instructions and takes 3300: the rest are the barrier, where
// wavefronts wait 550 for the last one, and what precedes the first matrix instruction behind it. What the vector unit does there and between
// tiles counts in full: offsets by the compiler's divisions were 0.7 to 1.1 us a tile (0.35 by Div), the epilogue's by 64-bit products 1.3
// (0.8). The 128 x 128 tile as eight wavefronts of 64 x 32 has two to a SIMD and, with a second workgroup, four (four of 64 x 64
// before: 0.75 us a stage, 0.55 now). us before -> now: 32768 tokens, 512 -> 1536 features 59.7 -> 57.6 (894 TFLOP/s), 1536 -> 512 52.7 -> 49.5,
// 512 -> 512 24.0 -> 22.7; 65536, 128 -> 384 19.4 -> 17.5; 2680, 896 -> 896 15.5 -> 12.2, 468, 2112 -> 704 17.1 -> 14.8.
template <int IM, int JN, int WM, int WN>
__global__ __launch_bounds__(64 * WM * WN, IM * JN >= 8 ? 1 : 2) void proj_nt_kernel(NtParams p) {
  typedef NtShape<IM, JN, WM, WN> SH;
  constexpr int TM = SH::TM, TNF = SH::TNF, ROWB = SH::ROWB;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  float* lds_bias = reinterpret_cast<float*>(smem + 2 * SH::STAGE);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int ln = lane & 31, kg = lane >> 5;
  const int wm = wave % WM, wn = wave / WM;
  const int wave_u = __builtin_amdgcn_readfirstlane(wave);

  // tiles of this workgroup (the grid is a multiple of 8)
  const int per_xcd = (p.tiles + 7) >> 3, wg_per_xcd = gridDim.x >> 3;
  const int t_begin = (blockIdx.x & 7) * per_xcd, slot = blockIdx.x >> 3;
  const int t_len = min(per_xcd, p.tiles - t_begin);
  if (slot >= t_len) return;
  const int my_tiles = (t_len - slot + wg_per_xcd - 1) / wg_per_xcd;
  auto tile_at = [&](int i) { return t_begin + slot + i * wg_per_xcd; };

  // ---- load cursor. Lane L of a transfer sits at row L / 8, chunk position L % 8, and fetches chunk
  // (L % 8) ^ (row / 2 % 8), the same one in every transfer (they are 16 rows or a multiple of it apart).
  const int chunk = (lane & 7) ^ ((wave & 1) << 2 | lane >> 4);
  uint32_t a_row[SH::DMA_A], w_row[SH::DMA_W];
  int ld_tile = -1, ld_ks = 0;
  uint16_t bias_next = 0;  // raw: converted when it goes to LDS, a use here would wait for the load
  const int nk = (p.K + BK - 1) / BK;
  auto enter_tile = [&]() {
    ++ld_tile;
    ld_ks = 0;
    const uint32_t t = tile_at(ld_tile), tm = quotient(t, p.by_tiles_n);
    const int n0 = (t - tm * p.tiles_n) * TNF;
#pragma unroll
    for (int i = 0; i < SH::DMA_A; ++i)  // a row past the end repeats the last one and is dropped
      a_row[i] = row_bytes<uint32_t>(p.am, min(tm * TM + (i * SH::WAVES + wave) * 8 + (lane >> 3), (uint32_t)p.rows - 1));
#pragma unroll
    for (int i = 0; i < SH::DMA_W; ++i) {
      const int n = min(n0 + (i * SH::WAVES + wave) * 8 + (lane >> 3), p.N - 1);
      w_row[i] = (uint32_t)n * (uint32_t)p.K * 2u;
    }
    if (p.bias != nullptr) bias_next = p.bias[min(n0 + tid, p.N - 1)];  // features past the end are dropped
  };
  const uint32_t lds_a = jg::lds_address(smem) + wave_u * 1024, lds_w = lds_a + SH::OP_A;
  uint32_t fa = 0, fw = 0;  // where the stage to fetch lies in a row
  auto enter_stage = [&]() {
    const int k = ld_ks * BK + chunk * 8;
    const int kk = k < p.K ? k : 0;  // a chunk past the contraction length is read at k = 0 and zeroed below
    fa = feat_bytes<uint32_t>(p.am, kk);
    fw = (uint32_t)kk * 2u;
  };
  constexpr int TRANSFERS = SH::DMA_A + SH::DMA_W;
  auto transfer = [&](int q, int buf) __attribute__((always_inline)) {
    if (q < SH::DMA_A) jg::to_lds_1k(p.a, a_row[q] + fa, lds_a + buf * SH::STAGE + q * SH::WAVES * 1024);
    else jg::to_lds_1k(p.w, w_row[q - SH::DMA_A] + fw, lds_w + buf * SH::STAGE + (q - SH::DMA_A) * SH::WAVES * 1024);
  };
  auto issue = [&](int buf) {
    enter_stage();
#pragma unroll
    for (int q = 0; q < TRANSFERS; ++q) transfer(q, buf);
  };
  // the last stage of a contraction length that is no multiple of BK: a lane clears what its transfers put past it
  auto clear_tail = [&](int buf, int ks) {
    if (ks * BK + chunk * 8 >= p.K) {
      u32x4* at = reinterpret_cast<u32x4*>(smem + buf * SH::STAGE + wave * 1024 + lane * 16);
#pragma unroll
      for (int i = 0; i < SH::DMA_A + SH::DMA_W; ++i) at[i * SH::WAVES * 64] = u32x4{0u, 0u, 0u, 0u};
    }
  };

  f32x16 acc[IM][JN];
  // acc[i][j] = w fragment (rows: features) x a fragment (columns: tokens). The fragments of
  // a 16-wide step are requested AHEAD steps before its MFMAs are issued.
  constexpr int AHEAD = IM * JN == 1 ? BK / 16 : IM * JN <= 4 ? 2 : 1;
  constexpr bool SPREAD = IM * JN > 1;
  constexpr int EVERY = IM * JN >= 8 ? 2 : 1;
  static_assert(EVERY * TRANSFERS <= BK / 16 * IM * JN, "every transfer has its place");
  // The transfers of a stage to come (buffer `to`, none: -1) go out one by one between them: eight wavefronts' 64 at the head of
  // a stage occupied the address unit for 1000 cycles in which no matrix instruction was issued.
  auto compute = [&](int buf, int to) {
    const unsigned char* sa = smem + buf * SH::STAGE + (wm * 32 * IM + ln) * ROWB;
    const unsigned char* sw = smem + buf * SH::STAGE + SH::OP_A + (wn * 32 * JN + ln) * ROWB;
    u32x4 fr[AHEAD + 1][IM + JN];
    auto fetch = [&](int kk, u32x4 (&f)[IM + JN]) {
      const int at = ((kk * 2 + kg) ^ ((ln >> 1) & 7)) << 4;
#pragma unroll
      for (int t = 0; t < IM; ++t) f[t] = *reinterpret_cast<const u32x4*>(sa + t * 32 * ROWB + at);
#pragma unroll
      for (int t = 0; t < JN; ++t) f[IM + t] = *reinterpret_cast<const u32x4*>(sw + t * 32 * ROWB + at);
    };
#pragma unroll
    for (int kk = 0; kk < AHEAD; ++kk) fetch(kk, fr[kk]);
#pragma unroll
    for (int kk = 0; kk < BK / 16; ++kk) {
      if (kk + AHEAD < BK / 16) fetch(kk + AHEAD, fr[(kk + AHEAD) % (AHEAD + 1)]);
      const u32x4(&f)[IM + JN] = fr[kk % (AHEAD + 1)];
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < IM; ++i)
#pragma unroll
        for (int j = 0; j < JN; ++j) {
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, f[IM + j]), __builtin_bit_cast(bf16x8, f[i]), acc[i][j], 0, 0, 0);
          const int at = (kk * IM + i) * JN + j;
          if (SPREAD && at % EVERY == EVERY - 1 && at / EVERY < TRANSFERS) {
            __builtin_amdgcn_sched_barrier(0);
            if (to >= 0) transfer(at / EVERY, to);
            __builtin_amdgcn_sched_barrier(0);
          }
        }
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  // Accumulator lane (ln, kg), register e of block (i, j): feature (wn*JN + j)*32 + 8*(e/4) +
  // 4*kg + e%4, token (wm*IM + i)*32 + ln. The sums start from the bias.
  auto init_acc = [&](int parity) {
    const float* b = lds_bias + parity * TNF + wn * JN * 32 + kg * 4;
#pragma unroll
    for (int j = 0; j < JN; ++j)
#pragma unroll
      for (int e4 = 0; e4 < 4; ++e4) {
        const f32x4 bq = *reinterpret_cast<const f32x4*>(b + j * 32 + e4 * 8);
#pragma unroll
        for (int i = 0; i < IM; ++i)
#pragma unroll
          for (int e = 0; e < 4; ++e) acc[i][j][e4 * 4 + e] = bq[e];
      }
  };
  // A wavefront's 32 tokens x 32 JN features pass through its slice of the stage just computed as bf16
  // [token][feature] and leave in 16-byte pieces of 8 features, whole rows of 64 JN bytes at a time.
  // What is read there (a residual, a saved pre-activation) is asked for a block of 32 tokens ahead: asked for where it
  // is used, every piece waited for the memory and for the stores issued before it (READS, see NtParams::epi).
  // y * gelu'(aux): 65536 tokens, 256 -> 1024 features 117 -> 102 us, 512 -> 2048 274 -> 240, 250000 of 128 -> 512 198 -> 157.
  auto epilogue = [&](int t, int buf, auto reads) __attribute__((always_inline)) {
    constexpr bool READS = decltype(reads)::value;
    unsigned char* block = smem + buf * SH::STAGE + wave * 32 * SH::OUT_PITCH;
    constexpr int CPR = JN * 4, RPI = 64 / CPR;  // pieces per token, tokens per store instruction
    const int fc = lane % CPR, trow = lane / CPR;
    const uint32_t tm = quotient(t, p.by_tiles_n);
    const int n = (t - tm * p.tiles_n) * TNF + wn * 32 * JN + fc * 8;
    const long long r0 = (long long)tm * TM + wm * 32 * IM + trow;
    const int left = n < p.N ? (int)min(p.rows - r0, (long long)TM) : 0;  // tokens from r0 on
    TokenWalk<uint64_t> out_at, ahead;
    out_at.start(p.om, r0);
    out_at.off += feat_bytes<uint64_t>(p.om, n < p.N ? n : 0);
    ahead = out_at;
    const char* const aux = reinterpret_cast<const char*>(p.aux);
    u32x4 saved[2][32 / RPI];
    auto fetch = [&](int i, u32x4 (&to)[32 / RPI]) __attribute__((always_inline)) {
#pragma unroll
      for (int q = 0; q < 32 / RPI; ++q) {
        to[q] = *reinterpret_cast<const u32x4*>(aux + (i * 32 + RPI * q < left ? ahead.off : 0));  // what is not there is not used either
        ahead.advance(RPI);
      }
    };
    if (READS) fetch(0, saved[0]);
#pragma unroll
    for (int i = 0; i < IM; ++i) {
      if (READS && i + 1 < IM) fetch(i + 1, saved[(i + 1) & 1]);
#pragma unroll
      for (int j = 0; j < JN; ++j)
#pragma unroll
        for (int e4 = 0; e4 < 4; ++e4) {
          const f32x2 lo = {acc[i][j][e4 * 4 + 0], acc[i][j][e4 * 4 + 1]}, hi = {acc[i][j][e4 * 4 + 2], acc[i][j][e4 * 4 + 3]};
          u32x2 pk;
          pk.x = __builtin_bit_cast(uint32_t, __builtin_convertvector(lo, bf16x2));
          pk.y = __builtin_bit_cast(uint32_t, __builtin_convertvector(hi, bf16x2));
          *reinterpret_cast<u32x2*>(block + ln * SH::OUT_PITCH + (j * 32 + e4 * 8 + kg * 4) * 2) = pk;
        }
      u32x4 piece[32 / RPI];
#pragma unroll
      for (int q = 0; q < 32 / RPI; ++q)
        piece[q] = *reinterpret_cast<const u32x4*>(block + (trow + RPI * q) * SH::OUT_PITCH + fc * 16);
#pragma unroll
      for (int q = 0; q < 32 / RPI; ++q) {
        if (i * 32 + RPI * q < left) {
          u32x4 y = piece[q];
          if (READS) {
            if (p.epi == EPI_DGELU) y = map8(y, saved[i & 1][q], [](float g, float h) { return g * dgelu_f(h); });
            else y = map8(y, saved[i & 1][q], [](float a, float b) { return a + b; });
          } else if (p.epi == EPI_GELU) {
            *reinterpret_cast<u32x4*>(reinterpret_cast<char*>(p.aux) + out_at.off) = map8(y, y, [](float h, float) { return gelu_f(h); });
          }
          *reinterpret_cast<u32x4*>(reinterpret_cast<char*>(p.out) + out_at.off) = y;
        }
        out_at.advance(RPI);
      }
    }
  };

  const bool tail = p.K % BK != 0;
  // the next stage of the stream, over the end of a tile too
  auto advance = [&]() {
    if (++ld_ks < nk) return true;
    if (ld_tile + 1 == my_tiles) return false;
    enter_tile();
    return true;
  };
  enter_tile();
  issue(0);
  bool more = true;
  int buf = 0;
  for (int ti = 0; ti < my_tiles; ++ti) {
    for (int ks = 0; ks < nk; ++ks) {
      transfers_landed();
      if (tail && ks == nk - 1) clear_tail(buf, ks);
      if (ks == 0 && tid < TNF) lds_bias[(ti & 1) * TNF + tid] = jg::bf16_to_f32(bias_next);
      __syncthreads();  // stage ks is in LDS, and every wavefront is done with the other buffer
      if (ks == 0) init_acc(ti & 1);
      if (more && (more = advance())) {
        if (SPREAD) enter_stage();
        else issue(buf ^ 1);
      }
      compute(buf, SPREAD && more ? buf ^ 1 : -1);
      buf ^= 1;
    }
    __syncthreads();  // the other wavefronts are done with the stage the results pass through
    if (p.epi >= EPI_DGELU) epilogue(tile_at(ti), buf ^ 1, std::true_type{});
    else epilogue(tile_at(ti), buf ^ 1, std::false_type{});
  }
}

template <int IM, int JN, int WM, int WN>
int launch_nt(NtParams& p, hipStream_t s, const char* who) {
  typedef NtShape<IM, JN, WM, WN> SH;
  p.tiles_n = jg::cdiv(p.N, SH::TNF);
  p.by_tiles_n = div_by(p.tiles_n);
  const long long tiles = (long long)jg::cdiv(p.rows, SH::TM) * p.tiles_n;
  JG_REQUIRE(tiles < (1ll << 30), "%s: too many tiles", who);
  p.tiles = (int)tiles;
  void (*kern)(NtParams) = &proj_nt_kernel<IM, JN, WM, WN>;
  if (hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, SH::LDS) != hipSuccess)
    JG_FAIL(JG_ERR_LAUNCH, "%s: cannot reserve %d bytes of LDS", who, SH::LDS);
  // as many workgroups as fit at once (a multiple of 8: one share per XCD)
  const long long fit = (long long)jg::cu_count() * (160 * 1024 / SH::LDS);
  const unsigned grid = (unsigned)(((tiles < fit ? tiles : fit) + 7) / 8 * 8);
  kern<<<grid, SH::THREADS, SH::LDS, s>>>(p);
  JG_CHECK_LAUNCH(who);
  return JG_OK;
}

// ------------------------------------------------------------------------ TN
constexpr int BR = 64;  // tokens per stage

struct TnParams {
  const uint16_t* g;  // tokens x N
  const uint16_t* x;  // tokens x C
  float* part;        // [split][N][C]
  float* bias_part;   // [split][N] or NULL
  Map gm, xm;
  long long rows;
  int N, C;
  int tiles_c, tiles;  // column tiles, all tiles; a workgroup is split * tiles + tile_n * tiles_c + tile_c
  Div by_tiles_c, by_tiles;
  int stages_per_split;
};

// WM x WN wavefronts, each with IM x JN blocks of 32 features of g x 32 features of x; the tile is square (T x T).
template <int IM, int JN, int WM, int WN>
struct TnShape {
  static constexpr int T = 32 * IM * WM;
  static_assert(T == 32 * JN * WN && IM <= WN, "square tile; block i of the bias gradient goes to wavefront column i");
  static constexpr int WAVES = WM * WN, THREADS = 64 * WAVES;
  static constexpr int ROWB = 2 * T;                  // bytes of a token's row in LDS
  static constexpr int OP = BR * ROWB, STAGE = 2 * OP, LDS = 2 * STAGE;
  static constexpr int CPR = T / 8, RPI = 64 / CPR;   // 16-byte chunks per row, rows per transfer
  static constexpr int DMA = OP / 1024 / WAVES;       // transfers of a wavefront per operand and stage
  static constexpr int JROWS = WAVES * RPI;           // rows between a wavefront's transfers
};

// Weight gradient. The tiles of g and x (64 tokens x T features) lie in LDS as they lie in memory, a token per row,
// brought there by direct transfers a stage ahead; the fragments, whose contraction runs over the tokens, come from
// transposing LDS reads (ds_read_b64_tr_b16, as in the attention backward). Chunk c of a row sits at c ^ 4 (row % 4): the
// four rows a transposing read of 16 lanes touches then cover all banks. No registers are staged and no vector
// instruction transposes: with its reduction 72 us for 32768 tokens, 1536 x 512 (101 us with both and a round more), 1132 us for
// 8192 x 8192 x 8192 (1294). A batch entry may be of any length: the octet-wise staging took multiples of 8 tokens
// only and left the rest to the FMA kernel (5 x 590 tokens, 896 features, qkv and output projection: 2247 -> 250 us). The bias gradient is one more matrix instruction with ones, in the first column of tiles.
// Around the stages: the tokens of a stage that lie a row apart share their offsets' products (walked token by token they were 0.3 of
// 0.75 us a stage), the partials leave by pointers that walk the rows (by index 2.6 us, 0.9 now), and tn_plan sets how many there are.
// us before -> now with the reduction: 924 tokens, 768 x 768 21.2 -> 13.6, 2560, 640 x 160 14.4 -> 10.9, 2680, 2688 x 896 37.7 -> 28.9, 32768,
// 512 x 512 42.4 -> 32.7, 65536, 512 x 128 26.3 -> 25.2. (A ring of four stages changed nothing, transfers between the matrix instructions, as in
// proj_nt_kernel, cost 5 % where the operands stream from memory.)
// OFF as in TokenWalk: 64-bit offsets from 2^32 bytes an operand on, at the same rate (2048 x 512 over 2^20 tokens 2.44 ms,
// 2040 x 512 with 32-bit ones 2.48; the FMA kernel, which the larger one would else fall to, 238 ms).
template <int IM, int JN, int WM, int WN, typename OFF>
__global__ __launch_bounds__(64 * WM * WN, IM * JN >= 8 ? 1 : 2) void proj_tn_kernel(TnParams p) {
  typedef TnShape<IM, JN, WM, WN> SH;
  constexpr int T = SH::T, ROWB = SH::ROWB;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int ln = lane & 31, kg = lane >> 5;
  const int wn = wave % WM, wc = wave / WM;
  const int wave_u = __builtin_amdgcn_readfirstlane(wave);
  // Workgroups go to the 8 XCDs round-robin. The few tiles of 128 x 128 of a split are gathered on one XCD, where they
  // meet in its L2 (65536 tokens, 512 x 128: 26.6 us, 29.5 spread). The 256-wide ones, which stream twice as much
  // per workgroup, are spread (32768 tokens, 1536 x 512 in 22 splits: 92 us, 113 gathered).
  int id = blockIdx.x;
  if (T == 128) {
    const int per_xcd = gridDim.x / 8;
    if (id < per_xcd * 8) id = (id % 8) * per_xcd + id / 8;
  }
  const int split = quotient(id, p.by_tiles), tile = id - split * p.tiles;
  const int tile_n = quotient(tile, p.by_tiles_c), tile_c = tile - tile_n * p.tiles_c;
  const int n0 = tile_n * T, c0 = tile_c * T;
  const long long r_first = (long long)split * p.stages_per_split * BR;
  long long r_last = r_first + (long long)p.stages_per_split * BR;
  if (r_last > p.rows) r_last = p.rows;
  const int nst = r_last > r_first ? (int)((r_last - r_first + BR - 1) / BR) : 0;

  // ---- transfers: number j of a wavefront carries rows j * JROWS + wave * RPI + lane / CPR
  const int my_row = wave * SH::RPI + lane / SH::CPR;
  const int chunk = (lane % SH::CPR) ^ ((my_row & 3) << 2);  // JROWS is a multiple of 4: the same for every j
  // a chunk past the last feature repeats the last one and is dropped
  const OFF gf = feat_bytes<OFF>(p.gm, min(n0 + chunk * 8, p.N - 8));
  const OFF xf = feat_bytes<OFF>(p.xm, min(c0 + chunk * 8, p.C - 8));
  const OFF g_row = (OFF)(p.gm.heads ? p.gm.D : p.gm.ld) * 2u, x_row = (OFF)(p.xm.heads ? p.xm.D : p.xm.ld) * 2u;
  const OFF g_lane = (OFF)my_row * g_row + gf, x_lane = (OFF)my_row * x_row + xf;
  // S = 0: the tokens of an operand lie a row apart throughout
  const int S = p.gm.heads ? p.gm.S : p.xm.heads ? p.xm.S : 0;
  const Div by_S = p.gm.heads ? p.gm.by_S : p.xm.by_S;
  const uint32_t lds_g = jg::lds_address(smem) + wave_u * 1024;
  auto entry_of = [&](long long r) { return sizeof(OFF) == 4 ? (long long)quotient((uint32_t)r, by_S) : r / S; };  // batch entry of a token
  auto row_at = [&](const Map& m, long long b, long long r) {  // first element of token r, which is of batch entry b
    return m.heads ? (b * m.H * m.S + (r - b * m.S)) * m.D : r * m.ld;
  };
  auto issue = [&](int st, int buf) {
    const long long first = r_first + (long long)st * BR, left = p.rows - first;
    const uint32_t dst = lds_g + buf * SH::STAGE;
    const long long b = S == 0 ? 0 : entry_of(first);
    if (left >= BR && (S == 0 || first - b * S + BR <= S)) {  // wave-uniform: the tokens of the stage lie a row apart
      OFF g_at = g_lane + (OFF)(row_at(p.gm, b, first) * 2), x_at = x_lane + (OFF)(row_at(p.xm, b, first) * 2);
#pragma unroll
      for (int j = 0; j < SH::DMA; ++j) {
        jg::to_lds_1k(p.g, g_at, dst + j * SH::WAVES * 1024);
        jg::to_lds_1k(p.x, x_at, dst + SH::OP + j * SH::WAVES * 1024);
        g_at += SH::JROWS * g_row;
        x_at += SH::JROWS * x_row;
      }
    } else {  // a batch entry ends in the stage, or the tokens do: a row past the end repeats the last token and is cleared below
#pragma unroll
      for (int j = 0; j < SH::DMA; ++j) {
        const long long r = min(first + j * SH::JROWS + my_row, p.rows - 1), e = S == 0 ? 0 : entry_of(r);
        jg::to_lds_1k(p.g, (OFF)(row_at(p.gm, e, r) * 2) + gf, dst + j * SH::WAVES * 1024);
        jg::to_lds_1k(p.x, (OFF)(row_at(p.xm, e, r) * 2) + xf, dst + SH::OP + j * SH::WAVES * 1024);
      }
    }
  };
  static_assert(SH::DMA * SH::JROWS == BR, "whole stages");
  auto clear_tail = [&](int st, int buf) {
    const long long left = p.rows - (r_first + (long long)st * BR);
    if (left >= BR) return;
    u32x4* at = reinterpret_cast<u32x4*>(smem + buf * SH::STAGE + wave * 1024 + lane * 16);
#pragma unroll
    for (int j = 0; j < SH::DMA; ++j)
      if (j * SH::JROWS + my_row >= left) {
        at[j * SH::WAVES * 64] = u32x4{0u, 0u, 0u, 0u};
        at[SH::OP / 16 + j * SH::WAVES * 64] = u32x4{0u, 0u, 0u, 0u};
      }
  };

  // ---- fragments: 32 features (block fb) x 16 tokens. Lane p of a group of 16 points at row 4 kg + p / 4, features
  // 16 (group % 2) + 4 (p % 4) of the block; a second read takes the rows 8 further on.
  auto frag_off = [&](int fb) {
    const int pp = lane & 15, g1 = (lane >> 4) & 1;
    const int c = 4 * fb + 2 * g1 + ((pp & 3) >> 1);
    return (4 * kg + (pp >> 2)) * ROWB + ((c ^ ((pp >> 2) << 2)) << 4) + 8 * (pp & 1);
  };
  int g_off[IM], x_off[JN];
#pragma unroll
  for (int i = 0; i < IM; ++i) g_off[i] = frag_off(wn * IM + i);
#pragma unroll
  for (int j = 0; j < JN; ++j) x_off[j] = SH::OP + frag_off(wc * JN + j);
  const int b_off = frag_off(wn * IM + min(wc, IM - 1));  // the block whose bias gradient this wavefront sums
  auto tr_frag = [&](const unsigned char* at) {
    typedef short i16x4 __attribute__((ext_vector_type(4)));
    typedef __attribute__((address_space(3))) i16x4* tr_ptr;
    const u32x2 lo = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((tr_ptr)(at)));
    const u32x2 hi = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((tr_ptr)(at + 8 * ROWB)));
    return __builtin_bit_cast(bf16x8, u32x4{lo.x, lo.y, hi.x, hi.y});
  };

  f32x16 acc[IM][JN], acc_b;
#pragma unroll
  for (int e = 0; e < 16; ++e) acc_b[e] = 0.0f;
#pragma unroll
  for (int i = 0; i < IM; ++i)
#pragma unroll
    for (int j = 0; j < JN; ++j) acc[i][j] = acc_b;
  bf16x8 ones;
#pragma unroll
  for (int e = 0; e < 8; ++e) ones[e] = (__bf16)1.0f;

  constexpr int AHEAD = IM * JN <= 4 ? 2 : 1;  // steps of 16 tokens between a fragment's request and its use
  auto compute = [&](int buf, auto with_bias) {
    const unsigned char* st = smem + buf * SH::STAGE;
    bf16x8 fr[AHEAD + 1][IM + JN + 1];
    auto fetch = [&](int kk, bf16x8 (&f)[IM + JN + 1]) {
      const unsigned char* at = st + kk * 16 * ROWB;
#pragma unroll
      for (int t = 0; t < IM; ++t) f[t] = tr_frag(at + g_off[t]);
#pragma unroll
      for (int t = 0; t < JN; ++t) f[IM + t] = tr_frag(at + x_off[t]);
      if (with_bias) f[IM + JN] = tr_frag(at + b_off);
    };
#pragma unroll
    for (int kk = 0; kk < AHEAD; ++kk) fetch(kk, fr[kk]);
#pragma unroll
    for (int kk = 0; kk < BR / 16; ++kk) {
      if (kk + AHEAD < BR / 16) fetch(kk + AHEAD, fr[(kk + AHEAD) % (AHEAD + 1)]);
      const bf16x8(&f)[IM + JN + 1] = fr[kk % (AHEAD + 1)];
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < IM; ++i)
#pragma unroll
        for (int j = 0; j < JN; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f[i], f[IM + j], acc[i][j], 0, 0, 0);
      if (with_bias) acc_b = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f[IM + JN], ones, acc_b, 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
    }
  };

  const bool want_bias = p.bias_part != nullptr && tile_c == 0;  // uniform over the workgroup
  auto run = [&](auto with_bias) {
    if (nst > 0) issue(0, 0);
    for (int st = 0; st < nst; ++st) {
      transfers_landed();
      if (st == nst - 1) clear_tail(st, st & 1);
      __syncthreads();  // stage st is in LDS, and every wavefront is done with the other buffer
      if (st + 1 < nst) issue(st + 1, (st + 1) & 1);
      compute(st & 1, with_bias);
    }
  };
  if (want_bias) run(std::true_type{});
  else run(std::false_type{});

  // register e of block (i, j): row n0 + (wn*IM + i)*32 + 8*(e/4) + 4*kg + e%4, column c0 + (wc*JN + j)*32 + ln
  {
    const int n_first = n0 + wn * IM * 32 + kg * 4, c_first = c0 + wc * JN * 32 + ln;
    const int rows_left = p.N - n_first, cols_left = p.C - c_first;
    auto store = [&](auto whole) __attribute__((always_inline)) {
      float* at = p.part + (size_t)split * p.N * p.C + (size_t)n_first * p.C + c_first;
#pragma unroll
      for (int i = 0; i < IM; ++i)
#pragma unroll
        for (int e4 = 0; e4 < 4; ++e4) {
#pragma unroll
          for (int e = 0; e < 4; ++e) {
#pragma unroll
            for (int j = 0; j < JN; ++j)
              if (whole || (i * 32 + e4 * 8 + e < rows_left && j * 32 < cols_left)) at[j * 32] = acc[i][j][e4 * 4 + e];
            at += p.C;
          }
          at += 4 * (size_t)p.C;
        }
    };
    if (n0 + T <= p.N && c0 + T <= p.C) store(std::true_type{});  // uniform over the workgroup
    else store(std::false_type{});
  }
  if (want_bias && wc < IM && ln == 0) {  // every column of acc_b holds the same sums
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      const int n = n0 + (wn * IM + wc) * 32 + (e >> 2) * 8 + kg * 4 + (e & 3);
      if (n < p.N) p.bias_part[(size_t)split * p.N + n] = acc_b[e];
    }
  }
}

// out[i] (bf16) = sum over the splits of part[split][i], for the weight gradient and (blocks behind
// it) the bias gradient in one launch. A block takes 256 consecutive outputs: 64 lanes x 4 values,
// and its W wavefronts (4, or 16 where there are many splits: a small weight matrix has few blocks,
// and each of their threads would walk the splits one load after the other) each add every W-th
// split; the W sums are then added in a fixed order, so the result does not depend on scheduling.
struct ReduceArgs {
  void* out_w;
  const float* part_w;
  size_t count_w;
  void* out_b;  // NULL: no bias gradient
  const float* part_b;
  size_t count_b;
  int splits;
  int out32;  // write fp32 instead of bf16
};

template <int W>
__global__ __launch_bounds__(64 * W) void proj_reduce_kernel(ReduceArgs a) {
  __shared__ float4 sm[W][64];
  const size_t blocks_w = (a.count_w + 255) / 256;
  const bool second = blockIdx.x >= blocks_w;
  void* const out = second ? a.out_b : a.out_w;
  const float* part = second ? a.part_b : a.part_w;
  const size_t count = second ? a.count_b : a.count_w;
  // every split's slice starts 16-byte aligned when the count is a multiple of 4 and the base is aligned
  const bool vec = jg::slices_vec(part, out, count), out32 = a.out32 != 0;
  jg::reduce_slices<W>(sm, part, count, a.splits, vec, blockIdx.x - (second ? blocks_w : 0), threadIdx.x >> 6, threadIdx.x & 63, [=](size_t i0, float4 t) {
    const float v[4] = {t.x, t.y, t.z, t.w};
    if (out32 && vec) {
      *reinterpret_cast<float4*>(static_cast<float*>(out) + i0) = t;
    } else if (vec) {
      u32x2 o;
      o.x = (uint32_t)jg::f32_to_bf16(v[0]) | ((uint32_t)jg::f32_to_bf16(v[1]) << 16);
      o.y = (uint32_t)jg::f32_to_bf16(v[2]) | ((uint32_t)jg::f32_to_bf16(v[3]) << 16);
      *reinterpret_cast<u32x2*>(static_cast<uint16_t*>(out) + i0) = o;
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (i0 + e < count) {
          if (out32) static_cast<float*>(out)[i0 + e] = v[e];
          else static_cast<uint16_t*>(out)[i0 + e] = jg::f32_to_bf16(v[e]);
        }
    }
  });
}

// ------------------------------------------------------------------- generic
template <int DT>
struct Elem;
template <>
struct Elem<JG_F32> {
  typedef float T;
  __device__ static __forceinline__ float up(float v) { return v; }
  __device__ static __forceinline__ float down(float v) { return v; }
};
template <>
struct Elem<JG_BF16> {
  typedef uint16_t T;
  __device__ static __forceinline__ float up(uint16_t v) { return jg::bf16_to_f32(v); }
  __device__ static __forceinline__ uint16_t down(float v) { return jg::f32_to_bf16(v); }
};
template <>
struct Elem<JG_F16> {
  typedef _Float16 T;
  __device__ static __forceinline__ float up(_Float16 v) { return (float)v; }
  __device__ static __forceinline__ _Float16 down(float v) { return (_Float16)v; }
};

struct GenParams {
  const void* p;   // NT: a (tokens x K);       TN: g (tokens x I)
  const void* q;   // NT: w (J, K) row-major;    TN: x (tokens x J)
  const void* bias;
  void* out;       // NT: tokens x J through om; TN: (I, J) row-major
  Map pm, qm, om;
  long long I;     // NT: tokens; TN: features of g
  int J;
  long long L;     // contraction length: NT: K; TN: tokens
  int out32;       // TN: write fp32 whatever the operands' dtype
};

// out(i, j) = sum_l P(i, l) * Q(j, l): 16 x 16 outputs per workgroup, the operands pass
// through LDS in tiles of 16 contraction steps. TRANS = 0: P(i, l) = a(i, l), Q(j, l) = w[j][l].
// TRANS = 1: P(i, l) = g(l, i), Q(j, l) = x(l, j).
template <int DT, bool TRANS>
__global__ __launch_bounds__(256) void proj_generic_kernel(GenParams p) {
  typedef typename Elem<DT>::T T;
  __shared__ float sp[16][17], sq[16][17];
  const int tx = threadIdx.x & 15, ty = threadIdx.x >> 4;
  const long long i0 = (long long)blockIdx.y * 16;
  const int j0 = blockIdx.x * 16;
  const T* P = static_cast<const T*>(p.p);
  const T* Q = static_cast<const T*>(p.q);
  float acc = 0.0f;
  for (long long l0 = 0; l0 < p.L; l0 += 16) {
    // thread (ty, tx) stages P(i0 + ty, l0 + tx) and Q(j0 + ty, l0 + tx)
    const long long l = l0 + tx;
    float pv = 0.0f, qv = 0.0f;
    if (l < p.L) {
      if (i0 + ty < p.I)
        pv = Elem<DT>::up(TRANS ? P[row_part(p.pm, l) + feat_part(p.pm, (int)(i0 + ty))]
                                : P[row_part(p.pm, i0 + ty) + feat_part(p.pm, (int)l)]);
      if (j0 + ty < p.J)
        qv = Elem<DT>::up(TRANS ? Q[row_part(p.qm, l) + feat_part(p.qm, j0 + ty)]
                                : Q[(long long)(j0 + ty) * p.L + l]);
    }
    sp[ty][tx] = pv;
    sq[ty][tx] = qv;
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 16; ++k) acc += sp[ty][k] * sq[tx][k];
    __syncthreads();
  }
  const long long i = i0 + ty;
  const int j = j0 + tx;
  if (i >= p.I || j >= p.J) return;
  T* out = static_cast<T*>(p.out);
  if (TRANS) {
    if (p.out32) static_cast<float*>(p.out)[i * p.J + j] = acc;
    else out[i * p.J + j] = Elem<DT>::down(acc);
  } else {
    if (p.bias != nullptr) acc += Elem<DT>::up(static_cast<const T*>(p.bias)[j]);
    out[row_part(p.om, i) + feat_part(p.om, j)] = Elem<DT>::down(acc);
  }
}

// gb[n] = sum over the tokens of g(r, n): one workgroup per feature, fixed order
template <int DT>
__global__ __launch_bounds__(256) void proj_colsum_kernel(void* gb, const void* g, Map gm, long long rows, bool out32) {
  typedef typename Elem<DT>::T T;
  __shared__ float red[256];
  const int n = blockIdx.x;
  const long long fo = feat_part(gm, n);
  float s = 0.0f;
  for (long long r = threadIdx.x; r < rows; r += 256) s += Elem<DT>::up(static_cast<const T*>(g)[row_part(gm, r) + fo]);
  red[threadIdx.x] = s;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    if (out32) static_cast<float*>(gb)[n] = red[0];
    else static_cast<T*>(gb)[n] = Elem<DT>::down(red[0]);
  }
}

// fp32 matrices to bf16 and to their transposes, a 64 x 64 tile per block, every matrix of the list in one launch
// (a block's parameters are a few hundred KB: what a cast costs is its launch)
constexpr int CAST_MOST = 16;
struct CastArgs {
  const float* src[CAST_MOST];
  uint16_t* dst[CAST_MOST];
  uint16_t* dst_t[CAST_MOST];
  int rows[CAST_MOST], cols[CAST_MOST];
  int end[CAST_MOST];  // blocks of this matrix and the ones before it
};
__global__ __launch_bounds__(256) void cast_params_kernel(CastArgs a) {
  __shared__ uint16_t tile[64][66];
  int m = 0;
  while ((int)blockIdx.x >= a.end[m]) ++m;
  const int t = blockIdx.x - (m == 0 ? 0 : a.end[m - 1]);
  const int rows = a.rows[m], cols = a.cols[m], tiles_c = (cols + 63) / 64;
  const int r0 = t / tiles_c * 64, c0 = t % tiles_c * 64;
  const int x = threadIdx.x & 63, y = threadIdx.x >> 6;
  const float* src = a.src[m];
  uint16_t* dst = a.dst[m];
  float v[16];  // all loads first: one memory latency a tile
#pragma unroll
  for (int i = 0; i < 16; ++i) v[i] = src[(size_t)min(r0 + y + 4 * i, rows - 1) * cols + min(c0 + x, cols - 1)];
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const int r = y + 4 * i;
    const uint16_t h = jg::f32_to_bf16(v[i]);
    if (r0 + r < rows && c0 + x < cols) dst[(size_t)(r0 + r) * cols + c0 + x] = h;
    tile[r][x] = h;
  }
  if (a.dst_t[m] == nullptr) return;
  __syncthreads();
  for (int i = y; i < 64; i += 4)
    if (c0 + i < cols && r0 + x < rows) a.dst_t[m][(size_t)(c0 + i) * rows + r0 + x] = tile[x][i];
}

// dst (cols, rows) = src (rows, cols)^T, 16-bit values, both sizes multiples of 8: a 64 x 64 tile per block, 16-byte
// pieces both ways, turned on the way into LDS. What a weight of some MB waits for is one memory latency and the
// launch: 1536 x 512 7.3 us with torch's copy, 3.4 here; 512 x 512 5.6 and 3.4.
__global__ __launch_bounds__(256) void transpose16_kernel(uint16_t* __restrict__ dst, const uint16_t* __restrict__ src,
                                                          long long rows, long long cols, int tiles_c) {
  __shared__ __attribute__((aligned(16))) uint16_t tile[64][72];
  const long long r0 = (long long)(blockIdx.x / tiles_c) * 64, c0 = (long long)(blockIdx.x % tiles_c) * 64;
  const int piece = threadIdx.x & 7, line = threadIdx.x >> 3;  // 8 values, and the row (or column) they are of
#pragma unroll
  for (int i = 0; i < 64; i += 32) {
    const long long r = r0 + line + i, c = c0 + piece * 8;
    if (r < rows && c < cols) {
      const u32x4 v = *reinterpret_cast<const u32x4*>(src + r * cols + c);
#pragma unroll
      for (int e = 0; e < 8; ++e) tile[piece * 8 + e][line + i] = (uint16_t)(v[e >> 1] >> (16 * (e & 1)));
    }
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < 64; i += 32) {
    const long long c = c0 + line + i, r = r0 + piece * 8;
    if (c < cols && r < rows) *reinterpret_cast<u32x4*>(dst + c * rows + r) = *reinterpret_cast<const u32x4*>(&tile[line + i][piece * 8]);
  }
}

// --------------------------------------------------------------------- host
int make_map(Map* m, int heads, long long features, long long rows, int B, int H, int S, int D, const char* who,
             const char* what) {
  m->heads = heads ? 1 : 0;
  m->ld = features;
  m->B = B; m->H = H; m->S = S; m->D = D;
  m->by_S = div_by(S); m->by_D = div_by(D); m->by_H = div_by(H);
  if (!heads) return JG_OK;
  JG_REQUIRE(B > 0 && H > 0 && S > 0 && D > 0, "%s: %s: heads layout needs positive B, H, S, D", who, what);
  JG_REQUIRE((long long)B * S == rows, "%s: %s: B * S = %lld does not match %lld tokens", who, what,
             (long long)B * S, rows);
  JG_REQUIRE(features % ((long long)H * D) == 0, "%s: %s: %lld features are not a multiple of H * D = %lld", who, what,
             features, (long long)H * D);
  return JG_OK;
}

bool aligned16(const void* ptr) { return (reinterpret_cast<uintptr_t>(ptr) & 15) == 0; }
// 16-byte chunks of 8 features stay inside one head and start aligned
bool map_vec_ok(const Map& m, long long features) {
  if (features % 8 != 0) return false;
  return m.heads ? (m.D % 8 == 0) : (m.ld % 8 == 0);
}
long long tn_stages(long long rows) { return (rows + BR - 1) / BR; }

// Tile edge of the weight-gradient kernel and the ranges of tokens (splits) the contraction is cut into: the pair with the least of
// what the figures of both say, us on 256 compute units (measured, the reduction included, and what the rule expects):
//   128   a stage takes 0.7 where a compute unit has one workgroup, 1 where some have two, and all of them together no less than
//         14.6 TB/s out of the caches allow; 5.4 around them. 32768 tokens, 512 x 512, 16 splits 32.3 (33.4), 32 33.7 (35.0), 1536 x 512, 8 splits
//         75.9 (77.8), 10 70.7 (71.0); 5000, 1024 x 1024, 4 splits 24.8 (25.0), 8 28.5 (27.9); 924, 768 x 768, 1 split 17.2 (16.9), 3 12.9 (11.3).
//   256   half the operand traffic per matrix instruction and one workgroup a compute unit: 1.7 a stage and 5 a round of workgroups.
//         8192 tokens, 3072 x 1024, 5 splits 70.7 (70.2; at 128 76.4), 32768 219 (201; at 128 238), 512 x 512, 48 splits 38.5 (40.5).
// and the partials written and read back at 6 TB/s. More splits only where they win a twentieth with the partials counted half as
// much again: a Swin block holds those of all its weights until the end of its backward. With at least eight stages a split, and 256 wherever
// its tiles filled most of the chip, 924 tokens, 768 x 768 took 17.1, 5000, 1024 x 1024 32.2, 32768, 512 x 512 39.7.
constexpr int TN_MOST_SPLITS = 64;
struct TnPlan {
  int tile, splits;
};
TnPlan tn_plan(long long rows, int n, int c) {
  const long long stages = tn_stages(rows), cus = jg::cu_count();
  const double partial = (double)n * c * 8.0 / 6.0e6;
  TnPlan best{128, 1};
  double best_us = 0.0;
  for (const int t : {128, 256}) {
    if (t == 256 && (n < 256 || c < 256)) break;
    const long long tiles = (long long)jg::cdiv(n, t) * jg::cdiv(c, t);
    // (with one to three tiles as many as put a workgroup on every compute unit)
    const long long most = std::min<long long>(stages, std::max<long long>(TN_MOST_SPLITS, cus / tiles));
    double least = 0.0, us = 0.0;
    int splits = 1;
    for (long long k = 1; k <= most; k += 1 + k / 8) {
      const long long walk = (stages + k - 1) / k, workgroups = tiles * k;
      double sums;
      if (t == 256) sums = (double)((workgroups + cus - 1) / cus) * (walk * 1.7 + 5.0);
      else sums = std::max(walk * (workgroups <= cus ? 0.7 : (double)((workgroups + 2 * cus - 1) / (2 * cus))), (double)tiles * stages * 32768.0 / 14.6e6) + 5.4;
      if (least == 0.0 || sums + 1.5 * k * partial < 0.95 * least) {
        least = sums + 1.5 * k * partial;
        us = sums + k * partial;
        splits = (int)((stages + walk - 1) / walk);  // (no empty ones)
      }
    }
    if (t == 128 || us < best_us) {
      best = TnPlan{t, splits};
      best_us = us;
    }
  }
  return best;
}

template <int IM, int JN, int WM, int WN, typename OFF>
int launch_tn(TnParams& p, int splits, hipStream_t s, const char* who) {
  typedef TnShape<IM, JN, WM, WN> SH;
  p.tiles_c = jg::cdiv(p.C, SH::T);
  p.tiles = jg::cdiv(p.N, SH::T) * p.tiles_c;
  p.by_tiles_c = div_by(p.tiles_c);
  p.by_tiles = div_by(p.tiles);
  void (*kern)(TnParams) = &proj_tn_kernel<IM, JN, WM, WN, OFF>;
  if (hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, SH::LDS) != hipSuccess)
    JG_FAIL(JG_ERR_LAUNCH, "%s: cannot reserve %d bytes of LDS", who, SH::LDS);
  kern<<<(unsigned)p.tiles * (unsigned)splits, SH::THREADS, SH::LDS, s>>>(p);
  JG_CHECK_LAUNCH(who);
  return JG_OK;
}

template <bool TRANS>
int launch_generic(const GenParams& gp, int dtype, hipStream_t s, const char* who) {
  dim3 grid((unsigned)jg::cdiv(gp.J, 16), (unsigned)jg::cdiv(gp.I, 16));
  JG_REQUIRE(grid.y <= 65535u, "%s: too many rows for the generic kernel", who);
  switch (dtype) {
    case JG_F32: proj_generic_kernel<JG_F32, TRANS><<<grid, 256, 0, s>>>(gp); break;
    case JG_BF16: proj_generic_kernel<JG_BF16, TRANS><<<grid, 256, 0, s>>>(gp); break;
    case JG_F16: proj_generic_kernel<JG_F16, TRANS><<<grid, 256, 0, s>>>(gp); break;
    default: JG_FAIL(JG_ERR_BAD_ARG, "%s: unknown dtype %d", who, dtype);
  }
  JG_CHECK_LAUNCH(who);
  return JG_OK;
}

}  // namespace

extern "C" {

static int proj_nt_common(const char* who, void* out, void* aux, int epi, const void* a, const void* w, const void* bias,
                          int dtype, int64_t rows, int n_out, int k_in, int a_heads, int out_heads, int B, int H, int S,
                          int D, void* stream) {
  JG_REQUIRE(out && a && w, "%s: null pointer", who);
  JG_REQUIRE(jg::dtype_size(dtype) != 0, "%s: unknown dtype %d", who, dtype);
  JG_REQUIRE(rows >= 0 && n_out > 0 && k_in > 0, "%s: bad sizes rows=%lld n_out=%d k_in=%d", who, (long long)rows, n_out,
             k_in);
  if (rows == 0) return JG_OK;
  Map am, om;
  int rc = make_map(&am, a_heads, k_in, rows, B, H, S, D, who, "input");
  if (rc) return rc;
  rc = make_map(&om, out_heads, n_out, rows, B, H, S, D, who, "output");
  if (rc) return rc;
  hipStream_t s = static_cast<hipStream_t>(stream);
  const bool fast = dtype == JG_BF16 && map_vec_ok(am, k_in) && map_vec_ok(om, n_out) && aligned16(a) &&
                    aligned16(w) && aligned16(out) && rows < (1ll << 31) - 256 &&
                    (unsigned long long)rows * k_in < (1ull << 31) && (unsigned long long)n_out * k_in < (1ull << 31);
  if (!fast) {
    if (epi != EPI_NONE)
      JG_FAIL(JG_ERR_UNSUPPORTED, "%s: the fused epilogues are built for bf16 operands on 16-byte aligned rows", who);
    GenParams gp;
    gp.p = a; gp.q = w; gp.bias = bias; gp.out = out;
    gp.pm = am; gp.qm = am; gp.om = om;
    gp.I = rows; gp.J = n_out; gp.L = k_in;
    gp.out32 = 0;
    return launch_generic<false>(gp, dtype, s, who);
  }
  NtParams p;
  p.epi = epi;
  p.aux = static_cast<uint16_t*>(aux);
  p.a = static_cast<const uint16_t*>(a);
  p.w = static_cast<const uint16_t*>(w);
  p.bias = static_cast<const uint16_t*>(bias);
  p.out = static_cast<uint16_t*>(out);
  p.am = am; p.om = om;
  p.rows = rows; p.N = n_out; p.K = k_in;
  // Tiles of 256 x 256 (half the operand traffic per MFMA), one workgroup a compute unit, where their rounds leave no more than two fifths of
  // the chip idle and the last column of tiles is more than half full; below a round only contractions of 1024 and more gain (us, 256 : 128:
  // 16000 tokens, 1024 -> 1024 34.6 : 39.8, 5000, 1024 -> 2048 30.3 : 33.8, 8000, 384 -> 768 14.9 : 10.8; 282 tiles, 12000, 512 -> 1536
  // 33.4 : 28.3; 512, 32768, 256 -> 1024 26.8 : 28.1). What is read on the way out and short contractions, which are little but their
  // epilogue, are better off with two workgroups a compute unit (y gelu'(aux), 65536, 128 -> 512 42.3 : 38.7, 55680, 256 -> 1024 91.2 : 86.8;
  // plain, 65536, 128 -> 512 21.5 : 19.6; with GELU, whose arithmetic bounds it, 250000, 128 -> 512 150 : 183).
  const long long cus = jg::cu_count(), tiles_256 = (long long)jg::cdiv(rows, 256) * jg::cdiv(n_out, 256);
  const int waste = jg::cdiv(n_out, 256) * 256 - n_out;
  const bool fills = tiles_256 * 5 >= (tiles_256 + cus - 1) / cus * cus * 3 && (tiles_256 >= cus || k_in >= 1024);
  const bool epilogue_only = epi == EPI_DGELU ? k_in <= 256 : epi != EPI_GELU && k_in <= 128;
  if (fills && waste < 128 && !epilogue_only) return launch_nt<4, 2, 2, 4>(p, s, who);
  // 64 x 64 where 128 x 128 tiles would leave a quarter of the chip idle (us, 64 : 128: 468 tokens, 704 -> 2112 7.2 : 9.7, 924, 768 -> 2304
  // 9.6 : 12.2, 4000, 640 -> 640 8.9 : 9.7; 224 tiles of 128, 3520, 256 -> 1024 7.5 : 6.9)
  if ((long long)jg::cdiv(rows, 128) * jg::cdiv(n_out, 128) < cus * 3 / 4) return launch_nt<1, 1, 2, 2>(p, s, who);
  return launch_nt<2, 1, 2, 4>(p, s, who);
}

int jg_proj_nt(void* out, const void* a, const void* w, const void* bias, int dtype, int64_t rows, int n_out,
               int k_in, int a_heads, int out_heads, int B, int H, int S, int D, void* stream) {
  return proj_nt_common("jg_proj_nt", out, nullptr, EPI_NONE, a, w, bias, dtype, rows, n_out, k_in, a_heads, out_heads,
                        B, H, S, D, stream);
}

int jg_proj_nt_fused_heads(void* out, void* aux, int epilogue, const void* a, const void* w, const void* bias, int dtype,
                           int64_t rows, int n_out, int k_in, int a_heads, int B, int H, int S, int D, void* stream) {
  const char* who = "jg_proj_nt_fused";
  JG_REQUIRE(epilogue == EPI_GELU || epilogue == EPI_DGELU || epilogue == EPI_ADD, "%s: unknown epilogue %d", who,
             epilogue);
  JG_REQUIRE(aux != nullptr && aligned16(aux), "%s: aux must be a 16-byte aligned tensor of the shape of out", who);
  return proj_nt_common(who, out, aux, epilogue, a, w, bias, dtype, rows, n_out, k_in, a_heads, 0, B, H, S, D, stream);
}

int jg_proj_nt_fused(void* out, void* aux, int epilogue, const void* a, const void* w, const void* bias, int dtype,
                     int64_t rows, int n_out, int k_in, void* stream) {
  return jg_proj_nt_fused_heads(out, aux, epilogue, a, w, bias, dtype, rows, n_out, k_in, 0, 1, 1, 1, 1, stream);
}

int jg_cast_params(void* const* dst, void* const* dst_t, const void* const* src, const int32_t* rows, const int32_t* cols,
                   int n, void* stream) {
  const char* who = "jg_cast_params";
  JG_REQUIRE(n >= 0 && n <= CAST_MOST, "%s: at most %d tensors, got %d", who, CAST_MOST, n);
  JG_REQUIRE(n == 0 || (dst && dst_t && src && rows && cols), "%s: null pointer", who);
  CastArgs a = {};
  long long blocks = 0;
  for (int i = 0; i < n; ++i) {
    JG_REQUIRE(dst[i] && src[i] && rows[i] >= 0 && cols[i] >= 0, "%s: tensor %d", who, i);
    a.src[i] = static_cast<const float*>(src[i]);
    a.dst[i] = static_cast<uint16_t*>(dst[i]);
    a.dst_t[i] = static_cast<uint16_t*>(dst_t[i]);
    a.rows[i] = rows[i];
    a.cols[i] = cols[i];
    blocks += (long long)jg::cdiv(rows[i], 64) * jg::cdiv(cols[i], 64);
    JG_REQUIRE(blocks < (1ll << 31), "%s: too large", who);
    a.end[i] = (int)blocks;
  }
  if (blocks == 0) return JG_OK;
  cast_params_kernel<<<(unsigned)blocks, 256, 0, static_cast<hipStream_t>(stream)>>>(a);
  JG_CHECK_LAUNCH(who);
  return JG_OK;
}

int jg_transpose16(void* dst, const void* src, int64_t rows, int64_t cols, void* stream) {
  const char* who = "jg_transpose16";
  JG_REQUIRE(rows >= 0 && cols >= 0, "%s: bad sizes rows=%lld cols=%lld", who, (long long)rows, (long long)cols);
  if (rows == 0 || cols == 0) return JG_OK;
  JG_REQUIRE(dst && src, "%s: null pointer", who);
  if (rows % 8 != 0 || cols % 8 != 0 || !aligned16(dst) || !aligned16(src))
    JG_FAIL(JG_ERR_UNSUPPORTED, "%s: sizes that are multiples of 8 and 16-byte aligned matrices only", who);
  const long long tiles_r = (rows + 63) / 64, tiles_c = (cols + 63) / 64;
  JG_REQUIRE(tiles_r < (1ll << 31) / tiles_c, "%s: too large", who);
  transpose16_kernel<<<(unsigned)(tiles_r * tiles_c), 256, 0, static_cast<hipStream_t>(stream)>>>(
      static_cast<uint16_t*>(dst), static_cast<const uint16_t*>(src), rows, cols, (int)tiles_c);
  JG_CHECK_LAUNCH(who);
  return JG_OK;
}

size_t jg_proj_tn_workspace(int64_t rows, int n, int c) {
  if (rows <= 0 || n <= 0 || c <= 0) return 0;
  const size_t splits = (size_t)tn_plan(rows, n, c).splits;
  return splits * ((size_t)n * c + n) * sizeof(float);
}

// later: NULL, or where the sums of the splits are left
static int proj_tn_common(const char* who, jg_reductions* later, void* gw, void* gb, const void* g, const void* x, int dtype, int grad_dtype, int64_t rows,
                          int n, int c, int g_heads, int x_heads, int B, int H, int S, int D, void* workspace, size_t workspace_bytes, void* stream) {
  JG_REQUIRE(gw && g && x, "%s: null pointer", who);
  JG_REQUIRE(jg::dtype_size(dtype) != 0, "%s: unknown dtype %d", who, dtype);
  JG_REQUIRE(grad_dtype == dtype || grad_dtype == JG_F32, "%s: gradient dtype %d with operand dtype %d", who, grad_dtype,
             dtype);
  const bool out32 = grad_dtype == JG_F32 && dtype != JG_F32;
  JG_REQUIRE(rows > 0 && n > 0 && c > 0, "%s: bad sizes rows=%lld n=%d c=%d", who, (long long)rows, n, c);
  JG_REQUIRE(n < (1 << 27) && c < (1 << 27), "%s: more than 2^27 features a row (n=%d c=%d)", who, n, c);
  Map gm, xm;
  int rc = make_map(&gm, g_heads, n, rows, B, H, S, D, who, "gradient");
  if (rc) return rc;
  rc = make_map(&xm, x_heads, c, rows, B, H, S, D, who, "input");
  if (rc) return rc;
  hipStream_t s = static_cast<hipStream_t>(stream);
  const bool fast = dtype == JG_BF16 && map_vec_ok(gm, n) && map_vec_ok(xm, c) && aligned16(g) && aligned16(x);
  if (!fast) {
    GenParams gp;
    gp.p = g; gp.q = x; gp.bias = nullptr; gp.out = gw;
    gp.pm = gm; gp.qm = xm; gp.om = gm;
    gp.I = n; gp.J = c; gp.L = rows;
    gp.out32 = out32 ? 1 : 0;
    rc = launch_generic<true>(gp, dtype, s, who);
    if (rc) return rc;
    if (gb != nullptr) {
      switch (dtype) {
        case JG_F32: proj_colsum_kernel<JG_F32><<<n, 256, 0, s>>>(gb, g, gm, rows, out32); break;
        case JG_BF16: proj_colsum_kernel<JG_BF16><<<n, 256, 0, s>>>(gb, g, gm, rows, out32); break;
        default: proj_colsum_kernel<JG_F16><<<n, 256, 0, s>>>(gb, g, gm, rows, out32); break;
      }
      JG_CHECK_LAUNCH(who);
    }
    return JG_OK;
  }
  const size_t need = jg_proj_tn_workspace(rows, n, c);
  if (workspace == nullptr || workspace_bytes < need)
    JG_FAIL(JG_ERR_WORKSPACE, "%s: workspace %zu < %zu bytes", who, workspace_bytes, need);
  JG_REQUIRE(aligned16(workspace), "%s: workspace must be 16-byte aligned", who);
  TnParams p;
  p.g = static_cast<const uint16_t*>(g);
  p.x = static_cast<const uint16_t*>(x);
  p.gm = gm; p.xm = xm;
  p.rows = rows; p.N = n; p.C = c;
  const TnPlan plan = tn_plan(rows, n, c);
  const int splits = plan.splits;
  const long long stages = (rows + BR - 1) / BR;
  p.stages_per_split = (int)((stages + splits - 1) / splits);
  p.part = static_cast<float*>(workspace);
  p.bias_part = gb != nullptr ? p.part + (size_t)splits * n * c : nullptr;
  const bool far = (unsigned long long)rows * (n > c ? n : c) >= (1ull << 31);
  if (plan.tile == 256)
    rc = far ? launch_tn<4, 2, 2, 4, uint64_t>(p, splits, s, who) : launch_tn<4, 2, 2, 4, uint32_t>(p, splits, s, who);
  else
    rc = far ? launch_tn<1, 2, 4, 2, uint64_t>(p, splits, s, who) : launch_tn<1, 2, 4, 2, uint32_t>(p, splits, s, who);
  if (rc) return rc;
  if (later != nullptr && out32) {
    rc = jg::add_reduction(later, jg::RED_SLICES, splits, (int64_t)n * c, p.part, static_cast<float*>(gw), nullptr);
    return rc != JG_OK || gb == nullptr ? rc : jg::add_reduction(later, jg::RED_SLICES, splits, n, p.bias_part, static_cast<float*>(gb), nullptr);
  }
  ReduceArgs ra{};
  ra.out_w = gw;
  ra.part_w = p.part;
  ra.count_w = (size_t)n * c;
  ra.out_b = gb;
  ra.part_b = p.bias_part;
  ra.count_b = gb != nullptr ? (size_t)n : 0;
  ra.splits = splits;
  ra.out32 = out32 ? 1 : 0;
  const size_t blocks = (ra.count_w + 255) / 256 + (ra.count_b + 255) / 256;
  if (jg::slice_waves(splits) == 16) proj_reduce_kernel<16><<<(unsigned)blocks, 1024, 0, s>>>(ra);
  else proj_reduce_kernel<4><<<(unsigned)blocks, 256, 0, s>>>(ra);
  JG_CHECK_LAUNCH(who);
  return JG_OK;
}

int jg_proj_tn(void* gw, void* gb, const void* g, const void* x, int dtype, int grad_dtype, int64_t rows, int n, int c,
               int g_heads, int x_heads, int B, int H, int S, int D, void* workspace, size_t workspace_bytes,
               void* stream) {
  return proj_tn_common("jg_proj_tn", nullptr, gw, gb, g, x, dtype, grad_dtype, rows, n, c, g_heads, x_heads, B, H, S, D, workspace, workspace_bytes, stream);
}

int jg_proj_tn_later(jg_reductions* later, void* gw, void* gb, const void* g, const void* x, int dtype, int grad_dtype, int64_t rows, int n, int c,
                     int g_heads, int x_heads, int B, int H, int S, int D, void* workspace, size_t workspace_bytes, void* stream) {
  const char* who = "jg_proj_tn_later";
  JG_REQUIRE(later != nullptr, "%s: null pointer", who);
  return proj_tn_common(who, later, gw, gb, g, x, dtype, grad_dtype, rows, n, c, g_heads, x_heads, B, H, S, D, workspace, workspace_bytes, stream);
}

}  // extern "C"
