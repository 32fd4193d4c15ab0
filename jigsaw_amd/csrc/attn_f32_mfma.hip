// fp32 attention core on the matrix cores (v_mfma_f32_32x32x2_f32): forward with the natural-log
// LSE and, optionally, the merge into a running (out_acc, lse_acc) pair of a ring of chunks; backward.
// Any lengths, head sizes that are multiples of 4 up to 128, one or several K / V chunks a launch, no bias.
// A wavefront owns 32 queries and walks the keys 32 at a time:
//
//   S^T = K Q^T      A = K (row = key), B = Q^T (column = query); the two contraction slots of an
//                    MFMA step belong to the two halves of the wavefront, and half g owns the
//                    head-size slice [g D/2, (g + 1) D/2), so a lane reads its K slice as 16-byte
//                    words and keeps its Q slice in registers, scaled by scale * log2(e).
//   softmax          a lane holds 16 keys of ONE query (column = lane % 32): the row maximum and
//                    sum are 16 values in registers plus one exchange with the other half.
//   O^T = V^T P^T    A = V^T (row = head-size index), B = P^T: step i contracts the two keys whose
//                    probabilities the two halves hold in element i, so P never moves.
//
// Workgroups of four wavefronts: R of them take 32 rows each of the resident side, and 4 / R groups of R
// share the streamed tiles out among themselves, each with a tile of its own in LDS; their partial
// results meet in LDS at the end. R = 4 reads the streamed side once for 128 rows; R = 1 gives a head of few
// rows four times the workgroups, each a quarter as long, and leaves fewer wavefronts without rows.
// The chunks of a ring are one launch: a launch a chunk held 90 workgroups at 45 heads x 171 tokens, and the
// backward's four launches a chunk a fifth of its time.
// D: the kernel's width, 32, 64, 96 or 128; a head size d below it (d % 4 == 0) has its missing columns as zeros
// in LDS and registers and no copies in memory.
//
// Reference behaviour restated here:
//   jigsaw/modules/attention/_functional/cores/math.py:69-78   (forward, lse = logsumexp of the scaled scores)
//   jigsaw/modules/attention/_functional/forward.py (merge of a chunk into the running output by its LSE)
#include "attn_chunks.h"

namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int kWaves = 4;
constexpr int kThreads = 64 * kWaves;
constexpr int kBK = 32;  // rows of the streamed side per step

// key row (inside a 32-key step) of accumulator element i in half g: the 32x32 result layout
__device__ __forceinline__ int row_of(int i, int g) { return (i >> 2) * 8 + g * 4 + (i & 3); }

template <int D, int R>
struct Shape {
  static constexpr int G = kWaves / R;            // groups that share the streamed tiles out
  static constexpr int H = D / 2;                 // contraction slots of one half
  static constexpr int PITCH = D + 4;             // LDS row pitch in floats: 16-byte rows, the b128 reads of 16 rows cover all banks
  static constexpr int NT = D / 32;               // 32-wide head-size tiles
  static constexpr int TG = 64 * R;               // threads of a group
  static constexpr int PIECES = kBK * D / 4 / TG; // 16-byte pieces of a 32 x D tile per thread
  static constexpr int TILE = kBK * PITCH;        // floats
  static constexpr int GROUP = 2 * TILE + 2 * kBK;  // two tiles; 32 lse and 32 delta
  static constexpr int LDS = G * GROUP * 4;
};

template <int D, int R>
using Pieces = f32x4[Shape<D, R>::PIECES];

// Where a wavefront stands.
template <int R>
struct Seat {
  int lane, g, n, group, row_wave, gt;
  __device__ __forceinline__ Seat() {
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    lane = tid & 63;
    g = lane >> 5;
    n = lane & 31;
    group = wave / R;
    row_wave = wave % R;
    gt = tid - group * 64 * R;
  }
};
// Workgroups go to the 8 XCDs round-robin; each XCD gets a contiguous range, so that the workgroups of a head meet in one L2.
__device__ __forceinline__ unsigned block_id() {
  const unsigned total = gridDim.x, id = blockIdx.x;
  return (total & 7u) == 0 ? (id & 7u) * (total >> 3) + (id >> 3) : id;
}
// The steps of a group: number group, group + G, ... of the chunks' steps in order.
struct Walk {
  int chunk, step, left;
  __device__ __forceinline__ Walk(int group, int G, int per_chunk, int chunks) : chunk(0), step(group) {
    const int total = per_chunk * chunks;
    left = total > group ? (total - group + G - 1) / G : 0;
    settle(per_chunk);
  }
  __device__ __forceinline__ void settle(int per_chunk) {
    while (step >= per_chunk) {
      step -= per_chunk;
      ++chunk;
    }
  }
  __device__ __forceinline__ void advance(int G, int per_chunk) {
    step += G;
    --left;
    settle(per_chunk);
  }
};

// A 32 x D tile of two tensors into registers (rows past `rows` read the last row; those of the
// second tensor become zero, and so do columns past d), and from there into LDS.
template <int D, int R>
__device__ __forceinline__ void fetch_tiles(Pieces<D, R>& a, Pieces<D, R>& b, const float* abase,
                                            const float* bbase, int row0, int rows, int d, int gt) {
  const f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int i = 0; i < Shape<D, R>::PIECES; ++i) {
    const int e = gt + Shape<D, R>::TG * i, row = e / (D / 4), c = e % (D / 4) * 4;
    const int r = row0 + row;
    const bool there = c < d;
    const long long at = (long long)(r < rows ? r : rows - 1) * d + (there ? c : 0);
    const f32x4 t = *reinterpret_cast<const f32x4*>(abase + at), u = *reinterpret_cast<const f32x4*>(bbase + at);
    a[i] = there ? t : zero;
    b[i] = there && r < rows ? u : zero;
  }
}
template <int D, int R>
__device__ __forceinline__ void store_tiles(float* as, float* bs, const Pieces<D, R>& a, const Pieces<D, R>& b, int gt) {
#pragma unroll
  for (int i = 0; i < Shape<D, R>::PIECES; ++i) {
    const int e = gt + Shape<D, R>::TG * i, row = e / (D / 4), c = e % (D / 4) * 4;
    *reinterpret_cast<f32x4*>(as + row * (D + 4) + c) = a[i];
    *reinterpret_cast<f32x4*>(bs + row * (D + 4) + c) = b[i];
  }
}
// This lane's slice of a row (columns g D/2 ..), times mul.
template <int D>
__device__ __forceinline__ void load_slice(float (&f)[D / 2], const float* row, int g, int d, float mul) {
#pragma unroll
  for (int j = 0; j < D / 2; j += 4) {
    const bool there = g * (D / 2) + j < d;
    const f32x4 t = *reinterpret_cast<const f32x4*>(row + (there ? g * (D / 2) + j : 0));
#pragma unroll
    for (int e = 0; e < 4; ++e) f[j + e] = there ? t[e] * mul : 0.0f;
  }
}
// acc of the groups behind the first into LDS, and from there onto the first group's (the caller's barriers).
template <int NT>
__device__ __forceinline__ void put_acc(float* at, const f32x16 (&acc)[NT]) {
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int i = 0; i < 16; ++i) at[(t * 16 + i) * 64] = acc[t][i];
}
template <int NT>
__device__ __forceinline__ void add_acc(f32x16 (&acc)[NT], const float* at, float mul) {
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[t][i] += at[(t * 16 + i) * 64] * mul;
}
template <int NT>
__device__ __forceinline__ void clear_acc(f32x16 (&acc)[NT]) {
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[t][i] = 0.0f;
}

// acc = acc * mul + A^T B over the 32 rows of a step: `rows` (LDS) holds A as rows of PITCH floats, of which this lane takes column 32 t + n; b
// is the other operand as it lies in the registers. The matrix cores sum a step from zero and the vector unit adds it to the steps before:
// output and dQ are sums over the keys of all chunks, which in the matrix cores' accumulators alone are one chain of roundings. Relative errors
// of the output and dQ, 64 heads x 1000 x 16 chunks at 64: one chain 2.3e-6 / 2.3e-6, a launch and a chain a chunk 8.3e-7 / 7.5e-7, this
// 6.1e-7 / 6.3e-7; 16 x 64 x 8 chunks 3.6e-7 / 3.9e-7 a chunk, this 2.5e-7 / 3.8e-7. It costs 1 to 3 % at widths up to 96 (16 x 700 x 4 at
// 64 489 -> 501 us both ways) and gains 3 to 5 % at 128, whose accumulators no longer wait for the factor (48 x 900 x 4 4871 -> 4641).
template <int NT, int PITCH>
__device__ __forceinline__ void add_step(f32x16 (&acc)[NT], const float* rows, const f32x16& b, int g, float mul) {
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    f32x16 sum;
#pragma unroll
    for (int i = 0; i < 16; ++i) sum[i] = 0.0f;
#pragma unroll
    for (int i = 0; i < 16; ++i) sum = __builtin_amdgcn_mfma_f32_32x32x2f32(rows[row_of(i, g) * PITCH + 32 * t], b[i], sum, 0, 0, 0);
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[t][i] = acc[t][i] * mul + sum[i];
  }
}

// Wavefronts a SIMD that the two kernels are held to where the compiler would take a few registers more than leave room for them: 64 heads x 1000 x 3
// chunks at 96 3162 -> 3018 us, x 4 at 32 1533 -> 1491.
constexpr int fwd_waves(int D, int R) { return D == 32 ? (R == 1 ? 3 : 4) : D == 64 || (D == 96 && R == 4) ? 2 : 1; }
constexpr int dq_waves(int D, int R) { return D == 32 ? (R == 4 ? 4 : 3) : (D == 64 && R > 1) || (D == 96 && R == 4) ? 2 : 1; }

struct F32Params {
  const float* q;      // (batch, sq, d)
  float* out;          // (batch, sq, d) or NULL
  float* lse;          // (batch, sq) or NULL
  float* out_acc;      // (batch, sq, d) merged in place, or NULL
  float* lse_acc;      // (batch, sq) merged in place, or NULL
  int sq, sk, d, chunks, blocks;  // blocks of 32 R queries of a batch entry
  float scale_log2;    // scale * log2(e)
};

template <int D, int R>
__global__ __launch_bounds__(kThreads, fwd_waves(D, R)) void attn_f32_mfma_fwd_kernel(jg::ChunkTable, F32Params p) {
  typedef Shape<D, R> S;
  constexpr int H = S::H, PITCH = S::PITCH, NT = S::NT, G = S::G;
  extern __shared__ __attribute__((aligned(16))) float smem[];
  const Seat<R> me;
  const int g = me.g, n = me.n;
  float* Ks = smem + me.group * S::GROUP;
  float* Vs = Ks + S::TILE;
  const unsigned id = block_id();
  const long long b = id / (unsigned)p.blocks;
  const int wave_row = (int)(id % (unsigned)p.blocks) * (32 * R) + me.row_wave * 32;
  const bool wave_live = wave_row < p.sq;  // uniform: a wavefront without rows only helps with the tiles
  const int qrow = wave_row + n;
  const bool q_live = qrow < p.sq;
  const long long kv_at = b * (long long)p.sk * p.d;

  float qf[H];  // this lane's slice of its query, scaled
  load_slice<D>(qf, p.q + (b * p.sq + (q_live ? qrow : p.sq - 1)) * (long long)p.d, g, p.d, p.scale_log2);

  f32x16 o[NT];
  clear_acc(o);
  float m = -INFINITY, l = 0.0f;

  const int per_chunk = (p.sk + kBK - 1) / kBK;
  Walk w(me.group, G, per_chunk, p.chunks);
  const int steps = (per_chunk * p.chunks + G - 1) / G;  // of the first group; the others have as many or one less
  Pieces<D, R> kreg, vreg;
  auto fetch = [&]() {
    if (w.left > 0)
      fetch_tiles<D, R>(kreg, vreg, reinterpret_cast<const float*>(jg::chunk_entry(0, w.chunk)) + kv_at,
                        reinterpret_cast<const float*>(jg::chunk_entry(1, w.chunk)) + kv_at, w.step * kBK, p.sk, p.d, me.gt);
  };
  fetch();
  for (int it = 0; it < steps; ++it) {
    const bool mine = w.left > 0;
    const int key0 = w.step * kBK;
    __syncthreads();  // every wavefront is done with the previous tile
    if (mine) store_tiles<D, R>(Ks, Vs, kreg, vreg, me.gt);
    __syncthreads();
    if (!mine) continue;  // (the last iteration, groups behind the first)
    w.advance(G, per_chunk);
    fetch();
    if (!wave_live) continue;

    // S^T[key][query], in units of log2
    f32x16 s;
#pragma unroll
    for (int i = 0; i < 16; ++i) s[i] = 0.0f;
#pragma unroll
    for (int j = 0; j < H; j += 4) {
      const f32x4 kv = *reinterpret_cast<const f32x4*>(Ks + n * PITCH + g * H + j);
      s = __builtin_amdgcn_mfma_f32_32x32x2f32(kv.x, qf[j], s, 0, 0, 0);
      s = __builtin_amdgcn_mfma_f32_32x32x2f32(kv.y, qf[j + 1], s, 0, 0, 0);
      s = __builtin_amdgcn_mfma_f32_32x32x2f32(kv.z, qf[j + 2], s, 0, 0, 0);
      s = __builtin_amdgcn_mfma_f32_32x32x2f32(kv.w, qf[j + 3], s, 0, 0, 0);
    }
    if (key0 + kBK > p.sk) {  // a chunk's last, ragged step
#pragma unroll
      for (int i = 0; i < 16; ++i)
        if (key0 + row_of(i, g) >= p.sk) s[i] = -INFINITY;
    }
    float mx = s[0];
#pragma unroll
    for (int i = 1; i < 16; ++i) mx = fmaxf(mx, s[i]);
    mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
    const float m_new = fmaxf(m, mx);
    const float ms = m_new == -INFINITY ? 0.0f : m_new;  // steps whose scores are all -inf (infinite keys) weigh nothing
    const float alpha = __builtin_amdgcn_exp2f(m - ms);
    float sum = 0.0f;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      s[i] = __builtin_amdgcn_exp2f(s[i] - ms);
      sum += s[i];
    }
    sum += __shfl_xor(sum, 32, 64);
    l = l * alpha + sum;
    m = m_new;
    add_step<NT, PITCH>(o, Vs + n, s, g, alpha);  // O^T[dv][query] += V^T P^T
  }

  if (G > 1) {  // the groups' results by their maxima, in the order of the groups
    constexpr int PART = (NT * 16 + 2) * 64;
    __syncthreads();
    if (me.group > 0) {
      float* at = smem + ((me.group - 1) * R + me.row_wave) * PART + me.lane;
      put_acc(at, o);
      at[NT * 16 * 64] = m;
      at[(NT * 16 + 1) * 64] = l;
    }
    __syncthreads();
    if (me.group > 0) return;
#pragma unroll
    for (int k = 1; k < G; ++k) {
      const float* at = smem + ((k - 1) * R + me.row_wave) * PART + me.lane;
      const float mk = at[NT * 16 * 64], lk = at[(NT * 16 + 1) * 64];
      if (per_chunk * p.chunks <= k) break;  // a group that had no step
      const float top = fmaxf(m, mk), ts = top == -INFINITY ? 0.0f : top;
      const float mine = __builtin_amdgcn_exp2f(m - ts), other = __builtin_amdgcn_exp2f(mk - ts);
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int i = 0; i < 16; ++i) o[t][i] *= mine;
      add_acc(o, at, other);
      l = l * mine + lk * other;
      m = top;
    }
  }
  if (!q_live) return;
  const bool none = l == 0.0f;  // no finite score: out 0, lse -inf, no weight in a merge (a score that is NaN makes l NaN)
  const float inv = none ? 0.0f : 1.0f / l;
  const float lse_j = none ? -INFINITY : fmaf(m, 0.6931471805599453f, __builtin_amdgcn_logf(l) * 0.6931471805599453f);  // v_log_f32 is log2
  const long long qi = b * p.sq + qrow;
  float wt = 0.0f;
  if (p.out_acc != nullptr && !none) {
    const float l_old = p.lse_acc[qi];
    wt = 1.0f / (1.0f + expf(l_old - lse_j));  // sigmoid(lse_j - l_old); l_old = -inf -> 1
    if (g == 0) p.lse_acc[qi] = fmaxf(l_old, lse_j) + log1pf(expf(-fabsf(l_old - lse_j)));
  }
  if (g == 0 && p.lse != nullptr) p.lse[qi] = lse_j;
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int i4 = 0; i4 < 4; ++i4) {
      const int c = 32 * t + 8 * i4 + 4 * g;
      if (c >= p.d) continue;
      const long long at = qi * p.d + c;
      f32x4 val = {o[t][4 * i4] * inv, o[t][4 * i4 + 1] * inv, o[t][4 * i4 + 2] * inv, o[t][4 * i4 + 3] * inv};
      if (p.out != nullptr) *reinterpret_cast<f32x4*>(p.out + at) = val;
      if (p.out_acc != nullptr) {
        f32x4 a = *reinterpret_cast<const f32x4*>(p.out_acc + at);
        a.x += wt * (val.x - a.x);
        a.y += wt * (val.y - a.y);
        a.z += wt * (val.z - a.z);
        a.w += wt * (val.w - a.w);
        *reinterpret_cast<f32x4*>(p.out_acc + at) = a;
      }
    }
}

// ------------------------------------------------------------------ backward
// From the global output and LSE (cores/math.py:125-149): delta = rowsum(dO * O),
// P = exp(S - lse), dS = P * (dO V^T - delta), dQ = scale dS K, dK = scale dS^T Q, dV = P^T dO.
// Two kernels with the forward's operand placement. attn_f32_mfma_dq_kernel: a wavefront owns 32
// queries (a lane: one query, 16 keys a step), S^T = K Q^T and dP^T = V dO^T with the Q and dO
// slices in registers, then dQ^T += K^T dS^T with dS^T as it lies in the registers, over all chunks; it
// leaves delta for the other. attn_f32_mfma_dkv_kernel: a wavefront owns 32 keys (a lane: one key, 16 queries a
// step) of one chunk, S = Q K^T and dP = dO V^T with the K and V slices in registers, then dV^T += dO^T P and
// dK^T += Q^T dS. Both recompute S and dP (6 + 8 matrix products of 32 x 32 x D per tile pair for
// the 5 the mathematics needs once).
struct F32BwdParams {
  float* dq;           // (batch, sq, d)
  const float* dout;   // (batch, sq, d)
  const float* q;
  const float* out;
  const float* lse;    // (batch, sq) natural log
  float* delta;        // (batch, sq)
  int sq, sk, d, chunks, blocks;  // blocks of 32 R resident rows
  float scale, scale_log2;
};

template <int D, int NT>
__device__ __forceinline__ void store_rows(float* row, const f32x16 (&acc)[NT], int g, int d, float mul) {
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int i4 = 0; i4 < 4; ++i4) {
      const int c = 32 * t + 8 * i4 + 4 * g;
      if (c >= d) continue;
      const f32x4 val = {acc[t][4 * i4] * mul, acc[t][4 * i4 + 1] * mul, acc[t][4 * i4 + 2] * mul, acc[t][4 * i4 + 3] * mul};
      *reinterpret_cast<f32x4*>(row + c) = val;
    }
}

template <int D, int R>
__global__ __launch_bounds__(kThreads, dq_waves(D, R)) void attn_f32_mfma_dq_kernel(jg::ChunkTable, F32BwdParams p) {
  typedef Shape<D, R> S;
  constexpr int H = S::H, PITCH = S::PITCH, NT = S::NT, G = S::G;
  extern __shared__ __attribute__((aligned(16))) float smem[];
  const Seat<R> me;
  const int g = me.g, n = me.n;
  float* Ks = smem + me.group * S::GROUP;
  float* Vs = Ks + S::TILE;
  const unsigned id = block_id();
  const long long b = id / (unsigned)p.blocks;
  const int wave_row = (int)(id % (unsigned)p.blocks) * (32 * R) + me.row_wave * 32;
  const bool wave_live = wave_row < p.sq;
  const int qrow = wave_row + n;
  const bool q_live = qrow < p.sq;
  const long long qi = b * p.sq + (q_live ? qrow : p.sq - 1);
  const long long kv_at = b * (long long)p.sk * p.d;

  float qf[H], dof[H];
  load_slice<D>(qf, p.q + qi * p.d, g, p.d, p.scale_log2);
  load_slice<D>(dof, p.dout + qi * p.d, g, p.d, 1.0f);
  const float lse2 = p.lse[qi] * 1.4426950408889634f;
  float dl = 0.0f;
#pragma unroll
  for (int j = 0; j < H; j += 4) {
    const bool there = g * H + j < p.d;
    const f32x4 t = *reinterpret_cast<const f32x4*>(p.out + qi * p.d + (there ? g * H + j : 0));
    if (there) dl += dof[j] * t.x + dof[j + 1] * t.y + dof[j + 2] * t.z + dof[j + 3] * t.w;
  }
  dl += __shfl_xor(dl, 32, 64);
  if (me.group == 0 && g == 0 && q_live) p.delta[qi] = dl;

  f32x16 dq[NT];
  clear_acc(dq);
  const int per_chunk = (p.sk + kBK - 1) / kBK;
  Walk w(me.group, G, per_chunk, p.chunks);
  const int steps = (per_chunk * p.chunks + G - 1) / G;
  Pieces<D, R> kreg, vreg;
  auto fetch = [&]() {
    if (w.left > 0)
      fetch_tiles<D, R>(kreg, vreg, reinterpret_cast<const float*>(jg::chunk_entry(0, w.chunk)) + kv_at,
                        reinterpret_cast<const float*>(jg::chunk_entry(1, w.chunk)) + kv_at, w.step * kBK, p.sk, p.d, me.gt);
  };
  fetch();
  for (int it = 0; it < steps; ++it) {
    const bool mine = w.left > 0;
    const int key0 = w.step * kBK;
    __syncthreads();
    if (mine) store_tiles<D, R>(Ks, Vs, kreg, vreg, me.gt);
    __syncthreads();
    if (!mine) continue;
    w.advance(G, per_chunk);
    fetch();
    if (!wave_live) continue;

    f32x16 s, dp;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      s[i] = 0.0f;
      dp[i] = 0.0f;
    }
#pragma unroll
    for (int j = 0; j < H; j += 4) {
      const f32x4 kv = *reinterpret_cast<const f32x4*>(Ks + n * PITCH + g * H + j);
      const f32x4 vv = *reinterpret_cast<const f32x4*>(Vs + n * PITCH + g * H + j);
      s = __builtin_amdgcn_mfma_f32_32x32x2f32(kv.x, qf[j], s, 0, 0, 0);
      dp = __builtin_amdgcn_mfma_f32_32x32x2f32(vv.x, dof[j], dp, 0, 0, 0);
      s = __builtin_amdgcn_mfma_f32_32x32x2f32(kv.y, qf[j + 1], s, 0, 0, 0);
      dp = __builtin_amdgcn_mfma_f32_32x32x2f32(vv.y, dof[j + 1], dp, 0, 0, 0);
      s = __builtin_amdgcn_mfma_f32_32x32x2f32(kv.z, qf[j + 2], s, 0, 0, 0);
      dp = __builtin_amdgcn_mfma_f32_32x32x2f32(vv.z, dof[j + 2], dp, 0, 0, 0);
      s = __builtin_amdgcn_mfma_f32_32x32x2f32(kv.w, qf[j + 3], s, 0, 0, 0);
      dp = __builtin_amdgcn_mfma_f32_32x32x2f32(vv.w, dof[j + 3], dp, 0, 0, 0);
    }
    const bool ragged = key0 + kBK > p.sk;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      float pr = __builtin_amdgcn_exp2f(s[i] - lse2);
      if (ragged && key0 + row_of(i, g) >= p.sk) pr = 0.0f;
      s[i] = pr * (dp[i] - dl);  // dS^T
    }
    add_step<NT, PITCH>(dq, Ks + n, s, g, 1.0f);
  }
  if (G > 1) {
    constexpr int PART = NT * 16 * 64;
    __syncthreads();
    if (me.group > 0) put_acc(smem + ((me.group - 1) * R + me.row_wave) * PART + me.lane, dq);
    __syncthreads();
    if (me.group > 0) return;
#pragma unroll
    for (int k = 1; k < G; ++k) add_acc(dq, smem + ((k - 1) * R + me.row_wave) * PART + me.lane, 1.0f);
  }
  if (q_live) store_rows<D>(p.dq + qi * p.d, dq, g, p.d, p.scale);
}

template <int D, int R>
__global__ __launch_bounds__(kThreads) void attn_f32_mfma_dkv_kernel(jg::ChunkTable, F32BwdParams p) {
  typedef Shape<D, R> S;
  constexpr int H = S::H, PITCH = S::PITCH, NT = S::NT, G = S::G;
  extern __shared__ __attribute__((aligned(16))) float smem[];
  const Seat<R> me;
  const int g = me.g, n = me.n;
  float* Qs = smem + me.group * S::GROUP;
  float* dOs = Qs + S::TILE;
  float* lse2s = dOs + S::TILE;
  float* deltas = lse2s + kBK;
  const unsigned id = block_id(), per_entry = (unsigned)p.blocks * (unsigned)p.chunks;
  const long long b = id / per_entry;
  const int chunk = __builtin_amdgcn_readfirstlane((int)(id % per_entry / (unsigned)p.blocks));
  const int wave_row = (int)(id % (unsigned)p.blocks) * (32 * R) + me.row_wave * 32;
  const bool wave_live = wave_row < p.sk;
  const int krow = wave_row + n;
  const bool k_live = krow < p.sk;
  const long long ki = b * p.sk + (k_live ? krow : p.sk - 1);
  const float* qb_base = p.q + b * (long long)p.sq * p.d;
  const float* dob_base = p.dout + b * (long long)p.sq * p.d;
  const float* lse_base = p.lse + b * (long long)p.sq;
  const float* delta_base = p.delta + b * (long long)p.sq;

  float kf[H], vf[H];
  load_slice<D>(kf, reinterpret_cast<const float*>(jg::chunk_entry(0, chunk)) + ki * p.d, g, p.d, p.scale_log2);
  load_slice<D>(vf, reinterpret_cast<const float*>(jg::chunk_entry(1, chunk)) + ki * p.d, g, p.d, 1.0f);
  f32x16 dk[NT], dv[NT];
  clear_acc(dk);
  clear_acc(dv);

  const int per_chunk = (p.sq + kBK - 1) / kBK;  // here the steps run over the queries, once
  Walk w(me.group, G, per_chunk, 1);
  const int steps = (per_chunk + G - 1) / G;
  Pieces<D, R> qreg, doreg;
  float lreg = 0.0f, dreg = 0.0f;
  auto fetch = [&]() {
    if (w.left <= 0) return;
    fetch_tiles<D, R>(qreg, doreg, qb_base, dob_base, w.step * kBK, p.sq, p.d, me.gt);
    if (me.gt < kBK) {  // the 32 queries' lse (in log2 units) and delta; 0 past the end
      const int r = w.step * kBK + me.gt;
      lreg = r < p.sq ? lse_base[r] * 1.4426950408889634f : 0.0f;
      dreg = r < p.sq ? delta_base[r] : 0.0f;
    }
  };
  fetch();
  for (int it = 0; it < steps; ++it) {
    const bool mine = w.left > 0;
    const int q0 = w.step * kBK;
    __syncthreads();
    if (mine) {
      store_tiles<D, R>(Qs, dOs, qreg, doreg, me.gt);
      if (me.gt < kBK) {
        lse2s[me.gt] = lreg;
        deltas[me.gt] = dreg;
      }
    }
    __syncthreads();
    if (!mine) continue;
    w.step += G;
    --w.left;
    fetch();
    if (!wave_live) continue;

    f32x16 s, dp;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      s[i] = 0.0f;
      dp[i] = 0.0f;
    }
#pragma unroll
    for (int j = 0; j < H; j += 4) {
      const f32x4 qv = *reinterpret_cast<const f32x4*>(Qs + n * PITCH + g * H + j);
      const f32x4 gv = *reinterpret_cast<const f32x4*>(dOs + n * PITCH + g * H + j);
      s = __builtin_amdgcn_mfma_f32_32x32x2f32(qv.x, kf[j], s, 0, 0, 0);
      dp = __builtin_amdgcn_mfma_f32_32x32x2f32(gv.x, vf[j], dp, 0, 0, 0);
      s = __builtin_amdgcn_mfma_f32_32x32x2f32(qv.y, kf[j + 1], s, 0, 0, 0);
      dp = __builtin_amdgcn_mfma_f32_32x32x2f32(gv.y, vf[j + 1], dp, 0, 0, 0);
      s = __builtin_amdgcn_mfma_f32_32x32x2f32(qv.z, kf[j + 2], s, 0, 0, 0);
      dp = __builtin_amdgcn_mfma_f32_32x32x2f32(gv.z, vf[j + 2], dp, 0, 0, 0);
      s = __builtin_amdgcn_mfma_f32_32x32x2f32(qv.w, kf[j + 3], s, 0, 0, 0);
      dp = __builtin_amdgcn_mfma_f32_32x32x2f32(gv.w, vf[j + 3], dp, 0, 0, 0);
    }
    const bool ragged = q0 + kBK > p.sq;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int qr = row_of(i, g);
      float pr = __builtin_amdgcn_exp2f(s[i] - lse2s[qr]);
      if (ragged && q0 + qr >= p.sq) pr = 0.0f;
      s[i] = pr;                          // P
      dp[i] = pr * (dp[i] - deltas[qr]);  // dS
    }
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const float* gorow = dOs + row_of(i, g) * PITCH + n;
      const float* qrow_ = Qs + row_of(i, g) * PITCH + n;
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        dv[t] = __builtin_amdgcn_mfma_f32_32x32x2f32(gorow[32 * t], s[i], dv[t], 0, 0, 0);
        dk[t] = __builtin_amdgcn_mfma_f32_32x32x2f32(qrow_[32 * t], dp[i], dk[t], 0, 0, 0);
      }
    }
  }
  if (G > 1) {
    constexpr int PART = 2 * NT * 16 * 64;
    __syncthreads();
    if (me.group > 0) {
      float* at = smem + ((me.group - 1) * R + me.row_wave) * PART + me.lane;
      put_acc(at, dk);
      put_acc(at + NT * 16 * 64, dv);
    }
    __syncthreads();
    if (me.group > 0) return;
#pragma unroll
    for (int k = 1; k < G; ++k) {
      const float* at = smem + ((k - 1) * R + me.row_wave) * PART + me.lane;
      add_acc(dk, at, 1.0f);
      add_acc(dv, at + NT * 16 * 64, 1.0f);
    }
  }
  if (!k_live) return;
  store_rows<D>(reinterpret_cast<float*>(const_cast<char*>(jg::chunk_entry(2, chunk))) + ki * p.d, dk, g, p.d, p.scale);
  store_rows<D>(reinterpret_cast<float*>(const_cast<char*>(jg::chunk_entry(3, chunk))) + ki * p.d, dv, g, p.d, 1.0f);
}

bool aligned16(const void* ptr) { return (reinterpret_cast<uintptr_t>(ptr) & 15) == 0; }

// Resident rows of a workgroup, in wavefronts: what the busiest compute unit has to do (its workgroups, each R / 4 of the
// streamed side long, whether they run beside each other or in turn), a little more where the streamed side is read more often,
// a little less at 32 columns, where several workgroups of one wavefront's tiles fit a compute unit. Forward / dQ / dK and dV, us,
// one against two wavefronts of rows where both leave two units of work, each summed in one chain: 45 x 171 x 6 chunks at 32 34 / 45 / - and
// 39 / 50 / -, 16 x 700 x 4 at 64 126 / 208 and 141 / 183, 12 x 800 x 3 at 96 302 / 364 and 165 / 219. Whole steps before (a launch a chunk of
// 128 rows each, 96 columns as 128 with copies) and now: 322 -> 122, 1061 -> 501, 1960 -> 594; a launch that filled the chip 1963 -> 1892
// (64 x 1000 x 3 at 64: 0.09 PFLOP/s of the matrix cores' 0.16).
int width(long long rows, long long entries, int d, int least) {
  int best = 4;
  long long best_cost = -1;
  for (int r = 4; r >= least; r /= 2) {
    const long long cost = jg::cdiv(jg::cdiv(rows, 32 * r) * entries, jg::cu_count()) * (long long)r * (d <= 32 ? (r == 1 ? 97 : 100) : r == 4 ? 100 : r == 2 ? 103 : 110);
    if (best_cost < 0 || cost < best_cost) {
      best = r;
      best_cost = cost;
    }
  }
  return best;
}

// kernel<D, R><<<>>> for run-time d and R
#define JG_F32_LAUNCH(KERNEL, DD, RR, BLOCKS, ...)                                                                             \
  do {                                                                                                                         \
    typedef Shape<DD, RR> S_;                                                                                                  \
    if (S_::LDS > 65536 && hipFuncSetAttribute(reinterpret_cast<const void*>(&KERNEL<DD, RR>),                                 \
                                               hipFuncAttributeMaxDynamicSharedMemorySize, S_::LDS) != hipSuccess)             \
      JG_FAIL(JG_ERR_LAUNCH, "jg_attn(fp32 mfma): cannot reserve %d bytes of LDS", S_::LDS);                                   \
    KERNEL<DD, RR><<<(unsigned)(BLOCKS), kThreads, S_::LDS, s>>>(__VA_ARGS__);                                                 \
  } while (0)
#define JG_F32_WIDTHS(KERNEL, DD, R, BLOCKS, ...)                              \
  do {                                                                         \
    if (R == 1) JG_F32_LAUNCH(KERNEL, DD, 1, BLOCKS, __VA_ARGS__);             \
    else if (R == 2) JG_F32_LAUNCH(KERNEL, DD, 2, BLOCKS, __VA_ARGS__);        \
    else JG_F32_LAUNCH(KERNEL, DD, 4, BLOCKS, __VA_ARGS__);                    \
  } while (0)
#define JG_F32_GO(KERNEL, D, R, BLOCKS, ...)                                   \
  do {                                                                         \
    if (D <= 32) JG_F32_WIDTHS(KERNEL, 32, R, BLOCKS, __VA_ARGS__);            \
    else if (D <= 64) JG_F32_WIDTHS(KERNEL, 64, R, BLOCKS, __VA_ARGS__);       \
    else if (D <= 96) JG_F32_WIDTHS(KERNEL, 96, R, BLOCKS, __VA_ARGS__);       \
    else JG_F32_WIDTHS(KERNEL, 128, R, BLOCKS, __VA_ARGS__);                   \
  } while (0)

}  // namespace

namespace jg {

bool attn_f32_mfma_supported(long long batch, int sq, int sk, int d, int chunks, int dtype, bool has_bias) {
  if (dtype != JG_F32 || has_bias || batch <= 0 || sq <= 0 || sk <= 0) return false;
  if (d < 4 || d > 128 || d % 4 != 0) return false;
  // workgroups of 32 rows, and the steps of all chunks, in 31 bits
  return batch < (1ll << 31) && batch * cdiv((long long)sq, 32ll) < (1ll << 31) && batch * chunks * cdiv((long long)sk, 32ll) < (1ll << 31);
}

int attn_f32_mfma_fwd_chunks(void* out, float* lse, const void* q, const void* const* k, const void* const* v, int chunks,
                             long long batch, int sq, int sk, int d, float scale, float* out_acc, float* lse_acc, hipStream_t s) {
  for (const void* ptr : {static_cast<const void*>(out), q, static_cast<const void*>(out_acc)})
    JG_REQUIRE(aligned16(ptr), "jg_attn_fwd: the fp32 matrix-core kernel needs 16-byte aligned tensors");
  const ChunkTable tab = chunk_table(k, v, nullptr, nullptr, chunks);
  const int r = width(sq, batch, d, 1);
  F32Params p = {};
  p.q = static_cast<const float*>(q);
  p.out = static_cast<float*>(out);
  p.lse = lse;
  p.out_acc = out_acc;
  p.lse_acc = lse_acc;
  p.sq = sq;
  p.sk = sk;
  p.d = d;
  p.chunks = chunks;
  p.blocks = (int)cdiv((long long)sq, 32ll * r);
  p.scale_log2 = scale * 1.4426950408889634f;
  JG_F32_GO(attn_f32_mfma_fwd_kernel, d, r, batch * p.blocks, tab, p);
  JG_CHECK_LAUNCH("jg_attn_fwd(fp32 mfma)");
  return JG_OK;
}

// workspace: (batch, sq) floats for delta
int attn_f32_mfma_bwd_chunks(void* dq, void* const* dk, void* const* dv, const void* dout, const void* q, const void* const* k,
                             const void* const* v, int chunks, const void* out, const float* lse, long long batch, int sq, int sk,
                             int d, float scale, void* workspace, hipStream_t s) {
  for (const void* ptr : {static_cast<const void*>(dq), dout, q, out})
    JG_REQUIRE(aligned16(ptr), "jg_attn_bwd: the fp32 matrix-core kernels need 16-byte aligned tensors");
  const ChunkTable tab = chunk_table(k, v, dk, dv, chunks);
  F32BwdParams p = {};
  p.dq = static_cast<float*>(dq);
  p.dout = static_cast<const float*>(dout);
  p.q = static_cast<const float*>(q);
  p.out = static_cast<const float*>(out);
  p.lse = lse;
  p.delta = static_cast<float*>(workspace);
  p.sq = sq;
  p.sk = sk;
  p.d = d;
  p.chunks = chunks;
  p.scale = scale;
  p.scale_log2 = scale * 1.4426950408889634f;
  // (dK / dV at 128 columns: no registers for tiles that one wavefront fetches alone)
  const int rq = width(sq, batch, d, 1), rk = width(sk, batch * chunks, d, d > 96 ? 2 : 1);
  p.blocks = (int)cdiv((long long)sq, 32ll * rq);
  JG_F32_GO(attn_f32_mfma_dq_kernel, d, rq, batch * p.blocks, tab, p);
  JG_CHECK_LAUNCH("jg_attn_bwd(fp32 mfma dq)");
  p.blocks = (int)cdiv((long long)sk, 32ll * rk);
  JG_F32_GO(attn_f32_mfma_dkv_kernel, d, rk, batch * chunks * p.blocks, tab, p);
  JG_CHECK_LAUNCH("jg_attn_bwd(fp32 mfma dk dv)");
  return JG_OK;
}

}  // namespace jg
