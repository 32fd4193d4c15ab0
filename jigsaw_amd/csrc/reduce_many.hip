// Every sum of partials that a backward has left, in one launch. On its own each is 4 to 6 us, most of it the start and the
// end of the launch: the eight of a Swin block's backward took 39 us at 65536 tokens of 128 channels, together they take
// 20 (60 MB of partials, which by then come from the last-level cache), at 4480 tokens of 256 channels 32 and 10.
// The step 466 -> 455 us, 4 x 104 x 232 tokens of 96 channels 496 -> 475, 2 x 40 x 56 of 256 (host time) 313 -> 298.
#include "reductions.h"

namespace {

struct ManyArgs {
  jg_reduction job[JG_MOST_REDUCTIONS];
  unsigned end[JG_MOST_REDUCTIONS];  // blocks of this job and the ones before it
};

__global__ __launch_bounds__(jg::RED_THREADS) void reduce_many_kernel(ManyArgs a) {
  __shared__ jg::ReduceShared sm;
  int m = 0;
  while (blockIdx.x >= a.end[m]) ++m;
  const unsigned block = blockIdx.x - (m == 0 ? 0 : a.end[m - 1]);
  const jg_reduction r = a.job[m];
  float* const out = r.out;
  float* const out2 = r.out2;
  if (r.kind == jg::RED_SLICES) {
    const bool vec = jg::slices_vec(r.part, out, (size_t)r.count);
    const size_t count = (size_t)r.count;
    auto store = [=](size_t i, float4 t) {
      if (vec) {
        *reinterpret_cast<float4*>(out + i) = t;
      } else {
        const float v[4] = {t.x, t.y, t.z, t.w};
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (i + e < count) out[i + e] = v[e];
      }
    };
    const int wave = threadIdx.x >> 6, q = threadIdx.x & 63;
    if (jg::slice_waves(r.parts) == 16) jg::reduce_slices<16>(sm.slices, r.part, count, r.parts, vec, block, wave, q, store);
    else jg::reduce_slices<4>(sm.slices + wave / 4 * 4, r.part, count, r.parts, vec, (size_t)block * 4 + wave / 4, wave % 4, q, store);
  } else if (r.kind == jg::RED_COLUMNS) {
    jg::reduce_columns(sm.columns, r.part, r.parts, r.count, block, [=](long long c, float w, float b) {
      if (out != nullptr) out[c] = w;
      if (out2 != nullptr) out2[c] = b;
    });
  } else {
    jg::reduce_table(sm.table, r.part, out, r.parts, (int)r.count, block);
  }
}

}  // namespace

extern "C" int jg_reduce_many(const jg_reductions* all, void* stream) {
  const char* who = "jg_reduce_many";
  JG_REQUIRE(all != nullptr && all->n >= 0 && all->n <= JG_MOST_REDUCTIONS, "%s: bad list", who);
  ManyArgs a = {};
  unsigned long long blocks = 0;
  for (int i = 0; i < all->n; ++i) {
    const jg_reduction& r = all->job[i];
    JG_REQUIRE(r.kind >= 0 && r.kind <= 2 && r.part != nullptr && r.count > 0 && r.parts >= 0 && (r.out != nullptr || (r.kind == jg::RED_COLUMNS && r.out2 != nullptr)),
               "%s: job %d", who, i);
    a.job[i] = r;
    blocks += jg::reduction_blocks(r);
    JG_REQUIRE(blocks < (1ull << 31), "%s: too large", who);
    a.end[i] = (unsigned)blocks;
  }
  if (blocks == 0) return JG_OK;
  reduce_many_kernel<<<(unsigned)blocks, jg::RED_THREADS, 0, static_cast<hipStream_t>(stream)>>>(a);
  JG_CHECK_LAUNCH(who);
  return JG_OK;
}
