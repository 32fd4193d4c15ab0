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

// Workgroup -> (batch entry, chunk, row block) of a grid (row blocks, batch entries, chunks). Consecutive
// workgroup ids go to the 8 XCDs in turn; each XCD is given a contiguous range of the flat order (batch entry,
// chunk, block), so the workgroups that stream the same K / V (or Q / dO) share one L2 instead of every L2
// holding every head. Falls back to the plain order when the count does not divide.
struct BlockOf {
  long long bh;
  int blk;
  int chunk;
};
__device__ __forceinline__ BlockOf block_of() {
  const unsigned nblk = gridDim.x, nch = gridDim.z, total = gridDim.x * gridDim.y * gridDim.z;
  unsigned id = (blockIdx.y * nch + blockIdx.z) * nblk + blockIdx.x;
  if ((total & 7u) == 0) id = (id & 7u) * (total >> 3) + (id >> 3);
  BlockOf b;
  b.blk = (int)(id % nblk);
  id /= nblk;
  b.chunk = (int)(id % nch);
  b.bh = id / nch;
  return b;
}

}  // namespace jg
