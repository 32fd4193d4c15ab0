// Memory -> LDS without registers (global_load_lds_dwordx4): one instruction of a wavefront lands 64 x 16 bytes contiguously, in lane order,
// at the LDS address in M0. Written in assembly: with the compiler's own form it waits for ALL outstanding transfers before every LDS
// read. The kernels order reads and transfers themselves, by their waits and barriers.
//
// The transfer reads M0 one wait state after a scalar instruction wrote it at the earliest: the compiler puts an s_nop between the two where
// it emits them itself, but does not look inside an asm statement. M0 is named as clobbered, so that no value of the compiler's own lives in it;
// memory is not: what was read in LDS before and what is read behind are kept apart by the waits and barriers, other accesses may move.
#pragma once
#include "jg_common.h"

namespace jg {

// A wave-uniform base plus a 32-bit byte offset of the lane; lds_dst: LDS address of the 1 KB block, wave-uniform.
__device__ __forceinline__ void to_lds_1k(const void* base, uint32_t lane_off, uint32_t lds_dst) {
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" : : "v"(lane_off), "s"(base), "s"(lds_dst) : "m0");
}
// The same for tensors of 2^32 bytes and more: 64-bit offsets, added to the base lane by lane.
__device__ __forceinline__ void to_lds_1k(const void* base, uint64_t lane_off, uint32_t lds_dst) {
  const char* at = static_cast<const char*>(base) + lane_off;
  asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" : : "v"(at), "s"(lds_dst) : "m0");
}
__device__ __forceinline__ uint32_t lds_address(const void* p) {
  typedef const __attribute__((address_space(3))) unsigned char* lds_bytes;
  return (uint32_t)(uintptr_t)((lds_bytes)p);
}

}  // namespace jg
