// Shared helpers for the jigsaw HIP kernels (gfx950 only).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <stdio.h>
#include <string.h>

#include "../../include/jigsaw_hip.h"

namespace jg {

// Thread-local message of the most recent failure on this host thread.
char* last_error_buf();
void set_error(const char* fmt, ...);

#define JG_FAIL(code, ...)        \
  do {                            \
    ::jg::set_error(__VA_ARGS__); \
    return (code);                \
  } while (0)

#define JG_REQUIRE(cond, ...)                         \
  do {                                                \
    if (!(cond)) JG_FAIL(JG_ERR_BAD_ARG, __VA_ARGS__); \
  } while (0)

// Launch check: picks up a launch-time error without synchronising the device.
#define JG_CHECK_LAUNCH(name)                                              \
  do {                                                                     \
    hipError_t e__ = hipGetLastError();                                    \
    if (e__ != hipSuccess)                                                 \
      JG_FAIL(JG_ERR_LAUNCH, "%s: launch failed: %s", (name),              \
              hipGetErrorString(e__));                                     \
  } while (0)

static inline size_t dtype_size(int dtype) {
  switch (dtype) {
    case JG_F32: return 4;
    case JG_BF16: return 2;
    case JG_F16: return 2;
    default: return 0;
  }
}

// ---- bf16 <-> f32 (round to nearest even, NaN kept quiet), as torch rounds ----
__host__ __device__ static inline float bf16_to_f32(uint16_t h) {
  union { uint32_t u; float f; } c;
  c.u = ((uint32_t)h) << 16;
  return c.f;
}
__host__ __device__ static inline uint16_t f32_to_bf16(float f) {
  union { uint32_t u; float f; } c;
  c.f = f;
  if ((c.u & 0x7fffffffu) > 0x7f800000u) return (uint16_t)0x7fc0;
  uint32_t r = c.u + 0x7fffu + ((c.u >> 16) & 1u);
  return (uint16_t)(r >> 16);
}

// Division by a number that holds for a whole launch, of numbers below 2^31: m = 2^(32 + s) / d rounded up, s < 0 for d = 1. A division of
// the compiler's own is 30 instructions and more, over 100 in 64 bits, and a tile's place takes half a dozen of them.
struct Div {
  uint32_t m;
  int s;
};
inline Div div_by(int d) {
  if (d <= 1) return {0u, -1};
  int bits = 0;
  while ((1ll << bits) < d) ++bits;
  return {(uint32_t)(((1ull << (31 + bits)) + d - 1) / d), bits - 1};
}
__device__ __forceinline__ uint32_t quotient(uint32_t n, const Div& d) { return d.s < 0 ? n : __umulhi(n, d.m) >> d.s; }

static inline int cdiv(int64_t a, int64_t b) { return (int)((a + b - 1) / b); }

// Compute units of the device (of a partition of it, where the device is one): what the host-side rules that fill the
// chip count with. Asked once; 256, a whole MI355X, where there is no device to ask (sizes of workspaces on the CPU).
inline int cu_count() {
  static const int count = [] {
    int dev = 0, n = 0;
    return hipGetDevice(&dev) == hipSuccess && hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess && n > 0 ? n : 256;
  }();
  return count;
}

}  // namespace jg
