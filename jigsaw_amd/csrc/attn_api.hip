// C entry points of the attention core: validate and route to the MFMA flash
// kernels (bf16 at head size 64; bf16 / fp16 at any head size that is a multiple of 8, up to 128)
// when they cover the problem, to the window or generic kernels otherwise.
#include <initializer_list>

#include "attn_chunks.h"

namespace jg {
bool attn_generic_supported(int d);
int attn_generic_fwd(void* out, float* lse, const void* q, const void* k, const void* v,
                     long long batch, int sq, int sk, int d, float scale, const float* bias,
                     long long bias_period, int dtype, hipStream_t s);
int attn_generic_bwd(void* dq, void* dk, void* dv, float* delta, float* dbias, const void* dout,
                     const void* q, const void* k, const void* v, const void* out,
                     const float* lse, long long batch, int sq, int sk, int d, float scale,
                     const float* bias, long long bias_period, int dtype, hipStream_t s);
bool attn_mfma_fwd_supported(long long batch, int sq, int sk, int d, int dtype, bool has_bias);
int attn_mfma_fwd_chunks(void* out, float* lse, const void* q, const void* const* k, const void* const* v, int nchunks,
                         long long batch, int sq, int sk, float scale, float* out_acc, float* lse_acc, hipStream_t s);
bool attn_mfma_bwd_supported(long long batch, int sq, int sk, int d, int dtype, bool has_bias);
int attn_mfma_bwd_chunks(void* dq, void* const* dk, void* const* dv, const void* dout, const void* q,
                         const void* const* k, const void* const* v, int nchunks, const void* out, const float* lse,
                         long long batch, int sq, int sk, float scale, void* ws, hipStream_t s);
int attn_mfma_bwd_one_launch_width(long long batch, int sq, int sk, int nchunks);
bool attn_wide_supported(long long batch, int sq, int sk, int d, int dtype, bool has_bias);
bool attn_f32_mfma_supported(long long batch, int sq, int sk, int d, int chunks, int dtype, bool has_bias);
int attn_f32_mfma_fwd_chunks(void* out, float* lse, const void* q, const void* const* k, const void* const* v, int chunks,
                             long long batch, int sq, int sk, int d, float scale, float* out_acc, float* lse_acc, hipStream_t s);
int attn_f32_mfma_bwd_chunks(void* dq, void* const* dk, void* const* dv, const void* dout, const void* q, const void* const* k,
                             const void* const* v, int chunks, const void* out, const float* lse, long long batch, int sq, int sk,
                             int d, float scale, void* workspace, hipStream_t s);
bool attn_window_supported(long long batch, int sq, int sk, int d, int dtype);
int attn_window_fwd(void* out, float* lse, const void* q, const void* k, const void* v,
                    long long batch, float scale, const float* bias, long long bias_period,
                    hipStream_t s);
int attn_window_bwd(void* dq, void* dk, void* dv, float* dbias, const void* dout, const void* q,
                    const void* k, const void* v, const void* out, const float* lse,
                    long long batch, float scale, const float* bias, long long bias_period,
                    hipStream_t s);
}  // namespace jg

namespace {
bool known(int dt) { return dt == JG_F32 || dt == JG_BF16 || dt == JG_F16; }

int check_shape(const char* who, int64_t batch, int64_t sq, int64_t sk, int64_t d, float scale,
                int dtype) {
  JG_REQUIRE(known(dtype), "%s: unknown dtype %d", who, dtype);
  JG_REQUIRE(batch >= 0 && sq >= 0 && sk >= 1 && d >= 1, "%s: bad shape", who);
  JG_REQUIRE(sq < (1ll << 30) && sk < (1ll << 30), "%s: sequence too long", who);
  JG_REQUIRE(scale > 0.0f, "%s: scale must be positive", who);
  return JG_OK;
}

// Every kernel but the one-thread-per-row ones moves 16 bytes per lane.
bool aligned16(std::initializer_list<const void*> ptrs) {
  for (const void* q : ptrs)
    if ((reinterpret_cast<uintptr_t>(q) & 15) != 0) return false;
  return true;
}

// Host arrays of n device pointers, one per chunk.
typedef std::initializer_list<const void* const*> ChunkArrays;
int check_chunks(const char* who, int64_t n, ChunkArrays arrays) {
  if (n > jg::ATTN_MAX_CHUNKS) JG_FAIL(JG_ERR_UNSUPPORTED, "%s: at most %d chunks a call, got %lld", who, jg::ATTN_MAX_CHUNKS, (long long)n);
  for (const void* const* a : arrays) {
    JG_REQUIRE(a, "%s: NULL pointer", who);
    for (int64_t c = 0; c < n; ++c) JG_REQUIRE(a[c], "%s: NULL pointer for chunk %lld", who, (long long)c);
  }
  return JG_OK;
}
bool chunks_aligned16(int64_t n, ChunkArrays arrays) {
  for (const void* const* a : arrays)
    for (int64_t c = 0; c < n; ++c)
      if (!aligned16({a[c]})) return false;
  return true;
}
}  // namespace

extern "C" int jg_attn_fwd(void* out, float* lse, const void* q, const void* k, const void* v,
                           int64_t batch, int64_t sq, int64_t sk, int64_t d, float scale,
                           const float* bias, int64_t bias_period, float* out_acc,
                           float* lse_acc, int dtype, void* stream) {
  const char* who = "jg_attn_fwd";
  int rc = check_shape(who, batch, sq, sk, d, scale, dtype);
  if (rc) return rc;
  JG_REQUIRE(q && k && v, "%s: NULL input", who);
  JG_REQUIRE((out_acc == nullptr) == (lse_acc == nullptr),
             "%s: out_acc and lse_acc go together", who);
  JG_REQUIRE(out_acc != nullptr || (out != nullptr && lse != nullptr),
             "%s: nowhere to write the result", who);
  JG_REQUIRE(bias == nullptr || bias_period >= 1, "%s: bias_period must be >= 1", who);
  if (batch == 0 || sq == 0) return JG_OK;
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (jg::attn_mfma_fwd_supported(batch, (int)sq, (int)sk, (int)d, dtype, bias != nullptr) &&
      aligned16({out, q, k, v, out_acc}))
    return jg::attn_mfma_fwd_chunks(out, lse, q, &k, &v, 1, batch, (int)sq, (int)sk, scale, out_acc, lse_acc, s);
  if (out_acc == nullptr && jg::attn_window_supported(batch, (int)sq, (int)sk, (int)d, dtype) &&
      aligned16({out, q, k, v, bias}))
    return jg::attn_window_fwd(out, lse, q, k, v, batch, scale, bias, bias_period, s);
  if (jg::attn_wide_supported(batch, (int)sq, (int)sk, (int)d, dtype, bias != nullptr) &&
      aligned16({out, q, k, v, out_acc}))
    return jg::attn_wide_fwd_chunks(out, lse, q, &k, &v, 1, batch, (int)sq, (int)sk, (int)d, dtype, scale, out_acc,
                                    lse_acc, s);
  if (jg::attn_f32_mfma_supported(batch, (int)sq, (int)sk, (int)d, 1, dtype, bias != nullptr) &&
      aligned16({out, q, k, v, out_acc}))
    return jg::attn_f32_mfma_fwd_chunks(out, lse, q, &k, &v, 1, batch, (int)sq, (int)sk, (int)d, scale, out_acc, lse_acc, s);
  if (!jg::attn_generic_supported((int)d))
    JG_FAIL(JG_ERR_UNSUPPORTED, "%s: head size %lld not in {8, 16, 32, 64, 96, 128}", who, (long long)d);
  if (out_acc != nullptr)
    JG_FAIL(JG_ERR_UNSUPPORTED,
            "%s: the fused merge needs an MFMA path (bf16 or fp16 with d a multiple of 8 up to 128,"
            " fp32 with d a multiple of 4 up to 128, no bias, 16-byte aligned tensors);"
            " call jg_lse_merge after the core instead", who);
  rc = jg::attn_generic_fwd(out, lse, q, k, v, batch, (int)sq, (int)sk, (int)d, scale, bias,
                            bias_period, dtype, s);
  if (rc) return rc;
  return JG_OK;
}

extern "C" size_t jg_attn_bwd_workspace_bytes(int64_t batch, int64_t sq, int64_t sk, int64_t d) {
  if (batch <= 0 || sq <= 0) return 0;
  (void)sk;
  (void)d;
  // delta (batch, sq) fp32; the MFMA path needs nothing beyond it
  return (size_t)batch * (size_t)sq * sizeof(float);
}

extern "C" int jg_attn_bwd(void* dq, void* dk, void* dv, const void* dout, const void* q,
                           const void* k, const void* v, const void* out, const float* lse,
                           int64_t batch, int64_t sq, int64_t sk, int64_t d, float scale,
                           const float* bias, int64_t bias_period, float* dbias, int dtype,
                           void* workspace, size_t workspace_bytes, void* stream) {
  const char* who = "jg_attn_bwd";
  int rc = check_shape(who, batch, sq, sk, d, scale, dtype);
  if (rc) return rc;
  JG_REQUIRE(dq && dk && dv && dout && q && k && v && out && lse, "%s: NULL pointer", who);
  JG_REQUIRE(bias == nullptr || bias_period >= 1, "%s: bias_period must be >= 1", who);
  if (batch == 0 || sq == 0) return JG_OK;
  if (workspace == nullptr || workspace_bytes < jg_attn_bwd_workspace_bytes(batch, sq, sk, d))
    JG_FAIL(JG_ERR_WORKSPACE, "%s: workspace %zu < %zu bytes", who, workspace_bytes,
            jg_attn_bwd_workspace_bytes(batch, sq, sk, d));
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (dbias == nullptr && jg::attn_mfma_bwd_supported(batch, (int)sq, (int)sk, (int)d, dtype, bias != nullptr) &&
      aligned16({dq, dk, dv, dout, q, k, v, out}))
    return jg::attn_mfma_bwd_chunks(dq, &dk, &dv, dout, q, &k, &v, 1, out, lse, batch, (int)sq, (int)sk, scale,
                                    workspace, s);
  if (jg::attn_window_supported(batch, (int)sq, (int)sk, (int)d, dtype) &&
      aligned16({dq, dk, dv, dout, q, k, v, out, bias, dbias}))
    return jg::attn_window_bwd(dq, dk, dv, dbias, dout, q, k, v, out, lse, batch, scale, bias,
                               bias_period, s);
  if (dbias == nullptr &&
      jg::attn_wide_supported(batch, (int)sq, (int)sk, (int)d, dtype, bias != nullptr) &&
      aligned16({dq, dk, dv, dout, q, k, v, out}))
    return jg::attn_wide_bwd_chunks(dq, &dk, &dv, dout, q, &k, &v, 1, out, lse, batch, (int)sq, (int)sk, (int)d,
                                    dtype, scale, workspace, s);
  if (dbias == nullptr && jg::attn_f32_mfma_supported(batch, (int)sq, (int)sk, (int)d, 1, dtype, bias != nullptr) &&
      aligned16({dq, dk, dv, dout, q, k, v, out}))
    return jg::attn_f32_mfma_bwd_chunks(dq, &dk, &dv, dout, q, &k, &v, 1, out, lse, batch, (int)sq, (int)sk, (int)d, scale,
                                        workspace, s);
  if (!jg::attn_generic_supported((int)d))
    JG_FAIL(JG_ERR_UNSUPPORTED, "%s: head size %lld not in {8, 16, 32, 64, 96, 128}", who, (long long)d);
  return jg::attn_generic_bwd(dq, dk, dv, static_cast<float*>(workspace), dbias, dout, q, k, v, out,
                              lse, batch, (int)sq, (int)sk, (int)d, scale, bias, bias_period, dtype,
                              s);
}

extern "C" int jg_attn_fwd_chunks(void* out, float* lse, const void* q, const void* const* k, const void* const* v,
                                  int64_t n_chunks, int64_t batch, int64_t sq, int64_t sk, int64_t d, float scale,
                                  int dtype, void* stream) {
  const char* who = "jg_attn_fwd_chunks";
  int rc = check_shape(who, batch, sq, sk, d, scale, dtype);
  if (rc) return rc;
  JG_REQUIRE(n_chunks >= 1, "%s: n_chunks must be at least 1", who);
  JG_REQUIRE(out && lse && q, "%s: NULL pointer", who);
  rc = check_chunks(who, n_chunks, {k, v});
  if (rc) return rc;
  if (batch == 0 || sq == 0) return JG_OK;
  hipStream_t s = static_cast<hipStream_t>(stream);
  const bool aligned = aligned16({out, q}) && chunks_aligned16(n_chunks, {k, v});
  if (aligned && jg::attn_mfma_fwd_supported(batch, (int)sq, (int)sk, (int)d, dtype, false))
    return jg::attn_mfma_fwd_chunks(out, lse, q, k, v, (int)n_chunks, batch, (int)sq, (int)sk, scale, nullptr, nullptr, s);
  if (aligned && jg::attn_wide_supported(batch, (int)sq, (int)sk, (int)d, dtype, false))
    return jg::attn_wide_fwd_chunks(out, lse, q, k, v, (int)n_chunks, batch, (int)sq, (int)sk, (int)d, dtype, scale,
                                    nullptr, nullptr, s);
  if (aligned && jg::attn_f32_mfma_supported(batch, (int)sq, (int)sk, (int)d, (int)n_chunks, dtype, false))
    return jg::attn_f32_mfma_fwd_chunks(out, lse, q, k, v, (int)n_chunks, batch, (int)sq, (int)sk, (int)d, scale, nullptr, nullptr, s);
  JG_FAIL(JG_ERR_UNSUPPORTED, "%s: bf16 or fp16, d a multiple of 8 up to 128, or fp32, d a multiple of 4 up to 128; 16-byte aligned tensors", who);
}

extern "C" int jg_attn_bwd_chunks(void* dq, void* const* dk, void* const* dv, const void* dout, const void* q,
                                  const void* const* k, const void* const* v, int64_t n_chunks, const void* out,
                                  const float* lse, int64_t batch, int64_t sq, int64_t sk, int64_t d, float scale,
                                  int dtype, void* workspace, size_t workspace_bytes, void* stream) {
  const char* who = "jg_attn_bwd_chunks";
  int rc = check_shape(who, batch, sq, sk, d, scale, dtype);
  if (rc) return rc;
  JG_REQUIRE(n_chunks >= 1, "%s: n_chunks must be at least 1", who);
  JG_REQUIRE(dq && dout && q && out && lse, "%s: NULL pointer", who);
  rc = check_chunks(who, n_chunks, {k, v, dk, dv});
  if (rc) return rc;
  if (batch == 0 || sq == 0) return JG_OK;
  if (workspace == nullptr || workspace_bytes < jg_attn_bwd_workspace_bytes(batch, sq, sk, d))
    JG_FAIL(JG_ERR_WORKSPACE, "%s: workspace %zu < %zu bytes", who, workspace_bytes,
            jg_attn_bwd_workspace_bytes(batch, sq, sk, d));
  hipStream_t s = static_cast<hipStream_t>(stream);
  const bool aligned = aligned16({dq, dout, q, out}) && chunks_aligned16(n_chunks, {k, v, dk, dv});
  if (aligned && jg::attn_mfma_bwd_supported(batch, (int)sq, (int)sk, (int)d, dtype, false))
    return jg::attn_mfma_bwd_chunks(dq, dk, dv, dout, q, k, v, (int)n_chunks, out, lse, batch, (int)sq, (int)sk, scale,
                                    workspace, s);
  if (aligned && jg::attn_wide_supported(batch, (int)sq, (int)sk, (int)d, dtype, false))
    return jg::attn_wide_bwd_chunks(dq, dk, dv, dout, q, k, v, (int)n_chunks, out, lse, batch, (int)sq, (int)sk, (int)d,
                                    dtype, scale, workspace, s);
  if (aligned && jg::attn_f32_mfma_supported(batch, (int)sq, (int)sk, (int)d, (int)n_chunks, dtype, false))
    return jg::attn_f32_mfma_bwd_chunks(dq, dk, dv, dout, q, k, v, (int)n_chunks, out, lse, batch, (int)sq, (int)sk, (int)d, scale,
                                        workspace, s);
  JG_FAIL(JG_ERR_UNSUPPORTED, "%s: bf16 or fp16, d a multiple of 8 up to 128, or fp32, d a multiple of 4 up to 128; 16-byte aligned tensors", who);
}

// Rows of a workgroup where jg_attn_bwd_chunks forms dQ, dK and dV of aligned tensors in one launch of attn_wide.hip, 0 where it does not: for
// tests, which have to know what they reach, and not in the interface.
extern "C" int jg_attn_bwd_one_launch_rows(int64_t n_chunks, int64_t batch, int64_t sq, int64_t sk, int64_t d, int dtype) {
  if (check_shape("jg_attn_bwd_one_launch_rows", batch, sq, sk, d, 1.0f, dtype) != JG_OK) return 0;
  if (jg::attn_mfma_bwd_supported(batch, (int)sq, (int)sk, (int)d, dtype, false)) return 32 * jg::attn_mfma_bwd_one_launch_width(batch, (int)sq, (int)sk, (int)n_chunks);
  if (!jg::attn_wide_supported(batch, (int)sq, (int)sk, (int)d, dtype, false)) return 0;
  return 32 * jg::attn_wide_bwd_one_launch_width(batch, (int)sq, (int)sk, (int)d, (int)n_chunks);
}
