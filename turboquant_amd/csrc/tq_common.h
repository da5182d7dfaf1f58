// tq_common.h -- host-side helpers shared by the C ABI launchers.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdarg>
#include <cstdint>
#include <cstdio>

#include "turboquant_amd.h"

namespace tqh {

// Records the calling thread's last error message and returns `code`.
int fail(int code, const char *fmt, ...);
// Maps a HIP error after a launch to TQ_ERR_DEVICE with its message.
int check_launch(const char *what);

inline bool valid_dtype(int dt) { return dt == TQ_DTYPE_F32 || dt == TQ_DTYPE_BF16 || dt == TQ_DTYPE_F16; }

// PQO codebook of the reference (src/cache/precomputed/codebooks.rs:51-88)
// evaluated in f32 exactly as there; outer = max centroid (mod.rs:78).
struct PqoCodebook {
  int bits = 0;
  int nc = 0;
  float c[16] = {};
  float b[15] = {};
  float outer = 0.f;
};
PqoCodebook pqo_codebook(int bits);

// Codec of one cache mode (CacheConfig, src/cache/config.rs:50-85;
// GpuPrecomputed, precomputed/mod.rs:45-98).  The outlier codebook has
// `bits` bits, the standard one bits - 1, its codes in bits-wide slots
// (packed_dim = head_dim * bits / 8).  outlier_blocks >= num_blocks (PQO):
// every block on the outlier codebook; 0 (PQ / TQ): every block on the
// standard one; in between, quantize_tensor.rs:118-150 sends the first
// n * outlier_blocks rows of the [n * num_blocks, 32] block matrix to the
// outlier boundaries while the scale sign (negative = outlier, which the
// dequantize dispatches on) marks the first outlier_blocks blocks of each
// vector.  MaxNorm divides by the outlier codebook's largest centroid
// (quantize_tensor.rs:103-108); L2Norm uses the Beta-optimal tables of
// dimension 32 (codebooks.rs:30-47).
struct PolarCodec {
  int bits = 0;         // slot width
  int cb_bits = 0;      // codebook width of uniform modes (bits or bits - 1)
  int norm_mode = 0;
  bool outlier = false; // every block on the outlier codebook
  bool mixed = false;   // 0 < outlier_blocks < num_blocks
  int num_blocks = 0;
  int eo = 0;           // min(outlier_blocks, num_blocks)
  PqoCodebook cb;       // the blocks' codebook in uniform modes
  PqoCodebook ocb, ncb; // outlier (bits) and standard (bits - 1) codebooks
  float outer = 0.f;    // MaxNorm divisor: the outlier codebook's largest centroid
  float scale_sign = 1.f;
};
// Fills `codec` for (bits, norm_mode, outlier_blocks) or returns an error
// status for an invalid mode.
int polar_codec(int bits, int norm_mode, size_t outlier_blocks, int num_blocks, PolarCodec &codec);

// One token's k and v, [num_heads][1][head_dim] of `dtype`, that a decode
// launch stores at record h * head_stride + offset of every head before it
// attends; the length it attends over includes it.  signs, norms and
// sign_matrix: a TQ cache's, whose key is sketched too; q and rq: its decode's
// query rows and where a launch of the append's own leaves R q.
struct AppendToken {
  const void *k, *v;
  int dtype, num_heads;
  uint8_t *k_idx, *v_idx;
  uint16_t *k_sc, *v_sc;
  uint8_t *signs;
  uint16_t *norms;
  const uint32_t *sign_matrix;
  long long head_stride, offset;
  int head_dim, bits;
  size_t outlier_blocks;
  int norm_mode;
  const void *q;
  int q_dtype;
  float *rq;
  size_t num_q_rows;
  int rc;  // status of a launch of its own, where the decode took one
};
// The same as a launch of its own, which projects q too.
int store_token(const AppendToken &t, hipStream_t stream);

// Fused decode attention (tq_cache_decode_attention) with the length given
// by the host: kv_lens null and host_len >= 0 means every sequence holds
// host_len tokens, no length is read on the device; max_kv_len fixes the
// workspace layout (a cache passes its capacity, so the layout stays put as
// the sequence grows).  append: a token to store first, inside the launch
// where that pays.
int decode_attention(const void *q, int q_dtype, const uint8_t *k_indices, const uint16_t *k_scales,
                     const uint8_t *v_indices, const uint16_t *v_scales, const float *rq, const uint8_t *qjl_signs,
                     const uint16_t *qjl_norms, const int *kv_lens, int host_len, int batch, int num_heads,
                     int num_kv_heads, int head_dim, int bits, size_t outlier_blocks, int norm_mode, int max_kv_len,
                     long long kv_head_stride, long long seq_stride, float softmax_scale, void *out, int out_dtype,
                     void *workspace, size_t workspace_bytes, hipStream_t stream, const uint32_t *rmat = nullptr,
                     AppendToken *append = nullptr);

// tq_polar_quantize_to_cache of x and, unless null, of x2 (the same shape and
// placement in its own buffers) in one launch per codebook.
int polar_quantize_to_cache(const void *x, const void *x2, int x_dtype, int num_heads, int tokens, uint8_t *packed,
                            uint16_t *scales, uint8_t *packed2, uint16_t *scales2, long long head_stride,
                            long long offset, int head_dim, int bits, size_t outlier_blocks, int norm_mode,
                            hipStream_t stream);

// tq_polar_dequantize_from_cache and, unless out2 is null, the same records of
// packed2 and scales2 into out2, in one launch.
int polar_dequantize_from_cache(const uint8_t *packed, const uint16_t *scales, const uint8_t *packed2,
                                const uint16_t *scales2, long long head_stride, int num_heads, int tokens, void *out,
                                void *out2, int out_dtype, int head_dim, int bits, size_t outlier_blocks,
                                int norm_mode, hipStream_t stream);

// A TQ cache's append in one launch: k and v [num_heads][tokens][head_dim]
// quantized into their records, the sketch of the keys' residuals
// (tq_qjl_cache_sketch) and, for num_q_rows > 0, rq = R q (tq_qjl_project).
// The standard codebook (outlier_blocks 0).
struct TqAppend {
  const void *k, *v;
  int dtype, num_heads, tokens;
  uint8_t *k_idx, *v_idx;
  uint16_t *k_sc, *v_sc;
  uint8_t *signs;
  uint16_t *norms;
  long long head_stride, offset;
  int head_dim, bits, norm_mode;
  const uint32_t *sign_matrix;
  const void *q;
  int q_dtype;
  float *rq;
  size_t num_q_rows;
};
int tq_append(const TqAppend &a, hipStream_t stream);

// One buffer of a cache layer that grows: [heads][capacity] records of
// rec_bytes (even), from src (null when nothing is stored) to dst.
constexpr int kGrowParts = 6;
struct GrowPart {
  const void *src = nullptr;
  void *dst = nullptr;
  int rec_bytes = 0;
};
// Copies the first `rows` records of every head into the new buffers and
// zeroes the others, one launch for all parts.
int grow_layer(const GrowPart *parts, int num_parts, int heads, long long old_cap, long long new_cap, long long rows,
               hipStream_t stream);

// compute_logit_bias (tq.rs:185-253) of query rows q [num_q_heads][q_len]
// [head_dim]: tq_qjl_project and tq_qjl_logit_bias (output in q's type) in one
// launch, the projection on the matrix cores from exact products.  q on a
// 16-byte boundary.
int query_logit_bias(const void *q, int q_dtype, const uint32_t *sign_matrix, int num_q_heads, int q_len,
                     const uint8_t *signs, const uint16_t *norms, int num_kv_heads, int kv_len, long long head_stride,
                     int head_dim, void *out, hipStream_t stream);

// fl(1 / fl(sqrt(dim))): the QJL projection's scale (1 / sqrt(d), qjl.rs),
// each step rounded to f32.
float inv_sqrt_dim(int dim);

// Per-boundary constants of the exact division threshold (see
// tqd::div_threshold): mu = midpoint of b and nextup(b), strict = b even.
struct DivThresholds {
  int nb = 0;
  double mu[15] = {};
  uint32_t strict_mask = 0;
  float mul = 0.f;  // fl(1 / outer), candle's affine(1/rhs) scalar division
};
DivThresholds div_thresholds(const float *b, int nb, float outer);

}  // namespace tqh
