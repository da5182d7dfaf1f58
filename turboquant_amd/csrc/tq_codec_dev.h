// tq_codec_dev.h -- lane-level core codec (quantize_vec / dequantize_vec,
// reference src/quantize.rs:142-316) shared by the codec and QJL kernels.
//
// A vector is spread over D / 32 neighbouring lanes, 32 elements each, so a
// lane's straight-line work does not grow with D: with one lane per vector
// (a pair for d = 256) a quantize of two 256-element vectors took 20.7 us,
// nearly all of it one wave issuing the 128-element unrolled code.  The
// reference's sequential parts stay sequential and bit-exact: the f32 sum of
// squares runs in element order through the lanes (quantize.rs:51-53), and
// the Walsh-Hadamard stages keep the reference's order (rotation.rs:22-40),
// those that pair elements of one lane on registers, the last ones across
// lanes.
//
// Bucketize: the reference compares (f64)v > B_k against f64 boundaries
// (codebook/mod.rs:66-87).  For f32 v that is v >= T_k with T_k the smallest
// f32 above B_k (computed on the host), so the lanes do f32 compares only and
// produce the same codes for every input.
#pragma once

#include "tq_codebooks.h"
#include "tq_common.h"
#include "tq_device.h"
#include "tq_mfma.h"

#include <cmath>
#include <type_traits>

namespace tqd {

constexpr float kMinNorm = 1e-10f;  // MIN_NORM, quantize.rs

struct CodecConsts {
  float thr[15];      // smallest f32 T with (double)T > boundary k
  float cent[16];     // (f32) centroid k
  float wht_norm;     // fl(1 / fl(sqrt(d)))  (rotation.rs:36-39)
  float sign_even;    // sign of even elements: +1 if the rotation seed is even
};

template <int D>
struct Geo {
  static constexpr int E = 32;       // elements per lane
  static constexpr int LPV = D / E;  // lanes per vector
};

// #{t : U[t] <= x} for the 2^BITS - 1 ascending thresholds U (bucket_bits).
template <int BITS>
__device__ __forceinline__ uint32_t bucket_sorted(float x, const float (&U)[(1 << BITS) - 1]) {
  bool bit[BITS];
  bucket_bits<BITS>(x, U, bit);
  uint32_t code = 0;
#pragma unroll
  for (int t = 0; t < BITS; t++) code |= bit[t] ? 1u << (BITS - 1 - t) : 0u;
  return code;
}

// Value of the lane before, inside rows of 16 (DPP row_shr:1).
__device__ __forceinline__ float lane_before(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x111, 0xF, 0xF, false));
}

// sum over the vector's elements of sq, in element order from `zero`: lane q
// continues the sum of lane q - 1, so after LPV rounds the last lane's has
// run over the whole vector; every lane gets it.  All lanes of a vector take
// part.
template <int LPV>
__device__ __forceinline__ float ordered_sum(const float (&sq)[32], int q, float zero) {
  float s = zero;
#pragma unroll
  for (int round = 0; round < LPV; round++) {
    if (round > 0) {
      const float before = lane_before(s);  // evaluated by every lane
      s = q == 0 ? zero : before;
    }
#pragma unroll
    for (int e = 0; e < 32; e++) s = s + sq[e];
  }
  if constexpr (LPV > 1) s = __shfl(s, (int)(threadIdx.x & 63) | (LPV - 1), 64);
  return s;
}

// The unnormalized transform of a vector spread over LPV lanes (lane q holds
// elements 32 q ..), stages in the order of butterfly<D>: h < 32 inside the
// lanes, h = 32 X between lanes q and q ^ X (the lower takes x + y, the upper
// x - y).
template <int LPV>
__device__ __forceinline__ void butterfly_lanes(float (&w)[32], int q) {
  butterfly<32>(w);
  auto cross = [&](auto xc) {
    constexpr int X = decltype(xc)::value;
    if constexpr (X < LPV) {
      const bool upper = (q & X) != 0;
#pragma unroll
      for (int e = 0; e < 32; e++) {
        const float o = tqm::lane_xor<X>(w[e]);
        w[e] = upper ? o - w[e] : w[e] + o;
      }
    }
  };
  cross(std::integral_constant<int, 1>{});
  cross(std::integral_constant<int, 2>{});
  cross(std::integral_constant<int, 4>{});
}

// A lane's packed words: 32 codes of BITS bits, on 4 BITS-byte boundaries.
template <int BITS>
__device__ __forceinline__ void store_codes(uint8_t *dst, const uint32_t (&w)[BITS]) {
  uint32_t *p = reinterpret_cast<uint32_t *>(dst);
  if constexpr (BITS == 4) *reinterpret_cast<uint4 *>(p) = make_uint4(w[0], w[1], w[2], w[3]);
  else if constexpr (BITS == 2) *reinterpret_cast<uint2 *>(p) = make_uint2(w[0], w[1]);
  else p[0] = w[0], p[1] = w[1], p[2] = w[2];
}
template <int BITS>
__device__ __forceinline__ void load_codes(const uint8_t *src, uint32_t (&w)[BITS]) {
  const uint32_t *p = reinterpret_cast<const uint32_t *>(src);
  if constexpr (BITS == 4) {
    const uint4 v = *reinterpret_cast<const uint4 *>(p);
    w[0] = v.x; w[1] = v.y; w[2] = v.z; w[3] = v.w;
  } else if constexpr (BITS == 2) {
    const uint2 v = *reinterpret_cast<const uint2 *>(p);
    w[0] = v.x; w[1] = v.y;
  } else {
    w[0] = p[0]; w[1] = p[1]; w[2] = p[2];
  }
}
__device__ __forceinline__ void load_elements(const float *src, float (&w)[32]) {
  const float4 *p = reinterpret_cast<const float4 *>(src);
#pragma unroll
  for (int i = 0; i < 8; i++) {
    const float4 f = p[i];
    w[4 * i] = f.x; w[4 * i + 1] = f.y; w[4 * i + 2] = f.z; w[4 * i + 3] = f.w;
  }
}

// Quantizes lane q's 32 elements of a vector into packed words; returns the
// vector's L2 norm.  `w` is overwritten.
template <int LPV, int BITS>
__device__ __forceinline__ float quantize_lanes(float (&w)[32], int q, const CodecConsts &k, uint32_t (&pk)[BITS]) {
  // l2_norm: f32 sum of squares in element order, from -0.0 (Rust's f32 sum)
  float sq[32];
#pragma unroll
  for (int e = 0; e < 32; e++) sq[e] = w[e] * w[e];
  const float norm = sqrtf(ordered_sum<LPV>(sq, q, -0.0f));
  // normalize_inplace (quantize.rs:60-71), then Forward rotation: sign, WHT
  if (norm < kMinNorm) {
#pragma unroll
    for (int e = 0; e < 32; e++) w[e] = 0.0f;
  } else {
    const float inv = 1.0f / norm;
#pragma unroll
    for (int e = 0; e < 32; e++) w[e] = w[e] * inv;
  }
  const float se = k.sign_even, so = -k.sign_even;  // 32 q is even: parity of element = parity of e
#pragma unroll
  for (int e = 0; e < 32; e++) w[e] = w[e] * ((e & 1) ? so : se);
  butterfly_lanes<LPV>(w, q);
  float thr[(1 << BITS) - 1];
#pragma unroll
  for (int b = 0; b < (1 << BITS) - 1; b++) thr[b] = k.thr[b];
#pragma unroll
  for (int i = 0; i < BITS; i++) pk[i] = 0u;
#pragma unroll
  for (int e = 0; e < 32; e++) {
    const uint32_t idx = bucket_sorted<BITS>(w[e] * k.wht_norm, thr);
    const int bit = e * BITS, wi = bit >> 5, sh = bit & 31;
    pk[wi] |= idx << sh;
    if (sh + BITS > 32) pk[wi + 1] |= idx >> (32 - sh);
  }
  return norm;
}

// Dequantizes lane q's 32 elements: centroid lookup (s_cent in LDS), then,
// with ROTATE, the inverse rotation (WHT with its normalization, then sign,
// rotation.rs:137-150); finally times the f32 scale.
template <int LPV, int BITS, bool ROTATE>
__device__ __forceinline__ void dequant_lanes(const uint32_t (&pk)[BITS], float sc, int q, const float *s_cent,
                                              const CodecConsts &k, float (&w)[32]) {
#pragma unroll
  for (int e = 0; e < 32; e++) w[e] = s_cent[field<BITS>(pk, e)];
  if constexpr (ROTATE) {
    butterfly_lanes<LPV>(w, q);
    const float se = k.sign_even, so = -k.sign_even;
#pragma unroll
    for (int e = 0; e < 32; e++) w[e] = (w[e] * k.wht_norm) * ((e & 1) ? so : se);
  }
#pragma unroll
  for (int e = 0; e < 32; e++) w[e] = w[e] * sc;
}

}  // namespace tqd

namespace tqh {
// Host constants of a TurboQuantConfig{bits, dim, rotation_seed}; a status
// (with tq_last_error set) for a config without a codebook table.
inline int make_codec_consts(int bits, int dim, uint64_t seed, tqd::CodecConsts &k) {
  if (bits < 2 || bits > 4) return fail(TQ_ERR_UNSUPPORTED_BITS, "bits must be 2, 3 or 4 (got %d)", bits);
  if (dim <= 0 || (dim & (dim - 1)) != 0)
    return fail(TQ_ERR_INVALID_DIMENSION, "dim must be a power of two (got %d)", dim);
  const double *c, *b;
  int nc;
  if (!core_codebook(bits, dim, &c, &b, &nc))
    return fail(TQ_ERR_INVALID_DIMENSION, "no codebook table for bits=%d dim=%d (tables: d = 32..256)", bits, dim);
  k = tqd::CodecConsts{};
  for (int i = 0; i < nc; i++) k.cent[i] = (float)c[i];
  for (int i = 0; i < nc - 1; i++) {
    float t = (float)b[i];
    if (!((double)t > b[i])) t = std::nextafter(t, INFINITY);
    k.thr[i] = t;
  }
  for (int i = nc - 1; i < 15; i++) k.thr[i] = INFINITY;
  volatile float fd = (float)dim;
  volatile float sq = sqrtf(fd);
  k.wht_norm = 1.0f / sq;
  k.sign_even = (seed & 1u) ? -1.0f : 1.0f;  // generate_sign_pattern, rotation.rs:47-70
  return TQ_OK;
}
}  // namespace tqh
