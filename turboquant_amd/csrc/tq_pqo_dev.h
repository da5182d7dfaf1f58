// tq_pqo_dev.h -- lane-level PQO / PQ block codec (block-32 MaxNorm or L2Norm)
// shared by the codec kernels and the TQ cache's append.
//
// One lane owns one 32-element qblock.  The block's values live in 32 VGPRs,
// so the Walsh-Hadamard rotation is five in-register butterfly stages with no
// cross-lane traffic, the max-abs is a register reduction, and the bucketized
// codes are shifted straight into the packed words (12 B for 3-bit, 16 B for
// 4-bit) that the lane stores.
//
// Exactness: the reference computes v = fl(r / scale) and counts v > b_k
// (quantize_tensor.rs:107-108, 161-176).  Here each block turns its 2^b - 1
// boundaries into exact thresholds U_k in the input domain once
// (tqd::div_threshold, f64), and the per-element work is r >= U_k: the same
// codes for every finite input, without a division per element.
#pragma once

#include "tq_common.h"
#include "tq_device.h"

#include <algorithm>
#include <cmath>
#include <cstring>

namespace tqp {

using namespace tqd;

constexpr float kInvSqrt32 = 0x1.6a09e6p-3f;  // fl(1 / fl(sqrt(32))) = 0.17677669f

struct QuantConsts {
  double mu[15];
  float b[15];
  float u[15];  // L2Norm: nextup(b), so x >= u <=> x > b
  uint32_t strict_mask;
  float mul;
  float scale_sign;
  int nb, eo;
  long long blk0;  // first block of this launch
  // Evenly spaced boundaries (the 4-bit MaxNorm codebook): b_k = b_0 + k D
  // up to a few ulps, and grid_step = fl(D), grid_off = fl(1 - b_0 / D).
  int grid;
  float grid_step, grid_off;
};

// Half-width of the band around an integer of the grid coordinate inside
// which the fast 4-bit path defers to the exact thresholds: 2^-16 = 256 u
// (u = 2^-24).  The coordinate's error is below 70 u (see quantize_grid).
constexpr float kGridBand = 0x1p-16f;

enum NormMode : int { kMaxNorm = 0, kL2Norm = 1 };

template <int BITS>
struct Packed {
  static constexpr int kWords = BITS;  // 32 * BITS / 32
  static constexpr int kBytes = 4 * BITS;
};

template <int IN_DT>
__device__ __forceinline__ void load_block(const void *__restrict__ x, long long blk, float (&r)[32]) {
  if constexpr (IN_DT == kF32) {
    const float4 *p = reinterpret_cast<const float4 *>(static_cast<const float *>(x) + blk * 32);
#pragma unroll
    for (int q = 0; q < 8; q++) {
      float4 v = p[q];
      r[4 * q + 0] = v.x;
      r[4 * q + 1] = v.y;
      r[4 * q + 2] = v.z;
      r[4 * q + 3] = v.w;
    }
  } else {
    const uint4 *p = reinterpret_cast<const uint4 *>(static_cast<const uint16_t *>(x) + blk * 32);
#pragma unroll
    for (int q = 0; q < 4; q++) {
      uint4 v = p[q];
      uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
      for (int k = 0; k < 4; k++) {
        if constexpr (IN_DT == kBF16) {
          r[8 * q + 2 * k] = u2f(w[k] << 16);
          r[8 * q + 2 * k + 1] = u2f(w[k] & 0xffff0000u);
        } else {
          r[8 * q + 2 * k] = f16_to_f32((uint16_t)(w[k] & 0xffffu));
          r[8 * q + 2 * k + 1] = f16_to_f32((uint16_t)(w[k] >> 16));
        }
      }
    }
  }
}

// acc = 2 acc + bit, with the bit taken straight from the comparison's lane
// mask as the carry-in of one v_addc (LLVM would rebuild it as a select, a
// shift and an or).  The s_nop covers the wait after a VALU write of the
// mask's SGPRs.
__device__ __forceinline__ uint32_t push_bit(uint32_t acc, bool bit) {
  uint32_t r;
  uint64_t carry_out;
  asm("s_nop 1\n\tv_addc_co_u32_e64 %0, %1, %2, %2, %3"
      : "=v"(r), "=s"(carry_out)
      : "v"(acc), "s"(__builtin_amdgcn_ballot_w64(bit)));
  return r;
}

// MaxNorm scale, exact bucketize and pack of one rotated block.  The packed
// LSB-first bitstream is built from its most significant bit down: code j's
// bits go to stream bits 3j+2 .. 3j (for 3-bit codes) and each 32-bit word
// is the last 32 bits pushed into it, so codes that straddle words need no
// special case.  CB < BITS: CB-bit codes (the standard codebook) in BITS-wide
// slots, whose top bits stay zero (quantize_tensor.rs:73, config.rs:82-84).
template <int BITS, int CB>
__device__ __forceinline__ void pack_codes(const float (&r)[32], const float (&U)[(1 << CB) - 1],
                                           uint32_t (&w)[Packed<BITS>::kWords]) {
  uint32_t acc[Packed<BITS>::kWords];
#pragma unroll
  for (int q = 0; q < Packed<BITS>::kWords; q++) acc[q] = 0;
#pragma unroll
  for (int j = 31; j >= 0; j--) {
    bool bit[CB];
    bucket_bits<CB>(r[j], U, bit);
#pragma unroll
    for (int t = 0; t < BITS; t++) {
      const int pos = j * BITS + (BITS - 1 - t);
      if (t < BITS - CB) acc[pos >> 5] <<= 1;
      else acc[pos >> 5] = push_bit(acc[pos >> 5], bit[t - (BITS - CB)]);
    }
  }
#pragma unroll
  for (int q = 0; q < Packed<BITS>::kWords; q++) w[q] = acc[q];
}

template <int BITS, int CB = BITS>
__device__ __forceinline__ float quantize_block(const float (&r)[32], const QuantConsts &k,
                                                uint32_t (&w)[Packed<BITS>::kWords]) {
  static_assert(CB <= BITS, "codes fit their slots");
  constexpr int NB = (1 << CB) - 1;
  float amax = 0.0f;
#pragma unroll
  for (int j = 0; j < 32; j++) amax = fmaxf(amax, fabsf(r[j]));
  float s = amax * k.mul;
  if (s < 1e-10f) s = 1e-10f;

  uint32_t idx[32];
  if (__builtin_isfinite(s)) {
    float U[NB];
#pragma unroll
    for (int t = 0; t < NB; t++) U[t] = div_threshold(k.mu[t], (k.strict_mask >> t) & 1u, s);
    pack_codes<BITS, CB>(r, U, w);
    return s;
  } else {
    // Infinite scale (an infinite input): follow the reference's division.
#pragma unroll
    for (int j = 0; j < 32; j++) {
      float v = r[j] / s;
      uint32_t c = 0;
#pragma unroll
      for (int t = 0; t < NB; t++) c += (v > k.b[t]) ? 1u : 0u;
      idx[j] = c;
    }
  }
#pragma unroll
  for (int q = 0; q < Packed<BITS>::kWords; q++) w[q] = 0;
#pragma unroll
  for (int j = 0; j < 32; j++) {
    const int pos = j * BITS, wi = pos >> 5, sh = pos & 31;
    w[wi] |= idx[j] << sh;
    if (sh + BITS > 32) w[wi + 1] |= idx[j] >> (32 - sh);
  }
  return s;
}

// Fast MaxNorm bucketize for evenly spaced boundaries, on the butterfly
// outputs x_j before the sign and 1/sqrt(32) factor f_j = +-fl(1/sqrt(32)).
// The reference code is q_j = #{k : fl(fl(x_j f_j) / s) > b_k}.  With
// W = x_j f_j / s (real) and D the boundary spacing, boundary k sits at
// T = (v - b_0) / D + 1 = k + 1 + d_k, |d_k| <= 11 u for this codebook
// (checked on the host, which sets k.grid only below 16 u).  The lane
// computes t = fma(x_j, +-fl(fl(1/sqrt(32)) / fl(s D)), fl(1 - b_0 / D)):
// the scale carries <= 3 u, v's two roundings 2 u, |W / D| <= outer / D =
// 7.5, the offset's rounding 8 u (|1 - b_0 / D| < 8.5) and t's own rounding
// 8 u (t < 16 near a boundary), so |t - T| <= 7.5 * 5 u + 8 u + 8 u + 16 u
// (d_k) < 70 u.  Where t is more than
// kGridBand = 256 u from every integer, each comparison v > b_k equals
// t > k + 1, so q_j = min(floor(t), 15) (0 for t < 1).  Returns false when
// some element of the block falls inside the band (or t is NaN); the caller
// then takes the exact path for the whole block.
__device__ __forceinline__ bool quantize_grid(const float (&x)[32], float s, const QuantConsts &k,
                                              uint32_t (&w)[4]) {
  const float a = kInvSqrt32 / (s * k.grid_step);
  bool clear = true;
#pragma unroll
  for (int q = 0; q < 4; q++) w[q] = 0;
#pragma unroll
  for (int j = 0; j < 32; j++) {
    const float t = __builtin_fmaf(x[j], pqo_neg(j) ? -a : a, k.grid_off);
    const uint32_t c = (uint32_t)__builtin_amdgcn_fmed3f(t, 0.0f, 15.5f);
    const float f = __builtin_amdgcn_fractf(t);
    clear = clear && (fabsf(f - 0.5f) < 0.5f - kGridBand);
    w[j >> 3] |= c << (4 * (j & 7));
  }
  return clear;
}

template <int BITS>
__device__ __forceinline__ void store_packed(uint8_t *__restrict__ packed, long long blk,
                                             const uint32_t (&w)[Packed<BITS>::kWords]) {
  uint32_t *p = reinterpret_cast<uint32_t *>(packed + blk * Packed<BITS>::kBytes);
  if constexpr (BITS == 4) {
    *reinterpret_cast<uint4 *>(p) = make_uint4(w[0], w[1], w[2], w[3]);
  } else if constexpr (BITS == 2) {
    *reinterpret_cast<uint2 *>(p) = make_uint2(w[0], w[1]);
  } else {
    p[0] = w[0];
    p[1] = w[1];
    p[2] = w[2];
  }
}

// Placement of contiguous [heads][tokens] vectors in a cache laid out
// [heads][head_stride] records (CompressedStorage, storage.rs:24-139):
// vector (h, t) <-> record h * head_stride + offset + t.
struct CacheMap {
  uint32_t qb_per_vec;  // head_dim / 32
  uint32_t tokens;
  long long head_stride;
  long long offset;
};

__device__ __forceinline__ long long cache_block(uint32_t blk, const CacheMap &m) {
  const uint32_t v = blk / m.qb_per_vec, j = blk - v * m.qb_per_vec;
  const uint32_t h = v / m.tokens, t = v - h * m.tokens;
  return ((long long)h * m.head_stride + m.offset + t) * m.qb_per_vec + j;
}


// One block of activations r (ROTATE: raw, with the forward rotation fused in
// butterfly order; otherwise already rotated), overwritten: its codes in w;
// returns its scale before the sign.
// NORM = kL2Norm: the block's L2 norm (sum of squares in element order,
// sqrt, clamped to 1e-10) divides it before the rotation and is its scale;
// codes count the boundaries strictly below the rotated value
// (normalize_and_rotate, quantize_tensor.rs:90-101, 161-176).
template <int BITS, int CB, bool ROTATE, int NORM>
__device__ __forceinline__ float encode_block(float (&r)[32], const QuantConsts &k,
                                              uint32_t (&w)[Packed<BITS>::kWords]) {
  float nrm = 0.f;
  if constexpr (NORM == kL2Norm) {
    float ss = 0.0f;
#pragma unroll
    for (int j = 0; j < 32; j++) ss = ss + r[j] * r[j];
    nrm = sqrtf(ss);
    nrm = nrm < 1e-10f ? 1e-10f : nrm;
#pragma unroll
    for (int j = 0; j < 32; j++) r[j] = r[j] / nrm;
  }
  float s = 0.0f;
  bool done = false;
  if constexpr (ROTATE) {
    butterfly<32>(r);
    if constexpr (NORM == kMaxNorm && BITS == 4 && CB == 4) {
      if (k.grid) {
        // max_j |fl(x_j f_j)| = fl(max_j |x_j| / sqrt(32)): rounding is monotone
        float am = 0.0f;
#pragma unroll
        for (int j = 0; j < 32; j++) am = fmaxf(am, fabsf(r[j]));
        s = (am * kInvSqrt32) * k.mul;
        if (s < 1e-10f) s = 1e-10f;
        done = __builtin_isfinite(s) && quantize_grid(r, s, k, w);
      }
    }
    if (!done) {
#pragma unroll
      for (int j = 0; j < 32; j++) r[j] = r[j] * (pqo_neg(j) ? -kInvSqrt32 : kInvSqrt32);
    }
  }
  if (done) {
  } else if constexpr (NORM == kL2Norm) {
    float U[(1 << CB) - 1];
#pragma unroll
    for (int t = 0; t < (1 << CB) - 1; t++) U[t] = k.u[t];
    pack_codes<BITS, CB>(r, U, w);
    s = nrm;
  } else {
    s = quantize_block<BITS, CB>(r, k, w);
  }
  return s;
}

inline QuantConsts make_quant_consts(const tqh::PqoCodebook &cb, float outer, float scale_sign) {
  tqh::DivThresholds t = tqh::div_thresholds(cb.b, cb.nc - 1, outer);
  QuantConsts k{};
  for (int i = 0; i < t.nb; i++) {
    k.mu[i] = t.mu[i];
    k.b[i] = cb.b[i];
    uint32_t u;
    std::memcpy(&u, &cb.b[i], 4);  // nextup(b) for finite b
    if ((u & 0x7fffffffu) == 0) u = 1u;
    else u = ((int32_t)u >= 0) ? u + 1u : u - 1u;
    std::memcpy(&k.u[i], &u, 4);
  }
  k.strict_mask = t.strict_mask;
  k.mul = t.mul;
  k.scale_sign = scale_sign;
  // Evenly spaced 15 boundaries whose offsets from the grid stay below 16 u
  // in grid units (11 u for the 4-bit MaxNorm codebook) and whose spacing
  // keeps |W / D| <= outer / D near 7.5 (the error budget of quantize_grid).
  if (cb.nc == 16) {
    const double d = ((double)cb.b[14] - (double)cb.b[0]) / 14.0;
    double dev = 0.0;
    for (int i = 0; i < 15; i++) dev = std::max(dev, std::fabs(((double)cb.b[i] - (double)cb.b[0]) / d - i));
    if (d > 0.0 && dev < 16.0 * 0x1p-24 && (double)outer / d < 7.6 && std::fabs(1.0 - (double)cb.b[0] / d) < 8.5) {
      k.grid = 1;
      k.grid_step = (float)d;
      k.grid_off = (float)(1.0 - (double)cb.b[0] / d);
    }
  }
  return k;
}

}  // namespace tqp
