// tq_pqo.hip -- PQO (block-32 MaxNorm) cache codec kernels for gfx950.
//
// Design: one lane owns one 32-element qblock (tq_pqo_dev.h); nothing needs
// atomics or LDS.  A wave covers 64 consecutive qblocks, so its stores of
// packed codes and f16 scales are contiguous.
#include "tq_pqo_dev.h"

namespace {

using namespace tqp;

// A second tensor of a launch (x null: none).
struct Second {
  const void *x = nullptr;
  uint8_t *packed = nullptr;
  uint16_t *scales = nullptr;
};

// ROTATE: input is raw activations (fused forward rotation, butterfly order).
// Otherwise input is already rotated f32 (the reference kernel's contract).
// MAP: outputs go to cache records (CacheMap) instead of block order; with a
// second tensor of the same shape (an append's keys and values) grid.y is 2
// and y = 1 takes it: one launch instead of two of about 3 us each.
// MIXED: one of the two launches of a mixed-outlier config (blocks from
// k.blk0, scale sign per block).
template <int BITS, int CB, int IN_DT, bool ROTATE, bool MAP, int NORM, bool MIXED>
__global__ __launch_bounds__(256) void pqo_quant_kernel(const void *__restrict__ x,
                                                        uint8_t *__restrict__ packed,
                                                        uint16_t *__restrict__ scales,
                                                        long long nblocks, QuantConsts k, CacheMap map,
                                                        Second second) {
  if (MAP && blockIdx.y) {
    x = second.x;
    packed = second.packed;
    scales = second.scales;
  }
  const long long b0 = MIXED ? k.blk0 : 0;
  const long long blk = b0 + (long long)blockIdx.x * 256 + threadIdx.x;
  if (blk >= b0 + nblocks) return;
  const long long ob = MAP ? cache_block((uint32_t)blk, map) : blk;
  float r[32];
  load_block<IN_DT>(x, blk, r);
  uint32_t w[Packed<BITS>::kWords];
  const float s = encode_block<BITS, CB, ROTATE, NORM>(r, k, w);
  store_packed<BITS>(packed, ob, w);
  const float sign = MIXED ? (((int)(blk % k.nb) < k.eo) ? -1.0f : 1.0f) : k.scale_sign;
  scales[ob] = f32_to_f16(s * sign);
}

// Reference-ABI variant: boundaries and outer centroid come from the caller
// (device boundaries), constants derived in-kernel per lane.
template <int BITS>
__global__ __launch_bounds__(256) void pqo_quant_rotated_dev_kernel(
    const float *__restrict__ rotated, const float *__restrict__ boundaries,
    uint8_t *__restrict__ packed, uint16_t *__restrict__ scales, long long nblocks, float outer,
    float scale_sign) {
  const long long blk = (long long)blockIdx.x * 256 + threadIdx.x;
  if (blk >= nblocks) return;
  constexpr int NB = (1 << BITS) - 1;
  QuantConsts k;
#pragma unroll
  for (int t = 0; t < NB; t++) {
    float b = boundaries[t];
    float up = next_up(b);
    k.b[t] = b;
    k.mu[t] = ((double)b + (double)up) * 0.5;
  }
  k.strict_mask = 0;
#pragma unroll
  for (int t = 0; t < NB; t++) k.strict_mask |= ((f2u(k.b[t]) & 1u) == 0 ? 1u : 0u) << t;
  k.mul = (float)(1.0 / (double)outer);
  k.scale_sign = scale_sign;
  float r[32];
  load_block<kF32>(rotated, blk, r);
  uint32_t w[Packed<BITS>::kWords];
  float s = quantize_block<BITS>(r, k, w);
  store_packed<BITS>(packed, blk, w);
  scales[blk] = f32_to_f16(s * scale_sign);
}

// A second set of records of a dequantize launch (out null: none).
struct SecondOut {
  const uint8_t *packed = nullptr;
  const uint16_t *scales = nullptr;
  void *out = nullptr;
};

struct DequantConsts {
  float cb[16];   // codebook values (f32); the outlier codebook when mixed
  float cbn[16];  // mixed: the standard codebook
  // the reference's sign factor of element j is fl(R_fwd[0][j] * sqrt(32)) =
  // (pqo_neg(j) ? -sgm : sgm): one magnitude for every j
  float sgm;
  int mixed;      // codebook per block by the scale's sign (quantize_tensor.rs:242-260)
  int nn;         // mixed: standard codebook size (codes are clamped into it)
};

// out_j = fl(fl(W_j * fl(1/sqrt(32))) * |scale|), W = butterfly(cb[idx] * sign):
// butterfly_wht_inverse_cpu (wht_tensor.rs:38-64) then the broadcast_mul by
// |scale| (quantize_tensor.rs:203, 217-218).
// MAP: inputs come from cache records (CacheMap); outputs in block order; a
// second set of records (a layer's values beside its keys) is taken by y = 1.
// MIXED: the codebook per block from the scale's sign (else one codebook).
// With the library's constants the table holds fl(cb * |sg|) and element j
// takes it negated where sg[j] < 0: fl(c * -m) = -fl(c * m), the same value
// as the per-element product, one multiply per table entry instead of per
// element.
template <int BITS, int OUT_DT, bool DEV_CONSTS, bool MAP = false, bool MIXED = false>
__global__ __launch_bounds__(256) void pqo_dequant_kernel(const uint8_t *__restrict__ packed,
                                                          const uint16_t *__restrict__ scales,
                                                          void *__restrict__ out, long long nblocks,
                                                          DequantConsts dc,
                                                          const float *__restrict__ dev_cb,
                                                          const float *__restrict__ dev_sg, CacheMap map = {},
                                                          SecondOut second = {}) {
  if (MAP && blockIdx.y) {
    packed = second.packed;
    scales = second.scales;
    out = second.out;
  }
  __shared__ float lut[32];
  constexpr int NC = 1 << BITS;
  if (threadIdx.x < NC) lut[threadIdx.x] = DEV_CONSTS ? dev_cb[threadIdx.x] : dc.cb[threadIdx.x] * dc.sgm;
  if (MIXED && threadIdx.x >= 16 && threadIdx.x < 32) lut[threadIdx.x] = dc.cbn[threadIdx.x - 16] * dc.sgm;
  __syncthreads();
  const long long blk = (long long)blockIdx.x * 256 + threadIdx.x;
  // lanes past the end still take part in the wave's output staging
  const bool valid = blk < nblocks;
  const long long ib = !valid ? 0 : (MAP ? cache_block((uint32_t)blk, map) : blk);
  uint32_t w[Packed<BITS>::kWords];
#pragma unroll
  for (int q = 0; q < Packed<BITS>::kWords; q++) w[q] = 0u;
  uint16_t sbits = 0;
  if (valid) {
    const uint32_t *p = reinterpret_cast<const uint32_t *>(packed + ib * Packed<BITS>::kBytes);
    if constexpr (BITS == 4) {
      uint4 v = *reinterpret_cast<const uint4 *>(p);
      w[0] = v.x; w[1] = v.y; w[2] = v.z; w[3] = v.w;
    } else if constexpr (BITS == 2) {
      uint2 v = *reinterpret_cast<const uint2 *>(p);
      w[0] = v.x; w[1] = v.y;
    } else {
#pragma unroll
      for (int q = 0; q < 3; q++) w[q] = p[q];
    }
    sbits = scales[ib];
  }
  const float ssig = f16_to_f32(sbits);
  const float s = fabsf(ssig);
  // mixed: a non-negative scale selects the standard codebook, codes clamped
  float z[32];
  if constexpr (MIXED) {
    const bool std_cb = !(ssig < 0.0f);
    const uint32_t base = std_cb ? 16u : 0u, cmax = std_cb ? (uint32_t)dc.nn - 1u : 15u;
#pragma unroll
    for (int j = 0; j < 32; j++) {
      const float c = lut[base + min(field<BITS>(w, j), cmax)];
      z[j] = pqo_neg(j) ? -c : c;
    }
  } else {
#pragma unroll
    for (int j = 0; j < 32; j++) {
      const float c = lut[field<BITS>(w, j)];
      if constexpr (DEV_CONSTS) z[j] = c * dev_sg[j];
      else z[j] = pqo_neg(j) ? -c : c;
    }
  }
  butterfly<32>(z);
#pragma unroll
  for (int j = 0; j < 32; j++) z[j] = (z[j] * kInvSqrt32) * s;
  // the block's output words
  constexpr int NDW = OUT_DT == kF32 ? 32 : 16;
  uint32_t v[NDW];
  if constexpr (OUT_DT == kF32) {
#pragma unroll
    for (int j = 0; j < 32; j++) v[j] = f2u(z[j]);
  } else {
#pragma unroll
    for (int k = 0; k < 16; k++) {
      const float a = z[2 * k], b = z[2 * k + 1];
      if constexpr (OUT_DT == kBF16) v[k] = pack_bf16x2(a, b);
      else v[k] = (uint32_t)f32_to_f16(a) | ((uint32_t)f32_to_f16(b) << 16);
    }
  }
  // A wave's 64 blocks are one contiguous run of 64 * NDW words: staged
  // through LDS (rows padded to RS words), each store instruction writes
  // 1 KB of it contiguously rather than 16 bytes into each of 64 lines.
  constexpr int RS = NDW + 4;
  __shared__ __attribute__((aligned(16))) uint32_t s_out[4][64 * RS];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  uint32_t *row = s_out[wave] + lane * RS;
#pragma unroll
  for (int k = 0; k < NDW / 4; k++)
    *reinterpret_cast<uint4 *>(row + 4 * k) = make_uint4(v[4 * k], v[4 * k + 1], v[4 * k + 2], v[4 * k + 3]);
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  const long long wb = (long long)blockIdx.x * 256 + wave * 64;  // the wave's first block
  uint32_t *dst = static_cast<uint32_t *>(out) + wb * NDW;
#pragma unroll
  for (int q = 0; q < NDW / 4; q++) {
    const int f = 256 * q + 4 * lane;  // word of the wave's run
    const int r = f / NDW, c = f % NDW;
    if (wb + r < nblocks)
      *reinterpret_cast<uint4 *>(dst + f) = *reinterpret_cast<const uint4 *>(s_out[wave] + r * RS + c);
  }
}

// One thread per output byte: gathers the codes overlapping bits [8i, 8i+8).
__global__ __launch_bounds__(256) void pack_indices_kernel(const uint8_t *__restrict__ idx,
                                                           uint8_t *__restrict__ out,
                                                           long long nvec, int block_size, int bits,
                                                           int bytes_per_block) {
  const long long g = (long long)blockIdx.x * 256 + threadIdx.x;
  if (g >= nvec * bytes_per_block) return;
  const long long v = g / bytes_per_block;
  const int byte = (int)(g % bytes_per_block);
  const uint8_t *src = idx + v * block_size;
  uint32_t acc = 0;
  const int lo = byte * 8, hi = lo + 8;
  const int mask = (1 << bits) - 1;
  for (int i = lo / bits; i * bits < hi && i < block_size; i++) {
    const int pos = i * bits - lo;  // may be negative for a code straddling in
    uint32_t c = (uint32_t)(src[i] & mask);
    acc |= pos >= 0 ? (c << pos) : (c >> -pos);
  }
  out[g] = (uint8_t)(acc & 0xffu);
}

// One launch of pqo_quant_kernel for (slot bits, codebook bits, input type):
// ROTATE for activations, MAP for cache placement.
template <bool ROTATE, bool MAP, int NORM, bool MIXED>
int launch_quant(const void *x, int dt, uint8_t *packed, uint16_t *scales, long long nblocks, int bits, int cb_bits,
                 const QuantConsts &k, const CacheMap &m, const Second &second, hipStream_t st) {
  if (nblocks <= 0) return TQ_OK;
  const dim3 grid((unsigned)((nblocks + 255) / 256), second.x ? 2 : 1), block(256);
#define QL(B, C, D) hipLaunchKernelGGL((pqo_quant_kernel<B, C, D, ROTATE, MAP, NORM, MIXED>), grid, block, 0, st, x, \
                                       packed, scales, nblocks, k, m, second)
#define QD(B, C) \
  do {                                      \
    if (!ROTATE || dt == kF32) QL(B, C, kF32); \
    else if (dt == kBF16) QL(B, C, kBF16);  \
    else QL(B, C, kF16);                    \
  } while (0)
  if (bits == 2) QD(2, 2);
  else if (bits == 3 && cb_bits == 3) QD(3, 3);
  else if (bits == 3) QD(3, 2);
  else if (cb_bits == 4) QD(4, 4);
  else QD(4, 3);
#undef QD
#undef QL
  return tqh::check_launch("pqo_quant_kernel");
}

// polar_quantize of nblocks blocks (vectors of codec.num_blocks blocks) in
// one launch per codebook: a mixed config's first nblocks / nb * eo blocks
// on the outlier codebook, the rest on the standard one.
template <bool MAP>
int launch_polar_quant(const void *x, int dt, uint8_t *packed, uint16_t *scales, long long nblocks,
                       const tqh::PolarCodec &codec, const CacheMap &m, const Second &second, hipStream_t st) {
  auto run = [&](const tqh::PqoCodebook &cb, int cb_bits, long long b0, long long n) {
    QuantConsts k = make_quant_consts(cb, codec.outer, codec.scale_sign);
    k.nb = codec.num_blocks;
    k.eo = codec.eo;
    k.blk0 = b0;
    if (codec.mixed) {
      if (codec.norm_mode == kL2Norm)
        return launch_quant<true, MAP, kL2Norm, true>(x, dt, packed, scales, n, codec.bits, cb_bits, k, m, second, st);
      return launch_quant<true, MAP, kMaxNorm, true>(x, dt, packed, scales, n, codec.bits, cb_bits, k, m, second, st);
    }
    if (codec.norm_mode == kL2Norm)
      return launch_quant<true, MAP, kL2Norm, false>(x, dt, packed, scales, n, codec.bits, cb_bits, k, m, second, st);
    return launch_quant<true, MAP, kMaxNorm, false>(x, dt, packed, scales, n, codec.bits, cb_bits, k, m, second, st);
  };
  if (!codec.mixed) return run(codec.cb, codec.cb_bits, 0, nblocks);
  const long long nout = nblocks / codec.num_blocks * codec.eo;  // bucketize_blocks' outlier rows
  int rc = run(codec.ocb, codec.bits, 0, nout);
  if (rc) return rc;
  return run(codec.ncb, codec.bits - 1, nout, nblocks - nout);
}

DequantConsts make_dequant_consts(const tqh::PqoCodebook &cb);

DequantConsts dequant_consts(const tqh::PolarCodec &codec) {
  DequantConsts dc = make_dequant_consts(codec.mixed ? codec.ocb : codec.cb);
  if (codec.mixed) {
    for (int i = 0; i < codec.ncb.nc; i++) dc.cbn[i] = codec.ncb.c[i];
    dc.nn = codec.ncb.nc;
    dc.mixed = 1;
  }
  return dc;
}

DequantConsts make_dequant_consts(const tqh::PqoCodebook &cb) {
  DequantConsts dc{};
  for (int i = 0; i < cb.nc; i++) dc.cb[i] = cb.c[i];
  dc.nn = cb.nc;
  // fl(R_fwd[0][j] * sqrt(32)) = fl(+-fl(1/sqrt(32)) * fl(sqrt(32))) (wht_tensor.rs:28-41)
  volatile float thirty_two = 32.0f;
  volatile float sq = sqrtf(thirty_two);  // fl(sqrt(32)), IEEE sqrt
  volatile float inv = 1.0f / sq;
  volatile float m = inv * sq;  // fl(+-inv * sq) = +-fl(inv * sq)
  dc.sgm = m;
  return dc;
}

}  // namespace

// ---------------------------------------------------------------------------
// C ABI
// ---------------------------------------------------------------------------

namespace {
int check_shape(int head_dim) {
  if (head_dim <= 0 || head_dim % 32 != 0)
    return tqh::fail(TQ_ERR_INVALID_ARGUMENT, "head_dim (%d) must be divisible by QUANT_BLOCK_SIZE (32)", head_dim);
  return TQ_OK;
}

template <bool MAP>
int launch_dequant(const uint8_t *packed, const uint16_t *scales, void *out, int out_dtype, long long nblocks,
                   int bits, const DequantConsts &dc, const CacheMap &m, const SecondOut &second,
                   hipStream_t stream) {
  const dim3 grid((unsigned)((nblocks + 255) / 256), second.out ? 2 : 1), block(256);
#define DL(B, D)                                                                                                  \
  do {                                                                                                            \
    if (dc.mixed)                                                                                                 \
      hipLaunchKernelGGL((pqo_dequant_kernel<B, D, false, MAP, true>), grid, block, 0, stream, packed, scales, out, \
                         nblocks, dc, nullptr, nullptr, m, second);                                               \
    else                                                                                                          \
      hipLaunchKernelGGL((pqo_dequant_kernel<B, D, false, MAP, false>), grid, block, 0, stream, packed, scales,     \
                         out, nblocks, dc, nullptr, nullptr, m, second);                                          \
  } while (0)
  if (bits == 3) {
    if (out_dtype == kF32) DL(3, kF32);
    else if (out_dtype == kBF16) DL(3, kBF16);
    else DL(3, kF16);
  } else {
    if (out_dtype == kF32) DL(4, kF32);
    else if (out_dtype == kBF16) DL(4, kBF16);
    else DL(4, kF16);
  }
#undef DL
  return tqh::check_launch("pqo_dequant_kernel");
}
}  // namespace

extern "C" int tq_polar_quantize(const void *x, int x_dtype, uint8_t *packed_out, uint16_t *scales_out,
                                 size_t num_vectors, int head_dim, int bits, size_t outlier_blocks, int norm_mode,
                                 hipStream_t stream) {
  int rc = check_shape(head_dim);
  if (rc) return rc;
  tqh::PolarCodec codec;
  rc = tqh::polar_codec(bits, norm_mode, outlier_blocks, head_dim / 32, codec);
  if (rc) return rc;
  if (!tqh::valid_dtype(x_dtype)) return tqh::fail(TQ_ERR_INVALID_ARGUMENT, "unknown dtype %d", x_dtype);
  if (num_vectors == 0) return TQ_OK;
  if (!x || !packed_out || !scales_out) return tqh::fail(TQ_ERR_INVALID_ARGUMENT, "null pointer");
  const long long nblocks = (long long)num_vectors * (head_dim / 32);
  return launch_polar_quant<false>(x, x_dtype, packed_out, scales_out, nblocks, codec, CacheMap{}, Second{}, stream);
}

extern "C" int tq_polar_dequantize(const uint8_t *packed, const uint16_t *scales, void *out, int out_dtype,
                                   size_t num_vectors, int head_dim, int bits, size_t outlier_blocks, int norm_mode,
                                   hipStream_t stream) {
  int rc = check_shape(head_dim);
  if (rc) return rc;
  tqh::PolarCodec codec;
  rc = tqh::polar_codec(bits, norm_mode, outlier_blocks, head_dim / 32, codec);
  if (rc) return rc;
  if (!tqh::valid_dtype(out_dtype)) return tqh::fail(TQ_ERR_INVALID_ARGUMENT, "unknown dtype %d", out_dtype);
  if (num_vectors == 0) return TQ_OK;
  if (!packed || !scales || !out) return tqh::fail(TQ_ERR_INVALID_ARGUMENT, "null pointer");
  const long long nblocks = (long long)num_vectors * (head_dim / 32);
  return launch_dequant<false>(packed, scales, out, out_dtype, nblocks, bits, dequant_consts(codec),
                               CacheMap{}, SecondOut{}, stream);
}

extern "C" int tq_pqo_quantize(const void *x, int x_dtype, uint8_t *packed_out, uint16_t *scales_out,
                               size_t num_vectors, int head_dim, int bits, hipStream_t stream) {
  return tq_polar_quantize(x, x_dtype, packed_out, scales_out, num_vectors, head_dim, bits, TQ_OUTLIER_ALL,
                           TQ_NORM_MAXNORM, stream);
}

extern "C" int tq_pqo_dequantize(const uint8_t *packed, const uint16_t *scales, void *out, int out_dtype,
                                 size_t num_vectors, int head_dim, int bits, hipStream_t stream) {
  return tq_polar_dequantize(packed, scales, out, out_dtype, num_vectors, head_dim, bits, TQ_OUTLIER_ALL,
                             TQ_NORM_MAXNORM, stream);
}

extern "C" int tq_quant_maxnorm_batch(const float *rotated_input, const float *boundaries, uint8_t *packed_out,
                                      uint16_t *scales_out, int num_blocks, int block_size, int bits,
                                      int num_boundaries, int bytes_per_block, float outer_centroid,
                                      float scale_sign, hipStream_t stream) {
  if (num_blocks == 0) return TQ_OK;  // tq_quant_kernel.cu:430
  if (num_blocks < 0) return tqh::fail(TQ_ERR_INVALID_ARGUMENT, "num_blocks < 0");
  if (block_size != 32) return tqh::fail(TQ_ERR_INVALID_ARGUMENT, "block_size must be QUANT_BLOCK_SIZE (32), got %d", block_size);
  if (bits < 2 || bits > 4) return tqh::fail(TQ_ERR_UNSUPPORTED_BITS, "unsupported bit width %d", bits);
  if (num_boundaries != (1 << bits) - 1)
    return tqh::fail(TQ_ERR_INVALID_ARGUMENT, "num_boundaries %d != 2^bits - 1", num_boundaries);
  if (bytes_per_block != 32 * bits / 8)
    return tqh::fail(TQ_ERR_INVALID_ARGUMENT, "bytes_per_block %d != 32*bits/8", bytes_per_block);
  if (!rotated_input || !boundaries || !packed_out || !scales_out)
    return tqh::fail(TQ_ERR_INVALID_ARGUMENT, "null pointer");
  const long long nb = num_blocks;
  const dim3 grid((unsigned)((nb + 255) / 256)), block(256);
  if (bits == 2)
    hipLaunchKernelGGL((pqo_quant_rotated_dev_kernel<2>), grid, block, 0, stream, rotated_input, boundaries,
                       packed_out, scales_out, nb, outer_centroid, scale_sign);
  else if (bits == 3)
    hipLaunchKernelGGL((pqo_quant_rotated_dev_kernel<3>), grid, block, 0, stream, rotated_input, boundaries,
                       packed_out, scales_out, nb, outer_centroid, scale_sign);
  else
    hipLaunchKernelGGL((pqo_quant_rotated_dev_kernel<4>), grid, block, 0, stream, rotated_input, boundaries,
                       packed_out, scales_out, nb, outer_centroid, scale_sign);
  return tqh::check_launch("pqo_quant_rotated_dev_kernel");
}

extern "C" int tq_dequant_batch(const uint8_t *packed_indices, const uint16_t *scales, const float *codebook,
                                const float *sign_pattern, float *output, int num_blocks, int block_size, int bits,
                                int bytes_per_block, hipStream_t stream) {
  if (num_blocks == 0) return TQ_OK;  // tq_dequant_kernel.cu:116
  if (num_blocks < 0) return tqh::fail(TQ_ERR_INVALID_ARGUMENT, "num_blocks < 0");
  if (block_size != 32) return tqh::fail(TQ_ERR_INVALID_ARGUMENT, "block_size must be QUANT_BLOCK_SIZE (32), got %d", block_size);
  if (bits < 2 || bits > 4) return tqh::fail(TQ_ERR_UNSUPPORTED_BITS, "unsupported bit width %d", bits);
  if (bytes_per_block != 32 * bits / 8)
    return tqh::fail(TQ_ERR_INVALID_ARGUMENT, "bytes_per_block %d != 32*bits/8", bytes_per_block);
  if (!packed_indices || !scales || !codebook || !sign_pattern || !output)
    return tqh::fail(TQ_ERR_INVALID_ARGUMENT, "null pointer");
  const long long nb = num_blocks;
  const dim3 grid((unsigned)((nb + 255) / 256)), block(256);
  DequantConsts dc{};
  if (bits == 2)
    hipLaunchKernelGGL((pqo_dequant_kernel<2, kF32, true>), grid, block, 0, stream, packed_indices, scales, output,
                       nb, dc, codebook, sign_pattern);
  else if (bits == 3)
    hipLaunchKernelGGL((pqo_dequant_kernel<3, kF32, true>), grid, block, 0, stream, packed_indices, scales, output,
                       nb, dc, codebook, sign_pattern);
  else
    hipLaunchKernelGGL((pqo_dequant_kernel<4, kF32, true>), grid, block, 0, stream, packed_indices, scales, output,
                       nb, dc, codebook, sign_pattern);
  return tqh::check_launch("pqo_dequant_kernel");
}

extern "C" int tq_pack_indices(const uint8_t *indices, uint8_t *packed_out, int num_vectors, int block_size,
                               int bits, int bytes_per_block, hipStream_t stream) {
  if (num_vectors == 0) return TQ_OK;
  if (num_vectors < 0 || block_size <= 0) return tqh::fail(TQ_ERR_INVALID_ARGUMENT, "negative size");
  if (bits < 2 || bits > 4) return tqh::fail(TQ_ERR_UNSUPPORTED_BITS, "unsupported bit width %d", bits);
  if (bytes_per_block * 8 < block_size * bits)
    return tqh::fail(TQ_ERR_INVALID_ARGUMENT, "bytes_per_block %d too small", bytes_per_block);
  if (!indices || !packed_out) return tqh::fail(TQ_ERR_INVALID_ARGUMENT, "null pointer");
  // whole vectors a launch, fewer than 2^32 lanes (bytes_per_block is an int)
  const long long most = std::max((1ll << 31) / bytes_per_block, 1ll);
  for (long long v = 0; v < num_vectors; v += most) {
    const long long n = std::min(num_vectors - v, most);
    hipLaunchKernelGGL(pack_indices_kernel, dim3((unsigned)((n * bytes_per_block + 255) / 256)), dim3(256), 0, stream,
                       indices + v * block_size, packed_out + v * bytes_per_block, n, block_size, bits, bytes_per_block);
    const int rc = tqh::check_launch("pack_indices_kernel");
    if (rc) return rc;
  }
  return TQ_OK;
}

// ---------------------------------------------------------------------------
// Cache placement (CompressedStorage append / full dequantize)
// ---------------------------------------------------------------------------

namespace {
int cache_map(int num_heads, int tokens, int head_dim, long long head_stride, long long offset, CacheMap &m) {
  if (num_heads < 0 || tokens < 0) return tqh::fail(TQ_ERR_INVALID_ARGUMENT, "negative shape");
  if (head_dim <= 0 || head_dim % 32 != 0)
    return tqh::fail(TQ_ERR_INVALID_ARGUMENT, "head_dim (%d) must be divisible by QUANT_BLOCK_SIZE (32)", head_dim);
  if (offset < 0 || head_stride < offset + tokens)
    return tqh::fail(TQ_ERR_RANGE_OUT_OF_BOUNDS, "cache rows [%lld, %lld) exceed head stride %lld", offset,
                     offset + tokens, head_stride);
  if ((long long)num_heads * tokens * (head_dim / 32) >= (1ll << 31))
    return tqh::fail(TQ_ERR_INVALID_ARGUMENT, "too many blocks in one call");
  m.qb_per_vec = (uint32_t)(head_dim / 32);
  m.tokens = (uint32_t)(tokens > 0 ? tokens : 1);
  m.head_stride = head_stride;
  m.offset = offset;
  return TQ_OK;
}
}  // namespace

namespace tqh {
int polar_quantize_to_cache(const void *x, const void *x2, int x_dtype, int num_heads, int tokens, uint8_t *packed,
                            uint16_t *scales, uint8_t *packed2, uint16_t *scales2, long long head_stride,
                            long long offset, int head_dim, int bits, size_t outlier_blocks, int norm_mode,
                            hipStream_t stream) {
  int rc = check_shape(head_dim);
  if (rc) return rc;
  PolarCodec codec;
  rc = polar_codec(bits, norm_mode, outlier_blocks, head_dim / 32, codec);
  if (rc) return rc;
  if (!valid_dtype(x_dtype)) return fail(TQ_ERR_INVALID_ARGUMENT, "unknown dtype %d", x_dtype);
  CacheMap m;
  rc = cache_map(num_heads, tokens, head_dim, head_stride, offset, m);
  if (rc) return rc;
  const long long nblocks = (long long)num_heads * tokens * (head_dim / 32);
  if (nblocks == 0) return TQ_OK;
  if (!x || !packed || !scales) return fail(TQ_ERR_INVALID_ARGUMENT, "null pointer");
  return launch_polar_quant<true>(x, x_dtype, packed, scales, nblocks, codec, m, Second{x2, packed2, scales2}, stream);
}

int store_token(const AppendToken &t, hipStream_t stream) {
  if (t.signs) {
    TqAppend a{};
    a.k = t.k;
    a.v = t.v;
    a.dtype = t.dtype;
    a.num_heads = t.num_heads;
    a.tokens = 1;
    a.k_idx = t.k_idx;
    a.v_idx = t.v_idx;
    a.k_sc = t.k_sc;
    a.v_sc = t.v_sc;
    a.signs = t.signs;
    a.norms = t.norms;
    a.head_stride = t.head_stride;
    a.offset = t.offset;
    a.head_dim = t.head_dim;
    a.bits = t.bits;
    a.norm_mode = t.norm_mode;
    a.sign_matrix = t.sign_matrix;
    a.q = t.q;
    a.q_dtype = t.q_dtype;
    a.rq = t.rq;
    a.num_q_rows = t.num_q_rows;
    return tq_append(a, stream);
  }
  return polar_quantize_to_cache(t.k, t.v, t.dtype, t.num_heads, 1, t.k_idx, t.k_sc, t.v_idx, t.v_sc, t.head_stride,
                                 t.offset, t.head_dim, t.bits, t.outlier_blocks, t.norm_mode, stream);
}
}  // namespace tqh

extern "C" int tq_polar_quantize_to_cache(const void *x, int x_dtype, int num_heads, int tokens,
                                          uint8_t *packed_cache, uint16_t *scales_cache, long long cache_head_stride,
                                          long long cache_offset, int head_dim, int bits, size_t outlier_blocks,
                                          int norm_mode, hipStream_t stream) {
  return tqh::polar_quantize_to_cache(x, nullptr, x_dtype, num_heads, tokens, packed_cache, scales_cache, nullptr,
                                      nullptr, cache_head_stride, cache_offset, head_dim, bits, outlier_blocks,
                                      norm_mode, stream);
}

namespace tqh {
int polar_dequantize_from_cache(const uint8_t *packed, const uint16_t *scales, const uint8_t *packed2,
                                const uint16_t *scales2, long long head_stride, int num_heads, int tokens, void *out,
                                void *out2, int out_dtype, int head_dim, int bits, size_t outlier_blocks,
                                int norm_mode, hipStream_t stream) {
  int rc = check_shape(head_dim);
  if (rc) return rc;
  PolarCodec codec;
  rc = polar_codec(bits, norm_mode, outlier_blocks, head_dim / 32, codec);
  if (rc) return rc;
  if (!valid_dtype(out_dtype)) return fail(TQ_ERR_INVALID_ARGUMENT, "unknown dtype %d", out_dtype);
  CacheMap m;
  rc = cache_map(num_heads, tokens, head_dim, head_stride, 0, m);
  if (rc) return rc;
  const long long nblocks = (long long)num_heads * tokens * (head_dim / 32);
  if (nblocks == 0) return TQ_OK;
  if (!packed || !scales || !out) return fail(TQ_ERR_INVALID_ARGUMENT, "null pointer");
  return launch_dequant<true>(packed, scales, out, out_dtype, nblocks, bits, dequant_consts(codec), m,
                              SecondOut{packed2, scales2, out2}, stream);
}
}  // namespace tqh

extern "C" int tq_polar_dequantize_from_cache(const uint8_t *packed_cache, const uint16_t *scales_cache,
                                              long long cache_head_stride, int num_heads, int tokens, void *out,
                                              int out_dtype, int head_dim, int bits, size_t outlier_blocks,
                                              int norm_mode, hipStream_t stream) {
  return tqh::polar_dequantize_from_cache(packed_cache, scales_cache, nullptr, nullptr, cache_head_stride, num_heads,
                                          tokens, out, nullptr, out_dtype, head_dim, bits, outlier_blocks, norm_mode,
                                          stream);
}

extern "C" int tq_pqo_quantize_to_cache(const void *x, int x_dtype, int num_heads, int tokens, uint8_t *packed_cache,
                                        uint16_t *scales_cache, long long cache_head_stride, long long cache_offset,
                                        int head_dim, int bits, hipStream_t stream) {
  return tq_polar_quantize_to_cache(x, x_dtype, num_heads, tokens, packed_cache, scales_cache, cache_head_stride,
                                    cache_offset, head_dim, bits, TQ_OUTLIER_ALL, TQ_NORM_MAXNORM, stream);
}

extern "C" int tq_pqo_dequantize_from_cache(const uint8_t *packed_cache, const uint16_t *scales_cache,
                                            long long cache_head_stride, int num_heads, int tokens, void *out,
                                            int out_dtype, int head_dim, int bits, hipStream_t stream) {
  return tq_polar_dequantize_from_cache(packed_cache, scales_cache, cache_head_stride, num_heads, tokens, out,
                                        out_dtype, head_dim, bits, TQ_OUTLIER_ALL, TQ_NORM_MAXNORM, stream);
}
