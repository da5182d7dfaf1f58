// tq_codec.hip -- core full-vector TurboQuant codec kernels (quantize_vec /
// dequantize_vec / dequantize_rotated, reference src/quantize.rs:142-316),
// batched on gfx950: d / 32 lanes per vector, see tq_codec_dev.h.  A wave
// covers 2048 / d consecutive vectors.
#include "tq_codec_dev.h"

namespace {

using namespace tqd;

constexpr int kBlock = 256;

// quantize_vec (quantize.rs:142-157) for `n` vectors of D f32.  Reads 4 D
// bytes per vector and writes about a tenth of it; small batches are bound by
// one lane's instructions, large ones by the reads.  10,000 vectors of 128 at
// 3 bits: 14.3 us with a lane per vector, 5.0 us now.
template <int D, int BITS>
__global__ __launch_bounds__(kBlock) void codec_quant_kernel(const float *__restrict__ x, uint8_t *__restrict__ packed,
                                                             uint16_t *__restrict__ scales, long long n,
                                                             CodecConsts k) {
  constexpr int LPV = Geo<D>::LPV;
  const long long t = (long long)blockIdx.x * kBlock + threadIdx.x;
  const long long v = t / LPV;
  const int q = (int)(t % LPV);
  if (v >= n) return;  // LPV divides 64: a vector's lanes leave together
  float w[32];
  load_elements(x + t * 32, w);
  uint32_t pk[BITS];
  const float norm = quantize_lanes<LPV, BITS>(w, q, k, pk);
  store_codes<BITS>(packed + t * (4 * BITS), pk);
  if (q == 0) scales[v] = f32_to_f16(norm < kMinNorm ? 0.0f : norm);  // select_scale, quantize.rs:123-126
}

// Batches of up to two waves, latency alone, store from the registers: the
// staging would only lengthen them (us, staged / direct: 100 vectors of 32 2.95
// / 2.77, 200 3.10 / 3.30; 64 of 64 3.12 / 2.95, 100 3.32 / 3.44; 32 of 128 3.21 /
// 3.16, 64 3.39 / 3.73; 8 of 256 3.52 / 3.38, 24 3.55 / 3.90).
constexpr long long kDirectLanes = 128;

// dequantize_vec (quantize.rs:225-240) or, ROTATE = false, dequantize_rotated
// (quantize.rs:306-316).  A wave's 64 lanes make one run of 8 KB: staged
// through LDS, each store instruction writes 1 KB of it.  10,000 vectors of
// 128 at 3 bits: 9.9 us (rotated 7.3) with a lane per vector, 4.6 us (3.6) now.
template <int D, int BITS, bool ROTATE>
__global__ __launch_bounds__(kBlock) void codec_dequant_kernel(const uint8_t *__restrict__ packed,
                                                               const uint16_t *__restrict__ scales,
                                                               float *__restrict__ out, long long n, CodecConsts k) {
  constexpr int LPV = Geo<D>::LPV, RS = 36;  // staged floats per lane, padded
  __shared__ float s_cent[16];
  __shared__ __attribute__((aligned(16))) float s_out[kBlock / 64][64 * RS];
  if (threadIdx.x < 16) s_cent[threadIdx.x] = k.cent[threadIdx.x & ((1 << BITS) - 1)];
  __syncthreads();
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const long long t = (long long)blockIdx.x * kBlock + threadIdx.x;
  const long long v = t / LPV;
  const int q = (int)(t % LPV);
  uint32_t pk[BITS] = {};
  float sc = 0.f;
  if (v < n) {  // the others still take part in the wave's staging
    load_codes<BITS>(packed + t * (4 * BITS), pk);
    sc = f16_to_f32(scales[v]);
  }
  float w[32];
  dequant_lanes<LPV, BITS, ROTATE>(pk, sc, q, s_cent, k, w);
  if (n * LPV <= kDirectLanes) {
    if (v < n) {
      float4 *o = reinterpret_cast<float4 *>(out + t * 32);
#pragma unroll
      for (int i = 0; i < 8; i++) o[i] = make_float4(w[4 * i], w[4 * i + 1], w[4 * i + 2], w[4 * i + 3]);
    }
    return;
  }
  float4 *row = reinterpret_cast<float4 *>(s_out[wave] + lane * RS);
#pragma unroll
  for (int i = 0; i < 8; i++) row[i] = make_float4(w[4 * i], w[4 * i + 1], w[4 * i + 2], w[4 * i + 3]);
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  const long long t0 = t - lane;  // the wave's first run of 32
#pragma unroll
  for (int i = 0; i < 8; i++) {
    const int f = 256 * i + 4 * lane, r = f / 32;
    if (t0 + r < n * LPV)
      *reinterpret_cast<float4 *>(out + t0 * 32 + f) = *reinterpret_cast<const float4 *>(s_out[wave] + r * RS + f % 32);
  }
}

template <template <int, int> class Launch, typename A>
int dispatch(int dim, int bits, const A &a) {
  switch (dim * 8 + bits) {
    case 32 * 8 + 2: return Launch<32, 2>::run(a);
    case 32 * 8 + 3: return Launch<32, 3>::run(a);
    case 32 * 8 + 4: return Launch<32, 4>::run(a);
    case 64 * 8 + 2: return Launch<64, 2>::run(a);
    case 64 * 8 + 3: return Launch<64, 3>::run(a);
    case 64 * 8 + 4: return Launch<64, 4>::run(a);
    case 128 * 8 + 2: return Launch<128, 2>::run(a);
    case 128 * 8 + 3: return Launch<128, 3>::run(a);
    case 128 * 8 + 4: return Launch<128, 4>::run(a);
    case 256 * 8 + 2: return Launch<256, 2>::run(a);
    case 256 * 8 + 3: return Launch<256, 3>::run(a);
    case 256 * 8 + 4: return Launch<256, 4>::run(a);
  }
  return tqh::fail(TQ_ERR_INVALID_DIMENSION, "unsupported dim %d", dim);
}

struct QuantArgs {
  const float *x;
  uint8_t *packed;
  uint16_t *scales;
  long long n;
  CodecConsts k;
  hipStream_t stream;
};

template <int D, int BITS>
struct QuantLaunch {
  static int run(const QuantArgs &a) {
    const long long threads = a.n * Geo<D>::LPV;
    hipLaunchKernelGGL((codec_quant_kernel<D, BITS>), dim3((unsigned)((threads + kBlock - 1) / kBlock)), dim3(kBlock),
                       0, a.stream, a.x, a.packed, a.scales, a.n, a.k);
    return tqh::check_launch("codec_quant_kernel");
  }
};

struct DequantArgs {
  const uint8_t *packed;
  const uint16_t *scales;
  float *out;
  long long n;
  CodecConsts k;
  bool rotate;
  hipStream_t stream;
};

template <int D, int BITS>
struct DequantLaunch {
  static int run(const DequantArgs &a) {
    const long long threads = a.n * Geo<D>::LPV;
    const dim3 grid((unsigned)((threads + kBlock - 1) / kBlock));
    if (a.rotate)
      hipLaunchKernelGGL((codec_dequant_kernel<D, BITS, true>), grid, dim3(kBlock), 0, a.stream, a.packed,
                         a.scales, a.out, a.n, a.k);
    else
      hipLaunchKernelGGL((codec_dequant_kernel<D, BITS, false>), grid, dim3(kBlock), 0, a.stream, a.packed,
                         a.scales, a.out, a.n, a.k);
    return tqh::check_launch("codec_dequant_kernel");
  }
};

constexpr long long kMaxVectors = (1ll << 31) / 2;

}  // namespace

extern "C" int tq_quantize_vec_batch(const float *data, uint8_t *packed_out, uint16_t *scales_out, size_t num_vectors,
                                     int bits, int dim, uint64_t rotation_seed, hipStream_t stream) {
  CodecConsts k;
  int rc = tqh::make_codec_consts(bits, dim, rotation_seed, k);
  if (rc) return rc;
  if (num_vectors == 0) return TQ_OK;
  if ((long long)num_vectors > kMaxVectors) return tqh::fail(TQ_ERR_INVALID_ARGUMENT, "too many vectors");
  if (!data || !packed_out || !scales_out) return tqh::fail(TQ_ERR_INVALID_ARGUMENT, "null pointer");
  return dispatch<QuantLaunch>(dim, bits, QuantArgs{data, packed_out, scales_out, (long long)num_vectors, k, stream});
}

static int dequant_common(const uint8_t *packed, const uint16_t *scales, float *out, size_t num_vectors, int bits,
                          int dim, uint64_t seed, bool rotate, hipStream_t stream) {
  CodecConsts k;
  int rc = tqh::make_codec_consts(bits, dim, seed, k);
  if (rc) return rc;
  if (num_vectors == 0) return TQ_OK;
  if ((long long)num_vectors > kMaxVectors) return tqh::fail(TQ_ERR_INVALID_ARGUMENT, "too many vectors");
  if (!packed || !scales || !out) return tqh::fail(TQ_ERR_INVALID_ARGUMENT, "null pointer");
  return dispatch<DequantLaunch>(dim, bits, DequantArgs{packed, scales, out, (long long)num_vectors, k, rotate, stream});
}

extern "C" int tq_dequantize_vec_batch(const uint8_t *packed, const uint16_t *scales, float *out, size_t num_vectors,
                                       int bits, int dim, uint64_t rotation_seed, hipStream_t stream) {
  return dequant_common(packed, scales, out, num_vectors, bits, dim, rotation_seed, true, stream);
}

extern "C" int tq_dequantize_rotated_batch(const uint8_t *packed, const uint16_t *scales, float *out,
                                           size_t num_vectors, int bits, int dim, hipStream_t stream) {
  return dequant_common(packed, scales, out, num_vectors, bits, dim, 0, false, stream);
}
