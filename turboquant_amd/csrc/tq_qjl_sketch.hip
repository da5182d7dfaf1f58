// tq_qjl_sketch.hip -- a TQ cache's append (codes, scales, sketch) and the
// query projection R q on gfx950 (reference src/cache/tq.rs:97-182, 233-234,
// 373-412; src/qjl.rs:196-208, 305-319).
//
// The reference sums a row product in column order from -0.0 with one
// rounding per term, and both the sketch's signs and rq have to be its bits.
// v_mfma_f32_16x16x4_f32 adds its four products one after the other, in k
// order, each step rounded as one fused multiply-add (checked on MI355X
// against fmaf chains: random values of widely mixed magnitudes, denormals
// and zeros, no difference in 100,000 sums of 128 terms), so a chain of them
// over the columns is that sum, for 16 vectors x 16 rows of R at a time and
// at twice the rate of the vector unit, which also needs no select per term:
// R's entry is 1.0 with the sign bit inserted.
//
// A workgroup takes 16 vectors: lane = qblock quantizes (keys in the first
// lanes, values in the next), the key lanes decode their codes again and
// leave the residual in LDS, then wave w sums rows 32 w .. + 31 of R for all
// 16 (two chains, so neither waits for its own last step; a projection of few
// rows by itself gives each wave one).  Bound by the chains: D / 4 steps of 32
// cycles for two tiles each, 0.9 us at D = 128; launches bound a short append
// (prefill, extension, a decode whose token the attention launch does not
// store), which took three (keys, values, sketch with projection: two of 3.8
// us and one of 4.0 us, 16 tokens) and takes one.
#include "tq_pqo_dev.h"

#include <type_traits>

namespace {

using namespace tqp;

typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kVecs = 16;  // vectors (or query rows) per workgroup

template <int D>
struct Geo {
  static constexpr int NQB = D / 32, NW = D / 32, WAVES = D / 32, THREADS = 64 * WAVES;
  static constexpr int RS = D + 4;  // floats per staged row: the chain's reads hit 64 banks
};

// Sign words of R's rows 16 (T wave + t) + l16, shifted so that column
// 4 k + lg of word w is bit 4 k.
template <int D, int T>
__device__ __forceinline__ void load_rows(const uint32_t *__restrict__ rbits, int wave, int l16, int lg,
                                          uint32_t (&rb)[T][Geo<D>::NW]) {
#pragma unroll
  for (int t = 0; t < T; t++)
#pragma unroll
    for (int w = 0; w < Geo<D>::NW; w++) rb[t][w] = rbits[(16 * (T * wave + t) + l16) * Geo<D>::NW + w] >> lg;
}

// acc[t][i] = sum_c R[16 (T wave + t) + 4 lg + i][c] v[l16][c] (R = +-1), in
// column order from -0.0, for the 16 vectors staged in LDS.
template <int D, int T>
__device__ __forceinline__ void row_products(const float *s_v, const uint32_t (&rb)[T][Geo<D>::NW], int l16, int lg,
                                             f32x4 (&acc)[T]) {
#pragma unroll
  for (int t = 0; t < T; t++) acc[t] = f32x4{-0.0f, -0.0f, -0.0f, -0.0f};
  const float *v = s_v + l16 * Geo<D>::RS + lg;
#pragma unroll
  for (int w = 0; w < Geo<D>::NW; w++) {
    float x[8];
#pragma unroll
    for (int k = 0; k < 8; k++) x[k] = v[32 * w + 4 * k];
#pragma unroll
    for (int k = 0; k < 8; k++)
#pragma unroll
      for (int t = 0; t < T; t++) {
        const float a = u2f(((rb[t][w] << (31 - 4 * k)) & 0x80000000u) | 0x3f800000u);
        acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(a, x[k], acc[t], 0, 0, 0);
      }
  }
}

__device__ __forceinline__ float load_elem(const void *p, long long i, int dtype) {
  if (dtype == kF32) return static_cast<const float *>(p)[i];
  const uint16_t h = static_cast<const uint16_t *>(p)[i];
  return dtype == kBF16 ? bf16_to_f32(h) : f16_to_f32(h);
}

// rq = R q for query rows row0 .. + 15 (precompute_query_projections,
// qjl.rs:488-492; r_q = q R^T of tq.rs:233-234).
template <int D, int T>
__device__ __forceinline__ void project_rows(const void *q, int q_dtype, float *rq, long long row0, long long nq,
                                             float inv, float *s_v, const uint32_t (&rb)[T][Geo<D>::NW], int tid,
                                             int wave, int l16, int lg) {
  // a thread's 4 T elements by one or two loads, from any element boundary (one
  // element a load, one after the other: 16 bf16 rows of d = 64 3.7 us, 2.6 so)
  constexpr int E = 4 * T;
  const int r = E * tid / D, e = E * tid % D;
  float x[E] = {};
  if (row0 + r < nq) {
    const long long i = row0 * D + E * tid;
    if (q_dtype == kF32) {
      __builtin_memcpy(x, static_cast<const float *>(q) + i, 4 * E);
    } else {
      uint16_t h[E];
      __builtin_memcpy(h, static_cast<const uint16_t *>(q) + i, 2 * E);
#pragma unroll
      for (int j = 0; j < E; j++) x[j] = q_dtype == kBF16 ? bf16_to_f32(h[j]) : f16_to_f32(h[j]);
    }
  }
  float4 *dst = reinterpret_cast<float4 *>(s_v + r * Geo<D>::RS + e);
#pragma unroll
  for (int j = 0; j < T; j++) dst[j] = make_float4(x[4 * j], x[4 * j + 1], x[4 * j + 2], x[4 * j + 3]);
  __syncthreads();
  f32x4 acc[T];
  row_products<D>(s_v, rb, l16, lg, acc);
  if (row0 + l16 >= nq) return;
#pragma unroll
  for (int t = 0; t < T; t++)
#pragma unroll
    for (int i = 0; i < 4; i++) rq[(row0 + l16) * D + 16 * (T * wave + t) + 4 * lg + i] = acc[t][i] * inv;
}

struct SketchArgs {
  const void *k, *v;  // v: APPEND only
  uint8_t *k_idx, *v_idx;
  uint16_t *k_sc, *v_sc;
  const uint32_t *rbits;
  uint32_t *signs;
  uint16_t *norms;
  long long nvec, head_stride, offset;
  int tokens;
  int key_blocks;      // workgroups of keys; those after them project query rows
  int k_vec;           // k on a 16-byte boundary
  float cb[16];        // the cache codec's centroids
  float decode_factor; // magnitude of the decode signs
  float inv_sqrt_d;
  const void *q;
  int q_dtype;
  float *rq;
  long long nq;
  QuantConsts qc;      // APPEND only
};

// compute_qjl_signs_and_norms (tq.rs:154-182, 373-412) for the keys that are
// stored in the records (!APPEND) or that this launch stores together with
// the values (APPEND: polar_quantize, quantize_tensor.rs:40-76, with (BITS -
// 1)-bit codes in BITS-wide slots).  The residual r = k - k_hat takes k_hat
// as polar_dequantize's CPU branch gives it (quantize_tensor.rs:197-219,
// butterflies); sum r^2 runs in element order through the key's lanes.
template <int D, int BITS, int IN_DT, int NORM, bool APPEND>
__global__ __launch_bounds__(Geo<D>::THREADS) void qjl_sketch_kernel(SketchArgs a) {
  using G = Geo<D>;
  constexpr int NQB = G::NQB;
  __shared__ __attribute__((aligned(16))) float s_v[kVecs * G::RS];
  __shared__ float s_cb[16];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l16 = lane & 15, lg = lane >> 4;
  uint32_t rb[2][G::NW];
  load_rows<D>(a.rbits, wave, l16, lg, rb);
  if ((int)blockIdx.x >= a.key_blocks) {
    project_rows<D>(a.q, a.q_dtype, a.rq, (long long)(blockIdx.x - a.key_blocks) * kVecs, a.nq, a.inv_sqrt_d, s_v, rb,
                    tid, wave, l16, lg);
    return;
  }
  // element j of a block decodes to +-(c * factor), negative where the sign pattern is
#pragma unroll
  for (int i = 0; i < 16; i++)
    if (tid == i) s_cb[i] = a.cb[i] * a.decode_factor;
  const long long vec0 = (long long)blockIdx.x * kVecs;
  auto record = [&](long long v) {
    if (a.nvec >> 32) {
      const long long h = v / a.tokens;
      return h * a.head_stride + a.offset + (v - h * a.tokens);
    }
    const uint32_t h = (uint32_t)v / (uint32_t)a.tokens;
    return (long long)h * a.head_stride + a.offset + (long long)((uint32_t)v - h * (uint32_t)a.tokens);
  };
  const int qb = tid % NQB, vi = (tid / NQB) % kVecs;
  const long long v = vec0 + vi;
  const bool is_v = APPEND && tid >= kVecs * NQB;
  const bool live = tid < (APPEND ? 2 : 1) * kVecs * NQB && v < a.nvec;
  uint32_t w[BITS];
  float x[32], s = 0.f;
  long long rec = 0;
  if (live) {
    rec = record(v);
    if constexpr (APPEND) {
      load_block<IN_DT>(is_v ? a.v : a.k, v * NQB + qb, x);
      float r[32];
#pragma unroll
      for (int j = 0; j < 32; j++) r[j] = x[j];
      s = encode_block<BITS, BITS - 1, true, NORM>(r, a.qc, w);
      store_packed<BITS>(is_v ? a.v_idx : a.k_idx, rec * NQB + qb, w);
      const uint16_t h = f32_to_f16(s * a.qc.scale_sign);
      (is_v ? a.v_sc : a.k_sc)[rec * NQB + qb] = h;
      s = fabsf(f16_to_f32(h));
    } else {
      const long long blk = v * NQB + qb;
      if (a.k_vec) {
        load_block<IN_DT>(a.k, blk, x);
      } else {
#pragma unroll
        for (int j = 0; j < 32; j++) x[j] = load_elem(a.k, blk * 32 + j, IN_DT);
      }
      const uint32_t *p = reinterpret_cast<const uint32_t *>(a.k_idx + (rec * NQB + qb) * (4 * BITS));
#pragma unroll
      for (int i = 0; i < BITS; i++) w[i] = p[i];
      s = fabsf(f16_to_f32(a.k_sc[rec * NQB + qb]));
    }
  }
  __syncthreads();
  if (live && !is_v) {
    float y[32];
#pragma unroll
    for (int j = 0; j < 32; j++) {
      const float c = s_cb[field<BITS>(w, j)];
      y[j] = pqo_neg(j) ? -c : c;
    }
    butterfly<32>(y);
#pragma unroll
    for (int j = 0; j < 32; j++) x[j] = x[j] - (y[j] * kInvSqrt32) * s;
    float4 *dst = reinterpret_cast<float4 *>(s_v + vi * G::RS + 32 * qb);
#pragma unroll
    for (int j = 0; j < 8; j++) dst[j] = make_float4(x[4 * j], x[4 * j + 1], x[4 * j + 2], x[4 * j + 3]);
    // lane qb continues the sum of lane qb - 1; after NQB rounds the last
    // lane's has run over the whole key
#pragma unroll
    for (int j = 0; j < 32; j++) x[j] = x[j] * x[j];
    float ss = 0.f;
#pragma unroll
    for (int round = 0; round < NQB; round++) {
      const float before = __shfl_up(ss, 1, 64);
      ss = qb == 0 ? 0.f : before;
#pragma unroll
      for (int j = 0; j < 32; j++) ss = ss + x[j];
    }
    if (qb == NQB - 1) a.norms[rec] = f32_to_f16(sqrtf(ss));
  }
  __syncthreads();
  f32x4 acc[2];
  row_products<D>(s_v, rb, l16, lg, acc);
  // sign bit j = (R r)_j >= 0 (qjl.rs:305-319): the wave's 32 rows are one word of the key
  uint32_t bits = 0;
#pragma unroll
  for (int t = 0; t < 2; t++)
#pragma unroll
    for (int i = 0; i < 4; i++) bits |= (acc[t][i] * a.inv_sqrt_d >= 0.0f ? 1u : 0u) << (16 * t + 4 * lg + i);
  bits |= __shfl_xor(bits, 16, 64);
  bits |= __shfl_xor(bits, 32, 64);
  if (lg == 0 && vec0 + l16 < a.nvec) a.signs[record(vec0 + l16) * G::NW + wave] = bits;
}

// T tiles of 16 rows of R a wave.  Up to kFewRows query rows the grid is small
// and a wave's chain is what it takes: one tile (us, two / one: d = 64, 100 rows
// 2.86 / 2.54, 4,000 3.04 / 2.69, 16,384 4.13 / 4.10; d = 128 3.73 / 3.36, 4.10 /
// 3.75, 8.81 / 8.66); more rows are bound by the staged vectors' reads, which two
// tiles share (131,072 rows, f32, d = 128 45.7 / 48.7, d = 256 162.5 / 173.9).
constexpr long long kFewRows = 8192;
template <int D, int T>
__global__ __launch_bounds__(4 * D / T) void qjl_project_kernel(const void *__restrict__ q, int q_dtype,
                                                                const uint32_t *__restrict__ rbits,
                                                                float *__restrict__ rq, long long nrows, float inv) {
  __shared__ __attribute__((aligned(16))) float s_v[kVecs * Geo<D>::RS];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  uint32_t rb[T][Geo<D>::NW];
  load_rows<D>(rbits, wave, lane & 15, lane >> 4, rb);
  project_rows<D>(q, q_dtype, rq, (long long)blockIdx.x * kVecs, nrows, inv, s_v, rb, tid, wave, lane & 15, lane >> 4);
}

int check_sketch_dim(int dim) {
  if (dim != 64 && dim != 128 && dim != 256)
    return tqh::fail(TQ_ERR_INVALID_DIMENSION, "cache QJL kernels take head_dim 64, 128 or 256 (got %d)", dim);
  return TQ_OK;
}

template <typename F>
int by_cache_dim(int dim, F &&f) {
  switch (dim) {
    case 64: return f(std::integral_constant<int, 64>{});
    case 128: return f(std::integral_constant<int, 128>{});
    case 256: return f(std::integral_constant<int, 256>{});
  }
  return tqh::fail(TQ_ERR_INVALID_DIMENSION, "unsupported head_dim %d", dim);
}

template <int D, int NORM, bool APPEND>
int launch_sketch(const SketchArgs &a, int bits, int dtype, unsigned grid, hipStream_t st) {
#define SK(B, T) \
  hipLaunchKernelGGL((qjl_sketch_kernel<D, B, T, NORM, APPEND>), dim3(grid), dim3(Geo<D>::THREADS), 0, st, a)
  if (bits == 3) {
    if (dtype == kF32) SK(3, kF32);
    else if (dtype == kBF16) SK(3, kBF16);
    else SK(3, kF16);
  } else {
    if (dtype == kF32) SK(4, kF32);
    else if (dtype == kBF16) SK(4, kBF16);
    else SK(4, kF16);
  }
#undef SK
  return tqh::check_launch("qjl_sketch_kernel");
}

// The arguments that both entries share, checked; a.nvec + a.nq = 0: nothing to do.
int sketch_args(SketchArgs &a, tqh::PolarCodec &codec, const void *k, int k_dtype, int num_heads, int tokens,
                const uint32_t *sign_matrix, uint8_t *signs, uint16_t *norms, long long head_stride, long long offset,
                int head_dim, int bits, size_t outlier_blocks, int norm_mode, const void *q, int q_dtype, float *rq,
                size_t num_q_rows, unsigned &grid) {
  int rc = check_sketch_dim(head_dim);
  if (rc) return rc;
  rc = tqh::polar_codec(bits, norm_mode, outlier_blocks, head_dim / 32, codec);
  if (rc) return rc;
  if (!tqh::valid_dtype(k_dtype)) return tqh::fail(TQ_ERR_INVALID_ARGUMENT, "unknown dtype %d", k_dtype);
  if (num_heads < 0 || tokens < 0) return tqh::fail(TQ_ERR_INVALID_ARGUMENT, "negative shape");
  if (offset < 0 || head_stride < offset + tokens)
    return tqh::fail(TQ_ERR_RANGE_OUT_OF_BOUNDS, "cache rows [%lld, %lld) exceed head stride %lld", offset,
                     offset + tokens, head_stride);
  a.nvec = (long long)num_heads * tokens;
  a.nq = (long long)num_q_rows;
  if (a.nvec + a.nq == 0) return TQ_OK;
  if (!sign_matrix || (a.nvec && (!k || !signs || !norms)))
    return tqh::fail(TQ_ERR_INVALID_ARGUMENT, "null pointer");
  if (a.nq && (!q || !rq || !tqh::valid_dtype(q_dtype)))
    return tqh::fail(TQ_ERR_INVALID_ARGUMENT, "query projection needs q (f32/bf16/f16) and rq");
  const long long key_blocks = (a.nvec + kVecs - 1) / kVecs, blocks = key_blocks + (a.nq + kVecs - 1) / kVecs;
  if (blocks * 2 * head_dim >= 1ll << 32)  // a launch holds fewer than 2^32 lanes
    return tqh::fail(TQ_ERR_INVALID_ARGUMENT, "too many vectors in one call");
  a.k = k;
  a.rbits = sign_matrix;
  a.signs = reinterpret_cast<uint32_t *>(signs);
  a.norms = norms;
  a.head_stride = head_stride;
  a.offset = offset;
  a.tokens = tokens > 0 ? tokens : 1;
  a.key_blocks = (int)key_blocks;
  a.k_vec = reinterpret_cast<uintptr_t>(k) % 16 == 0;
  for (int i = 0; i < codec.cb.nc; i++) a.cb[i] = codec.cb.c[i];
  {
    volatile float thirty_two = 32.0f;
    volatile float sq = sqrtf(thirty_two);
    volatile float inv = 1.0f / sq;
    a.decode_factor = inv * sq;  // fl(fl(1/sqrt 32) * sqrt 32) (wht_tensor.rs:28-41)
  }
  a.inv_sqrt_d = tqh::inv_sqrt_dim(head_dim);
  a.q = q;
  a.q_dtype = q_dtype;
  a.rq = rq;
  grid = (unsigned)blocks;
  return TQ_OK;
}

}  // namespace

namespace tqh {

int tq_append(const TqAppend &p, hipStream_t stream) {
  SketchArgs a{};
  PolarCodec codec;
  unsigned grid = 0;
  int rc = sketch_args(a, codec, p.k, p.dtype, p.num_heads, p.tokens, p.sign_matrix, p.signs, p.norms, p.head_stride,
                       p.offset, p.head_dim, p.bits, 0, p.norm_mode, p.q, p.q_dtype, p.rq, p.num_q_rows, grid);
  if (rc || grid == 0) return rc;
  if (a.nvec * (p.head_dim / 32) >= (1ll << 31))
    return fail(TQ_ERR_INVALID_ARGUMENT, "too many blocks in one call");
  if (a.nvec && (!p.v || !p.k_idx || !p.v_idx || !p.k_sc || !p.v_sc))
    return fail(TQ_ERR_INVALID_ARGUMENT, "null pointer");
  a.v = p.v;
  a.k_idx = p.k_idx;
  a.v_idx = p.v_idx;
  a.k_sc = p.k_sc;
  a.v_sc = p.v_sc;
  a.qc = make_quant_consts(codec.cb, codec.outer, codec.scale_sign);
  return by_cache_dim(p.head_dim, [&](auto d) {
    constexpr int D = decltype(d)::value;
    if (p.norm_mode == kL2Norm) return launch_sketch<D, kL2Norm, true>(a, p.bits, p.dtype, grid, stream);
    return launch_sketch<D, kMaxNorm, true>(a, p.bits, p.dtype, grid, stream);
  });
}

}  // namespace tqh

extern "C" int tq_qjl_cache_sketch_project(const void *k, int k_dtype, int num_heads, int tokens,
                                           const uint8_t *packed_cache, const uint16_t *scales_cache,
                                           const uint32_t *sign_matrix, uint8_t *signs_cache, uint16_t *norms_cache,
                                           long long cache_head_stride, long long cache_offset, int head_dim, int bits,
                                           size_t outlier_blocks, int norm_mode, const void *q, int q_dtype, float *rq,
                                           size_t num_q_rows, hipStream_t stream) {
  SketchArgs a{};
  tqh::PolarCodec codec;
  unsigned grid = 0;
  int rc = sketch_args(a, codec, k, k_dtype, num_heads, tokens, sign_matrix, signs_cache, norms_cache,
                       cache_head_stride, cache_offset, head_dim, bits, outlier_blocks, norm_mode, q, q_dtype, rq,
                       num_q_rows, grid);
  if (rc || grid == 0) return rc;
  if (a.nvec && (!packed_cache || !scales_cache)) return tqh::fail(TQ_ERR_INVALID_ARGUMENT, "null pointer");
  a.k_idx = const_cast<uint8_t *>(packed_cache);   // read only
  a.k_sc = const_cast<uint16_t *>(scales_cache);
  return by_cache_dim(head_dim, [&](auto d) {
    return launch_sketch<decltype(d)::value, kMaxNorm, false>(a, bits, k_dtype, grid, stream);
  });
}

extern "C" int tq_qjl_cache_sketch(const void *k, int k_dtype, int num_heads, int tokens, const uint8_t *packed_cache,
                                   const uint16_t *scales_cache, const uint32_t *sign_matrix, uint8_t *signs_cache,
                                   uint16_t *norms_cache, long long cache_head_stride, long long cache_offset,
                                   int head_dim, int bits, size_t outlier_blocks, int norm_mode, hipStream_t stream) {
  return tq_qjl_cache_sketch_project(k, k_dtype, num_heads, tokens, packed_cache, scales_cache, sign_matrix,
                                     signs_cache, norms_cache, cache_head_stride, cache_offset, head_dim, bits,
                                     outlier_blocks, norm_mode, nullptr, TQ_DTYPE_F32, nullptr, 0, stream);
}

extern "C" int tq_qjl_project(const void *q, int q_dtype, const uint32_t *sign_matrix, float *rq, size_t num_rows,
                              int dim, hipStream_t stream) {
  int rc = check_sketch_dim(dim);
  if (rc) return rc;
  if (!tqh::valid_dtype(q_dtype)) return tqh::fail(TQ_ERR_INVALID_ARGUMENT, "unknown dtype %d", q_dtype);
  if (num_rows == 0) return TQ_OK;
  if (!q || !sign_matrix || !rq) return tqh::fail(TQ_ERR_INVALID_ARGUMENT, "null pointer");
  const long long n = (long long)num_rows;
  if ((n + kVecs - 1) / kVecs * 2 * dim >= 1ll << 32) return tqh::fail(TQ_ERR_INVALID_ARGUMENT, "too many rows in one call");
  return by_cache_dim(dim, [&](auto d) {
    constexpr int D = decltype(d)::value;
    const dim3 grid((unsigned)((n + kVecs - 1) / kVecs));
    const float inv = tqh::inv_sqrt_dim(dim);
    if (n <= kFewRows)
      hipLaunchKernelGGL((qjl_project_kernel<D, 1>), grid, dim3(4 * D), 0, stream, q, q_dtype, sign_matrix, rq, n, inv);
    else
      hipLaunchKernelGGL((qjl_project_kernel<D, 2>), grid, dim3(2 * D), 0, stream, q, q_dtype, sign_matrix, rq, n, inv);
    return tqh::check_launch("qjl_project_kernel");
  });
}
