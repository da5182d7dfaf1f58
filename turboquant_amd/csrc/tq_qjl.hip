// tq_qjl.hip -- QJL inner-product estimator (reference src/qjl.rs,
// src/attention.rs) on gfx950: key quantization with the 1-bit sign sketch,
// query projections, batched score estimation, softmax and weighted values.
//
// The Rademacher matrix R[j][c] = sign(j, c) / sqrt(d) is implicit in the
// reference (a SplitMix64 hash per entry, qjl.rs:143-189).  A workgroup hashes
// the sign bits it needs; a row product is d fused multiply-adds with a +-1
// factor in column order, which is exactly the reference's sequential sum of
// sign * value (the product is exact, so fma(sign, v, s) == fl(s + sign * v)).
//
// Scores use the rotated domain: <q, x_mse> = scale * <qt, c[idx]> with
// qt = H(s * q) / sqrt(d), the forward rotation of the query, so keys are
// never inverse-rotated, and both of a score's sums are matrix products.
#include "tq_codec_dev.h"
#include "tq_mfma.h"

#include <algorithm>
#include <type_traits>

namespace {

using namespace tqd;

constexpr int kBlock = 256;
constexpr uint64_t kGolden = 0x9E3779B97F4A7C15ull;

// qjl.rs:143-147
__device__ __forceinline__ uint64_t mix_seed(uint64_t seed, uint64_t row) {
  const uint64_t m = seed * 0x517CC1B727220A95ull + row;
  return m ^ (m >> 32) ^ 0x6C62272E07BB0142ull;
}

// qjl.rs:157-171: true where sign(row, col) = -1 (SplitMix64 finalizer odd),
// base = row_seed + row * golden.  Only bits 0 and 31 of the last product
// reach the parity, so its low word is enough.
__device__ __forceinline__ bool sign_negative(uint64_t base, uint32_t col) {
  uint64_t z = base + col;
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  const uint32_t p = (uint32_t)(z ^ (z >> 27)) * 0x133111EBu;
  return ((p ^ (p >> 31)) & 1u) != 0;
}
__device__ __forceinline__ uint64_t sign_base(uint64_t seed, uint64_t row) { return mix_seed(seed, row) + row * kGolden; }

struct QjlConsts {
  CodecConsts polar;   // (total_bits - 1)-bit codec of the same dimension
  uint64_t qjl_seed;
  float inv_sqrt_d;    // fl(1 / fl(sqrt(d)))
  float sqrt_d;        // fl(sqrt(d))
};

// +-1 for the four sign bits of a nibble (bit i set <=> element i negative)
__device__ __forceinline__ float4 nibble_signs(int nib) {
  return make_float4((nib & 1) ? -1.0f : 1.0f, (nib & 2) ? -1.0f : 1.0f, (nib & 4) ? -1.0f : 1.0f,
                     (nib & 8) ? -1.0f : 1.0f);
}

// quantize_with_qjl (qjl.rs:355-377) for 32 keys per workgroup of D / 16
// waves.  D / 32 lanes of a key quantize it (polar codes, scale, residual r =
// x - dequantized x, |r|) and stage r in LDS; meanwhile every wave hashes the
// signs of its 16 rows of R straight into the lanes that use them; then it
// sums those rows for the 32 keys on the matrix cores.  A row is summed in
// column order from -0.0 as rademacher_vector_product does (qjl.rs:196-208):
// v_mfma_f32_16x16x4_f32 adds its four products one after the other in k
// order, each step one fused multiply-add (checked on MI355X against fmaf
// chains), and fma(+-1, r_c, s) is the reference's fl(s + sign * r_c).
//
// Bound by the instructions of one workgroup: 32 hashes a lane, the codec of
// 32 elements, 2 x 32 matrix steps of 32 cycles.  8,192 keys of d = 128, 3
// bits: 36.2 us with the codec on one lane per key, all of R hashed into LDS
// by every workgroup and the sums on the vector unit; 11.1 us now.
template <int D, int PB>
__global__ __launch_bounds__(4 * D) void qjl_quant_kernel(const float *__restrict__ x, uint8_t *__restrict__ polar,
                                                          uint16_t *__restrict__ polar_scales,
                                                          uint16_t *__restrict__ signs,
                                                          uint16_t *__restrict__ residual_norms, long long n,
                                                          QjlConsts k) {
  constexpr int KB = 32, LPV = D / 32, RS = D + 4;  // floats per staged row: the sums' reads hit 64 banks
  __shared__ float s_cent[16];
  __shared__ __attribute__((aligned(16))) float s_res[KB * RS];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l16 = lane & 15, lg = lane >> 4;
  const long long key0 = (long long)blockIdx.x * KB;
  const long long v = key0 + tid / LPV;
  const int q = tid % LPV;
  const bool live = tid < KB * LPV && v < n;
  float w[32];
  if (live) load_elements(x + v * D + 32 * q, w);
  if (tid < 16) s_cent[tid] = k.polar.cent[tid & ((1 << PB) - 1)];
  // bit i: sign of (row 16 wave + l16, column 4 i + lg) is -1
  uint32_t rb = 0;
  const uint64_t base = sign_base(k.qjl_seed, (uint64_t)(16 * wave + l16));
#pragma unroll 8
  for (int i = 0; i < D / 4; i++) rb |= (sign_negative(base, (uint32_t)(4 * i + lg)) ? 1u : 0u) << i;
  __syncthreads();
  if (live) {
    float r[32];
#pragma unroll
    for (int e = 0; e < 32; e++) r[e] = w[e];
    uint32_t pk[PB];
    const float norm = quantize_lanes<LPV, PB>(w, q, k.polar, pk);
    const uint16_t sc = f32_to_f16(norm < kMinNorm ? 0.0f : norm);
    store_codes<PB>(polar + (v * LPV + q) * (4 * PB), pk);
    // x_mse = dequantize_vec(polar block), residual r = x - x_mse (qjl.rs:362-368)
    dequant_lanes<LPV, PB, true>(pk, f16_to_f32(sc), q, s_cent, k.polar, w);
#pragma unroll
    for (int e = 0; e < 32; e++) r[e] = r[e] - w[e];
    float4 *dst = reinterpret_cast<float4 *>(s_res + (tid / LPV) * RS + 32 * q);
#pragma unroll
    for (int i = 0; i < 8; i++) dst[i] = make_float4(r[4 * i], r[4 * i + 1], r[4 * i + 2], r[4 * i + 3]);
#pragma unroll
    for (int e = 0; e < 32; e++) r[e] = r[e] * r[e];
    const float rs = ordered_sum<LPV>(r, q, -0.0f);
    if (q == 0) {
      polar_scales[v] = sc;
      residual_norms[v] = f32_to_f16(sqrtf(rs));
    }
  }
  __syncthreads();
  // compute_qjl_signs + pack_sign_bits (qjl.rs:305-319, 245-256): bit j = p_j >= 0
  tqm::f32x4 acc[2];
#pragma unroll
  for (int g = 0; g < 2; g++) acc[g] = tqm::f32x4{-0.0f, -0.0f, -0.0f, -0.0f};
  const float *res = s_res + l16 * RS + lg;
#pragma unroll
  for (int i = 0; i < D / 4; i++) {
    const float a = u2f(((rb << (31 - i)) & 0x80000000u) | 0x3f800000u);
#pragma unroll
    for (int g = 0; g < 2; g++)
      acc[g] = __builtin_amdgcn_mfma_f32_16x16x4f32(a, res[16 * g * RS + 4 * i], acc[g], 0, 0, 0);
  }
#pragma unroll
  for (int g = 0; g < 2; g++) {  // lane: key l16 of the group, rows 4 lg .. + 3 of the wave's 16
    uint32_t bits = 0;
#pragma unroll
    for (int i = 0; i < 4; i++) bits |= (acc[g][i] * k.inv_sqrt_d >= 0.0f ? 1u : 0u) << (4 * lg + i);
    bits |= __shfl_xor(bits, 16, 64);
    bits |= __shfl_xor(bits, 32, 64);
    const long long key = key0 + 16 * g + l16;
    if (lg == 0 && key < n) signs[key * (D / 16) + wave] = (uint16_t)bits;
  }
}

// EstimationContext for a batch of queries (qjl.rs:488-492, 561-572):
// ctx[q] = { qt[D] = forward rotation of q (no normalization), rq[D] = R q }.
// A workgroup serves 8 queries x 32 projection rows, lane = (query, row): it
// hashes only its rows' sign bits; each lane sums its row in column order
// from -0.0 (rademacher_vector_product, qjl.rs:196-208).  The workgroups of
// the first row block also rotate their queries (one lane per query).
template <int D>
__global__ __launch_bounds__(kBlock) void qjl_query_kernel(const float *__restrict__ queries, float *__restrict__ ctx,
                                                           long long nq, QjlConsts k) {
  constexpr int RB = 32, QB = kBlock / RB;
  __shared__ uint32_t s_bits[RB * (D / 32)];
  __shared__ __attribute__((aligned(16))) float s_q[QB * D];
  __shared__ __attribute__((aligned(16))) float4 s_sgn[16];
  const int tid = threadIdx.x, qq = tid / RB, jj = tid % RB;
  if (tid < 16) s_sgn[tid] = nibble_signs(tid);
  const int jb = blockIdx.x * RB;
  const long long q0 = (long long)blockIdx.y * QB;
  // one sign per lane, 64 consecutive (row, column) entries per wave and step,
  // gathered into two words by a ballot
  for (int base = (tid >> 6) * 64; base < RB * D; base += kBlock) {
    const int f = base + (tid & 63), j = jb + f / D, col = f % D;
    const uint64_t m = __ballot(sign_negative(sign_base(k.qjl_seed, (uint64_t)j), (uint32_t)col));
    if ((tid & 63) == 0) {
      s_bits[base / 32] = (uint32_t)m;
      s_bits[base / 32 + 1] = (uint32_t)(m >> 32);
    }
  }
  for (int e = tid; e < QB * D; e += kBlock) {
    const long long qi = q0 + e / D;
    s_q[e] = qi < nq ? queries[qi * D + e % D] : 0.0f;
  }
  __syncthreads();
  const long long qi = q0 + qq;
  if (qi >= nq) return;
  const float *qv = s_q + qq * D;
  float s = -0.0f;
#pragma unroll
  for (int w = 0; w < D / 32; w++) {
    const uint32_t bits = s_bits[jj * (D / 32) + w];
#pragma unroll
    for (int nb = 0; nb < 8; nb++) {  // the signs of four columns by one table read
      const float4 sg = s_sgn[(bits >> (4 * nb)) & 15u];
      const float4 v = *reinterpret_cast<const float4 *>(qv + 32 * w + 4 * nb);
      s = __builtin_fmaf(sg.x, v.x, s);
      s = __builtin_fmaf(sg.y, v.y, s);
      s = __builtin_fmaf(sg.z, v.z, s);
      s = __builtin_fmaf(sg.w, v.w, s);
    }
  }
  float *out = ctx + qi * 2 * D;
  out[D + jb + jj] = s * k.inv_sqrt_d;
  if (blockIdx.x == 0) {
    // forward rotation, the query's 32 lanes holding E = D / 32 consecutive
    // elements each: butterfly stages h < E inside a lane, h >= E with the
    // lane jj ^ (h / E) (the lower element takes x + y, the upper x - y, in
    // the stage order of butterfly<D>, so every value is the same)
    constexpr int E = D / 32;
    const float se = k.polar.sign_even, so = -k.polar.sign_even;
    float q[E];
#pragma unroll
    for (int i = 0; i < E; i++) q[i] = qv[E * jj + i] * (((E * jj + i) & 1) ? so : se);
#pragma unroll
    for (int h = 1; h < E; h *= 2)
#pragma unroll
      for (int i = 0; i < E; i += 2 * h)
#pragma unroll
        for (int t = i; t < i + h; t++) {
          const float x = q[t], y = q[t + h];
          q[t] = x + y;
          q[t + h] = x - y;
        }
    auto cross = [&](auto xc) {
      constexpr int X = decltype(xc)::value;
      const bool upper = (jj & X) != 0;
#pragma unroll
      for (int i = 0; i < E; i++) {
        const float o = tqm::lane_xor<X>(q[i]);
        q[i] = upper ? o - q[i] : q[i] + o;
      }
    };
    cross(std::integral_constant<int, 1>{});
    cross(std::integral_constant<int, 2>{});
    cross(std::integral_constant<int, 4>{});
    cross(std::integral_constant<int, 8>{});
    cross(std::integral_constant<int, 16>{});
#pragma unroll
    for (int i = 0; i < E; i++) out[E * jj + i] = q[i] * k.polar.wht_norm;
  }
}

// Scores, 16 queries x 16 keys per wave:
//   est = scale_k * sum_i qt_i c[idx_i] + c_k * sum_j rq_j (2 b_j - 1),
//   c_k = |r_k| * sqrt(pi/2) / sqrt(d)   (qjl.rs:263-265, 512-519, 585-606).
// Both sums run on v_mfma_f32_16x16x32_f16 with every f32 operand as three f16
// parts that hold all of its 24 significant bits (a query's on its row's
// power-of-two scale, the centroids' times 2^8; the signs are exact).  Six part
// products for the first sum (the parts below 2^-33 of it dropped), three for
// the second.  With two parts (22 bits) scores of 32 elements were further from
// the f64 result than f32 sums are: 1.16e-7 against 9.0e-8 (2-norm, 2-bit
// codes); with three 6.3e-8.
//
// Lane (l16, lg) holds elements lg D / 4 .. + D / 4 - 1 of query l16 and of key
// l16, 8 for each of the D / 32 slices, so a row is read in whole runs, its
// largest magnitude needs two lane exchanges and the queries' operands stay in
// registers.  A slice's centroids are byte permutes: 4 codes as the selector
// bytes, tables of the parts' low and high bytes in registers.
// 64 queries x 8,192 keys, d = 128, 3 bits: 18 us with a lane per key adding LDS
// table entries (96 a score), 7.5 us in two parts with the queries staged in LDS
// for four waves, 7.4 in three parts and registers, 6.4 with a wave walking
// several key tiles (below).
constexpr int kCentExp = 8;
// The workgroups of a launch: one per compute unit, whose waves then walk
// several key tiles for one split of their queries, and two, as many as the
// registers hold at d = 128, above 6 tiles a wave (us, one / two: 64 queries x
// 8,192 keys 6.4 / 7.9, x 24,576 10.5 / 11.0, x 49,152 16.2 / 15.7, x 262,144
// 57.8 / 52.7; with a tile per wave 123).
constexpr int kScoreBlocks = 256;
constexpr int kScoreTiles = 6;
struct CentroidParts {
  uint32_t tab[3][2][2];  // [part][low, high byte][entries 0..3, 4..7]
};
template <int PB>
__device__ __forceinline__ uint32_t spread_codes(uint32_t x) {  // 4 codes -> 4 bytes
  constexpr uint32_t M = (1u << PB) - 1u;
  x &= (1u << (4 * PB)) - 1u;
  x = (x | x << (16 - 2 * PB)) & ((M | M << PB) * 0x00010001u);
  return (x | x << (8 - PB)) & (M * 0x01010101u);
}

template <int D, int PB>
__global__ __launch_bounds__(kBlock) void qjl_scores_kernel(const float *__restrict__ ctx, long long nq,
                                                            const uint8_t *__restrict__ polar,
                                                            const uint16_t *__restrict__ polar_scales,
                                                            const uint8_t *__restrict__ signs,
                                                            const uint16_t *__restrict__ residual_norms, long long nk,
                                                            float *__restrict__ scores, QjlConsts k, CentroidParts cent) {
  using namespace tqm;
  constexpr int NS = D / 32, E = D / 4, CBITS = E * PB;  // slices; elements and code bits of a lane
  constexpr int RW = D * PB / 32, NCW = D == 128 ? PB : PB - 1;  // words of a record; that hold a lane's codes
  __shared__ __attribute__((aligned(16))) u32x4 s_sign[256];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l16 = lane & 15, lg = lane >> 4;
  const long long q0 = (long long)blockIdx.y * 16;
  const int nql = (int)min<long long>(16, nq - q0);
  // the wave's key tiles: the lane's quarter of a record's codes and signs
  struct Keys {
    uint32_t raw[NCW], sgn;
    uint16_t scale, norm;
  };
  const int bit0 = CBITS * lg, wi0 = bit0 >> 5, sh0 = bit0 & 31;
  auto load_keys = [&](long long tile) {
    Keys r;
    const long long kc = min(tile * 16 + l16, nk - 1);
    const uint32_t *rec = reinterpret_cast<const uint32_t *>(polar + kc * (D * PB / 8));
#pragma unroll
    for (int i = 0; i < NCW; i++) r.raw[i] = rec[min(wi0 + i, RW - 1)];
    const uint8_t *sg = signs + kc * (D / 8) + lg * (E / 8);
    if constexpr (E == 32) r.sgn = *reinterpret_cast<const uint32_t *>(sg);
    else if constexpr (E == 16) r.sgn = *reinterpret_cast<const uint16_t *>(sg);
    else r.sgn = *sg;
    r.scale = polar_scales[kc];
    r.norm = residual_norms[kc];
    return r;
  };
  const long long tiles = (nk + 15) / 16, step = (long long)gridDim.x * (kBlock / 64);
  long long tile = (long long)blockIdx.x * (kBlock / 64) + wave;
  Keys next = load_keys(min(tile, tiles - 1));
  // the queries' rows qt and rq
  float x[2][E];
  {
    const float *row = ctx + (q0 + min(l16, nql - 1)) * 2 * D + lg * E;
#pragma unroll
    for (int p = 0; p < 2; p++)
#pragma unroll
      for (int e = 0; e < E; e++) x[p][e] = row[p * D + e];
  }
  // +-1 in f16 for the eight sign bits of a byte, LSB first (bit set: +1)
  {
    auto pm1 = [&](int bit) { return ((tid >> bit) & 1) ? 0x3C00u : 0xBC00u; };
    s_sign[tid] = u32x4{pm1(0) | (pm1(1) << 16), pm1(2) | (pm1(3) << 16), pm1(4) | (pm1(5) << 16), pm1(6) | (pm1(7) << 16)};
  }
  uint32_t tab[3][2][PB - 1];
#pragma unroll
  for (int p = 0; p < 3; p++)
#pragma unroll
    for (int h = 0; h < 2; h++)
#pragma unroll
      for (int i = 0; i < PB - 1; i++) tab[p][h][i] = cent.tab[p][h][i];
  float mone = -1.f;
  asm("" : "+v"(mone));
  u32x4 q[2][NS][3];
  int ex[2];  // row l16's exponents
#pragma unroll
  for (int p = 0; p < 2; p++) {
    float m = 0.f;
#pragma unroll
    for (int e = 0; e < E; e++) m = fmaxf(m, fabsf(x[p][e]));
    ex[p] = row_exponent(max_xor32(max_xor16(m)));
#pragma unroll
    for (int s = 0; s < NS; s++)
#pragma unroll
      for (int w = 0; w < 4; w++) {
        uint32_t part[3];
        split3(x[p][8 * s + 2 * w], x[p][8 * s + 2 * w + 1], -ex[p], mone, part);
#pragma unroll
        for (int i = 0; i < 3; i++) q[p][s][i][w] = part[i];
      }
  }
  int e0[4], e1[4];  // the exponents of the rows 4 lg .. + 3 that the lane's sums belong to
#pragma unroll
  for (int i = 0; i < 4; i++) {
    e0[i] = __shfl(ex[0], 4 * lg + i, 64) - kCentExp;
    e1[i] = __shfl(ex[1], 4 * lg + i, 64);
  }
  __syncthreads();
#pragma unroll 1
  for (; tile < tiles; tile += step) {
    const Keys cur = next;
    if (tile + step < tiles) next = load_keys(tile + step);  // in flight during this tile's products
    uint32_t code[NCW];
#pragma unroll
    for (int i = 0; i < NCW; i++)
      code[i] = i + 1 < NCW ? __builtin_amdgcn_alignbit(cur.raw[i + 1], cur.raw[i], sh0) : cur.raw[i] >> sh0;
    const float scale = f16_to_f32(cur.scale);
    const float ck = (f16_to_f32(cur.norm) * 1.2533141f) / k.sqrt_d;
    f32x4 base[3], corr[2];  // products of about the same size together
#pragma unroll
    for (int i = 0; i < 3; i++) base[i] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < 2; i++) corr[i] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < NS; s++) {
      u32x4 c[3];
#pragma unroll
      for (int h = 0; h < 2; h++) {  // 4 codes each
        const int bit = (8 * s + 4 * h) * PB, wi = bit >> 5, sh = bit & 31;
        const uint32_t sel = spread_codes<PB>(sh + 4 * PB > 32 ? __builtin_amdgcn_alignbit(code[wi + 1], code[wi], sh) : code[wi] >> sh);
#pragma unroll
        for (int p = 0; p < 3; p++) {
          const uint32_t lo = __builtin_amdgcn_perm(tab[p][0][PB - 2], tab[p][0][0], sel);
          const uint32_t hi = __builtin_amdgcn_perm(tab[p][1][PB - 2], tab[p][1][0], sel);
          c[p][2 * h] = __builtin_amdgcn_perm(hi, lo, 0x05010400u);
          c[p][2 * h + 1] = __builtin_amdgcn_perm(hi, lo, 0x07030602u);
        }
      }
      const u32x4 sg = s_sign[(cur.sgn >> (8 * s)) & 0xffu];
      const u32x4(&qt)[3] = q[0][s], (&rq)[3] = q[1][s];
      base[2] = mfma(qt[2], c[0], base[2]);
      corr[1] = mfma(rq[2], sg, corr[1]);
      base[1] = mfma(qt[1], c[0], base[1]);
      base[0] = mfma(qt[0], c[0], base[0]);
      base[2] = mfma(qt[0], c[2], base[2]);
      corr[1] = mfma(rq[1], sg, corr[1]);
      base[1] = mfma(qt[0], c[1], base[1]);
      corr[0] = mfma(rq[0], sg, corr[0]);
      base[2] = mfma(qt[1], c[1], base[2]);
    }
    const long long key = tile * 16 + l16;
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const int r = 4 * lg + i;
      const float b = __builtin_amdgcn_ldexpf(base[0][i] + (base[1][i] + base[2][i]), e0[i]);
      const float c = __builtin_amdgcn_ldexpf(corr[0][i] + corr[1][i], e1[i]);
      if (r < nql && key < nk) scores[(q0 + r) * nk + key] = scale * b + ck * c;
    }
  }
}

// The same scores for a few queries over many keys: lane = key, the sums of a
// query over code pairs and sign nibbles in LDS tables, D / 2 + D / 4 entries a
// score added in f32.  A 16-query tile's cost does not fall with its rows, a
// table's does.  By tables / by tiles, us, 262,144 keys at 3 bits: d = 128 one
// query 7.4 / 12.3, two 11.3 / 12.9, three 15.4 / 13.5; d = 64 one 4.2 / 8.7,
// four 8.4 / 10.2, six 11.2 / 10.5; d = 32 one 3.4 / 6.9, six 7.3 / 8.5, eight
// 8.8 / 8.9.  Few keys are latency, which tiles have less of: 8,192 keys, d =
// 128, one query 4.1 / 3.9, two 6.0 / 4.0.  A 3-bit code's pair tables are four
// times as large (4 bits in all, d = 128, one query x 49,152 keys 6.1 / 5.7,
// 262,144 keys 8.5 / 13.1, two queries 13.5 / 13.6).
template <int D, int PB>
constexpr int kTableQueries = (PB == 2 ? 256 : 128) / D;
// ... and the queries of a workgroup (their tables' LDS)
template <int PB>
constexpr int kTableBlockQueries = PB == 2 ? 8 : 2;
// the keys from which one query's table is no slower, and more for each other query
template <int D, int PB>
constexpr int kTableKeys = PB == 2 ? (D == 32 ? 1 : D == 64 ? 8192 : 24576) : (D == 32 ? 24576 : D == 64 ? 49152 : 57344);
template <int D>
constexpr int kTableKeysPerQuery = D == 32 ? 24576 : 32768;

template <int D, int PB>
__global__ __launch_bounds__(kBlock) void qjl_scores_table_kernel(const float *__restrict__ ctx, long long nq,
                                                                  const uint8_t *__restrict__ polar,
                                                                  const uint16_t *__restrict__ polar_scales,
                                                                  const uint32_t *__restrict__ signs,
                                                                  const uint16_t *__restrict__ residual_norms,
                                                                  long long nk, float *__restrict__ scores, QjlConsts k) {
  constexpr int QB = kTableBlockQueries<PB>;
  constexpr int PE = 1 << (2 * PB);         // entries per pair table
  constexpr int BT = (D / 2) * PE;          // pair tables per query
  constexpr int CT = (D / 4) * 16;          // sign-nibble tables per query
  constexpr int SW = D / 32, NW = SW * PB;  // sign and code words of a key
  __shared__ float s_tab[QB * (BT + CT)];
  __shared__ float s_cent[16];
  if (threadIdx.x < 16) s_cent[threadIdx.x] = k.polar.cent[threadIdx.x & ((1 << PB) - 1)];
  __syncthreads();
  const long long q0 = (long long)blockIdx.y * QB;
  const int nql = (int)min<long long>(QB, nq - q0);
  // pair (g, code) -> qt[2g] c[lo] + qt[2g+1] c[hi]; nibble (c, m) -> sum_b rq[4c+b] (m_b ? 1 : -1)
  for (int e = threadIdx.x; e < nql * (BT + CT); e += kBlock) {
    const int ql = e / (BT + CT), r = e % (BT + CT);
    const float *cq = ctx + (q0 + ql) * 2 * D;
    float val;
    if (r < BT) {
      const int g = r / PE, code = r % PE;
      val = cq[2 * g] * s_cent[code & ((1 << PB) - 1)] + cq[2 * g + 1] * s_cent[code >> PB];
    } else {
      const int c = (r - BT) / 16, m = (r - BT) % 16;
      const float *rq = cq + D + 4 * c;
      val = -0.0f;
#pragma unroll
      for (int b = 0; b < 4; b++) val = val + ((m >> b) & 1 ? rq[b] : -rq[b]);
    }
    s_tab[e] = val;
  }
  __syncthreads();
  const long long key = (long long)blockIdx.x * kBlock + threadIdx.x;
  if (key >= nk) return;
  uint32_t pk[NW], sg[SW];
#pragma unroll
  for (int i = 0; i < NW; i++) pk[i] = reinterpret_cast<const uint32_t *>(polar + key * (4 * NW))[i];
#pragma unroll
  for (int i = 0; i < SW; i++) sg[i] = signs[key * SW + i];
  const float scale = f16_to_f32(polar_scales[key]);
  const float ck = (f16_to_f32(residual_norms[key]) * 1.2533141f) / k.sqrt_d;
  for (int ql = 0; ql < nql; ql++) {
    const float *tb = s_tab + ql * (BT + CT);
    float base = 0.0f, corr = 0.0f;
#pragma unroll
    for (int g = 0; g < D / 2; g++) {
      const int bit = 2 * g * PB, wi = bit >> 5, sh = bit & 31;
      uint32_t code = pk[wi] >> sh;
      if (sh + 2 * PB > 32) code |= pk[wi + 1] << (32 - sh);
      base += tb[g * PE + (code & (PE - 1))];
    }
#pragma unroll
    for (int c = 0; c < D / 4; c++) corr += tb[BT + c * 16 + ((sg[c >> 3] >> ((c & 7) * 4)) & 15u)];
    scores[(q0 + ql) * nk + key] = scale * base + ck * corr;
  }
}

// Row softmax: probs = exp(scale * (s - max)) / sum (textbook; the reference
// returns raw scores, attention.rs:344-352).
constexpr int kSoftmaxBlock = 1024;
// One workgroup per row.  KEEP > 0: a row of at most kSoftmaxBlock KEEP columns
// is read once, held in KEEP registers a thread and written once; longer ones
// (KEEP 0) are read twice, their exponentials kept in the output and scaled in
// place.  The order of every sum is the same.  64 x 8,192: 6.5 us in place, 4.8
// us kept; short rows are bound by the code they run through: 1,000 rows x 100
// columns 8.7 us with 16 registers, 5.9 in place, 5.4 with one.
template <int KEEP>
__global__ __launch_bounds__(kSoftmaxBlock) void softmax_rows_kernel(const float *__restrict__ s,
                                                                     float *__restrict__ p, long long cols,
                                                                     float scale) {
  __shared__ float red[2][kSoftmaxBlock / 64];
  const float *row = s + (long long)blockIdx.x * cols;
  float *out = p + (long long)blockIdx.x * cols;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  float v[KEEP ? KEEP : 1];
  float m = -INFINITY;
  if constexpr (KEEP > 0) {
#pragma unroll
    for (int i = 0; i < KEEP; i++) {
      const long long c = threadIdx.x + (long long)i * kSoftmaxBlock;
      v[i] = c < cols ? row[c] : -INFINITY;
    }
#pragma unroll
    for (int i = 0; i < KEEP; i++) m = fmaxf(m, v[i]);
  } else {
    for (long long c = threadIdx.x; c < cols; c += kSoftmaxBlock) m = fmaxf(m, row[c]);
  }
  for (int o = 32; o > 0; o >>= 1) m = fmaxf(m, __shfl_xor(m, o, 64));
  if (lane == 0) red[0][wave] = m;
  __syncthreads();
  m = red[0][0];
  for (int w = 1; w < kSoftmaxBlock / 64; w++) m = fmaxf(m, red[0][w]);
  float sum = 0.0f;
  if constexpr (KEEP > 0) {
#pragma unroll
    for (int i = 0; i < KEEP; i++)
      if (threadIdx.x + i * kSoftmaxBlock < cols) {
        v[i] = expf(scale * (v[i] - m));
        sum += v[i];
      }
  } else {
    for (long long c = threadIdx.x; c < cols; c += kSoftmaxBlock) {
      const float e = expf(scale * (row[c] - m));
      out[c] = e;
      sum += e;
    }
  }
  for (int o = 32; o > 0; o >>= 1) sum += __shfl_xor(sum, o, 64);
  if (lane == 0) red[1][wave] = sum;
  __syncthreads();
  sum = 0.0f;
  for (int w = 0; w < kSoftmaxBlock / 64; w++) sum += red[1][w];
  const float inv = 1.0f / sum;
  if constexpr (KEEP > 0) {
#pragma unroll
    for (int i = 0; i < KEEP; i++) {
      const long long c = threadIdx.x + (long long)i * kSoftmaxBlock;
      if (c < cols) out[c] = v[i] * inv;
    }
  } else {
    for (long long c = threadIdx.x; c < cols; c += kSoftmaxBlock) out[c] = out[c] * inv;
  }
}

// weighted_values (attention.rs:371-408), rotated domain: sum_t w_t scale_t
// c[idx_t,e] over one chunk of values for 16 queries per workgroup; the finish
// kernel adds the chunks and applies the inverse rotation once.
constexpr int kWvChunk = 256;
constexpr int kWvQueries = 16;

// Wave w takes elements 16 w .. + 15 on v_mfma_f32_16x16x4_f32, whose steps
// add four values one after the other as fused multiply-adds in f32: the sums
// of a lane that walks the chunk, for 16 queries x 16 elements at a time.
// The scaled weights and the code words of the chunk are staged in LDS in the
// order the steps take them (value 4 s + g at [g][s]), so one 16-byte read
// feeds four steps.  Bound by the latency of the staging: 128 workgroups of
// 64 queries x 8,192 values, d = 128, 2-bit codes, take 16.7 us with a lane
// per element and 4 queries per workgroup, 9.5 us with each staged value
// loaded under its own bounds check, 6.3 us with all loads in flight at once.
// CHUNK: kWvChunk, or kWvFew for lists of no more values (4 values, d = 32,
// 16 queries: 5.6 us staging 256 places, 4.6 staging 32; a lane per element 4.7;
// with the finish's launch).
constexpr int kWvFew = 32;
template <int D, int PB, int CHUNK>
__global__ __launch_bounds__(4 * D) void qjl_wv_partial_kernel(const uint8_t *__restrict__ polar,
                                                               const uint16_t *__restrict__ polar_scales,
                                                               long long nv, long long nq,
                                                               const float *__restrict__ weights,
                                                               float *__restrict__ partial, int chunk0, int nchunks,
                                                               QjlConsts k) {
  constexpr int RW = D * PB / 32, THREADS = 4 * D, ST = CHUNK / 4;  // words per value, steps
  constexpr int GS = ST + 4;                                           // [g] stride
  __shared__ __attribute__((aligned(16))) uint32_t s_codes[RW][4 * GS];
  __shared__ __attribute__((aligned(16))) float s_w[kWvQueries][4 * GS];
  __shared__ float s_cent[16];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l16 = lane & 15, lg = lane >> 4;
  const int chunk = chunk0 + (int)blockIdx.x;
  const long long t0 = (long long)chunk * CHUNK, q0 = (long long)blockIdx.y * kWvQueries;
  const int cnt = (int)min<long long>(CHUNK, nv - t0);
  if (tid < 16) s_cent[tid] = k.polar.cent[tid & ((1 << PB) - 1)];
  // every load goes out before the first is used; places past the end read
  // the last value or query and are stored as zeros
  constexpr int CW = CHUNK * RW, NC = (CW + THREADS - 1) / THREADS, NWT = CHUNK * kWvQueries / THREADS;
  static_assert(NWT * THREADS == CHUNK * kWvQueries, "whole rounds");
  uint32_t cd[NC];
  float wt[NWT];
  uint16_t sc[NWT];
#pragma unroll
  for (int j = 0; j < NC; j++) {
    const int i = tid + j * THREADS;
    cd[j] = reinterpret_cast<const uint32_t *>(polar + (t0 + min(i / RW, cnt - 1)) * (D * PB / 8))[i % RW];
  }
#pragma unroll
  for (int j = 0; j < NWT; j++) {
    const int i = tid + j * THREADS;
    const long long t = t0 + min(i % CHUNK, cnt - 1);
    wt[j] = weights[min<long long>(q0 + i / CHUNK, nq - 1) * nv + t];
    sc[j] = polar_scales[t];
  }
#pragma unroll
  for (int j = 0; j < NC; j++) {
    const int i = tid + j * THREADS, t = i / RW;
    if (CW % THREADS == 0 || i < CW) s_codes[i % RW][(t & 3) * GS + (t >> 2)] = t < cnt ? cd[j] : 0u;
  }
#pragma unroll
  for (int j = 0; j < NWT; j++) {
    const int i = tid + j * THREADS, t = i % CHUNK, qq = i / CHUNK;
    s_w[qq][(t & 3) * GS + (t >> 2)] = t < cnt && q0 + qq < nq ? wt[j] * f16_to_f32(sc[j]) : 0.f;
  }
  __syncthreads();
  // the wave's 16 elements start at bit 16 PB w of a value's words
  const int bit = (16 * wave + l16) * PB, wi = bit >> 5, sh = bit & 31;
  const uint32_t *lo = s_codes[wi] + lg * GS, *hi = s_codes[min(wi + 1, RW - 1)] + lg * GS;
  const float *wp = s_w[l16] + lg * GS;
  tqm::f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  const int steps = (cnt + 3) / 4;
#pragma unroll 4
  for (int s = 0; s < steps; s += 4) {  // steps past the last add 0 * c
    const float4 a4 = *reinterpret_cast<const float4 *>(wp + s);
    const uint4 l4 = *reinterpret_cast<const uint4 *>(lo + s);
    const float a[4] = {a4.x, a4.y, a4.z, a4.w};
    uint32_t code[4] = {l4.x >> sh, l4.y >> sh, l4.z >> sh, l4.w >> sh};
    if constexpr (PB == 3) {
      const uint4 h4 = *reinterpret_cast<const uint4 *>(hi + s);
      code[0] = __builtin_amdgcn_alignbit(h4.x, l4.x, sh);
      code[1] = __builtin_amdgcn_alignbit(h4.y, l4.y, sh);
      code[2] = __builtin_amdgcn_alignbit(h4.z, l4.z, sh);
      code[3] = __builtin_amdgcn_alignbit(h4.w, l4.w, sh);
    }
#pragma unroll
    for (int u = 0; u < 4; u++)
      acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a[u], s_cent[code[u] & ((1u << PB) - 1u)], acc, 0, 0, 0);
  }
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const long long qi = q0 + 4 * lg + i;
    if (qi < nq) partial[(qi * nchunks + chunk) * D + 16 * wave + l16] = acc[i];
  }
}

// One workgroup of D lanes per query: lane e adds its element over the chunks
// (chunk order, from 0; 16 loads in flight: 8.1 -> 3.6 us for 32 chunks); then 32 lanes of E = D / 32 consecutive elements
// each apply the inverse rotation (butterfly<D>'s stages in its order: h < E
// inside a lane, h >= E with lane ^ (h / E); then the norm and the signs).
template <int D>
__global__ __launch_bounds__(D) void qjl_wv_finish_kernel(const float *__restrict__ partial, int nchunks,
                                                          float *__restrict__ out, long long nq, QjlConsts k) {
  constexpr int E = D / 32;
  __shared__ float s_a[D];
  const long long qi = blockIdx.x;
  const int e = threadIdx.x;
  float a = 0.0f;
  for (int c0 = 0; c0 < nchunks; c0 += 16) {
    float v[16];
#pragma unroll
    for (int i = 0; i < 16; i++) v[i] = c0 + i < nchunks ? partial[(qi * nchunks + c0 + i) * D + e] : 0.f;
#pragma unroll
    for (int i = 0; i < 16; i++)
      if (c0 + i < nchunks) a += v[i];
  }
  s_a[e] = a;
  __syncthreads();
  if (e >= 32) return;
  float q[E];
#pragma unroll
  for (int i = 0; i < E; i++) q[i] = s_a[E * e + i];
#pragma unroll
  for (int h = 1; h < E; h *= 2)
#pragma unroll
    for (int i = 0; i < E; i += 2 * h)
#pragma unroll
      for (int t = i; t < i + h; t++) {
        const float x = q[t], y = q[t + h];
        q[t] = x + y;
        q[t + h] = x - y;
      }
  auto cross = [&](auto xc) {
    constexpr int X = decltype(xc)::value;
    const bool upper = (e & X) != 0;
#pragma unroll
    for (int i = 0; i < E; i++) {
      const float o = tqm::lane_xor<X>(q[i]);
      q[i] = upper ? o - q[i] : q[i] + o;
    }
  };
  cross(std::integral_constant<int, 1>{});
  cross(std::integral_constant<int, 2>{});
  cross(std::integral_constant<int, 4>{});
  cross(std::integral_constant<int, 8>{});
  cross(std::integral_constant<int, 16>{});
  const float se = k.polar.sign_even, so = -k.polar.sign_even;
#pragma unroll
  for (int i = 0; i < E; i++) {
    const int el = E * e + i;
    out[qi * D + el] = (q[i] * k.polar.wht_norm) * ((el & 1) ? so : se);
  }
}

// The d x d sign bits of R once, for kernels that read rather than hash them:
// out[j * D/32 + w] bit b set <=> sign(j, 32 w + b) = -1.
template <int D>
__global__ __launch_bounds__(kBlock) void qjl_sign_matrix_kernel(uint32_t *__restrict__ out, uint64_t seed) {
  const int it = blockIdx.x * kBlock + threadIdx.x;
  if (it >= D * D / 32) return;
  const int j = it / (D / 32), w = it % (D / 32);
  const uint64_t base = sign_base(seed, (uint64_t)j);
  uint32_t bits = 0;
  for (int b = 0; b < 32; b++) bits |= (sign_negative(base, (uint32_t)(32 * w + b)) ? 1u : 0u) << b;
  out[it] = bits;
}

int qjl_consts(int polar_bits, int dim, uint64_t rot_seed, uint64_t qjl_seed, QjlConsts &k) {
  if (dim != 32 && dim != 64 && dim != 128)
    return tqh::fail(TQ_ERR_INVALID_DIMENSION, "QJL kernels take dim 32, 64 or 128 (got %d)", dim);
  if (polar_bits != 2 && polar_bits != 3)
    return tqh::fail(TQ_ERR_UNSUPPORTED_BITS, "QJL total bits must be 3 or 4 (polar bits %d)", polar_bits);
  int rc = tqh::make_codec_consts(polar_bits, dim, rot_seed, k.polar);
  if (rc) return rc;
  k.qjl_seed = qjl_seed;
  volatile float fd = (float)dim;
  volatile float sq = sqrtf(fd);
  k.sqrt_d = sq;
  k.inv_sqrt_d = 1.0f / sq;
  return TQ_OK;
}

// |v| < 2^15 cut to an f16's 11 significant bits (2^-24 for values below 2^-14).
double f16_cut(double v, uint16_t &bits) {
  const double a = std::fabs(v);
  const int e = a < 0x1p-14 ? -14 : std::ilogb(a);
  const double m = std::trunc(std::ldexp(a, 10 - e));  // [0, 2^11)
  const int field = m < 1024.0 ? 0 : e + 15;
  bits = (uint16_t)((v < 0 ? 0x8000 : 0) | (field << 10) | ((int)m & 0x3ff));
  return std::copysign(std::ldexp(m, e - 10), v);
}
CentroidParts centroid_parts(const CodecConsts &polar, int polar_bits) {
  CentroidParts c{};
  for (int i = 0; i < (1 << polar_bits); i++) {
    double v = std::ldexp((double)polar.cent[i], kCentExp);
    for (int p = 0; p < 3; p++) {
      uint16_t h;
      v -= f16_cut(v, h);
      c.tab[p][0][i >> 2] |= (uint32_t)(h & 0xff) << (8 * (i & 3));
      c.tab[p][1][i >> 2] |= (uint32_t)(h >> 8) << (8 * (i & 3));
    }
  }
  return c;
}

template <typename F>
int by_dim(int dim, F &&f) {
  switch (dim) {
    case 32: return f(std::integral_constant<int, 32>{});
    case 64: return f(std::integral_constant<int, 64>{});
    case 128: return f(std::integral_constant<int, 128>{});
  }
  return tqh::fail(TQ_ERR_INVALID_DIMENSION, "unsupported dim %d", dim);
}

template <typename F>
int by_dim_bits(int dim, int pb, F &&f) {
  return by_dim(dim, [&](auto d) {
    if (pb == 2) return f(d, std::integral_constant<int, 2>{});
    return f(d, std::integral_constant<int, 3>{});
  });
}

}  // namespace

extern "C" int tq_qjl_quantize_batch(const float *data, uint8_t *polar_packed, uint16_t *polar_scales,
                                     uint8_t *signs, uint16_t *residual_norms, size_t num_vectors, int total_bits,
                                     int dim, uint64_t rotation_seed, uint64_t qjl_seed, hipStream_t stream) {
  if (total_bits != 3 && total_bits != 4)
    return tqh::fail(TQ_ERR_UNSUPPORTED_BITS, "QJL total bits must be 3 or 4 (got %d)", total_bits);
  QjlConsts k;
  int rc = qjl_consts(total_bits - 1, dim, rotation_seed, qjl_seed, k);
  if (rc) return rc;
  if (num_vectors == 0) return TQ_OK;
  if (!data || !polar_packed || !polar_scales || !signs || !residual_norms)
    return tqh::fail(TQ_ERR_INVALID_ARGUMENT, "null pointer");
  const long long n = (long long)num_vectors;
  return by_dim_bits(dim, total_bits - 1, [&](auto d, auto pb) {
    constexpr int D = decltype(d)::value, PB = decltype(pb)::value;
    // 32 vectors a workgroup of 4 D lanes, fewer than 2^32 lanes a launch
    constexpr long long kMost = 32ll * ((1ll << 31) / (4 * D));
    for (long long v = 0; v < n; v += kMost) {
      const long long m = std::min(n - v, kMost);
      hipLaunchKernelGGL((qjl_quant_kernel<D, PB>), dim3((unsigned)((m + 31) / 32)), dim3(4 * D), 0, stream, data + v * D,
                         polar_packed + v * (D * PB / 8), polar_scales + v,
                         reinterpret_cast<uint16_t *>(signs + v * (D / 8)), residual_norms + v, m, k);
      const int rc2 = tqh::check_launch("qjl_quant_kernel");
      if (rc2) return rc2;
    }
    return (int)TQ_OK;
  });
}

extern "C" int tq_qjl_query_context(const float *queries, float *ctx_out, size_t num_queries, int dim,
                                    uint64_t rotation_seed, uint64_t qjl_seed, hipStream_t stream) {
  QjlConsts k;
  int rc = qjl_consts(2, dim, rotation_seed, qjl_seed, k);
  if (rc) return rc;
  if (num_queries == 0) return TQ_OK;
  if (!queries || !ctx_out) return tqh::fail(TQ_ERR_INVALID_ARGUMENT, "null pointer");
  const long long nq = (long long)num_queries;
  if (nq > 8LL * 65535) return tqh::fail(TQ_ERR_INVALID_ARGUMENT, "too many queries (%lld > %d)", nq, 8 * 65535);
  return by_dim(dim, [&](auto d) {
    constexpr int D = decltype(d)::value;
    hipLaunchKernelGGL((qjl_query_kernel<D>), dim3(D / 32, (unsigned)((nq + 7) / 8)), dim3(kBlock), 0, stream,
                       queries, ctx_out, nq, k);
    return tqh::check_launch("qjl_query_kernel");
  });
}

extern "C" int tq_qjl_scores(const float *ctx, size_t num_queries, const uint8_t *polar_packed,
                             const uint16_t *polar_scales, const uint8_t *signs, const uint16_t *residual_norms,
                             size_t num_keys, int polar_bits, int dim, uint64_t rotation_seed, float *scores,
                             hipStream_t stream) {
  QjlConsts k;
  int rc = qjl_consts(polar_bits, dim, rotation_seed, 0, k);
  if (rc) return rc;
  if (num_queries == 0 || num_keys == 0) return TQ_OK;
  if (!ctx || !polar_packed || !polar_scales || !signs || !residual_norms || !scores)
    return tqh::fail(TQ_ERR_INVALID_ARGUMENT, "null pointer");
  const long long nq = (long long)num_queries, nk = (long long)num_keys;
  return by_dim_bits(dim, polar_bits, [&](auto d, auto pb) {
    constexpr int D = decltype(d)::value, PB = decltype(pb)::value;
    // (a lane a key, and a launch holds fewer than 2^32)
    if (nq <= kTableQueries<D, PB> && nk >= kTableKeys<D, PB> + kTableKeysPerQuery<D> * (nq - 1) &&
        nk <= (1ll << 32) - 2 * kBlock) {
      constexpr int QB = kTableBlockQueries<PB>;
      hipLaunchKernelGGL((qjl_scores_table_kernel<D, PB>),
                         dim3((unsigned)((nk + kBlock - 1) / kBlock), (unsigned)((nq + QB - 1) / QB)), dim3(kBlock), 0,
                         stream, ctx, nq, polar_packed, polar_scales, reinterpret_cast<const uint32_t *>(signs),
                         residual_norms, nk, scores, k);
      return tqh::check_launch("qjl_scores_table_kernel");
    }
    const long long qblocks = (nq + 15) / 16, tiles = (nk + 15) / 16 * qblocks;
    const long long blocks = tiles > (long long)kScoreBlocks * (kBlock / 64) * kScoreTiles ? 2 * kScoreBlocks : kScoreBlocks;
    const long long room = std::max(1ll, blocks / qblocks);
    hipLaunchKernelGGL((qjl_scores_kernel<D, PB>), dim3((unsigned)std::min((nk + 63) / 64, room), (unsigned)qblocks),
                       dim3(kBlock), 0, stream, ctx, nq, polar_packed, polar_scales, signs, residual_norms, nk, scores,
                       k, centroid_parts(k.polar, polar_bits));
    return tqh::check_launch("qjl_scores_kernel");
  });
}

extern "C" int tq_softmax_rows(const float *scores, float *probs, size_t rows, size_t cols, float scale,
                               hipStream_t stream) {
  if (rows == 0 || cols == 0) return TQ_OK;
  if (!scores || !probs) return tqh::fail(TQ_ERR_INVALID_ARGUMENT, "null pointer");
  if (rows > 0x7fffffffu) return tqh::fail(TQ_ERR_INVALID_ARGUMENT, "too many rows");
  const size_t keep = (cols + kSoftmaxBlock - 1) / kSoftmaxBlock;  // columns per thread
  const auto kernel = keep <= 1    ? softmax_rows_kernel<1>
                      : keep <= 4  ? softmax_rows_kernel<4>
                      : keep <= 16 ? softmax_rows_kernel<16>
                                   : softmax_rows_kernel<0>;
  constexpr size_t kMost = (1ull << 31) / kSoftmaxBlock;  // rows: fewer than 2^32 lanes a launch
  for (size_t r = 0; r < rows; r += kMost) {
    hipLaunchKernelGGL(kernel, dim3((unsigned)std::min(rows - r, kMost)), dim3(kSoftmaxBlock), 0, stream,
                       scores + r * cols, probs + r * cols, (long long)cols, scale);
    const int rc = tqh::check_launch("softmax_rows_kernel");
    if (rc) return rc;
  }
  return TQ_OK;
}

extern "C" size_t tq_qjl_weighted_values_workspace_size(size_t num_queries, size_t num_values, int dim) {
  if (dim <= 0) return 0;
  const size_t chunks = (num_values + kWvChunk - 1) / kWvChunk;
  return num_queries * chunks * (size_t)dim * sizeof(float);
}

extern "C" int tq_qjl_weighted_values(const uint8_t *polar_packed, const uint16_t *polar_scales, size_t num_values,
                                      const float *weights, size_t num_queries, int polar_bits, int dim,
                                      uint64_t rotation_seed, float *out, void *workspace, size_t workspace_bytes,
                                      hipStream_t stream) {
  QjlConsts k;
  int rc = qjl_consts(polar_bits, dim, rotation_seed, 0, k);
  if (rc) return rc;
  if (num_queries == 0) return TQ_OK;
  if (!out || (num_values && (!polar_packed || !polar_scales || !weights)))
    return tqh::fail(TQ_ERR_INVALID_ARGUMENT, "null pointer");
  const size_t need = tq_qjl_weighted_values_workspace_size(num_queries, num_values, dim);
  if (need > 0 && (!workspace || workspace_bytes < need))
    return tqh::fail(TQ_ERR_INVALID_ARGUMENT, "workspace too small: %zu < %zu", workspace_bytes, need);
  const long long nv = (long long)num_values, nq = (long long)num_queries;
  const int nchunks = (int)((nv + kWvChunk - 1) / kWvChunk);
  if (nq > 65535) return tqh::fail(TQ_ERR_INVALID_ARGUMENT, "too many queries (%lld > 65535)", nq);
  float *partial = static_cast<float *>(workspace);
  return by_dim_bits(dim, polar_bits, [&](auto d, auto pb) {
    constexpr int D = decltype(d)::value, PB = decltype(pb)::value;
    const auto kernel = nv <= kWvFew ? qjl_wv_partial_kernel<D, PB, kWvFew> : qjl_wv_partial_kernel<D, PB, kWvChunk>;
    constexpr int kMost = (1 << 29) / D;  // chunks: fewer than 2^32 lanes a launch
    for (int c = 0; c < nchunks; c += kMost) {
      hipLaunchKernelGGL(kernel, dim3((unsigned)std::min(nchunks - c, kMost), (unsigned)((nq + kWvQueries - 1) / kWvQueries)),
                         dim3(4 * D), 0, stream, polar_packed, polar_scales, nv, nq, weights, partial, c, nchunks, k);
      int rc2 = tqh::check_launch("qjl_wv_partial_kernel");
      if (rc2) return rc2;
    }
    hipLaunchKernelGGL((qjl_wv_finish_kernel<D>), dim3((unsigned)nq), dim3(D), 0, stream, partial, nchunks, out, nq, k);
    return tqh::check_launch("qjl_wv_finish_kernel");
  });
}

// ---------------------------------------------------------------------------
// TqCache building blocks
// ---------------------------------------------------------------------------

extern "C" int tq_qjl_sign_matrix(uint32_t *bits_out, int dim, uint64_t qjl_seed, hipStream_t stream) {
  if (dim != 32 && dim != 64 && dim != 128 && dim != 256)
    return tqh::fail(TQ_ERR_INVALID_DIMENSION, "sign matrix dim must be 32, 64, 128 or 256 (got %d)", dim);
  if (!bits_out) return tqh::fail(TQ_ERR_INVALID_ARGUMENT, "null pointer");
  const unsigned grid = (unsigned)((dim * dim / 32 + kBlock - 1) / kBlock);
  switch (dim) {
    case 32: hipLaunchKernelGGL((qjl_sign_matrix_kernel<32>), dim3(grid), dim3(kBlock), 0, stream, bits_out, qjl_seed); break;
    case 64: hipLaunchKernelGGL((qjl_sign_matrix_kernel<64>), dim3(grid), dim3(kBlock), 0, stream, bits_out, qjl_seed); break;
    case 128: hipLaunchKernelGGL((qjl_sign_matrix_kernel<128>), dim3(grid), dim3(kBlock), 0, stream, bits_out, qjl_seed); break;
    default: hipLaunchKernelGGL((qjl_sign_matrix_kernel<256>), dim3(grid), dim3(kBlock), 0, stream, bits_out, qjl_seed); break;
  }
  return tqh::check_launch("qjl_sign_matrix_kernel");
}
