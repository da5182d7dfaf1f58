// tq_qjl_bias.hip -- the TQ cache's logit bias (compute_logit_bias, reference
// src/cache/tq.rs:185-253) on the matrix cores, with the query projection
// R q formed in the launch or given by the caller.
//
// bias[h][i][t] = (sum_j rq[h][i][j] (2 b_tj - 1)) * (|r_t| * sf), query head
// h over KV head h / n_rep.  The n_rep q_len query rows that read one KV head
// are consecutive, so per KV head this is one product of [rows][D] with
// [D][kv_len], whose right operand is +-1.
//
// What bounds it: the output (2 or 4 bytes per row and token against 128
// useful multiply-adds), so the product has to stay below the store rate.
// One workgroup makes 64 rows x 512 tokens (x 128 tokens where the grid would
// be small; one to four positions of given rows are sums of table entries
// instead, both below): the rows are staged once in LDS as two f16 parts (hi =
// x rounded to f16, lo = the rest rounded to f16, 22 to 23 significant bits
// together, on a power-of-two scale per row), each of its 8 waves expands the
// sign bits of its 64 tokens once into registers (f16 +-1) and keeps them for
// all rows.  Both part products are exact in the f32 accumulator.  A lane
// holds 4 tokens that follow each other for each of its rows, so a wave's
// store is 128 bytes (16-bit outputs) per row; rows of a kv_len that is no
// multiple of 4 are stored unaligned (513 x 1537 17.9 us, x 1536 13.3 us, 16
// heads).  512 tokens a workgroup instead of 256 halve the projection's work
// per row: 25.2 -> 16.1 us at 16 x 1024 x 1024.
//
// Mean of 16 heads x 1024 x 1024 and 16 x 513 x 1537 over 8 KV heads, d =
// 128, bf16: 49.2 us with one lane per token adding LDS table entries, plus
// 18.7 us for the projection's own launch, against 18.8 us for both.  Error
// against f64, f32 output: 2.0e-7 before, 1.1e-7 now (rq's own sum included).
#include "tq_common.h"
#include "tq_mfma.h"

#include <cmath>

namespace {

using namespace tqd;
using namespace tqm;

constexpr int kRows = 64, kThreads = 512;
// Given rows in a grid of at most this many workgroups of 512 tokens take 128
// tokens a workgroup instead (16 a wave): a fourth of the operands to expand
// and four times the workgroups (us, 512 / 128 tokens, 16 query heads on 8: 8
// rows x 1,000 tokens, d = 128 4.7 / 3.5, d = 256 7.7 / 4.7; 40 x 1,000 d = 64
// 5.8 / 4.0; at 128 workgroups, 16 x 8,000, d = 64 4.6 / 4.3, at 256, 40 x 8,000,
// 6.7 / 8.3).
constexpr int kFewBlocks = 128;
// And 16 rows a workgroup instead of 64 while there is at most one for every
// compute unit: a row tile a wave instead of four (us, 64 / 16 rows: 64 rows of one KV
// head x 1,000 tokens d = 64 3.75 / 2.94, d = 256 6.76 / 4.66; in 512 workgroups of
// 16 rows, 16 heads x 100 positions on 8 x 1,000 tokens, d = 256 7.8 / 10.2).
constexpr int kFewRowBlocks = 256;

// Where the staged rows come from: rq as given (f32), or R q of bf16, f16 or
// f32 query rows.
enum Source : int { kGiven = 0, kFromBF16 = 1, kFromF16 = 2, kFromF32 = 3 };

struct BiasArgs {
  const void *src;        // rq or q, [num_kv_heads][rows][D]
  const uint32_t *rbits;  // sign bits of R (bit set: -1), for a query source
  float inv;              // fl(1 / fl(sqrt(D)))
  int rows;               // query rows per KV head
  const uint32_t *signs;
  const uint16_t *norms;
  int kv_len;
  long long head_stride;
  float sf;
  void *out;
  int token_blocks, kv_heads, q_heads, block_rows;
};

// Four values as consecutive elements of type OUT.  Rows of kv_len elements
// start anywhere, so the store is of unaligned bytes.
template <int OUT>
__device__ __forceinline__ void store4(char *p, const float *v) {
  if constexpr (OUT == kF32) {
    __builtin_memcpy(p, v, 16);
  } else {
    const uint2 w = OUT == kBF16 ? make_uint2(pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]))
                                 : make_uint2(pack_pair(f32_to_f16(v[0]), f32_to_f16(v[1])),
                                              pack_pair(f32_to_f16(v[2]), f32_to_f16(v[3])));
    __builtin_memcpy(p, &w, 8);
  }
}
template <int OUT>
__device__ __forceinline__ void store1(char *p, float v) {
  if constexpr (OUT == kF32) *reinterpret_cast<float *>(p) = v;
  else *reinterpret_cast<uint16_t *>(p) = OUT == kBF16 ? f32_to_bf16(v) : f32_to_f16(v);
}

template <int D, int SRC, int OUT, int TT>
__global__ __launch_bounds__(kThreads, D == 256 && TT == 4 ? 2 : 4) void qjl_logit_bias_kernel(BiasArgs a) {
  constexpr int NS = D / 32, JH = D / 32, OB = OUT == kF32 ? 4 : 2;
  constexpr int RS = D + 8;  // halves per staged row: 16-byte chunks of 16 rows in different banks
  __shared__ uint2 s_nib[16];
  __shared__ __attribute__((aligned(16))) uint16_t s_hi[kRows * RS], s_lo[kRows * RS];
  __shared__ __attribute__((aligned(16))) int s_exp[kRows];
  __shared__ float s_max[2][kRows];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l16 = lane & 15, lg = lane >> 4;
  const int g = blockIdx.z;
  const int rblk = (int)(blockIdx.x / (unsigned)a.token_blocks), tblk = (int)(blockIdx.x % (unsigned)a.token_blocks);
  const int block = TT == 1 ? a.block_rows : kRows, r0 = rblk * block, nrows = min(block, a.rows - r0);
  const long long row0 = (long long)g * a.rows + r0;

  // the wave's tokens: column l16 of tile T is token t0 + TT l16 + T
  const int t0 = (tblk * (kThreads / 64) + wave) * (16 * TT);
  uint32_t sw[TT][NS];
  float c[TT];
#pragma unroll
  for (int T = 0; T < TT; T++) {
    const long long rec = (long long)g * a.head_stride + min(t0 + TT * l16 + T, a.kv_len - 1);
#pragma unroll
    for (int s = 0; s < NS; s++) sw[T][s] = a.signs[rec * NS + s];
    c[T] = f16_to_f32(a.norms[rec]) * a.sf;
  }
  // +-1 in f16 for the four sign bits of a nibble, LSB first (bit set: +1)
  if (tid < 16) {
    auto pm1 = [&](int bit) { return ((tid >> bit) & 1) ? 0x3C00u : 0xBC00u; };
    s_nib[tid] = make_uint2(pm1(0) | (pm1(1) << 16), pm1(2) | (pm1(3) << 16));
  }

  if constexpr (SRC == kGiven) {
    // wave w stages rows 8 w .. + 7, D / 4 lanes of 4 elements per row; a step
    // past the last row stages nothing (its outputs are not stored)
    constexpr int LPR = D / 4, RPS = 64 / LPR, STEPS = 8 / RPS;
    const int e0 = 4 * (lane % LPR), left = nrows - 8 * wave;
    float x[STEPS][4], m[STEPS];
#pragma unroll
    for (int step = 0; step < STEPS; step++) {  // every load goes out before the first is used
      const int row = 8 * wave + step * RPS + lane / LPR;
#pragma unroll
      for (int i = 0; i < 4; i++) x[step][i] = 0.f;
      if (row < nrows) {
        const float *p = static_cast<const float *>(a.src) + (row0 + row) * D + e0;
#pragma unroll
        for (int i = 0; i < 4; i++) x[step][i] = p[i];
      }
    }
    if (left > 0) {
#pragma unroll
      for (int step = 0; step < STEPS; step++)
        m[step] = fmaxf(fmaxf(fabsf(x[step][0]), fabsf(x[step][1])), fmaxf(fabsf(x[step][2]), fabsf(x[step][3])));
      auto fold = [&](auto op) {  // the steps' lane exchanges side by side
#pragma unroll
        for (int step = 0; step < STEPS; step++) m[step] = op(m[step]);
      };
      fold([](float v) { return fmaxf(v, lane_xor<1>(v)); });
      fold([](float v) { return fmaxf(v, lane_xor<2>(v)); });
      fold([](float v) { return fmaxf(v, lane_xor<4>(v)); });
      fold([](float v) { return fmaxf(v, lane_xor<8>(v)); });
      if constexpr (LPR > 16) fold([](float v) { return max_xor16(v); });
      if constexpr (LPR > 32) fold([](float v) { return max_xor32(v); });
#pragma unroll
      for (int step = 0; step < STEPS; step++) {
        if (step * RPS >= left) break;  // uniform
        const int row = 8 * wave + step * RPS + lane / LPR, e = row_exponent(m[step]);
        uint16_t hi[4], lo[4];
#pragma unroll
        for (int i = 0; i < 4; i++) split2(x[step][i], -e, hi[i], lo[i]);
        *reinterpret_cast<uint2 *>(s_hi + row * RS + e0) = make_uint2(pack_pair(hi[0], hi[1]), pack_pair(hi[2], hi[3]));
        *reinterpret_cast<uint2 *>(s_lo + row * RS + e0) = make_uint2(pack_pair(lo[0], lo[1]), pack_pair(lo[2], lo[3]));
        if (lane % LPR == 0) s_exp[row] = e;
      }
    }
  } else {
    // Waves w and w + 4 project rows 16 w .. + 15, each for half of R's
    // rows j: D[j][row] over 16-row tiles of R as the left operand (+-1,
    // exact) and the query rows as the right one: a bf16 or f16 query as it
    // is, an f32 query cut into three bf16 parts that sum to it exactly, so
    // every product is exact and only the f32 accumulation order differs
    // from the serial sum of precompute_query_projections (qjl.rs:196-208).
    constexpr int PARTS = SRC == kFromF32 ? 3 : 1;
    const int row = 16 * (wave & 3) + l16, jh = wave >> 2;
    const bool live = 16 * (wave & 3) < nrows;  // uniform
    f32x4 rq[JH];
    uint32_t rw[JH][NS];  // R's sign words of row 16 (JH jh + jt) + l16
    u32x4 q[NS][PARTS];
    int qexp = 0;  // an f32 row's exponent: its bf16 parts are cut from q 2^-qexp
    if (live) {
#pragma unroll
      for (int jt = 0; jt < JH; jt++)
#pragma unroll
        for (int s = 0; s < NS; s++) rw[jt][s] = a.rbits[(16 * (JH * jh + jt) + l16) * NS + s];
      float v[SRC == kFromF32 ? NS : 1][8];
      if constexpr (SRC == kFromF32) {
        float m = 0.f;
#pragma unroll
        for (int s = 0; s < NS; s++) {
          const float4 *p = reinterpret_cast<const float4 *>(static_cast<const float *>(a.src) + (row0 + row) * D + 32 * s + 8 * lg);
          const float4 none = make_float4(0.f, 0.f, 0.f, 0.f), v0 = row < nrows ? p[0] : none, v1 = row < nrows ? p[1] : none;
          v[s][0] = v0.x; v[s][1] = v0.y; v[s][2] = v0.z; v[s][3] = v0.w;
          v[s][4] = v1.x; v[s][5] = v1.y; v[s][6] = v1.z; v[s][7] = v1.w;
#pragma unroll
          for (int j = 0; j < 8; j++) m = fmaxf(m, fabsf(v[s][j]));
        }
        qexp = row_exponent(max_xor32(max_xor16(m)));
      }
#pragma unroll
      for (int s = 0; s < NS; s++) {
        const long long xi = (row0 + row) * D + 32 * s + 8 * lg;
        if constexpr (SRC == kFromF32) {
#pragma unroll
          for (int j = 0; j < 8; j++) v[s][j] = __builtin_amdgcn_ldexpf(v[s][j], -qexp);
#pragma unroll
          for (int p = 0; p < 3; p++) {
            uint32_t cut[8];
#pragma unroll
            for (int j = 0; j < 8; j++) {
              cut[j] = f2u(v[s][j]) & 0xffff0000u;  // the leading 8 significand bits
              v[s][j] -= u2f(cut[j]);               // exact: the rest
            }
            q[s][p] = u32x4{__builtin_amdgcn_perm(cut[1], cut[0], 0x07060302u),
                            __builtin_amdgcn_perm(cut[3], cut[2], 0x07060302u),
                            __builtin_amdgcn_perm(cut[5], cut[4], 0x07060302u),
                            __builtin_amdgcn_perm(cut[7], cut[6], 0x07060302u)};
          }
        } else {
          q[s][0] = u32x4{0u, 0u, 0u, 0u};
          if (row < nrows) {
            const uint4 v = *reinterpret_cast<const uint4 *>(static_cast<const uint16_t *>(a.src) + xi);
            q[s][0] = u32x4{v.x, v.y, v.z, v.w};
          }
        }
      }
    }
    __syncthreads();  // the nibble table
    if (live) {
      float m = 0.f;
#pragma unroll
      for (int jt = 0; jt < JH; jt++) {
        rq[jt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int s = 0; s < NS; s++) {
          const uint32_t byte = (rw[jt][s] >> (8 * lg)) & 0xffu;
          const uint2 n0 = s_nib[byte & 15u], n1 = s_nib[byte >> 4];
          // f16 +-1 to bf16 +-1 flips the exponent bits 0x0380
          constexpr uint32_t F = SRC == kFromF16 ? 0u : 0x03800380u;
          const u32x4 am = {n0.x ^ F, n0.y ^ F, n1.x ^ F, n1.y ^ F};
#pragma unroll
          for (int p = 0; p < PARTS; p++)
            rq[jt] = SRC == kFromF16 ? mfma(am, q[s][p], rq[jt]) : mfma_bf16(am, q[s][p], rq[jt]);
        }
#pragma unroll
        for (int i = 0; i < 4; i++) {
          rq[jt][i] = -rq[jt][i] * a.inv;  // R's set bits are -1, the table's +1
          m = fmaxf(m, fabsf(rq[jt][i]));
        }
      }
      m = max_xor32(max_xor16(m));
      if (lg == 0) s_max[jh][row] = m;
    }
    __syncthreads();
    if (live) {
      const int e = row_exponent(fmaxf(s_max[0][row], s_max[1][row]));
#pragma unroll
      for (int jt = 0; jt < JH; jt++) {
        uint16_t hi[4], lo[4];
#pragma unroll
        for (int i = 0; i < 4; i++) split2(rq[jt][i], -e, hi[i], lo[i]);
        const int at = row * RS + 16 * (JH * jh + jt) + 4 * lg;
        *reinterpret_cast<uint2 *>(s_hi + at) = make_uint2(pack_pair(hi[0], hi[1]), pack_pair(hi[2], hi[3]));
        *reinterpret_cast<uint2 *>(s_lo + at) = make_uint2(pack_pair(lo[0], lo[1]), pack_pair(lo[2], lo[3]));
      }
      if (jh == 0 && lg == 0) s_exp[row] = e + qexp;
    }
  }
  __syncthreads();
  if (t0 >= a.kv_len) return;

  // the tokens' signs as the right operand of every slice
  u32x4 b[TT][NS];
#pragma unroll
  for (int T = 0; T < TT; T++)
#pragma unroll
    for (int s = 0; s < NS; s++) {
      const uint32_t byte = (sw[T][s] >> (8 * lg)) & 0xffu;
      const uint2 n0 = s_nib[byte & 15u], n1 = s_nib[byte >> 4];
      b[T][s] = u32x4{n0.x, n0.y, n1.x, n1.y};
    }

  const int t = t0 + TT * l16;
  const long long pitch = (long long)a.kv_len * OB;  // bytes of an output row
  char *base = static_cast<char *>(a.out) + row0 * pitch;
  const long long at = 4 * lg * pitch + (long long)t * OB;  // the lane's first row, first token
#pragma unroll 1
  for (int rt = 0; 16 * rt < nrows; rt++, base += 16 * pitch) {
    f32x4 acc[TT];
#pragma unroll
    for (int T = 0; T < TT; T++) acc[T] = f32x4{0.f, 0.f, 0.f, 0.f};
    const uint16_t *ph = s_hi + (16 * rt + l16) * RS + 8 * lg, *pl = s_lo + (16 * rt + l16) * RS + 8 * lg;
#pragma unroll
    for (int s = 0; s < NS; s++) {
      const u32x4 lo = *reinterpret_cast<const u32x4 *>(pl + 32 * s);
#pragma unroll
      for (int T = 0; T < TT; T++) acc[T] = mfma(lo, b[T][s], acc[T]);
    }
#pragma unroll
    for (int s = 0; s < NS; s++) {
      const u32x4 hi = *reinterpret_cast<const u32x4 *>(ph + 32 * s);
#pragma unroll
      for (int T = 0; T < TT; T++) acc[T] = mfma(hi, b[T][s], acc[T]);
    }
    const int4 e4 = *reinterpret_cast<const int4 *>(s_exp + 16 * rt + 4 * lg);
    const int ex[4] = {e4.x, e4.y, e4.z, e4.w};
    const int left = nrows - 16 * rt - 4 * lg;  // rows of this tile that the lane still has
#pragma unroll
    for (int i = 0; i < 4; i++) {
      float v[TT];
#pragma unroll
      for (int T = 0; T < TT; T++) v[T] = __builtin_amdgcn_ldexpf(acc[T][i], ex[i]) * c[T];
      char *p = base + i * pitch + at;
      if (i < left) {
        if (TT == 4 && t + 4 <= a.kv_len) {
          store4<OUT>(p, v);
        } else {
#pragma unroll
          for (int T = 0; T < TT; T++)
            if (t + T < a.kv_len) store1<OUT>(p + T * OB, v[T]);
        }
      }
    }
  }
}

// One or two positions of given rows: lane = token, a query's sum over sign
// nibbles in LDS tables, D / 4 entries a value added in f32.  The products
// above first split and exchange their rows, a chain that so few rows do not
// repay, and at head_dim 256 a long sequence's grid runs in two rounds (us,
// products / tables, 16 query heads on 8, one position: d = 128, 1,000 tokens
// 3.0 / 2.8, 32,768 tokens 5.4 / 4.6; d = 256 3.8 / 3.5, 11.5 / 7.4; two
// positions d = 256 x 32,768 13.1 / 10.7).  Every query head reads the signs
// again, so more than 2^20 values stay with the products (32 heads, two
// positions x 32,768, d = 128 6.6 / 9.9), unless a KV head has no more than
// kTableRows rows: a product's cost is its tokens', whatever its rows (8 heads on
// 8, three positions x 65,536, d = 64 6.7 / 5.2, d = 128 9.1 / 7.6, d = 256 23.8 /
// 12.9; two x 131,072 10.6 / 6.6, 14.1 / 9.5, 42.8 / 20.1).  At d = 64 and 128 not
// with four query heads a KV head, which read the signs four times (32 heads on
// 8 x 65,536 7.0 / 8.3, 9.5 / 11.9; d = 256 24.6 / 19.8), and at d = 128 with four
// rows from 2^20 tokens on (8 heads, four positions x 32,768 6.0 / 6.4, x 131,072
// 16.0 / 14.8).
template <int D>
constexpr int kTablePositions = D == 256 ? 4 : 2;  // (3 and 4 from 16,384 tokens on: 8 heads x 32,768 13.1 / 9.9)
constexpr long long kTableValues = 1 << 20;
constexpr int kTableRows = 4;
constexpr long long kTableTokens = 1 << 18;  // of all KV heads: 512 workgroups of products
// At d = 256 five waves a SIMD at most: registers for more LDS reads in flight
// (eight waves: 1,000 tokens 4.6 us against 3.5).
template <int D>
__global__ __launch_bounds__(256)
__attribute__((amdgpu_waves_per_eu(1, D == 256 ? 5 : 8))) void qjl_logit_bias_table_kernel(
    const float *__restrict__ rq, int q_len, const uint32_t *__restrict__ signs, const uint16_t *__restrict__ norms,
    int kv_len, long long head_stride, int n_rep, float sf, void *__restrict__ out, int out_dtype) {
  constexpr int CT = (D / 4) * 16;
  __shared__ float s_tab[kTableRows * CT];
  const int h = blockIdx.z;
  for (int e = threadIdx.x; e < q_len * CT; e += 256) {
    const int ql = e / CT, rr = e % CT, c = rr / 16, m = rr % 16;
    const float *rp = rq + (((long long)h * q_len + ql) * D) + 4 * c;
    float val = -0.0f;
#pragma unroll
    for (int b = 0; b < 4; b++) val = val + (((m >> b) & 1) ? rp[b] : -rp[b]);
    s_tab[e] = val;
  }
  __syncthreads();
  const int t = blockIdx.x * 256 + threadIdx.x;
  if (t >= kv_len) return;
  const long long rec = (long long)(h / n_rep) * head_stride + t;
  uint32_t sgn[D / 32];
#pragma unroll
  for (int w = 0; w < D / 32; w++) sgn[w] = signs[rec * (D / 32) + w];
  const float c = f16_to_f32(norms[rec]) * sf;
  for (int ql = 0; ql < q_len; ql++) {
    const float *tb = s_tab + ql * CT;
    float raw = 0.0f;
#pragma unroll
    for (int cc = 0; cc < D / 4; cc++) raw += tb[cc * 16 + ((sgn[cc >> 3] >> ((cc & 7) * 4)) & 15u)];
    const float val = raw * c;
    const long long oi = ((long long)h * q_len + ql) * kv_len + t;
    if (out_dtype == kF32) static_cast<float *>(out)[oi] = val;
    else if (out_dtype == kBF16) static_cast<uint16_t *>(out)[oi] = f32_to_bf16(val);
    else static_cast<uint16_t *>(out)[oi] = f32_to_f16(val);
  }
}

template <int D, int SRC, int OUT, int TT = 4>
int launch_one(BiasArgs &a, hipStream_t st) {
  constexpr int TOKENS = kThreads / 64 * 16 * TT;
  const long long tblocks = ((long long)a.kv_len + TOKENS - 1) / TOKENS, rblocks = ((long long)a.rows + a.block_rows - 1) / a.block_rows;
  if (tblocks * rblocks > 0x7fffffffll)
    return tqh::fail(TQ_ERR_INVALID_ARGUMENT, "too many query rows (%d) for %d tokens", a.rows, a.kv_len);
  a.token_blocks = (int)tblocks;
  hipLaunchKernelGGL((qjl_logit_bias_kernel<D, SRC, OUT, TT>), dim3((unsigned)(tblocks * rblocks), 1, (unsigned)a.kv_heads),
                     dim3(kThreads), 0, st, a);
  return tqh::check_launch("qjl_logit_bias_kernel");
}

// Query sources write their own type; rows that were given any.
template <int D>
int launch_bias(BiasArgs &a, int source, int out_dtype, hipStream_t st) {
  if (source == kFromF32) return launch_one<D, kFromF32, kF32>(a, st);
  if (source == kFromBF16) return launch_one<D, kFromBF16, kBF16>(a, st);
  if (source == kFromF16) return launch_one<D, kFromF16, kF16>(a, st);
  const int n_rep = a.q_heads / a.kv_heads, q_len = a.rows / n_rep;
  const long long tokens = (long long)a.kv_heads * a.kv_len;
  const bool few = q_len <= (a.kv_len >= 16384 ? kTablePositions<D> : 2) && a.rows * tokens <= kTableValues;
  // (grid.z counts query heads here, KV heads in the products)
  const int rows = D == 128 && tokens < 4 * kTableTokens ? 3 : kTableRows;
  if (a.q_heads <= 65535 && (few || (a.rows <= rows && (n_rep <= 2 || D == 256) && tokens >= kTableTokens))) {
    hipLaunchKernelGGL((qjl_logit_bias_table_kernel<D>), dim3((unsigned)((a.kv_len + 255) / 256), 1, (unsigned)a.q_heads),
                       dim3(256), 0, st, static_cast<const float *>(a.src), q_len, a.signs, a.norms, a.kv_len,
                       a.head_stride, n_rep, a.sf, a.out, out_dtype);
    return tqh::check_launch("qjl_logit_bias_table_kernel");
  }
  const long long blocks = (long long)((a.kv_len + kThreads - 1) / kThreads) * ((a.rows + kRows - 1) / kRows) * a.kv_heads;
  if (blocks <= kFewBlocks) {
    if ((long long)((a.kv_len + 127) / 128) * ((a.rows + 15) / 16) * a.kv_heads <= kFewRowBlocks) a.block_rows = 16;
    if (out_dtype == kF32) return launch_one<D, kGiven, kF32, 1>(a, st);
    if (out_dtype == kBF16) return launch_one<D, kGiven, kBF16, 1>(a, st);
    return launch_one<D, kGiven, kF16, 1>(a, st);
  }
  if (out_dtype == kF32) return launch_one<D, kGiven, kF32>(a, st);
  if (out_dtype == kBF16) return launch_one<D, kGiven, kBF16>(a, st);
  return launch_one<D, kGiven, kF16>(a, st);
}

int bias(const void *src, int source, const uint32_t *rbits, int num_q_heads, int q_len, const uint8_t *signs,
         const uint16_t *norms, int num_kv_heads, int kv_len, long long head_stride, int head_dim, void *out,
         int out_dtype, hipStream_t stream) {
  if (head_dim != 64 && head_dim != 128 && head_dim != 256)
    return tqh::fail(TQ_ERR_INVALID_DIMENSION, "cache QJL kernels take head_dim 64, 128 or 256 (got %d)", head_dim);
  if (!tqh::valid_dtype(out_dtype)) return tqh::fail(TQ_ERR_INVALID_ARGUMENT, "unknown dtype %d", out_dtype);
  if (num_kv_heads <= 0 || num_q_heads <= 0 || num_q_heads % num_kv_heads != 0)
    return tqh::fail(TQ_ERR_INVALID_ARGUMENT, "num_q_heads (%d) must be a multiple of num_kv_heads (%d)", num_q_heads,
                     num_kv_heads);
  if (q_len < 0 || kv_len < 0 || head_stride < kv_len) return tqh::fail(TQ_ERR_INVALID_ARGUMENT, "bad shape");
  if (q_len == 0 || kv_len == 0) return TQ_OK;
  if (!src || !signs || !norms || !out) return tqh::fail(TQ_ERR_INVALID_ARGUMENT, "null pointer");
  const long long rows = (long long)(num_q_heads / num_kv_heads) * q_len;
  if (rows > 0x7fffffffll)
    return tqh::fail(TQ_ERR_INVALID_ARGUMENT, "too many query rows (%lld) for %d tokens", rows, kv_len);
  BiasArgs a{};
  a.src = src;
  a.rbits = rbits;
  a.inv = tqh::inv_sqrt_dim(head_dim);
  a.rows = (int)rows;
  a.signs = reinterpret_cast<const uint32_t *>(signs);
  a.norms = norms;
  a.kv_len = kv_len;
  a.head_stride = head_stride;
  a.sf = tq_qjl_bias_scale(head_dim);
  a.out = out;
  a.kv_heads = num_kv_heads;
  a.q_heads = num_q_heads;
  a.block_rows = kRows;
  if (head_dim == 64) return launch_bias<64>(a, source, out_dtype, stream);
  if (head_dim == 128) return launch_bias<128>(a, source, out_dtype, stream);
  return launch_bias<256>(a, source, out_dtype, stream);
}

}  // namespace

extern "C" float tq_qjl_bias_scale(int head_dim) {
  // tq.rs:213-214: f32(sqrt(pi / 2)) / sqrt(head_dim as f32)
  volatile float sp = (float)std::sqrt(3.14159265358979323846 / 2.0);
  volatile float fd = (float)head_dim;
  volatile float sq = sqrtf(fd);
  return sp / sq;
}

extern "C" int tq_qjl_logit_bias(const float *rq, int num_q_heads, int q_len, const uint8_t *signs_cache,
                                 const uint16_t *norms_cache, int num_kv_heads, int kv_len,
                                 long long cache_head_stride, int head_dim, void *out, int out_dtype,
                                 hipStream_t stream) {
  return bias(rq, kGiven, nullptr, num_q_heads, q_len, signs_cache, norms_cache, num_kv_heads, kv_len,
              cache_head_stride, head_dim, out, out_dtype, stream);
}

namespace tqh {

int query_logit_bias(const void *q, int q_dtype, const uint32_t *sign_matrix, int num_q_heads, int q_len,
                     const uint8_t *signs, const uint16_t *norms, int num_kv_heads, int kv_len, long long head_stride,
                     int head_dim, void *out, hipStream_t stream) {
  const int source = q_dtype == TQ_DTYPE_F32 ? kFromF32 : q_dtype == TQ_DTYPE_BF16 ? kFromBF16 : kFromF16;
  return bias(q, source, sign_matrix, num_q_heads, q_len, signs, norms, num_kv_heads, kv_len, head_stride, head_dim,
              out, q_dtype, stream);
}

}  // namespace tqh
