// attention_split_kernels.h — gfx950 self-attention of f32 tensors on the 16-bit matrix units, without
// a mask or dropout: the forward, and the fused backward (head_dim 32, up to 32 kAtFusedBlocks rows).
//
// v_mfma_f32_32x32x2_f32 takes 64 cycles for 4096 flops and bounded the f32 kernels
// (attention_kernels.h). Here every operand, the softmax weights and dS included, is split into three
// bf16 terms, each the rounding of what the ones before left, which together hold the 24 significand
// bits of a value of any size from 2^-109 up (below, to a unit of 2^-133). Of the products of terms t
// and u the six with t + u <= 2 are summed, the five small ones before or beside the main one; what is
// left out is below 2^-25 of a product, under the rounding of an f32 product. bf16 products run at 16
// times the rate of f32 ones (10 times measured: dense bf16 MFMAs reach 1.6 PFLOP/s here); sums are f32.
// A workgroup whose results are not all finite (an infinity, or a value that rounds to one in bf16,
// leaves the split as NaN), or that meets a non-zero element of its inputs below 2^-100, does its work
// again in the f32 kernel's body. Such a workgroup takes the time of both.
// (Two f16 terms, scaled into f16's range, took 62 us where three bf16 terms take 84, and lost bits: the
// low ones of a quarter of all values, and of rows far below the size that the scale was taken from,
// with relative errors of 1e-2 at a spread of 1e8.)
//
// Measured (20 calls a graph, f32, f32 kernel -> these; relative 2-norm against float64 of the output
// and of grad_q, grad_k, grad_v):
//   104 slices x 8 heads, 300 x 32: forward 119 -> 84 us, backward 317 -> 228; 3.1e-7 -> 1.7e-7,
//     4.8, 5.5, 5.5e-7 -> 2.3, 2.0, 1.9e-7
//   forward 32 x 8, 300 x 32: 40 -> 29;  2 x 8: 16.9 -> 13.6;  52 x 8, 128 x 32: 14.2 -> 12.6;  2 x 8, 50 x 32: 5.8, 5.8
//   forward 4 x 8, 600 x 32: 30 -> 23;  104 x 4, 300 x 64: 119 -> 75;  8 x 8, 300 x 64: 29 -> 21.6
//   backward 32 x 8, 300 x 32: 83 -> 63;  2 x 8: 78 -> 53;  52 x 8, 128 x 32: 39 -> 35
#pragma once

#include <type_traits>

#include "attention_kernels.h"

namespace msda {

// ---- operands of three bf16 terms --------------------------------------------------------------
constexpr int kAtTerms = 3;

// N f32 values (r, left as what the terms do not hold) as three bf16 terms packed in pairs, largest
// first. Written on the packed words: element by element the compiler converts twice, once to pack
// and once to subtract.
template <int N>
__device__ __forceinline__ void at_split(float (&r)[N], uint32_t (&t)[kAtTerms][N / 2]) {
  typedef __bf16 bf2 __attribute__((ext_vector_type(2)));
  typedef float f2 __attribute__((ext_vector_type(2)));
#pragma unroll
  for (int u = 0; u < kAtTerms; ++u)
#pragma unroll
    for (int i = 0; i < N / 2; ++i) {
      t[u][i] = __builtin_bit_cast(uint32_t, __builtin_convertvector(f2{r[2 * i], r[2 * i + 1]}, bf2));
      if (u + 1 < kAtTerms) {
        r[2 * i] -= __uint_as_float(t[u][i] << 16);
        r[2 * i + 1] -= __uint_as_float(t[u][i] & 0xffff0000u);
      }
    }
}

__device__ __forceinline__ void at_split8(const at_f8& f, at_bf8 (&t)[kAtTerms]) {
  float r[8] = {f[0], f[1], f[2], f[3], f[4], f[5], f[6], f[7]};
  uint32_t w[kAtTerms][4];
  at_split(r, w);
#pragma unroll
  for (int u = 0; u < kAtTerms; ++u) t[u] = __builtin_bit_cast(at_bf8, uint4{w[u][0], w[u][1], w[u][2], w[u][3]});
}

__device__ __forceinline__ void at_split4(const at_f4& f, uint2 (&t)[kAtTerms]) {
  float r[4] = {f[0], f[1], f[2], f[3]};
  uint32_t w[kAtTerms][2];
  at_split(r, w);
#pragma unroll
  for (int u = 0; u < kAtTerms; ++u) t[u] = uint2{w[u][0], w[u][1]};
}

// result registers i0 .. i0 + 7
__device__ __forceinline__ void at_split_regs(const at_f16& v, int i0, at_bf8 (&t)[kAtTerms]) {
  at_split8(at_f8{v[i0], v[i0 + 1], v[i0 + 2], v[i0 + 3], v[i0 + 4], v[i0 + 5], v[i0 + 6], v[i0 + 7]}, t);
}

// Whether a non-zero element is below 2^-100, where the third term leaves bf16's range, by the first terms
// (packed pairs): the least of (16 bits shifted past the sign) - 1, unsigned, so that 0 wraps to the
// largest. One multiply-add and one minimum a pair; on the f32 values, which takes three operations a
// pair, the backward's dQ waves made it 231 us where this way and no check are both 222.
typedef uint16_t at_u2 __attribute__((ext_vector_type(2)));
constexpr int kAtLeastLog2 = 100;
__device__ __forceinline__ void at_least(at_u2& least, uint32_t pair) {
  least = __builtin_elementwise_min(least, __builtin_bit_cast(at_u2, pair) * static_cast<uint16_t>(2) - static_cast<uint16_t>(1));
}
__device__ __forceinline__ void at_least(at_u2& least, const at_bf8& t) {
  const uint4 w = __builtin_bit_cast(uint4, t);
  at_least(least, w.x);
  at_least(least, w.y);
  at_least(least, w.z);
  at_least(least, w.w);
}
__device__ __forceinline__ bool at_too_small(const at_u2& least) { return min(least.x, least.y) < (127 - kAtLeastLog2) * 256; }
constexpr at_u2 kAtNoneSmall = {0xffff, 0xffff};

// channels 16 s + 8 grp .. + 7 of a 16-byte aligned f32 row, s < D / 16
template <int D>
__device__ __forceinline__ void at_row_split(at_bf8 (&t)[D / 16][kAtTerms], const float* row, int grp, at_u2& least) {
#pragma unroll
  for (int s = 0; s < D / 16; ++s) {
    const at_f4 a = *reinterpret_cast<const at_f4*>(row + 16 * s + 8 * grp), b = *reinterpret_cast<const at_f4*>(row + 16 * s + 8 * grp + 4);
    at_split8(at_f8{a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]}, t[s]);
    at_least(least, t[s][0]);
  }
}

__device__ __forceinline__ void at_mfma(at_f16& c, const at_bf8& a, const at_bf8& b) {
  c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

// small += the five small term products, smallest first
__device__ __forceinline__ void at_mfma_small(at_f16& small, const at_bf8 (&a)[kAtTerms], const at_bf8 (&b)[kAtTerms]) {
  at_mfma(small, a[0], b[2]);
  at_mfma(small, a[1], b[1]);
  at_mfma(small, a[2], b[0]);
  at_mfma(small, a[0], b[1]);
  at_mfma(small, a[1], b[0]);
}

// Result-layout products of the 32 rows at row x of the swizzled term tiles X (`stride` elements
// apart) and the lane's register row: the small products of all channels first, then the main ones.
template <int D>
__device__ __forceinline__ at_f16 at_scores_split(const uint16_t* X, int stride, int x, const at_bf8 (&r)[D / 16][kAtTerms], int col, int grp) {
  at_bf8 a[D / 16][kAtTerms];
#pragma unroll
  for (int s = 0; s < D / 16; ++s)
#pragma unroll
    for (int u = 0; u < kAtTerms; ++u)
      a[s][u] = __builtin_bit_cast(at_bf8, *reinterpret_cast<const uint4*>(&X[u * stride + at_swo<D>(x + col, 16 * s + 8 * grp)]));
  at_f16 acc = at_zero16();
#pragma unroll
  for (int s = 0; s < D / 16; ++s) at_mfma_small(acc, a[s], r[s]);
#pragma unroll
  for (int s = 0; s < D / 16; ++s) at_mfma(acc, a[s][0], r[s][0]);
  return acc;
}

// Operand of X^T for MFMA (nd, s) of at_accum_tr: channel 32 nd + l % 32 at the rows of result
// registers 8 s .. 8 s + 7, by transposing reads of the term tiles at row x.
template <int D>
__device__ __forceinline__ void at_operand_tr(at_bf8 (&a)[kAtTerms], const uint16_t* X, int stride, int x, int nd, int s, int lane) {
  const int g = lane >> 4, r = lane & 15, grp = lane >> 5;
  const int c = 32 * nd + 16 * (g & 1) + 4 * (r & 3), ro = x + 16 * s + 4 * grp + (r >> 2);
#pragma unroll
  for (int u = 0; u < kAtTerms; ++u) a[u] = at_bf8_of(at_read_tr(X + u * stride + at_swo<D>(ro, c)), at_read_tr(X + u * stride + at_swo<D>(ro + 8, c)));
}

// Asks the scheduler to follow each of the block's N MFMAs by up to V vector operations: it would
// issue the dependent MFMAs back to back and the vector work after them.
template <int N, int V>
__device__ __forceinline__ void at_interleave() {
#pragma unroll
  for (int i = 0; i < N; ++i) {
    __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
    __builtin_amdgcn_sched_group_barrier(0x2, V, 0);
  }
}

// ---- forward ------------------------------------------------------------------------------------
// An AtChunk (64 f32 rows in registers) as swizzled term tiles [term][64][D] (at_swo); rows past L are 0.
template <int D, int NT>
__device__ __forceinline__ void at_store_split(const AtChunk<float, D, NT>& ch, uint16_t* dst, int r0, int L, at_u2& least) {
#pragma unroll
  for (int u = 0; u < AtChunk<float, D, NT>::NV; ++u) {
    const int idx = threadIdx.x + NT * u, row = idx / (D / 4), c4 = idx - row * (D / 4);
    uint2 t[kAtTerms];
    at_split4(r0 + row < L ? ch.v[u] : at_f4{0.0f, 0.0f, 0.0f, 0.0f}, t);
    at_least(least, t[0].x);
    at_least(least, t[0].y);
#pragma unroll
    for (int q = 0; q < kAtTerms; ++q) *reinterpret_cast<uint2*>(&dst[q * kAtChunk * D + at_swo<D>(row, 4 * c4)]) = t[q];
  }
}

// Key and value term tiles. head_dim 32 has two buffers (three workgroups a CU); two of head_dim 64 would leave one workgroup a CU.
template <int D>
constexpr int at_split_buffers() { return D == 32 ? 2 : 1; }
template <int D>
constexpr int at_split_lds_bytes() { return at_split_buffers<D>() * 2 * kAtTerms * kAtChunk * D * 2; }
static_assert(at_split_lds_bytes<32>() >= at_lds_floats<32>() * 4 && at_split_lds_bytes<64>() >= at_lds_floats<64>() * 4, "the f32 body fits");

// Forward (attn_fwd_kernel's work split and streaming). A workgroup splits each chunk once, at head_dim 32
// into one of two buffers in the shadow of the chunk before's MFMAs. The softmax reference m is moved
// when a chunk's largest weight would leave [2^3, 2^15] (the first chunk) or exceed 2^15.
template <int D, int RB>
__global__ void __launch_bounds__(64 * RB, D == 32 ? 3 : 2) attn_fwd_split_kernel(const AttnParams p) {
  constexpr int NT = 64 * RB, ND = D / 32, TS = kAtChunk * D, NBUF = at_split_buffers<D>();  // TS: elements of a term tile
  extern __shared__ __align__(16) float at_lds[];
  uint16_t* Kt = reinterpret_cast<uint16_t*>(at_lds);  // [buffer][K, V][term][64][D]
  const int L = p.len, nb = (L + 31) / 32, nchunks = (L + kAtChunk - 1) / kAtChunk;
  const AttnWork w(p, (nb + RB - 1) / RB);
  const float* kp = static_cast<const float*>(p.k) + w.sl.base(p, kAtK);
  const float* vp = static_cast<const float*>(p.v) + w.sl.base(p, kAtV);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, grp = lane >> 5, col = lane & 31;
  const int qb = w.rc * RB + wave, qi = qb * 32 + col;
  const bool qv = qi < L;
  using Chunk = AtChunk<float, D, NT>;
  Chunk kc, vc;
  kc.load(kp, p.st[kAtK][3], 0, L);
  vc.load(vp, p.st[kAtV][3], 0, L);
  at_u2 least = kAtNoneSmall;
  at_bf8 qt[D / 16][kAtTerms];
  {
    const float* qp = static_cast<const float*>(p.q) + w.sl.base(p, kAtQ) + at_row_off(min(qi, L - 1), p.st[kAtQ][3]);
    at_row_split<D>(qt, qp, grp, least);
  }
  float m = 0.0f, l = 0.0f;  // reference score; sum of the weights
  at_f16 o[ND], os[ND];      // O^T: main and small products
#pragma unroll
  for (int nd = 0; nd < ND; ++nd) o[nd] = os[nd] = at_zero16();
  auto stage = [&](int j) {
    uint16_t* dst = Kt + (j % NBUF) * 2 * kAtTerms * TS;
    at_store_split<D, NT>(kc, dst, j * kAtChunk, L, least);
    at_store_split<D, NT>(vc, dst + kAtTerms * TS, j * kAtChunk, L, least);
    kc.load(kp, p.st[kAtK][3], (j + 1) * kAtChunk, L);  // past L: row L - 1 again
    vc.load(vp, p.st[kAtV][3], (j + 1) * kAtChunk, L);
  };
  stage(0);
  __syncthreads();
  // One chunk; `last` (a constant): the chunk with the keys past L, which stages nothing.
  auto chunk = [&](auto last, int j) {
    constexpr bool LAST = decltype(last)::value;
    const uint16_t* Kj = Kt + (j % NBUF) * 2 * kAtTerms * TS;
    const uint16_t* Vj = Kj + kAtTerms * TS;
    at_f16 s0 = at_scores_split<D>(Kj, TS, 0, qt, col, grp), s1 = at_scores_split<D>(Kj, TS, 32, qt, col, grp);  // the chunk's two key blocks
    if constexpr (!LAST && NBUF == 2) stage(j + 1);
    float bm = -INFINITY;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      s0[i] = fmaf(s0[i], p.scale2, -m);
      s1[i] = fmaf(s1[i], p.scale2, -m);
      if (LAST) {
        const int key = j * kAtChunk + 8 * (i >> 2) + 4 * grp + (i & 3);
        s0[i] = key < L ? s0[i] : -INFINITY;
        s1[i] = key + 32 < L ? s1[i] : -INFINITY;
      }
      bm = at_max3(bm, s0[i], s1[i]);
    }
    bm = at_max_halves(bm);  // relative to m; finite: every chunk holds a key below L
    if (bm > 15.0f || (l == 0.0f && bm < 3.0f)) {
      bm -= 7.0f;
      const float alpha = l == 0.0f ? 0.0f : at_exp2(-bm);
      m += bm;
      l *= alpha;
      s0 -= bm;
      s1 -= bm;
#pragma unroll
      for (int nd = 0; nd < ND; ++nd) {
        o[nd] *= alpha;
        os[nd] *= alpha;
      }
    }
    float rs = 0.0f;
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        at_f16& sc = h == 0 ? s0 : s1;
#pragma unroll
        for (int i = 8 * s; i < 8 * s + 8; ++i) {
          sc[i] = at_exp2(sc[i]);
          rs += sc[i];
        }
        at_bf8 b[kAtTerms];
        at_split_regs(sc, 8 * s, b);
#pragma unroll
        for (int nd = 0; nd < ND; ++nd) {  // O^T += V^T P^T
          at_bf8 a[kAtTerms];
          at_operand_tr<D>(a, Vj, TS, 32 * h, nd, s, lane);
          at_mfma_small(os[nd], a, b);
          at_mfma(o[nd], a[0], b[0]);
        }
      }
    l += at_sum_halves(rs);
  };
  for (int j = 0; j + 1 < nchunks; ++j) {
    if (qb < nb) chunk(std::false_type{}, j);
    if constexpr (NBUF == 1) {
      __syncthreads();  // every wave is done with chunk j
      stage(j + 1);
    } else if (qb >= nb) {
      stage(j + 1);
    }
    __syncthreads();  // chunk j + 1 is staged, and every wave is done with chunk j
  }
  if (qb < nb) chunk(std::true_type{}, nchunks - 1);
  const float inv = 1.0f / l;
  float z = 0.0f;  // NaN if a result is not finite
#pragma unroll
  for (int nd = 0; nd < ND; ++nd) {
    o[nd] = (o[nd] + os[nd]) * inv;
#pragma unroll
    for (int i = 0; i < 16; ++i) z = fmaf(o[nd][i], 0.0f, z);
  }
  if (__syncthreads_or(at_too_small(least) || (z != z && qv))) {  // and every wave is done with the tiles
    attn_fwd_body<float, D, false, RB, false>(p, w, at_lds);
    return;
  }
  if (qb < nb) {
    float* op = static_cast<float*>(p.out) + w.sl.base(p, kAtO);
#pragma unroll
    for (int nd = 0; nd < ND; ++nd) at_store_block<float>(op + 32 * nd, p.st[kAtO][3], qb * 32, L, o[nd], 1.0f, at_lds + wave * (at_scratch_bytes<float>() / 4), lane);
    if (qv && grp == 0) {
      float* stats = p.stats + (static_cast<int64_t>(w.zh) * L + qi) * 4;
      // The weights sum to l = 2^e f, f in [1, 2): m + e, and log2 f with what m + e rounds off. The
      // backward's s - stats[0] - stats[1] is then rounded at the size of the weight's own log2; with m
      // and log2 l (3 to 24) the rounding of these was most of the gradients' error against float64:
      // 300 x 32 4.3, 4.1, 4.2e-7 (grad_q, grad_k, grad_v) -> 2.3, 2.0, 1.9e-7; 50 x 32 3.0 -> 1.7e-7;
      // 300 x 64 (backward on f32 MFMAs) 5.7, 6.0, 5.8e-7 -> 4.4, 4.7, 4.5e-7.
      const float e = static_cast<float>(static_cast<int>(__float_as_uint(l) >> 23) - 127);
      const float f = __uint_as_float((__float_as_uint(l) & 0x007fffffu) | 0x3f800000u);
      const float me = m + e, t = me - m;
      stats[0] = me;
      stats[1] = log2f(f) + ((m - (me - t)) + (e - t));
    }
  }
}

// ---- fused backward -----------------------------------------------------------------------------
// Fused backward: one workgroup per (slice, head), one phase per 32-row query block. Key waves (one
// per key block, K and V terms in registers) form S, dP, P and dS of their block against the
// phase's query block, write dS as three term tiles [32 keys][32 queries], and accumulate dV and dK.
// The two dQ waves stage the query rows (Q and dO terms, rowsum(dO * O)) one block ahead and form
// 16 channels each of the previous block's dQ^T = K^T dS^T over all key blocks
// (v_mfma_f32_16x16x32_bf16, one key block per product), straight to memory. The dS tiles of one
// block fill 61 KB at 320 rows, as much as the key terms, so there is one set of them: between the
// two barriers of a phase the key waves write their tiles, and dV, dK and the next block's scores
// overlap the dQ waves' products. The query rows have three buffers: the dQ waves write one while
// key waves may still read the two before it.
// A key wave's vector work is asked between its MFMAs where it does not depend on them: the softmax
// weights beside dP's products, the split of the weights beside dK's (left to the compiler each came
// after its MFMAs, and the three waves of a SIMD are in the same stage; also 8 registers spilled instead
// of 15): 104 slices x 8 heads of 300 rows 228 -> 222 us. dV's products moved before the barriers, beside
// the split of dS, took 236 to 243 (24 registers spilled).
constexpr int kAtSchedReads = 0x100;  // __builtin_amdgcn_sched_barrier: only LDS reads may cross
constexpr int kAtSplitRow = 32 * 32;  // elements of one term of a 32-row tile
constexpr int at_fused_split_lds_bytes(int nb) {
  return 3 * (2 * kAtTerms * kAtSplitRow * 2 + 3 * 32 * 4) + 16 + 2 * nb * kAtTerms * kAtSplitRow * 2;
}

__global__ void __launch_bounds__(64 * (kAtFusedBlocks + 2), 3) attn_bwd_fused_split_kernel(const AttnParams p) {
  constexpr int D = 32, TR = kAtSplitRow;
  extern __shared__ __align__(16) float at_lds[];
  const int L = p.len, nb = (L + 31) / 32;
  float* Ms = at_lds;                     // [3][32][2]: m, log2 l (rows past L: +inf)
  float* Ds = Ms + 3 * 64;                // [3][32]: rowsum(dO * O)
  int* bad = reinterpret_cast<int*>(Ds + 3 * 32);  // a result is not finite
  uint16_t* Qt = reinterpret_cast<uint16_t*>(bad + 4);  // [3][term][32][32]
  uint16_t* Gt = Qt + 3 * kAtTerms * TR;
  uint16_t* Kt = Gt + 3 * kAtTerms * TR;  // [term][32 nb][32] (0 past L)
  uint16_t* St = Kt + kAtTerms * nb * TR;  // [key block][term][32][32]
  const int zh = xcd_logical(static_cast<int>(blockIdx.x), static_cast<int>(gridDim.x));  // as the bf16 kernel
  const AttnSlice sl(p, zh);
  const float* kp = static_cast<const float*>(p.k) + sl.base(p, kAtK);
  const int t = threadIdx.x, wave = t >> 6, lane = t & 63, grp = lane >> 5, col = lane & 31;
  if (t == 0) *bad = 0;
  float z = 0.0f;  // NaN if a result of this lane is not finite
  if (wave < nb) {  // key block kb = wave (uniform per wave)
    const int kb = wave, kcl = min(kb * 32 + col, L - 1);
    at_bf8 kt[D / 16][kAtTerms], vt[D / 16][kAtTerms];
    at_u2 least = kAtNoneSmall;
    {
      at_f4 kc[4];  // the block's rows of the key copy: row 8 u + lane / 8, channels 4 (lane % 8) .. + 3
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int row = kb * 32 + 8 * u + (lane >> 3);
        kc[u] = row < L ? *reinterpret_cast<const at_f4*>(kp + at_row_off(row, p.st[kAtK][3]) + 4 * (lane & 7)) : at_f4{0.0f, 0.0f, 0.0f, 0.0f};
      }
      at_row_split<D>(kt, kp + at_row_off(kcl, p.st[kAtK][3]), grp, least);
      at_row_split<D>(vt, static_cast<const float*>(p.v) + sl.base(p, kAtV) + at_row_off(kcl, p.st[kAtV][3]), grp, least);
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        uint2 x[kAtTerms];
        at_split4(kc[u], x);
#pragma unroll
        for (int q = 0; q < kAtTerms; ++q) *reinterpret_cast<uint2*>(&Kt[q * nb * TR + at_swo<D>(kb * 32 + 8 * u + (lane >> 3), 4 * (lane & 7))]) = x[q];
      }
    }
    at_f16 dk = at_zero16(), dv = at_zero16();
    __syncthreads();  // query block 0 staged, key terms written, the flag cleared
    if (at_too_small(least)) *bad = 1;
    for (int j = 0, b = 0; j < nb; ++j, b = b == 2 ? 0 : b + 1) {
      const uint16_t* Qb = Qt + b * kAtTerms * TR;
      const uint16_t* Gb = Gt + b * kAtTerms * TR;
      if (kb == 0 && lane < 32 && j * 32 + lane < L)  // rowsum(dO * O) into the statistics (their entry 2)
        p.stats[(static_cast<int64_t>(zh) * L + j * 32 + lane) * 4 + 2] = Ds[32 * b + lane];
      at_f16 s = at_scores_split<D>(Qb, TR, 0, kt, col, grp);  // S = Q K^T
      __builtin_amdgcn_sched_barrier(kAtSchedReads);
      const at_f16 dp = at_scores_split<D>(Gb, TR, 0, vt, col, grp);  // dP = dO V^T
      at_f16 pw;
#pragma unroll
      for (int c4 = 0; c4 < 4; ++c4) {
        const int ql = 8 * c4 + 4 * grp;
        const at_f4 ms0 = *reinterpret_cast<const at_f4*>(&Ms[64 * b + 2 * ql]), ms1 = *reinterpret_cast<const at_f4*>(&Ms[64 * b + 2 * ql + 4]);
        const float mq[4] = {ms0[0], ms0[2], ms1[0], ms1[2]}, lq[4] = {ms0[1], ms0[3], ms1[1], ms1[3]};
        // a lane past L holds the clamped last key: finite weights, and its rows of the key copy
        // are 0, so it adds nothing to dQ; rows past L have m = +inf: weight 0
#pragma unroll
        for (int jj = 0; jj < 4; ++jj) pw[4 * c4 + jj] = at_exp2(fmaf(s[4 * c4 + jj], p.scale2, -mq[jj]) - lq[jj]);
      }
      at_interleave<12, 5>();
      __builtin_amdgcn_sched_barrier(kAtSchedReads);
#pragma unroll
      for (int c4 = 0; c4 < 4; ++c4) {
        const at_f4 dd = *reinterpret_cast<const at_f4*>(&Ds[32 * b + 8 * c4 + 4 * grp]);
#pragma unroll
        for (int jj = 0; jj < 4; ++jj) s[4 * c4 + jj] = pw[4 * c4 + jj] * (dp[4 * c4 + jj] - dd[jj]);  // dS
      }
      at_bf8 ds[2][kAtTerms];
      at_split_regs(s, 0, ds[0]);
      at_split_regs(s, 8, ds[1]);
      __syncthreads();  // the dQ waves are done with the previous block's tiles
      uint16_t* T = St + kb * kAtTerms * TR;  // row = key (this lane's col), columns = the block's queries
#pragma unroll
      for (int u = 0; u < kAtTerms; ++u)
#pragma unroll
        for (int s2 = 0; s2 < 2; ++s2) {
          const uint4 x = __builtin_bit_cast(uint4, ds[s2][u]);
          *reinterpret_cast<uint2*>(&T[u * TR + at_swo<D>(col, 16 * s2 + 4 * grp)]) = uint2{x.x, x.y};
          *reinterpret_cast<uint2*>(&T[u * TR + at_swo<D>(col, 16 * s2 + 8 + 4 * grp)]) = uint2{x.z, x.w};
        }
      __syncthreads();  // the block's tiles are written
      // dK^T += Q^T dS and dV^T += dO^T P: the block's sums by themselves, then added
      at_bf8 pt[2][kAtTerms];
      {
        at_f16 acc = at_zero16();
        at_bf8 a0[kAtTerms], a1[kAtTerms];
        at_operand_tr<D>(a0, Qb, TR, 0, 0, 0, lane);
        at_operand_tr<D>(a1, Qb, TR, 0, 0, 1, lane);
        at_mfma_small(acc, a0, ds[0]);
        at_mfma_small(acc, a1, ds[1]);
        at_mfma(acc, a0[0], ds[0][0]);
        at_mfma(acc, a1[0], ds[1][0]);
        at_split_regs(pw, 0, pt[0]);
        at_split_regs(pw, 8, pt[1]);
        at_interleave<12, 8>();
        dk += acc;
      }
      __builtin_amdgcn_sched_barrier(kAtSchedReads);
      {
        at_f16 acc = at_zero16();
        at_bf8 a0[kAtTerms], a1[kAtTerms];
        at_operand_tr<D>(a0, Gb, TR, 0, 0, 0, lane);
        at_operand_tr<D>(a1, Gb, TR, 0, 0, 1, lane);
        at_mfma_small(acc, a0, pt[0]);
        at_mfma_small(acc, a1, pt[1]);
        at_mfma(acc, a0[0], pt[0][0]);
        at_mfma(acc, a1[0], pt[1][0]);
        dv += acc;
      }
    }
#pragma unroll
    for (int i = 0; i < 16; ++i) z = fmaf(dk[i], 0.0f, fmaf(dv[i], 0.0f, z));
    if (z != z) *bad = 1;
    __syncthreads();  // the dQ waves are done with the tiles and the key terms
    if (*bad == 0) {
      float* sc = reinterpret_cast<float*>(Kt) + kb * (at_scratch_bytes<float>() / 4);  // output scratch
      if (p.gk != nullptr) at_store_block<float>(static_cast<float*>(p.gk) + sl.base(p, kAtGK), p.st[kAtGK][3], kb * 32, L, dk, p.scale, sc, lane);
      if (p.gv != nullptr) at_store_block<float>(static_cast<float*>(p.gv) + sl.base(p, kAtGV), p.st[kAtGV][3], kb * 32, L, dv, 1.0f, sc, lane);
    }
  } else {
    // The two dQ waves. Staging: thread tq holds row tq / 4 of a block, channels 8 (tq % 4) .. + 7.
    const int tq = t - 64 * nb, ch0 = 16 * (tq >> 6);  // this wave's channels of dQ
    const float* qp = static_cast<const float*>(p.q) + sl.base(p, kAtQ);
    const float* gop = static_cast<const float*>(p.go) + sl.base(p, kAtGO);
    const float* opp = static_cast<const float*>(p.o) + sl.base(p, kAtO);
    const float* stats = p.stats + static_cast<int64_t>(zh) * L * 4;
    const int srow = tq >> 2, sq4 = tq & 3;
    at_f8 qv, gv, ov;
    float2 sq = {0.0f, 0.0f};  // m, log2 l
    at_u2 least = kAtNoneSmall;
    auto ld8 = [](const float* e) {
      const at_f4 a = *reinterpret_cast<const at_f4*>(e), b = *reinterpret_cast<const at_f4*>(e + 4);
      return at_f8{a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]};
    };
    auto prefetch = [&](int r0) {
      const int r = min(r0 + srow, L - 1);
      qv = ld8(qp + at_row_off(r, p.st[kAtQ][3]) + 8 * sq4);
      gv = ld8(gop + at_row_off(r, p.st[kAtGO][3]) + 8 * sq4);
      ov = ld8(opp + at_row_off(r, p.st[kAtO][3]) + 8 * sq4);
      if (sq4 == 0) sq = *reinterpret_cast<const float2*>(&stats[4 * r]);
    };
    auto stage = [&](int r0, int b) {
      const bool in = r0 + srow < L;
      float dd = 0.0f;
#pragma unroll
      for (int e = 0; e < 8; ++e) dd += gv[e] * ov[e];
      const at_f8 zero = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
      at_bf8 qs[kAtTerms], gs[kAtTerms];
      at_split8(in ? qv : zero, qs);
      at_split8(in ? gv : zero, gs);
#pragma unroll
      for (int u = 0; u < kAtTerms; ++u) {
        *reinterpret_cast<uint4*>(&Qt[(b * kAtTerms + u) * TR + at_swo<D>(srow, 8 * sq4)]) = __builtin_bit_cast(uint4, qs[u]);
        *reinterpret_cast<uint4*>(&Gt[(b * kAtTerms + u) * TR + at_swo<D>(srow, 8 * sq4)]) = __builtin_bit_cast(uint4, gs[u]);
      }
      at_least(least, qs[0]);
      at_least(least, gs[0]);
      // the row's four quarters: neighbouring lanes (DPP quad_perm [1, 0, 3, 2], then [2, 3, 0, 1])
      dd += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(dd), 0xB1, 0xF, 0xF, false));
      dd += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(dd), 0x4E, 0xF, 0xF, false));
      if (sq4 == 0) {
        Ms[64 * b + 2 * srow] = in ? sq.x : INFINITY;
        Ms[64 * b + 2 * srow + 1] = in ? sq.y : 0.0f;
        Ds[32 * b + srow] = in ? dd : 0.0f;
      }
    };
    float* gqp = static_cast<float*>(p.gq) + sl.base(p, kAtGQ);
    const bool gq16 = (reinterpret_cast<uintptr_t>(gqp) & 15) == 0 && (p.st[kAtGQ][3] & 3) == 0;
    const int g = lane >> 4, i16 = lane & 15;
    // dQ^T of query block jq, channels ch0 .. + 15: lane l of v_mfma_f32_16x16x32_bf16 supplies row
    // (or column) l % 16 at reduction slots 8 (l / 16) .. + 7, here the keys of a block, each half of
    // them by one transposing read; its results are channels ch0 + 4 (l / 16) .. + 3 of query l % 16
    auto dq = [&](int jq) {
      at_f4 acc[2], small[2];
#pragma unroll
      for (int h = 0; h < 2; ++h) acc[h] = small[h] = at_f4{0.0f, 0.0f, 0.0f, 0.0f};
      const int ro = 8 * g + (i16 >> 2), co = 4 * (i16 & 3);
      for (int kb = 0; kb < nb; ++kb) {
        at_bf8 a[kAtTerms], x[2][kAtTerms];
#pragma unroll
        for (int u = 0; u < kAtTerms; ++u) {
          const uint16_t* K = Kt + (u * nb + kb) * TR;
          const uint16_t* T = St + (kb * kAtTerms + u) * TR;
          a[u] = at_bf8_of(at_read_tr(K + at_swo<D>(ro, ch0 + co)), at_read_tr(K + at_swo<D>(ro + 4, ch0 + co)));
#pragma unroll
          for (int h = 0; h < 2; ++h) x[h][u] = at_bf8_of(at_read_tr(T + at_swo<D>(ro, 16 * h + co)), at_read_tr(T + at_swo<D>(ro + 4, 16 * h + co)));
        }
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          auto mm = [&](at_f4& c, int u, int v) { c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[u], x[h][v], c, 0, 0, 0); };
          mm(small[h], 0, 2);
          mm(small[h], 1, 1);
          mm(small[h], 2, 0);
          mm(small[h], 0, 1);
          mm(small[h], 1, 0);
          mm(acc[h], 0, 0);
        }
      }
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int q = 32 * jq + 16 * h + i16;
        const at_f4 v = (acc[h] + small[h]) * p.scale;
#pragma unroll
        for (int e = 0; e < 4; ++e) z = q < L ? fmaf(v[e], 0.0f, z) : z;
        if (q >= L) continue;
        float* dst = gqp + at_row_off(q, p.st[kAtGQ][3]) + ch0 + 4 * g;
        if (gq16) {
          *reinterpret_cast<at_f4*>(dst) = v;
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e) dst[e] = v[e];
        }
      }
    };
    prefetch(0);
    stage(0, 0);
    if (nb > 1) prefetch(32);
    __syncthreads();  // query block 0 staged, key terms written
    for (int j = 0, b = 1; j < nb; ++j, b = b == 2 ? 0 : b + 1) {
      if (j > 0) dq(j - 1);
      if (j + 1 < nb) {  // read from the second barrier of phase j on
        stage((j + 1) * 32, b);
        if (j + 2 < nb) prefetch((j + 2) * 32);
      }
      __syncthreads();
      __syncthreads();
    }
    dq(nb - 1);
    if (z != z || at_too_small(least)) *bad = 1;
    __syncthreads();
  }
  if (*bad != 0) {  // the same for every thread: read after the last barrier
    __syncthreads();  // every wave has read the flag: the f32 body takes the LDS over
    attn_bwd_fused_f32_body(p, zh, at_lds);
  }
}

}  // namespace msda
