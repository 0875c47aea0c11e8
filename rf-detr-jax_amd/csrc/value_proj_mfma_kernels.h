// value_proj_mfma_kernels.h — gfx950 value projection on the bf16 matrix unit, for K and head_dim
// multiples of 8 and 16-byte aligned tensors (value_proj_kernels.h handles the rest, and f32 calls too
// small to gain).
//
// bf16 inputs enter v_mfma_f32_32x32x16_bf16 as they are (the weight rounded to bf16 first, as
// weight.astype(x.dtype) does); sums are f32. f32 operands are split into three bf16 terms, each the
// rounding of what the ones before left, which together hold the 24 significand bits; the six
// products of terms t and u with t + u <= 2 are summed. What is left out is below 2^-25 of a product,
// under the rounding of an f32 sum. Relative 2-norm against float64 at K = N = 256, 576 x 8 to 6800 x
// 16 rows (v_mfma_f32_32x32x2_f32 in brackets): output 7e-8 (1.1e-7), grad_input 9e-8 (1.5e-7),
// grad_weight 1.1e-7 to 2.5e-7 (1.6e-7 to 3.9e-7). The split turns an infinity (or a value that
// rounds to one in bf16) into NaN, and of values below 2^-109 the third term leaves bf16's range, so a
// wave with a sum that is not finite, or not zero and below 2^-105, computes its block again in plain
// f32, runs of 8 columns and indices at a time: with such a row the 4608-row forward takes 61 us instead
// of 17, grad_weight 45 instead of 19, at 108800 rows 235 (94) and 397 (124), with one in the weights,
// which every row meets, 88 and 1200. (One product at a time took 393 and 540 us, 893 and 3750, 947 and
// 13300.)
//
// Measured (graph replays, 256 -> 16 x 16, us; v_mfma_f32 kernels before -> these):
//   bf16 16 x 6800 rows: forward 207 -> 34, grad_input 221 -> 31, grad_weight and bias 219 -> 44
//        (111 MB each: 21 us at the rate of a device copy)
//   bf16 8 x 576:        17.3 -> 6.4, 17.3 -> 5.6, 19.8 -> 12.4
//   f32 16 x 6800:       161 -> 97, 187 -> 92, 217 -> 145 (six products: 54 us each at the measured
//        1.6 PFLOP/s of dense bf16 MFMAs)
//   f32 16 x 1026:       33 -> 24, 37 -> 22, 59 -> 42;  f32 8 x 576: 13.6 -> 13.5, 14.1 -> 12.0, 20.0 -> 18.4
#pragma once

#include "value_proj_kernels.h"

namespace msda {

typedef __bf16 vp_b2 __attribute__((ext_vector_type(2)));
typedef __bf16 vp_b8 __attribute__((ext_vector_type(8)));
typedef float vp_f2 __attribute__((ext_vector_type(2)));

template <typename VT>
struct VpTerms {
  static constexpr int kTerms = sizeof(VT) == 2 ? 1 : 3;
};

__device__ __forceinline__ uint32_t vp_pk(float a, float b) {  // v_cvt_pk_bf16_f32, nearest even
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(vp_f2{a, b}, vp_b2));
}

// Eight values as bf16 operand chunks: out[t] is term t, summed values first to smallest last.
template <int TERMS>
__device__ __forceinline__ void vp_split8(const float (&f)[8], uint4 (&out)[TERMS]) {
  float r[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) r[i] = f[i];
#pragma unroll
  for (int t = 0; t < TERMS; ++t) {
    uint32_t w[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      w[i] = vp_pk(r[2 * i], r[2 * i + 1]);
      if (t + 1 < TERMS) {
        r[2 * i] -= __uint_as_float(w[i] << 16);
        r[2 * i + 1] -= __uint_as_float(w[i] & 0xffff0000u);
      }
    }
    out[t] = uint4{w[0], w[1], w[2], w[3]};
  }
}

// One 32 x 32 block of sums. The split's five small products have sums of their own, 2^-8 of the
// main ones: added to the main ones at every step they would cost five more roundings at its size.
template <int TERMS>
struct VpAcc {
  vp_f16 main, small;
  __device__ __forceinline__ void clear() {
#pragma unroll
    for (int i = 0; i < 16; ++i) main[i] = small[i] = 0.0f;
  }
  // += A B over 16 reduction indices
  __device__ __forceinline__ void mfma(const uint4 (&a)[TERMS], const uint4 (&b)[TERMS]) {
    auto mm = [&](int i, int j, vp_f16& c) {
      c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(vp_b8, a[i]), __builtin_bit_cast(vp_b8, b[j]), c, 0, 0, 0);
    };
    if constexpr (TERMS == 3) {
      mm(0, 2, small);
      mm(1, 1, small);
      mm(2, 0, small);
      mm(0, 1, small);
      mm(1, 0, small);
    }
    mm(0, 0, main);
  }
  // the same into the other sums: one product, half as long a chain of roundings (TERMS = 1)
  __device__ __forceinline__ void odd(const uint4 (&a)[TERMS], const uint4 (&b)[TERMS]) {
    small = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(vp_b8, a[0]), __builtin_bit_cast(vp_b8, b[0]), small, 0, 0, 0);
  }
  __device__ __forceinline__ float at(int i) const { return main[i] + small[i]; }
};

// Whether a sum of the wave is not finite, or is below 2^-105 and not zero: operands that small have lost
// their low bits (the third term of a value below 2^-109 leaves bf16's range).
constexpr int kVpLeastLog2 = 105;
template <int TERMS, int NB>
__device__ __forceinline__ bool vp_any_lost(const VpAcc<TERMS> (&acc)[NB], bool ignore) {
  float s = 0.0f;
  uint32_t least = 0xffffffffu;  // of (bits shifted past the sign) - 1, unsigned: a zero wraps to the largest
#pragma unroll
  for (int j = 0; j < NB; ++j)
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const float v = acc[j].at(i);
      s = fmaf(v, 0.0f, s);
      least = min(least, (__float_as_uint(v) << 1) - 1u);
    }
  return __any((s != s || least < (static_cast<uint32_t>(127 - kVpLeastLog2) << 24) - 1u) && !ignore) != 0;
}

__device__ __forceinline__ float vp_sum8(const float (&f)[8]) {
  return ((f[0] + f[1]) + (f[2] + f[3])) + ((f[4] + f[5]) + (f[6] + f[7]));
}

// Hardware workgroup h (dispatched to the 8 XCDs in turn) to a logical id such that each XCD runs a
// contiguous range: workgroups that read the same rows share an L2.
__device__ __forceinline__ int vp_xcd_id() {
  const int g = static_cast<int>(gridDim.x), h = static_cast<int>(blockIdx.x), per = g >> 3, rem = g & 7, xcd = h & 7;
  return xcd * per + min(xcd, rem) + (h >> 3);
}

// ---- forward and grad_input -------------------------------------------------------------------
// Out[m][c] = sum_r Act[m][r] Wt[c][r]: X against W (forward), dY against W^T (grad_input).
//
// At many rows the product is bound by memory (bf16, M = 108800, K = N = 256: 111 MB), so a
// workgroup keeps the weights of its CB 32-column blocks in LDS for its whole life and its waves
// walk 32-row tiles without a barrier: the activations go from global memory into the operand
// registers of the MFMA, two batches of PB reduction steps ahead. The product runs transposed (A =
// weights, B = activations), so a lane owns one output row m and, with operand row rho holding
// column vp_col_of(rho), runs of 8 consecutive columns: 16-byte stores, two lanes covering a 32-byte
// head cell at head_dim 16.
// In operand order a load of X takes 32 bytes from each of 32 rows (bf16; 64 bytes in f32, and whole
// runs for dY, whose head cells of consecutive rows are adjacent): the bf16 forward took 55 us that
// way against 33 us of grad_input. kScratch: it loads four rows of 256 bytes at a time instead and
// passes them through 8 KB of LDS per wave (16-byte pieces swizzled by row).
// At few rows it is bound by latency (M = 4608: 0.6 GFLOP): one column block per workgroup (CB = 1)
// makes the most workgroups, each staging least, and PB = 8 has the whole row of K = 256 in flight.
template <int KIND, typename VT, int CB>
struct VpRows {
  static constexpr int kWaves = CB == 1 ? 4 : 8;
  static constexpr int kThreads = 64 * kWaves;
  static constexpr int kTerms = VpTerms<VT>::kTerms;
  static constexpr int kRaw = kTerms == 1 ? 1 : 2;            // 16-byte loads per step and lane
  static constexpr bool kScratch = KIND == kGemmForward && kTerms == 1;
  static constexpr int kPB = CB == 1 && kTerms == 1 ? 8 : 4;                 // reduction steps (of 16) of a batch
  static constexpr int kPieces = 2 * kPB * kRaw;              // 16-byte pieces of a row in a batch
  // reduction steps: whole pairs of batches (zero weights past the end)
  __host__ __device__ static constexpr int steps(int red) { return (red + 32 * kPB - 1) / (32 * kPB) * 2 * kPB; }
  // LDS rows of 2 steps + 1 16-byte chunks: an odd stride puts 16 consecutive rows into 16 bank groups
  static constexpr int64_t lds_bytes(int red) {
    return (int64_t{32} * CB * kTerms * (2 * steps(red) + 1) + (kScratch ? kWaves * 32 * kPieces : 0) + 8 * CB) * 16;
  }
};

// Column (of 32) that operand row rho of a block holds: bits 2 and 3 swapped, so result registers
// 0..7 and 8..15 of lane half h are columns 8 h .. and 16 + 8 h .. .
__device__ __forceinline__ int vp_col_of(int rho) { return (rho & 0x13) | ((rho & 4) << 1) | ((rho & 8) >> 1); }

template <int KIND, typename VT, int CB>
__global__ void __launch_bounds__((VpRows<KIND, VT, CB>::kThreads)) vp_rows_kernel(const ValueProjParams p) {
  using Cfg = VpRows<KIND, VT, CB>;
  constexpr int T = Cfg::kThreads, TERMS = Cfg::kTerms, PB = Cfg::kPB, RAW = Cfg::kRaw, BN = 32 * CB;
  constexpr bool bf = sizeof(VT) == 2;
  extern __shared__ __align__(16) uint4 vp_lds[];
  const int M = p.batch * p.seq, K = p.k, N = p.n;
  const int C = KIND == kGemmForward ? N : K, rc = (KIND == kGemmForward ? K : N) / 8;  // columns, reduction chunks
  const int steps = Cfg::steps(8 * rc), ld = 2 * steps + 1;
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6, half = lane >> 5;
  const int cgroups = (C + BN - 1) / BN, rgroups = static_cast<int>(gridDim.x) / cgroups;
  const int id = vp_xcd_id();
  const int c0 = (id % cgroups) * BN, stride = rgroups * Cfg::kWaves;
  const int tiles = (M + 31) / 32, pairs = steps / (2 * PB);
  const void* act = KIND == kGemmForward ? p.x : p.gvalue;

  struct Raw {
    uint4 v[PB * RAW];
  };
  // The loads of batch b of a tile, clamped into the tensor; past the last tile one address for all lanes.
  auto load = [&](int tile, int b, Raw& r) {
    const bool none = tile >= tiles;
    if constexpr (Cfg::kScratch) {
      constexpr int PC = Cfg::kPieces;
      const int j = none ? 0 : min(b * PC + lane % PC, rc - 1);
#pragma unroll
      for (int i = 0; i < PB; ++i) {
        const int m = none ? 0 : min(tile * 32 + 64 / PC * i + lane / PC, M - 1);
        r.v[i] = *reinterpret_cast<const uint4*>(static_cast<const uint16_t*>(act) + static_cast<uint32_t>(m) * static_cast<uint32_t>(K) + 8 * j);
      }
    } else {
      const int m = none ? 0 : min(tile * 32 + (lane & 31), M - 1);
      const uint32_t row = KIND == kGemmForward ? static_cast<uint32_t>(m) * static_cast<uint32_t>(K) : vp_row_part(p, m);
#pragma unroll
      for (int u = 0; u < PB; ++u) {
        const int j = none ? 0 : min(2 * (b * PB + u) + half, rc - 1);
        const uint32_t at = row + (KIND == kGemmForward ? static_cast<uint32_t>(8 * j) : vp_col_part(p, 8 * j));
        const uint4* src = bf ? reinterpret_cast<const uint4*>(static_cast<const uint16_t*>(act) + at)
                              : reinterpret_cast<const uint4*>(static_cast<const float*>(act) + at);
#pragma unroll
        for (int w = 0; w < RAW; ++w) r.v[u * RAW + w] = src[w];
      }
    }
  };
  int tile = (id / cgroups) * Cfg::kWaves + wave;
  Raw buf0, buf1;
  load(tile, 0, buf0);  // in flight while the weights are staged
  load(tile, 1, buf1);

  // Weights: chunk j (8 reduction indices) of column c, zero outside the matrix.
  {
    constexpr int U = 4;
    const int total = BN * 2 * steps;
    for (int e0 = t; e0 < total; e0 += T * U) {
      float f[U][8];
      int at[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int e = min(e0 + u * T, total - 1);
        // forward: W[c][8 j ..] is contiguous, consecutive threads take consecutive chunks;
        // grad_input: W[8 j + i][c], consecutive threads take consecutive columns
        const int c = KIND == kGemmForward ? e / (2 * steps) : e % BN, j = KIND == kGemmForward ? e - c * 2 * steps : e / BN;
        at[u] = c * ld + j;
        const bool ok = c0 + c < C && j < rc;
        const int cc = min(c0 + c, C - 1), jj = min(j, rc - 1);
        if constexpr (KIND == kGemmForward) {
          const vp_f4* src = reinterpret_cast<const vp_f4*>(p.w + static_cast<uint32_t>(cc) * static_cast<uint32_t>(K) + static_cast<uint32_t>(8 * jj));
          const vp_f4 a = src[0], b = src[1];
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            f[u][i] = ok ? a[i] : 0.0f;
            f[u][4 + i] = ok ? b[i] : 0.0f;
          }
        } else {
#pragma unroll
          for (int i = 0; i < 8; ++i) {
            const float w = p.w[static_cast<uint32_t>(8 * jj + i) * static_cast<uint32_t>(K) + static_cast<uint32_t>(cc)];
            f[u][i] = ok ? w : 0.0f;
          }
        }
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        if (e0 + u * T >= total) break;
        uint4 o[TERMS];
        vp_split8<TERMS>(f[u], o);
#pragma unroll
        for (int s = 0; s < TERMS; ++s) vp_lds[s * BN * ld + at[u]] = o[s];
      }
    }
  }
  vp_f4* const bias = reinterpret_cast<vp_f4*>(vp_lds + TERMS * BN * ld + (Cfg::kScratch ? Cfg::kWaves * 32 * Cfg::kPieces : 0));
  if (KIND == kGemmForward && p.bias != nullptr && t < BN) reinterpret_cast<float*>(bias)[t] = vp_wv<VT>(p.bias[min(c0 + t, C - 1)]);
  __syncthreads();

  const uint4* wrow = vp_lds + vp_col_of(lane & 31) * ld + half;
  uint4* const scratch = vp_lds + TERMS * BN * ld + wave * 32 * Cfg::kPieces;
  VpAcc<TERMS> acc[CB];
  auto step = [&](const Raw& r, int u, int s) {
    uint4 x[TERMS];
    const bool in = 2 * s + half < rc;  // what lies past the reduction's end has zero weights, but may not be finite
    if constexpr (bf) {
      x[0] = uint4{in ? r.v[u].x : 0u, in ? r.v[u].y : 0u, in ? r.v[u].z : 0u, in ? r.v[u].w : 0u};
    } else {
      float f[8];
#pragma unroll
      for (int w = 0; w < 2; ++w) {
        const vp_f4 v = __builtin_bit_cast(vp_f4, r.v[2 * u + w]);
#pragma unroll
        for (int i = 0; i < 4; ++i) f[4 * w + i] = in ? v[i] : 0.0f;
      }
      vp_split8<TERMS>(f, x);
    }
#pragma unroll
    for (int j = 0; j < CB; ++j) {
      uint4 w[TERMS];
#pragma unroll
      for (int q = 0; q < TERMS; ++q) w[q] = wrow[(q * BN + 32 * j) * ld + 2 * s];
      acc[j].mfma(w, x);
    }
    if constexpr (!bf) __builtin_amdgcn_sched_barrier(0);  // else the compiler reads the weights of many steps ahead
  };
  // the products of batch b (the wave's LDS accesses are in order: no barrier around the scratch)
  auto compute = [&](Raw& r, int b) {
    if constexpr (Cfg::kScratch) {
      constexpr int PC = Cfg::kPieces;
#pragma unroll
      for (int i = 0; i < PB; ++i) {
        const int row = 64 / PC * i + lane / PC;
        scratch[row * PC + ((lane % PC) ^ (row & (PC - 1) & 15))] = r.v[i];
      }
#pragma unroll
      for (int u = 0; u < PB; ++u) r.v[u] = scratch[(lane & 31) * PC + ((2 * u + half) ^ (lane & (PC - 1) & 15))];
    }
#pragma unroll
    for (int u = 0; u < PB; ++u) step(r, u, b * PB + u);
  };
  // column (from c0) of register i of block j
  auto col = [&](int j, int i) { return 32 * j + 16 * (i >> 3) + 8 * half + (i & 7); };
  // The tile's sums as plain f32 products, eight reduction indices at a time.
  auto redo = [&](int mc) {
    const uint32_t row = KIND == kGemmForward ? static_cast<uint32_t>(mc) * static_cast<uint32_t>(K) : vp_row_part(p, mc);
#pragma unroll
    for (int j = 0; j < CB; ++j) acc[j].clear();
#pragma unroll 1
    for (int r = 0; r < 8 * rc; r += 8) {
      const vp_f4* src = reinterpret_cast<const vp_f4*>(static_cast<const float*>(act) + row +
                                                        (KIND == kGemmForward ? static_cast<uint32_t>(r) : vp_col_part(p, r)));
      const vp_f4 x[2] = {src[0], src[1]};
#pragma unroll
      for (int j = 0; j < CB; ++j)
#pragma unroll
        for (int g = 0; g < 2; ++g) {
          const uint32_t c = static_cast<uint32_t>(min(c0 + col(j, 8 * g), C - 8));  // a run of 8 columns
#pragma unroll
          for (int i = 0; i < 8; ++i) {
            // forward: column c + i at the eight indices; grad_input: the eight columns at index r + i
            const uint32_t at = KIND == kGemmForward ? (c + static_cast<uint32_t>(i)) * static_cast<uint32_t>(K) + static_cast<uint32_t>(r)
                                                     : static_cast<uint32_t>(r + i) * static_cast<uint32_t>(K) + c;
            const vp_f4* w = reinterpret_cast<const vp_f4*>(p.w + at);
            const vp_f4 lo = w[0], hi = w[1];
#pragma unroll
            for (int q = 0; q < 8; ++q) {
              const float wq = q < 4 ? lo[q & 3] : hi[q & 3];
              if (KIND == kGemmForward) acc[j].main[8 * g + i] = fmaf(x[q >> 2][q & 3], wq, acc[j].main[8 * g + i]);
              else acc[j].main[8 * g + q] = fmaf(x[i >> 2][i & 3], wq, acc[j].main[8 * g + q]);
            }
          }
        }
    }
  };
  auto finish = [&](int tl, bool padded) {
    asm volatile("" ::: "memory");  // keeps the bias reads here: hoisted out of the loop they take 16 CB registers
    const int m = tl * 32 + (lane & 31);
    const int mc = min(m, M - 1);
    if constexpr (!bf) {
      if (vp_any_lost(acc, padded || m >= M)) redo(mc);
    }
    const uint32_t row = KIND == kGemmForward ? vp_row_part(p, mc) : static_cast<uint32_t>(mc) * static_cast<uint32_t>(K);
#pragma unroll
    for (int j = 0; j < CB; ++j)
#pragma unroll
      for (int g = 0; g < 2; ++g) {
        const int c = c0 + col(j, 8 * g);  // C is a multiple of 8: the run is inside or outside as a whole
        if (m >= M || c >= C) continue;
        float y[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) y[i] = acc[j].at(8 * g + i);
        if (KIND == kGemmForward && p.bias != nullptr) {
          const vp_f4 lo = bias[8 * j + 4 * g + 2 * half], hi = bias[8 * j + 4 * g + 2 * half + 1];
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            y[i] += lo[i];
            y[4 + i] += hi[i];
          }
        }
        if (padded) {  // where(mask, 0, value) (ops.py:377-378), and its gradient
#pragma unroll
          for (int i = 0; i < 8; ++i) y[i] = 0.0f;
        }
        const uint32_t at = row + (KIND == kGemmForward ? vp_col_part(p, c) : static_cast<uint32_t>(c));
        void* dst = KIND == kGemmForward ? p.value : p.gx;
        if constexpr (bf) {
          *reinterpret_cast<uint4*>(static_cast<uint16_t*>(dst) + at) = uint4{vp_pk(y[0], y[1]), vp_pk(y[2], y[3]), vp_pk(y[4], y[5]), vp_pk(y[6], y[7])};
        } else {
          vp_f4* d = reinterpret_cast<vp_f4*>(static_cast<float*>(dst) + at);
          d[0] = vp_f4{y[0], y[1], y[2], y[3]};
          d[1] = vp_f4{y[4], y[5], y[6], y[7]};
        }
      }
  };
  for (; tile < tiles; tile += stride) {
    const bool padded = p.mask != nullptr && p.mask[min(tile * 32 + (lane & 31), M - 1)] != 0;
#pragma unroll
    for (int j = 0; j < CB; ++j) acc[j].clear();
    for (int q = 0; q < pairs; ++q) {
      const bool last = q + 1 == pairs;
      const int nt = last ? tile + stride : tile, nb = last ? 0 : 2 * q + 2;
      compute(buf0, 2 * q);
      load(nt, nb, buf0);
      compute(buf1, 2 * q + 1);
      load(nt, nb + 1, buf1);
    }
    finish(tile, padded);
  }
}

// ---- grad_weight and grad_bias ----------------------------------------------------------------
// dW[n][k] = sum_m dY[m][n] X[m][k] over one slice of the rows per workgroup, TILE x TILE outputs.
// Both operands are stored along n and k, the product reduces over m: a thread loads 8 rows of EC
// consecutive columns (16-byte loads), forms the 8-row operand chunks in registers (bf16: a byte
// permute per two values; f32: the conversion of two rows to bf16 packs them) and writes them to
// LDS as 16-byte chunks. Column c is LDS row (c % EC) * GS + c / EC of ST chunks (ST odd, GS = 16 /
// EC modulo 16), so a wave's chunk writes and its reads of 32 consecutive columns both spread over
// all bank groups. The next step's loads are in flight during a step's products.
// TILE 128 (bf16, many rows): two reads of X and dY through L2 instead of four, 8 waves; TILE 64
// otherwise, for more workgroups (f32: three terms of a 128-row tile would not fit the LDS).
template <typename VT, int TILE>
struct VpGw {
  static constexpr int kTerms = VpTerms<VT>::kTerms;
  static constexpr int kEC = kTerms == 1 ? 8 : 4;       // columns per 16-byte load
  static constexpr int kMS = kTerms == 1 ? 128 : 64;    // rows per step
  static constexpr int kWaves = TILE == 128 ? 8 : 4;
  static constexpr int kThreads = 64 * kWaves;
  static constexpr int kGroups = TILE / kEC;            // column groups of a tile
  static constexpr int kGS = kGroups + 16 / kEC;
  static constexpr int kST = kMS / 8 + 1;
  static constexpr int kOp = kEC * kGS * kST;           // chunks of one operand term
  static constexpr int kWC = TILE / 32 / 2;             // 32-column blocks of a wave
  static constexpr int kLdsBytes = 2 * kTerms * kOp * 16;
  static_assert(2 * (kMS / 8) * kGroups == kThreads, "one 8-row block of one operand per thread");
  static_assert(kWaves * kWC * 32 * 32 == TILE * TILE, "the waves cover the tile");
};

template <typename VT, int TILE, bool MASK>
__global__ void __launch_bounds__((VpGw<VT, TILE>::kThreads)) vp_gw_kernel(const ValueProjParams p) {
  using Cfg = VpGw<VT, TILE>;
  constexpr int TERMS = Cfg::kTerms, EC = Cfg::kEC, MS = Cfg::kMS, T = Cfg::kThreads, ST = Cfg::kST, GS = Cfg::kGS, WC = Cfg::kWC, G = Cfg::kGroups;
  constexpr bool bf = sizeof(VT) == 2;
  extern __shared__ __align__(16) uint4 vp_lds[];
  const int M = p.batch * p.seq, K = p.k, N = p.n;
  const int tk = (K + TILE - 1) / TILE, tiles = (N + TILE - 1) / TILE * tk;
  const int id = vp_xcd_id();
  const int split = id / tiles, tile = id - split * tiles;  // the tiles of a slice of rows share an L2
  const int n0 = tile / tk * TILE, k0 = tile % tk * TILE;
  const int per = ((M + p.splits - 1) / p.splits + 7) / 8 * 8;
  const int m_lo = min(M, split * per), m_hi = min(M, m_lo + per);
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6, half = lane >> 5;
  const bool is_x = t >= T / 2;
  // Chunk mb holds rows mb + (MS / 8) i of a step, i < 8, of X and dY alike, so that load i of
  // consecutive mb reads consecutive rows: whole runs of dY's head cells at head_dim 16, with the CL
  // column groups of a cell side by side.
  constexpr int CL = 16 / EC, MB = MS / 8;
  const int tt = t % (T / 2);
  const int cg = is_x ? tt % G : tt % CL + tt / (CL * MB) * CL, mb = is_x ? tt / G : tt / CL % MB;
  // the thread's columns (N and K are multiples of 8: inside or outside as a whole)
  const int col0 = (is_x ? k0 : n0) + EC * cg, ncol = is_x ? K : N;
  const bool col_ok = col0 < ncol;
  const uint32_t cpart = is_x ? static_cast<uint32_t>(min(col0, ncol - EC)) : vp_col_part(p, min(col0, ncol - EC));
  const void* src = is_x ? p.x : p.gvalue;
  struct Raw {
    uint4 v[8];
    uint8_t pad[8];
  };
  auto row_at = [&](int m) { return is_x ? static_cast<uint32_t>(m) * static_cast<uint32_t>(K) : vp_row_part(p, m); };
  // past the slice one address for all lanes
  auto load = [&](int ms, Raw& r) {
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const uint32_t at = ms < m_hi ? row_at(min(ms + mb + MB * i, M - 1)) + cpart : 0u;
      if (MASK) r.pad[i] = p.mask[min(ms + mb + MB * i, M - 1)];
      r.v[i] = bf ? *reinterpret_cast<const uint4*>(static_cast<const uint16_t*>(src) + at)
                  : *reinterpret_cast<const uint4*>(static_cast<const float*>(src) + at);
    }
  };
  float bsum[EC];
#pragma unroll
  for (int i = 0; i < EC; ++i) bsum[i] = 0.0f;
  const bool bias_rows = k0 == 0 && !is_x;
  uint4* const op = vp_lds + (is_x ? TERMS * Cfg::kOp : 0);
  // the loaded block as operand chunks; rows past the slice are zero, padded rows are zero in dY
  auto store = [&](int ms, Raw& r) {
    const bool whole = ms + MS <= m_hi;
    if (!whole || !col_ok || (MASK && !is_x)) {
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const int m = ms + mb + MB * i;
        const bool ok = m < m_hi && col_ok && (!MASK || is_x || r.pad[i] == 0);
        r.v[i] = uint4{ok ? r.v[i].x : 0u, ok ? r.v[i].y : 0u, ok ? r.v[i].z : 0u, ok ? r.v[i].w : 0u};
      }
    }
    if constexpr (bf) {
#pragma unroll
      for (int c2 = 0; c2 < 4; ++c2) {
        uint32_t w[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) w[i] = reinterpret_cast<const uint32_t*>(&r.v[i])[c2];
        // columns 2 c2 (low halves) and 2 c2 + 1 (high halves) of the 8 rows
        op[((2 * c2) * GS + cg) * ST + mb] = uint4{__builtin_amdgcn_perm(w[1], w[0], 0x05040100u), __builtin_amdgcn_perm(w[3], w[2], 0x05040100u),
                                                   __builtin_amdgcn_perm(w[5], w[4], 0x05040100u), __builtin_amdgcn_perm(w[7], w[6], 0x05040100u)};
        op[((2 * c2 + 1) * GS + cg) * ST + mb] = uint4{__builtin_amdgcn_perm(w[1], w[0], 0x07060302u), __builtin_amdgcn_perm(w[3], w[2], 0x07060302u),
                                                       __builtin_amdgcn_perm(w[5], w[4], 0x07060302u), __builtin_amdgcn_perm(w[7], w[6], 0x07060302u)};
        if (bias_rows) {
          float lo[8], hi[8];
#pragma unroll
          for (int i = 0; i < 8; ++i) {
            lo[i] = __uint_as_float(w[i] << 16);
            hi[i] = __uint_as_float(w[i] & 0xffff0000u);
          }
          bsum[2 * c2] += vp_sum8(lo);
          bsum[2 * c2 + 1] += vp_sum8(hi);
        }
      }
    } else {
#pragma unroll
      for (int c = 0; c < EC; ++c) {
        float f[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) f[i] = __uint_as_float(reinterpret_cast<const uint32_t*>(&r.v[i])[c]);
        if (bias_rows) bsum[c] += vp_sum8(f);
        uint4 o[TERMS];
        vp_split8<TERMS>(f, o);
#pragma unroll
        for (int q = 0; q < TERMS; ++q) op[q * Cfg::kOp + (c * GS + cg) * ST + mb] = o[q];
      }
    }
  };
  // a wave's blocks: rows n of block wave / 2, WC column blocks from WC (wave % 2)
  const int wn = 32 * (wave >> 1), wk = 32 * WC * (wave & 1);
  auto lds_row = [&](int c) { return ((c % EC) * GS + c / EC) * ST; };
  const uint4* arow = vp_lds + lds_row(wn + (lane & 31)) + half;
  const uint4* brow[WC];
#pragma unroll
  for (int j = 0; j < WC; ++j) brow[j] = vp_lds + TERMS * Cfg::kOp + lds_row(wk + 32 * j + (lane & 31)) + half;
  VpAcc<TERMS> acc[WC];
#pragma unroll
  for (int j = 0; j < WC; ++j) acc[j].clear();
  Raw buf0, buf1;
  load(m_lo, buf0);
  load(m_lo + MS, buf1);
  auto turn = [&](int ms, Raw& r) {
    store(ms, r);
    __syncthreads();
    load(ms + 2 * MS, r);
#pragma unroll
    for (int s = 0; s < MS / 16; ++s) {
      uint4 a[TERMS];
#pragma unroll
      for (int q = 0; q < TERMS; ++q) a[q] = arow[q * Cfg::kOp + 2 * s];
#pragma unroll
      for (int j = 0; j < WC; ++j) {
        uint4 b[TERMS];
#pragma unroll
        for (int q = 0; q < TERMS; ++q) b[q] = brow[j][q * Cfg::kOp + 2 * s];
        if (TERMS == 1 && s % 2 != 0) acc[j].odd(a, b);
        else acc[j].mfma(a, b);
      }
    }
    __syncthreads();
  };
  for (int ms = m_lo; ms < m_hi; ms += 2 * MS) {
    turn(ms, buf0);
    turn(ms + MS, buf1);  // past the slice's end: zeros
  }
  if constexpr (!bf) {
    if (vp_any_lost(acc, false)) {  // the sums again as plain f32 products
      uint32_t n[4], k[WC];  // the lane's runs of 4 rows n, its columns
#pragma unroll
      for (int g = 0; g < 4; ++g) n[g] = vp_col_part(p, min(n0 + wn + 8 * g + 4 * half, N - 4));
#pragma unroll
      for (int j = 0; j < WC; ++j) {
        k[j] = static_cast<uint32_t>(min(k0 + wk + 32 * j + (lane & 31), K - 1));
        acc[j].clear();
      }
#pragma unroll 4
      for (int m = m_lo; m < m_hi; ++m) {
        const float* y = static_cast<const float*>(p.gvalue) + vp_row_part(p, m);
        const float* x = static_cast<const float*>(p.x) + static_cast<uint32_t>(m) * static_cast<uint32_t>(K);
        const bool off = MASK && p.mask[m] != 0;
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const vp_f4 v = *reinterpret_cast<const vp_f4*>(y + n[g]);
#pragma unroll
          for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int j = 0; j < WC; ++j) acc[j].main[4 * g + i] = fmaf(off ? 0.0f : v[i], x[k[j]], acc[j].main[4 * g + i]);
        }
      }
    }
  }
#pragma unroll
  for (int j = 0; j < WC; ++j) {
    const int k = k0 + wk + 32 * j + (lane & 31);
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int n = n0 + wn + 8 * (i >> 2) + 4 * half + (i & 3);
      if (n < N && k < K) p.gw_part[(static_cast<int64_t>(split) * N + n) * K + k] = acc[j].at(i);
    }
  }
  if (k0 == 0) {  // bias: the row blocks' sums of each column, added in order
    float* red = reinterpret_cast<float*>(vp_lds);  // free: the loop ends with a barrier
    if (!is_x) {
#pragma unroll
      for (int i = 0; i < EC; ++i) red[mb * TILE + EC * cg + i] = bsum[i];
    }
    __syncthreads();
    if (t < TILE && n0 + t < N) {
      float s = 0.0f;
      for (int q = 0; q < MS / 8; ++q) s += red[q * TILE + t];
      p.gw_part[static_cast<int64_t>(N) * K * p.splits + static_cast<int64_t>(split) * N + n0 + t] = s;
    }
  }
}

}  // namespace msda
