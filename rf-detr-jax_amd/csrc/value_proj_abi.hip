// value_proj_abi.hip — C ABI of the value projection with its fused epilogue (include/msda.h):
// validation, launch planning, kernel launches. Validation runs before any HIP call.
#include "msda.h"
#include "msda_launch.h"
#include "msda_kernels.h"  // bf16_t
#include "value_proj_kernels.h"
#include "value_proj_mfma_kernels.h"

#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cstdlib>

namespace {

using msda_host::aligned_to;
using msda_host::fail;

int vp_validate(int dtype, int batch, int len_in, int in_features, int n_heads, int head_dim) {
  if (dtype != MSDA_DTYPE_F32 && dtype != MSDA_DTYPE_BF16) return fail(MSDA_ERR_UNSUPPORTED, "input: unsupported dtype code %d", dtype);
  if (batch < 0 || len_in < 0) return fail(MSDA_ERR_INVALID_ARGUMENT, "batch (%d) and len_in (%d) must be >= 0", batch, len_in);
  if (in_features < 1 || n_heads < 1 || head_dim < 1)
    return fail(MSDA_ERR_INVALID_ARGUMENT, "in_features (%d), n_heads (%d) and head_dim (%d) must be >= 1", in_features, n_heads, head_dim);
  const int64_t m = static_cast<int64_t>(batch) * len_in, n = static_cast<int64_t>(n_heads) * head_dim;
  if (m >= (int64_t{1} << 31) || n >= (int64_t{1} << 24) || in_features >= (1 << 24) || m * std::max<int64_t>(n, in_features) >= (int64_t{1} << 40))
    return fail(MSDA_ERR_UNSUPPORTED, "value projection too large");
  // channel n of a row splits into (head, d), and row m into (batch, position), by multiply-highs,
  // exact while n * head_dim and m * len_in stay below 2^32; element offsets are 32-bit
  if (n * head_dim >= (int64_t{1} << 32) || m * len_in >= (int64_t{1} << 32))
    return fail(MSDA_ERR_UNSUPPORTED, "n_heads * head_dim^2 or batch * len_in^2 reaches 2^32");
  if (m * n >= (int64_t{1} << 32) || m * in_features >= (int64_t{1} << 32) || n * (static_cast<int64_t>(in_features) + 1) >= (int64_t{1} << 32))
    return fail(MSDA_ERR_UNSUPPORTED, "a value-projection tensor reaches 2^32 elements");
  return MSDA_OK;
}

// ceil(2^32 / divisor) for the kernels' multiply-high divisions (vp_div); 0 marks a divisor of 1
// (and an empty extent), whose magic 2^32 does not fit 32 bits.
uint32_t vp_magic(int divisor) {
  return divisor > 1 ? static_cast<uint32_t>(((uint64_t{1} << 32) + static_cast<uint64_t>(divisor) - 1) / static_cast<uint64_t>(divisor)) : 0u;
}

// grad_weight's product is split over m into slices of at least 256 rows (at most 64 slices); the
// partial sums [splits][N][K + 1] are the workspace. A function of the shape only.
int vp_splits(int64_t m) { return static_cast<int>(std::max<int64_t>(1, std::min<int64_t>(64, (m + 255) / 256))); }

int64_t vp_workspace(int batch, int len_in, int in_features, int n_heads, int head_dim) {
  const int64_t m = static_cast<int64_t>(batch) * len_in;
  return static_cast<int64_t>(vp_splits(m)) * n_heads * head_dim * (in_features + 1) * 4;
}

// The 16-byte operand kernels need every 4-element vector they load contiguous and aligned: the
// reduction and column extents K and D multiples of 4 (so N is too), and the tensors they read
// aligned to 4 elements. MSDA_VP_SCALAR forces the element-wise kernels.
bool vec_path(const msda::ValueProjParams& p, size_t eb, const void* a, const void* b) {
  if (msda_host::env_flag("MSDA_VP_SCALAR")) return false;
  return p.k % 4 == 0 && p.dim % 4 == 0 && aligned_to(p.w, 16) && (a == nullptr || aligned_to(a, 4 * eb)) &&
         (b == nullptr || aligned_to(b, 4 * eb));
}

template <int KIND, typename VT, int BM>
int launch_g4(const msda::ValueProjParams& p, int grid, hipStream_t st) {
  static std::atomic<int> granted[msda_host::kMaxDevices];  // per instantiation
  auto k = msda::gemm4_kernel<KIND, VT, BM>;
  using Cfg = msda::G4<BM>;
  const int rc = msda_host::allow_lds(k, Cfg::kLdsBytes, granted);
  if (rc != MSDA_OK) return rc;
  hipLaunchKernelGGL(k, dim3(grid), dim3(Cfg::kThreads), Cfg::kLdsBytes, st, p);
  return MSDA_OK;
}

// The bf16-matrix-unit kernels (value_proj_mfma_kernels.h) need runs of 8 elements of every tensor
// contiguous and 16-byte aligned: K and D multiples of 8, every tensor they touch on 16 bytes.
// MSDA_VP_SCALAR and MSDA_VP_BM select the other kernels.
bool mfma_path(const msda::ValueProjParams& p, const void* a, const void* b) {
  if (msda_host::env_flag("MSDA_VP_SCALAR") || msda_host::knob("MSDA_VP_BM", 0) != 0) return false;
  return p.k % 8 == 0 && p.dim % 8 == 0 && aligned_to(p.w, 16) && aligned_to(a, 16) && aligned_to(b, 16);
}

template <int KIND, typename VT, int CB>
int launch_rows(const msda::ValueProjParams& p, int lds_limit, int cus, hipStream_t st) {
  using Cfg = msda::VpRows<KIND, VT, CB>;
  static std::atomic<int> granted[msda_host::kMaxDevices];  // per instantiation
  const int64_t m = static_cast<int64_t>(p.batch) * p.seq;
  const int cols = KIND == msda::kGemmForward ? p.n : p.k, red = KIND == msda::kGemmForward ? p.k : p.n;
  const int lds = static_cast<int>(Cfg::lds_bytes(red));
  auto k = msda::vp_rows_kernel<KIND, VT, CB>;
  const int rc = msda_host::allow_lds(k, lds, granted);
  if (rc != MSDA_OK) return rc;
  // workgroups a CU holds at once (LDS, and registers: two waves per SIMD with 256, four with 128)
  const int resident = std::max(1, std::min(lds_limit / lds, 16 / Cfg::kWaves));
  const int64_t cgroups = (cols + 32 * CB - 1) / (32 * CB), tiles = (m + 31) / 32;
  const int64_t rgroups = std::max<int64_t>(1, std::min<int64_t>((tiles + Cfg::kWaves - 1) / Cfg::kWaves, int64_t{cus} * resident / cgroups));
  hipLaunchKernelGGL(k, dim3(static_cast<unsigned>(cgroups * rgroups)), dim3(Cfg::kThreads), lds, st, p);
  return MSDA_OK;
}

template <typename VT, int TILE, bool MASK>
int launch_gw(const msda::ValueProjParams& p, hipStream_t st) {
  using Cfg = msda::VpGw<VT, TILE>;
  static std::atomic<int> granted[msda_host::kMaxDevices];  // per instantiation
  auto k = msda::vp_gw_kernel<VT, TILE, MASK>;
  const int rc = msda_host::allow_lds(k, Cfg::kLdsBytes, granted);
  if (rc != MSDA_OK) return rc;
  const int64_t tiles = static_cast<int64_t>((p.n + TILE - 1) / TILE) * ((p.k + TILE - 1) / TILE);
  hipLaunchKernelGGL(k, dim3(static_cast<unsigned>(tiles * p.splits)), dim3(Cfg::kThreads), Cfg::kLdsBytes, st, p);
  return MSDA_OK;
}

// The product on the bf16 matrix unit, or MSDA_ERR_UNSUPPORTED (no message) where it would not pay
// (f32) or one 32-column block of weights does not fit the LDS.
//   * Rows: two column blocks a workgroup where that leaves four waves (32-row tiles) a CU, else one:
//     bf16 8 x 576 rows forward 6.4 (one) against 6.6 us, 16 x 6800 42 against 33; four and eight
//     blocks were slower at every size (52 and 55 us), their LDS leaving room for 8 waves a CU.
//     f32 (256 -> 256, forward): two blocks with more than four waves a CU (8192 rows, four: 18.1, one block
//     15.4; 9216: 18.3 and 21.9, gemm4_kernel 20.3), else one from four waves a CU on. From more than six it is
//     the faster kernel (6800 rows 15.0 and 17.3), from four to six the closer one to float64 (7e-8 and
//     1.1e-7; 4608 rows 14.6 and 13.6, grad_input 14.7 and 14.1; 128 columns, 9216 rows 10.7 and 9.3).
//   * grad_weight: 128-wide tiles (bf16) where they make one workgroup a CU. f32 from 16 slices (4096
//     rows) on (1152 rows 11.8 us by gemm4_kernel, 15.4), with workgroups for 5 of 8 CUs (64 x 64, one tile
//     and 64 slices, at 108800 rows 42 and 56; 128 x 128 at 8192 rows, half the CUs, 12.7 and 14.6; at 16416,
//     all of them, 21.2 and 20.0; 512 x 64 at 16416, two for each, 33 and 23; 160 x 160 at 4096, 9 of 16, 12.0
//     and 14.0; 256 x 256 at 4608, 20.3 and 17.3).
// MSDA_VP_CB=1 or 2 forces the path and the column blocks.
template <int KIND, typename VT>
int launch_mfma(const msda::ValueProjParams& p, hipStream_t st) {
  int lds = 0, cus = 0;
  const int rc = msda_host::device_attrs(&lds, &cus);
  if (rc != MSDA_OK) return rc;
  constexpr bool bf = sizeof(VT) == 2;
  const int cb = msda_host::knob("MSDA_VP_CB", 0);
  if constexpr (KIND == msda::kGemmGradWeight) {
    if constexpr (bf) {
      const int64_t t128 = static_cast<int64_t>((p.n + 127) / 128) * ((p.k + 127) / 128) * p.splits;
      if (t128 >= cus) return p.mask != nullptr ? launch_gw<VT, 128, true>(p, st) : launch_gw<VT, 128, false>(p, st);
    } else if (cb == 0) {
      const int64_t tiles = static_cast<int64_t>((p.n + 63) / 64) * ((p.k + 63) / 64);
      if (p.splits < 16 || 8 * tiles * p.splits < 5 * int64_t{cus}) return MSDA_ERR_UNSUPPORTED;
    }
    return p.mask != nullptr ? launch_gw<VT, 64, true>(p, st) : launch_gw<VT, 64, false>(p, st);
  } else {
    const int cols = KIND == msda::kGemmForward ? p.n : p.k, red = KIND == msda::kGemmForward ? p.k : p.n;
    const int64_t tiles = (static_cast<int64_t>(p.batch) * p.seq + 31) / 32;
    const int64_t two = tiles * ((cols + 63) / 64), one = tiles * ((cols + 31) / 32);  // waves
    if (msda::VpRows<KIND, VT, 2>::lds_bytes(red) <= lds && (cb ? cb == 2 : bf ? two >= 4 * int64_t{cus} : two > 4 * int64_t{cus}))
      return launch_rows<KIND, VT, 2>(p, lds, cus, st);
    if (msda::VpRows<KIND, VT, 1>::lds_bytes(red) <= lds && (cb ? cb == 1 : bf || one >= 4 * int64_t{cus}))
      return launch_rows<KIND, VT, 1>(p, lds, cus, st);
    return MSDA_ERR_UNSUPPORTED;
  }
}

// One product: rows x cols outputs (times `splits` slices of the reduction). The 16-byte kernels
// take 32-row tiles when 64-row tiles would be fewer than four per CU (a CU with one tile more
// than another finishes a whole tile later; smaller tiles even that out), else 64-row tiles;
// MSDA_VP_BM=32 or 64 forces one.
template <int KIND, typename VT>
int launch_gemm(const msda::ValueProjParams& p, int64_t rows, int64_t cols, int splits, bool vec, hipStream_t st, const char* what) {
  int rc = MSDA_OK;
  const int64_t ct = (cols + msda::kGemmBN - 1) / msda::kGemmBN;
  if (vec) {
    int lds = 0, cus = 0;
    if ((rc = msda_host::device_attrs(&lds, &cus)) != MSDA_OK) return rc;
    const int64_t t64 = (rows + 63) / 64 * ct * splits;
    int bm = t64 < 4 * static_cast<int64_t>(cus) ? 32 : 64;
    const int e = msda_host::knob("MSDA_VP_BM", 0);
    bm = e == 32 ? 32 : e == 64 ? 64 : bm;
    if (bm == 32) rc = launch_g4<KIND, VT, 32>(p, static_cast<int>((rows + 31) / 32 * ct * splits), st);
    else rc = launch_g4<KIND, VT, 64>(p, static_cast<int>(t64), st);
    if (rc != MSDA_OK) return rc;
  } else {
    hipLaunchKernelGGL((msda::gemm_kernel<KIND, VT>), dim3(static_cast<unsigned>((rows + 63) / 64 * ct * splits)), dim3(256), 0, st, p);
  }
  return msda_host::check_launch(what);
}

template <int KIND>
int launch_gemm_dt(const msda::ValueProjParams& p, int64_t rows, int64_t cols, int splits, bool vec, bool mfma, hipStream_t st,
                   const char* what) {
  if (mfma) {
    const int rc = p.bf16 ? launch_mfma<KIND, msda::bf16_t>(p, st) : launch_mfma<KIND, float>(p, st);
    if (rc != MSDA_ERR_UNSUPPORTED) return rc != MSDA_OK ? rc : msda_host::check_launch(what);
  }
  return p.bf16 ? launch_gemm<KIND, msda::bf16_t>(p, rows, cols, splits, vec, st, what)
                : launch_gemm<KIND, float>(p, rows, cols, splits, vec, st, what);
}

}  // namespace

extern "C" {

int msda_value_proj_fwd(const void* input, int dtype, const float* weight, const float* bias, const uint8_t* padding_mask, void* value,
                        int batch, int len_in, int in_features, int n_heads, int head_dim, void* stream) {
  msda_host::clear_error();
  int rc = vp_validate(dtype, batch, len_in, in_features, n_heads, head_dim);
  if (rc != MSDA_OK) return rc;
  if (batch == 0 || len_in == 0) return MSDA_OK;
  if (input == nullptr || weight == nullptr || value == nullptr) return fail(MSDA_ERR_INVALID_ARGUMENT, "msda_value_proj_fwd: NULL tensor pointer");
  const size_t eb = dtype == MSDA_DTYPE_BF16 ? 2 : 4;
  if (!aligned_to(input, eb) || !aligned_to(value, eb) || !aligned_to(weight, 4) || !aligned_to(bias, 4))
    return fail(MSDA_ERR_INVALID_ARGUMENT, "tensors must be aligned to their element size");
  msda::ValueProjParams p{};
  p.x = input;
  p.w = weight;
  p.bias = bias;
  p.mask = padding_mask;
  p.value = value;
  p.bf16 = dtype == MSDA_DTYPE_BF16;
  p.batch = batch;
  p.seq = len_in;
  p.k = in_features;
  p.n = n_heads * head_dim;
  p.heads = n_heads;
  p.dim = head_dim;
  p.dim_magic = vp_magic(head_dim);
  p.seq_magic = vp_magic(len_in);
  return launch_gemm_dt<msda::kGemmForward>(p, static_cast<int64_t>(batch) * len_in, p.n, 1, vec_path(p, eb, input, nullptr),
                                            mfma_path(p, input, value), static_cast<hipStream_t>(stream), "value projection forward");
}

int64_t msda_value_proj_bwd_workspace_size(int batch, int len_in, int in_features, int n_heads, int head_dim) {
  msda_host::clear_error();
  const int rc = vp_validate(MSDA_DTYPE_F32, batch, len_in, in_features, n_heads, head_dim);
  if (rc != MSDA_OK) return rc;
  return vp_workspace(batch, len_in, in_features, n_heads, head_dim);
}

int msda_value_proj_bwd(const void* input, int dtype, const float* weight, const uint8_t* padding_mask, const void* grad_value,
                        void* grad_input, float* grad_weight, float* grad_bias, int batch, int len_in, int in_features, int n_heads,
                        int head_dim, void* workspace, int64_t workspace_bytes, void* stream) {
  msda_host::clear_error();
  int rc = vp_validate(dtype, batch, len_in, in_features, n_heads, head_dim);
  if (rc != MSDA_OK) return rc;
  const bool want_w = grad_weight != nullptr || grad_bias != nullptr;
  if (grad_input == nullptr && !want_w) return MSDA_OK;
  const int64_t m = static_cast<int64_t>(batch) * len_in;
  const size_t eb = dtype == MSDA_DTYPE_BF16 ? 2 : 4;
  if (m > 0) {
    if (grad_value == nullptr || weight == nullptr || (want_w && input == nullptr))
      return fail(MSDA_ERR_INVALID_ARGUMENT, "msda_value_proj_bwd: NULL tensor pointer");
    if (!aligned_to(input, eb) || !aligned_to(grad_value, eb) || !aligned_to(grad_input, eb) || !aligned_to(weight, 4) ||
        !aligned_to(grad_weight, 4) || !aligned_to(grad_bias, 4))
      return fail(MSDA_ERR_INVALID_ARGUMENT, "tensors must be aligned to their element size");
  }
  const int64_t ws = vp_workspace(batch, len_in, in_features, n_heads, head_dim);
  if (want_w) {
    if (workspace == nullptr) return fail(MSDA_ERR_INVALID_ARGUMENT, "workspace is NULL (see msda_value_proj_bwd_workspace_size)");
    if (!aligned_to(workspace, 16)) return fail(MSDA_ERR_INVALID_ARGUMENT, "workspace must be 16-byte aligned");
    if (workspace_bytes < ws)
      return fail(MSDA_ERR_INVALID_ARGUMENT, "workspace of %lld bytes needed, got %lld", static_cast<long long>(ws),
                  static_cast<long long>(workspace_bytes));
  }
  msda::ValueProjParams p{};
  p.x = input;
  p.w = weight;
  p.mask = padding_mask;
  p.gvalue = grad_value;
  p.gx = grad_input;
  p.gw = grad_weight;
  p.gb = grad_bias;
  p.gw_part = static_cast<float*>(workspace);
  p.bf16 = dtype == MSDA_DTYPE_BF16;
  p.batch = batch;
  p.seq = len_in;
  p.k = in_features;
  p.n = n_heads * head_dim;
  p.heads = n_heads;
  p.dim = head_dim;
  p.splits = vp_splits(m);
  p.dim_magic = vp_magic(head_dim);
  p.seq_magic = vp_magic(len_in);
  hipStream_t st = static_cast<hipStream_t>(stream);
  if (grad_input != nullptr && m > 0) {
    const bool vec = vec_path(p, eb, grad_value, nullptr);
    if ((rc = launch_gemm_dt<msda::kGemmGradInput>(p, m, in_features, 1, vec, mfma_path(p, grad_value, grad_input),
                                                    st, "value projection backward (input)")) != MSDA_OK)
      return rc;
  }
  if (want_w) {
    // with no rows the partial sums are zero: the product still runs (every partial is written).
    // The element-wise kernel forms the bias gradient as a column of ones (K + 1 columns); the
    // 16-byte kernel sums dY^T rows instead (K columns).
    const bool vec = vec_path(p, eb, grad_value, input), mfma = m > 0 && mfma_path(p, grad_value, input);
    if ((rc = launch_gemm_dt<msda::kGemmGradWeight>(p, p.n, static_cast<int64_t>(in_features) + (vec ? 0 : 1), p.splits, vec, mfma, st,
                                                     "value projection backward (weight)")) != MSDA_OK)
      return rc;
    const int64_t total = static_cast<int64_t>(p.n) * (in_features + 1);
    hipLaunchKernelGGL(msda::wg_reduce_kernel, dim3(static_cast<unsigned>(std::min<int64_t>((total + 255) / 256, 4096))), dim3(256), 0, st,
                       p);
    if ((rc = msda_host::check_launch("value projection backward (weight reduction)")) != MSDA_OK) return rc;
  }
  return MSDA_OK;
}

}  // extern "C"
