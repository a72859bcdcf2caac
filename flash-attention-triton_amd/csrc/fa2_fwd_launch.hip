// Instantiates and launches the forward kernels: compiled twice, with FA2_F32_OUT 0 and 1 (kF32).
#include "fa2_fwd.hpp"
#include "fa2_launch.hpp"

namespace fa2 {
namespace {

constexpr bool kF32 = FA2_F32_OUT;

template <typename T, bool VEC>
void launch_generic(int dp, const FwdParams &p, dim3 grid, dim3 block, hipStream_t s) {
  switch (dp) {
    case 32: hipLaunchKernelGGL((fwd_kernel<T, 32, kFwdBlockKV, VEC, kF32>), grid, block, 0, s, p); break;
    case 64: hipLaunchKernelGGL((fwd_kernel<T, 64, kFwdBlockKV, VEC, kF32>), grid, block, 0, s, p); break;
    case 96: hipLaunchKernelGGL((fwd_kernel<T, 96, kFwdBlockKV, VEC, kF32>), grid, block, 0, s, p); break;
    case 128: hipLaunchKernelGGL((fwd_kernel<T, 128, kFwdBlockKV, VEC, kF32>), grid, block, 0, s, p); break;
    case 192: hipLaunchKernelGGL((fwd_kernel<T, 192, kFwdBlockKV, VEC, kF32>), grid, block, 0, s, p); break;
    default: hipLaunchKernelGGL((fwd_kernel<T, 256, kFwdBlockKV, VEC, kF32>), grid, block, 0, s, p); break;
  }
}

// PRE (exponents straight from the score MFMAs) is instantiated up to 128 columns.  The kernels of 160 columns and more live in a
// translation unit of their own (fa2_fwd_launch_wide.hip), for the time that they take to compile.
template <typename T, int DP, int COLS, bool PRE, int KG>
void launch_cols(const FwdParams &p, dim3 grid, dim3 block, hipStream_t s) {
  if constexpr (KG == 4) {
    if (p.headdim == COLS)
      hipLaunchKernelGGL((fwd_quad_kernel<T, DP, false, PRE, kF32, COLS>), grid, block, 0, s, p);
    else
      hipLaunchKernelGGL((fwd_quad_kernel<T, DP, true, PRE, kF32, COLS>), grid, block, 0, s, p);
  } else if (p.headdim == COLS)
    hipLaunchKernelGGL((fwd_direct_kernel<T, DP, kFwdBlockKV, false, PRE, KG, COLS, kF32>), grid, block, 0, s, p);
  else
    hipLaunchKernelGGL((fwd_direct_kernel<T, DP, kFwdBlockKV, true, PRE, KG, COLS, kF32>), grid, block, 0, s, p);
}

template <typename T, bool PRE, int KG>
void launch_direct(int dp, const FwdParams &p, dim3 grid, dim3 block, hipStream_t s) {
  switch (direct_columns(dp, p.headdim)) {
    case 32: launch_cols<T, 32, 32, PRE, KG>(p, grid, block, s); break;
    case 48: launch_cols<T, 64, 48, PRE, KG>(p, grid, block, s); break;
    case 64: launch_cols<T, 64, 64, PRE, KG>(p, grid, block, s); break;
    case 80: launch_cols<T, 96, 80, PRE, KG>(p, grid, block, s); break;
    case 96: launch_cols<T, 96, 96, PRE, KG>(p, grid, block, s); break;
    case 128: launch_cols<T, 128, 128, PRE, KG>(p, grid, block, s); break;
    default:  // (there are two key groups at most)
      launch_fwd_direct_wide<kF32>(std::is_same<T, __bf16>::value, dp, KG, p, grid, block, s);
      break;
  }
}

template <typename T, bool PRE>
void launch_mixed(const FwdParams &p, dim3 grid, dim3 block, hipStream_t s) {
  switch (p.headdim) {
    case 64: hipLaunchKernelGGL((fwd_mixed_kernel<T, 64, PRE, kF32>), grid, block, 0, s, p); break;
    case 80: hipLaunchKernelGGL((fwd_mixed_kernel<T, 96, PRE, kF32, 80>), grid, block, 0, s, p); break;
    case 96: hipLaunchKernelGGL((fwd_mixed_kernel<T, 96, PRE, kF32>), grid, block, 0, s, p); break;
    default: hipLaunchKernelGGL((fwd_mixed_kernel<T, 128, PRE, kF32>), grid, block, 0, s, p); break;
  }
}

template <typename T, int KG>
void launch_groups(int dp, const FwdParams &p, dim3 grid, dim3 block, hipStream_t s) {
  if (p.folded)
    launch_direct<T, true, KG>(dp, p, grid, block, s);
  else
    launch_direct<T, false, KG>(dp, p, grid, block, s);
}

template <typename T>
void launch(int dp, const FwdParams &p, dim3 grid, hipStream_t s) {
  const dim3 block(64 * kFwdWaves);
  if (p.mixed_singles > 0) {
    if (p.folded)
      launch_mixed<T, true>(p, grid, block, s);
    else
      launch_mixed<T, false>(p, grid, block, s);
    return;
  }
  if (fwd_direct_ok(dp, p)) {
    const int groups = fwd_key_groups(dp, p);
    if (groups == 4)
      launch_groups<T, 4>(dp, p, grid, block, s);
    else if (groups == 2)
      launch_groups<T, 2>(dp, p, grid, block, s);
    else
      launch_groups<T, 1>(dp, p, grid, block, s);
    return;
  }
  if (p.vec)
    launch_generic<T, true>(dp, p, grid, block, s);
  else
    launch_generic<T, false>(dp, p, grid, block, s);
}

}  // namespace

template <>
void launch_fwd<kF32>(bool bf16, int dp, const FwdParams &p, dim3 grid, hipStream_t s) {
  if (bf16)
    launch<__bf16>(dp, p, grid, s);
  else
    launch<_Float16>(dp, p, grid, s);
}

}  // namespace fa2
