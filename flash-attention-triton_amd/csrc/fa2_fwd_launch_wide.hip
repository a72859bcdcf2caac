// The LDS-direct forward kernels for 160 to 256 columns (one wave per SIMD, all 512 registers), in a
// translation unit of their own: see launch_direct in fa2_fwd_launch.hip.
#include "fa2_fwd.hpp"
#include "fa2_launch.hpp"

namespace fa2 {
namespace {

constexpr bool kF32 = FA2_F32_OUT;

template <typename T, int DP, int COLS, int KG>
void launch_cols(const FwdParams &p, dim3 grid, dim3 block, hipStream_t s) {
  if (p.headdim == COLS)
    hipLaunchKernelGGL((fwd_direct_kernel<T, DP, kFwdBlockKV, false, false, KG, COLS, kF32>), grid, block, 0, s, p);
  else
    hipLaunchKernelGGL((fwd_direct_kernel<T, DP, kFwdBlockKV, true, false, KG, COLS, kF32>), grid, block, 0, s, p);
}

template <typename T, int KG>
void launch_wide(int dp, const FwdParams &p, dim3 grid, dim3 block, hipStream_t s) {
  switch (direct_columns(dp, p.headdim)) {
    case 160: launch_cols<T, 192, 160, KG>(p, grid, block, s); break;
    case 192: launch_cols<T, 192, 192, KG>(p, grid, block, s); break;
    case 224: launch_cols<T, 256, 224, KG>(p, grid, block, s); break;
    default: launch_cols<T, 256, 256, KG>(p, grid, block, s); break;
  }
}

template <typename T>
void launch_groups(int dp, int key_groups, const FwdParams &p, dim3 grid, dim3 block, hipStream_t s) {
  if (key_groups == 2)
    launch_wide<T, 2>(dp, p, grid, block, s);
  else
    launch_wide<T, 1>(dp, p, grid, block, s);
}

}  // namespace

template <>
void launch_fwd_direct_wide<kF32>(bool bf16, int dp, int key_groups, const FwdParams &p, dim3 grid, dim3 block, hipStream_t s) {
  if (bf16)
    launch_groups<__bf16>(dp, key_groups, p, grid, block, s);
  else
    launch_groups<_Float16>(dp, key_groups, p, grid, block, s);
}

}  // namespace fa2
