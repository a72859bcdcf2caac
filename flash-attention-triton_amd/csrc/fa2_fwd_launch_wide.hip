// The LDS-direct forward kernels for 192 and 256 columns (one wave per SIMD, all 512 registers), in a
// translation unit of their own: see launch_direct in fa2_fwd_launch.hip.
#include "fa2_fwd.hpp"
#include "fa2_launch.hpp"

namespace fa2 {
namespace {

// At 256 columns only the padded variant is instantiated, also for a head dimension of exactly 256
// (it then switches no lane off): with the number of columns a run-time value the compiler keeps the
// kernel within its 512 registers, with a constant 256 it spills about forty of them, with reloads
// inside the tile loop, where they queue behind the tile loads (same counter).
template <typename T, bool PAD, int KG>
void launch_wide(int dp, const FwdParams &p, dim3 grid, dim3 block, hipStream_t s) {
  if (dp == 192)
    hipLaunchKernelGGL((fwd_direct_kernel<T, 192, kFwdBlockKV, PAD, false, KG>), grid, block, 0, s, p);
  else
    hipLaunchKernelGGL((fwd_direct_kernel<T, 256, kFwdBlockKV, true, false, KG>), grid, block, 0, s, p);
}

template <typename T>
void launch_groups(int dp, bool pad, int key_groups, const FwdParams &p, dim3 grid, dim3 block, hipStream_t s) {
  if (key_groups == 2) {
    if (pad) launch_wide<T, true, 2>(dp, p, grid, block, s); else launch_wide<T, false, 2>(dp, p, grid, block, s);
  } else {
    if (pad) launch_wide<T, true, 1>(dp, p, grid, block, s); else launch_wide<T, false, 1>(dp, p, grid, block, s);
  }
}

}  // namespace

void launch_fwd_direct_wide(bool bf16, int dp, bool pad, int key_groups, const FwdParams &p, dim3 grid, dim3 block, hipStream_t s) {
  if (bf16)
    launch_groups<__bf16>(dp, pad, key_groups, p, grid, block, s);
  else
    launch_groups<_Float16>(dp, pad, key_groups, p, grid, block, s);
}

}  // namespace fa2
