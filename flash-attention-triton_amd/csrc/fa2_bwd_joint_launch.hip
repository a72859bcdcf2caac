// Instantiates and launches the kernels that form dQ, dK and dV in one grid: compiled once per type, with FA2_BF16 0
// and 1 (Type).
#include "fa2_bwd_joint.hpp"
#include "fa2_launch.hpp"

namespace fa2 {
namespace {

#if FA2_BF16
typedef __bf16 Type;
#else
typedef _Float16 Type;
#endif

template <typename T, int KG, int DP, int COLS>
void launch_cols(const JointParams &p, dim3 grid, dim3 block, hipStream_t s) {
  if (p.both.headdim == COLS)
    hipLaunchKernelGGL((bwd_joint_kernel<T, DP, false, KG, COLS>), grid, block, 0, s, p);
  else
    hipLaunchKernelGGL((bwd_joint_kernel<T, DP, true, KG, COLS>), grid, block, 0, s, p);
}

template <typename T, int KG>
void launch_groups(int dp, const JointParams &p, dim3 grid, hipStream_t s) {
  const dim3 block(64 * kDqWaves);
  switch (direct_columns(dp, p.both.headdim)) {
    case 32: launch_cols<T, KG, 32, 32>(p, grid, block, s); break;
    case 48: launch_cols<T, KG, 64, 48>(p, grid, block, s); break;
    case 80: launch_cols<T, KG, 96, 80>(p, grid, block, s); break;
    case 96: launch_cols<T, KG, 96, 96>(p, grid, block, s); break;
    case 160: launch_cols<T, KG, 192, 160>(p, grid, block, s); break;
    case 192: launch_cols<T, KG, 192, 192>(p, grid, block, s); break;
    case 224: launch_cols<T, KG, 256, 224>(p, grid, block, s); break;
    case 64: launch_cols<T, KG, 64, 64>(p, grid, block, s); break;
    case 128: launch_cols<T, KG, 128, 128>(p, grid, block, s); break;
    default: launch_cols<T, KG, 256, 256>(p, grid, block, s); break;
  }
}

}  // namespace

template <>
void launch_joint<Type>(int dp, const JointParams &p, int key_groups, dim3 grid, hipStream_t s) {
  if (key_groups == 2)
    launch_groups<Type, 2>(dp, p, grid, s);
  else
    launch_groups<Type, 1>(dp, p, grid, s);
}

}  // namespace fa2
