// Instantiates and launches the dQ kernels, the delta preprocess and the fp32 casts.
#include "fa2_bwd_dq.hpp"
#include "fa2_cast.hpp"
#include "fa2_launch.hpp"

namespace fa2 {
namespace {

template <typename T, bool FUSE_DELTA, int KG, int DP, int COLS>
void launch_cols(const BwdParams &p, dim3 grid, dim3 block, hipStream_t s) {
  if (p.headdim == COLS)
    hipLaunchKernelGGL((bwd_dq_direct_kernel<T, DP, kDqBlockKV, FUSE_DELTA, false, KG, COLS>), grid, block, 0, s, p);
  else
    hipLaunchKernelGGL((bwd_dq_direct_kernel<T, DP, kDqBlockKV, FUSE_DELTA, true, KG, COLS>), grid, block, 0, s, p);
}

template <typename T, bool FUSE_DELTA, int KG>
void launch_direct_groups(int dp, const BwdParams &p, dim3 grid, dim3 block, hipStream_t s) {
  switch (direct_columns(dp, p.headdim)) {
    case 32: launch_cols<T, FUSE_DELTA, KG, 32, 32>(p, grid, block, s); break;
    case 48: launch_cols<T, FUSE_DELTA, KG, 64, 48>(p, grid, block, s); break;
    case 64: launch_cols<T, FUSE_DELTA, KG, 64, 64>(p, grid, block, s); break;
    case 80: launch_cols<T, FUSE_DELTA, KG, 96, 80>(p, grid, block, s); break;
    case 96: launch_cols<T, FUSE_DELTA, KG, 96, 96>(p, grid, block, s); break;
    case 128: launch_cols<T, FUSE_DELTA, KG, 128, 128>(p, grid, block, s); break;
    case 160: launch_cols<T, FUSE_DELTA, KG, 192, 160>(p, grid, block, s); break;
    case 192: launch_cols<T, FUSE_DELTA, KG, 192, 192>(p, grid, block, s); break;
    case 224: launch_cols<T, FUSE_DELTA, KG, 256, 224>(p, grid, block, s); break;
    default: launch_cols<T, FUSE_DELTA, KG, 256, 256>(p, grid, block, s); break;
  }
}

template <typename T, bool FUSE_DELTA>
void launch_direct(int dp, const BwdParams &p, int key_groups, dim3 grid, dim3 block, hipStream_t s) {
  if (key_groups == 2)
    launch_direct_groups<T, FUSE_DELTA, 2>(dp, p, grid, block, s);
  else
    launch_direct_groups<T, FUSE_DELTA, 1>(dp, p, grid, block, s);
}

template <typename T>
void launch(int dp, const BwdParams &p, int key_groups, dim3 grid, bool fuse_delta, hipStream_t s) {
  const dim3 block(64 * kDqWaves);
  if (dq_direct_ok(dp, p)) {
    if (fuse_delta)
      launch_direct<T, true>(dp, p, key_groups, grid, block, s);
    else
      launch_direct<T, false>(dp, p, key_groups, grid, block, s);
    return;
  }
  switch (dp) {
    case 32: hipLaunchKernelGGL((bwd_dq_kernel<T, 32, kDqBlockKV>), grid, block, 0, s, p); break;
    case 64: hipLaunchKernelGGL((bwd_dq_kernel<T, 64, kDqBlockKV>), grid, block, 0, s, p); break;
    case 96: hipLaunchKernelGGL((bwd_dq_kernel<T, 96, kDqBlockKV>), grid, block, 0, s, p); break;
    case 128: hipLaunchKernelGGL((bwd_dq_kernel<T, 128, kDqBlockKV>), grid, block, 0, s, p); break;
    case 192: hipLaunchKernelGGL((bwd_dq_kernel<T, 192, kDqBlockKV>), grid, block, 0, s, p); break;
    default: hipLaunchKernelGGL((bwd_dq_kernel<T, 256, kDqBlockKV>), grid, block, 0, s, p); break;
  }
}

}  // namespace

void launch_dq(bool bf16, int dp, const BwdParams &p, int key_groups, dim3 grid, bool fuse_delta, hipStream_t s) {
  if (bf16)
    launch<__bf16>(dp, p, key_groups, grid, fuse_delta, s);
  else
    launch<_Float16>(dp, p, key_groups, grid, fuse_delta, s);
}

void launch_cast(const CastParams &p, dim3 grid, hipStream_t s) {
  hipLaunchKernelGGL(cast_f16_kernel, grid, dim3(kCastThreads), 0, s, p);
}

void launch_preprocess(bool bf16, const PreParams &p, dim3 grid, hipStream_t s) {
  if (bf16)
    hipLaunchKernelGGL((bwd_preprocess_kernel<__bf16>), grid, dim3(256), 0, s, p);
  else
    hipLaunchKernelGGL((bwd_preprocess_kernel<_Float16>), grid, dim3(256), 0, s, p);
}

template <typename T>
static void launch_delta_steps(const PreParams &p, dim3 grid, hipStream_t s) {
  if (p.headdim <= 32)
    hipLaunchKernelGGL((bwd_delta_kernel<T, 2>), grid, dim3(64), 0, s, p);
  else if (p.headdim <= 64)
    hipLaunchKernelGGL((bwd_delta_kernel<T, 4>), grid, dim3(64), 0, s, p);
  else if (p.headdim <= 128)
    hipLaunchKernelGGL((bwd_delta_kernel<T, 8>), grid, dim3(64), 0, s, p);
  else
    hipLaunchKernelGGL((bwd_delta_kernel<T, 16>), grid, dim3(64), 0, s, p);
}

void launch_delta(bool bf16, const PreParams &p, dim3 grid, hipStream_t s) {
  if (bf16)
    launch_delta_steps<__bf16>(p, grid, s);
  else
    launch_delta_steps<_Float16>(p, grid, s);
}

}  // namespace fa2
