// dQ, dK and dV in one grid: workgroups of bwd_dq_direct and of bwd_dkdv_pair side by side, behind a launch that forms delta.
//
// Why: a grid that does not fill the chip takes as long as its longest workgroup's chain of blocks, whatever the CUs beside
// it do, and a kernel starts when the one before it has drained.  Two launches are two chains; in one grid the two kinds of
// workgroup share the chip and the longer chain hides the other (bf16, backward: 2 x 3968 D=128 102 -> 61 us, 16 x 333 D=128
// 20.2 -> 12.7, 4 x 1024 D=256 62.7 -> 34.2).  On grids of one to two rounds the second kind fills the CUs that the end of the
// first leaves idle (8 x 4096 D=128 132 -> 116, 40 x 1024 58.7 -> 50.7, 16 x 2048 D=64 45.2 -> 38.5), and at 128 and 256 columns also on
// larger ones (200 x 512 D=256 218 -> 195).  The price is the launch in front, since dQ can no longer form delta for dK/dV.  The heaviest workgroups of both
// kinds come first.  Where each is the faster one: joint_key_groups.
//
// Registers and LDS are the larger of the two kernels', whose workgroups share a CU equally often.  The compiler keeps a
// value or two more than it has registers for across the choice of the kind (20 bytes of scratch at 128 columns, stored and read
// back once per workgroup, outside the loops).
#pragma once

#include "fa2_bwd_dkdv_pair.hpp"
#include "fa2_bwd_dq.hpp"
#include "fa2_launch.hpp"

namespace fa2 {

template <typename T, int DP, bool PAD, int KG, int COLS = DP>
__global__ __launch_bounds__(64 * kDqWaves, (dkdv_pair_wg_per_cu(DP))) void bwd_joint_kernel(const JointParams p) {
  static_assert(kDqWaves == kDkvWaves, "one block size");
  constexpr int DQ_LDS = DqDirectLayout<DP, kDqBlockKV>::TOTAL_ELEMS, DKV_LDS = DkvPairLayout<DP>::TOTAL_ELEMS;
  __shared__ __attribute__((aligned(1024))) short smem[DQ_LDS > DKV_LDS ? DQ_LDS : DKV_LDS];
  const JointPlace at = joint_place(p.both.resident_grid ? balanced_index(blockIdx.x, p.both.resident_grid) : blockIdx.x,
                                    joint_period(KG));
  const int index = at.index;
  if (at.dq) {
    if (index >= p.n_dq) return;
    BwdParams dq = p.both;
    dq.n_tiles = p.dq_tiles;
    bwd_dq_direct<T, DP, kDqBlockKV, false, PAD, KG, COLS>(dq, smem, [=]() { return index; });
    return;
  }
  if (index >= p.n_dkdv) return;
  if (__builtin_amdgcn_readfirstlane(threadIdx.x >> 6) & 1)
    bwd_dkdv_pair<T, DP, PAD, 1, COLS>(p.both, smem, [=]() { return index; });
  else
    bwd_dkdv_pair<T, DP, PAD, 0, COLS>(p.both, smem, [=]() { return index; });
}

}  // namespace fa2
