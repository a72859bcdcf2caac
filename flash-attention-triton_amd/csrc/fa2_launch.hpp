// Kernel launchers, one translation unit per kernel family so that the library builds in parallel.
// `dp` is the padded head dimension of the table row in use (32, 64, 96, 128, 192 or 256); the
// launchers pick the LDS-direct fast kernel when the tensors allow it and the generic one otherwise.
#pragma once

#include <hip/hip_runtime.h>

#include <climits>

#include "fa2_params.hpp"

namespace fa2 {

// The fast kernels need a head dimension that is a multiple of 8 (whole 16-byte chunks), 16-byte aligned
// rows and row offsets inside a tile that fit 32 bits (direct_stride_ok).
inline bool direct_headdim(int dp, int headdim) {
  return headdim % 8 == 0 && headdim <= dp && (dp == 32 || dp == 64 || dp == 96 || dp == 128);
}
// The rows of 192 and 256 columns (one wave per SIMD, most or all of the 160 KiB of LDS): forward, dQ and
// paired dK/dV kernels.
inline bool direct_headdim_wide(int dp, int headdim) {
  return direct_headdim(dp, headdim) || (headdim % 8 == 0 && headdim <= dp && (dp == 192 || dp == 256));
}
// Columns the forward, dQ and paired dK/dV kernels of a row multiply: the head dimension rounded up to a step of 16
// up to 96 columns and of 32 above (against the row's own number: fa2_fwd.hpp).  The row still gives the LDS tiles, of pitch
// lds_pitch(dp) (32, 64, 128 or 256).  A head dimension that is one of these counts needs no zero-filled tiles: what lies behind
// a row is multiplied into accumulator rows that are not stored.  Any other runs the padded variant of the next count.
// Steps of 16 above 96 columns are not instantiated (each count is 36 to 52 kernels).  What they would save, time at the next
// count over its own, forward / dQ / paired dK/dV, bf16: 112 columns 1.03 / 1.04 / 1.03 (32 x 4096) to 1.06 / 1.05 / 1.09
// (256 x 512), 144 columns 1.05 / 1.03 / 1.05, 208 columns 1.05 / 1.04 / 1.04 (32 x 4096); 176 and 240 not measured.
inline int direct_columns(int dp, int headdim) {
  const int less = dp == 64 || dp == 96 ? dp - 16 : dp > 128 ? dp - 32 : dp;
  return headdim <= less ? less : dp;
}
// Key groups of the forward and dQ kernels.  With two, a workgroup owns 64 query rows instead of 128 and two
// waves share 32 of them, one taking the even and the other the odd 32-key blocks; they merge their results
// through LDS at the end.  Every wave's chain of blocks is half as long and the grid has twice the
// workgroups, but every K and V tile is loaded for half the rows and every block ends at a barrier.  So two
// groups win while the grid leaves CUs idle.  Heads that do not divide by 8 have their tiles spread over the XCDs, so
// that the same K and V tiles are fetched into several L2s: with odd numbers of heads the doubled loads cost more.
// Time of one group over two, bf16, (batch, head) pairs x tokens, forward / dQ, by workgroups of 128 rows:
//   to 128      0.94-1.00 / 0.80-1.00 (64 tokens: half the workgroups would have no rows); from 65 tokens on
//               1.04-1.2 / 0.99-1.2 (but dQ at 256 columns 0.95 at 65, 1.10 at 100), 1.3-1.7 / 1.25-1.65 beyond
//   to 256      32 columns 1.20 / 1.12 (128 x 256); 64 columns 1.15 / 1.10 (128 x 256), 1.13 (77 x 333);
//               96 columns 1.11 / 1.12 (128 x 256), 1.09 / 1.01 (59 x 333), 0.94 / 0.96 (77 x 384), 1.08 / 1.15 (58 x 512);
//               128 columns 1.06 / 0.98 (128 x 256), 0.96 / 0.92 (116 x 256), 1.16 / 1.00 (72 x 384), 0.92 / 0.97
//               (59 x 384), 0.96 / 0.98 (39 x 512), 0.92 / 1.01 (51 x 512), 0.91 (47 x 640), 1.05 / 1.07 (29 x 1024);
//               192 and 256 columns (one workgroup per CU either way) 1.02 / 1.02 and 1.08 / 0.99 (32 x 1024),
//               0.94 / 0.97 and 0.94 / 0.88 (29 x 1024), 1.18 / 1.21 and 1.25 / 1.14 (14 x 2048)
//   to 384      32 columns 1.11 / 1.10 (from 512 tokens); 64 columns 1.09 / 1.08 (96 x 512), 0.92 / 0.95 (75 x 512),
//               1.07 / 1.13 (43 x 1024); 96 columns 1.10 / 1.09 (24 x 2048), 0.96 / 0.95-1.08 at 1024 tokens;
//               128 columns 1.14 / 1.04 (12 x 4096), 1.08 / 0.94 (24 x 2048)
//   to 512      32 columns 1.08 / 1.03 (from 1024 tokens); 64 columns 1.04 / 1.05 (16 x 4096), 0.98 / 0.99-1.02 (2048 tokens);
//               128 columns 0.98 / 0.94 (16 x 4096)
//   beyond      0.75-0.98
// `cols` are the columns multiplied (direct_columns).  At 160 and 224 the lines of 192 and 256 hold.  Those of 64 and 96
// hold at 48 and 80 but for dQ with odd heads to 256 workgroups.  Time of the whole backward (delta formed by dQ), dQ with one
// group over two:
//   48 columns  1.03 (59 x 333), 1.00 (77 x 333), 1.02 (85 x 257), 1.04 (65 x 300), 1.02 (63 x 500): as with even heads
//   64 columns  0.98 (59 x 333), 0.98 (77 x 333), 0.97 (65 x 300), 0.98 (83 x 384), 1.00 (67 x 384), 0.99 (63 x 500), although
//               dQ by itself gains (1.15 at 59 x 333): the dK/dV kernel behind it takes longer by more
//   80 columns  1.05 (59 x 333), 1.03 (77 x 333), 1.04 (65 x 300), 1.03 (83 x 384), 1.04 (63 x 500): as with even heads
//   96 columns  1.02 (59 x 333), 1.01 (77 x 333), 1.01 (65 x 300), 1.01 (83 x 384), 1.00 (63 x 500), dQ by itself 0.92-1.06
inline int key_groups(int dp, int cols, int64_t heads, int seqlen_q, bool dq) {
  const int64_t wgs = heads * ((seqlen_q + kFwdBlockQ - 1) / kFwdBlockQ);
  static_assert(kFwdBlockQ == kDqBlockQ, "the same grid for both kernels");
  const bool odd = heads % 2 != 0;
  int from = INT_MAX;  // query rows from which two groups win
  if (wgs <= kCUs / 2) {
    from = dq && dp == 256 ? 97 : 65;
  } else if (wgs <= kCUs) {
    if (dp > 128)
      from = odd && wgs > kCUs * 3 / 4 ? 2048 : 1024;
    else if (dp == 128)
      from = (odd && wgs > kCUs * 9 / 16) || (heads % 8 != 0 && wgs > kCUs * 13 / 16) ? 1024 : dq ? 384 : 256;
    else
      from = odd && (dq ? cols == 64 || cols == 96 : dp == 96 && wgs > kCUs * 3 / 4) ? 512 : 256;
  } else if (wgs <= 3 * kCUs / 2 && dp <= 128) {
    from = dp == 128 ? 4096 : dp == 96 ? 2048 : dp == 64 && odd ? 1024 : 512;
  } else if (wgs <= 2 * kCUs && dp <= 64) {
    from = dp == 64 ? 4096 : 1024;
  }
  return seqlen_q >= from ? 2 : 1;
}
inline bool fwd_direct_ok(int dp, const FwdParams &p) {
  return p.vec && direct_headdim_wide(dp, p.headdim) && direct_stride_ok(p.q) && direct_stride_ok(p.k) &&
         direct_stride_ok(p.v);
}
// Four key groups (fwd_quad_kernel), to 128 columns: 32 query rows to a workgroup, again half the chain for twice the loads per
// row, in tiles of 128 keys that leave room for four workgroups per CU at 32 columns, two at 64 and one from 80 on.  Time of the faster
// of the other forms over its own, bf16, by workgroups of 32 rows, the row a backward follows / the folded one (the sizes:
// profiles/forward_forms_sweep.txt): while they are all resident it grows with the chain, and past that it is lost.
//   32 columns        to 512 1.02-1.65 / 1.01-1.52, to 768 from 1024 tokens on 1.02-1.50 / 1.00-1.40, to 1024 from 2048 on 1.17-1.36; 0.88-1.0
//                     beyond
//   48, 64 columns    to 512 1.02-1.63 / 1.02-1.55, to 640 from 2048 on 1.02-1.39 / 0.99-1.39, to 768 from 3000 on 1.01-1.55 / 0.99-1.55; to 768
//                     of 1024 to 2500 tokens 0.75-1.33 / 0.74-1.28
//   40, 56 columns    to 512 1.00-1.56 / 1.00-1.52, but 0.97-1.00 / 0.98-1.01 of up to 600 tokens beyond 256; to 576 from 2048 on 1.09-1.40 / 1.08-
//                     1.37, to 640 from 2500 on 1.05-1.42 / 1.05-1.39 (of 2048 0.93-0.99), to 704 from 3000 on 1.09-1.35 / 1.10-1.33, to 768
//                     from 3500 on 1.03-1.52 (of 3000 0.95-0.98)
//   80, 96 columns    to 256 from 2048 on 1.00-1.13 / 0.95-1.03, 1500 and 1750 0.97-1.01 / 0.93-0.95, below 0.92-0.97 / 0.87-0.92; to 384 from
//                     4096 on 1.05-1.29 / 0.99-1.23, below 0.66-1.18
//   72, 88 columns    to 256 from 1000 on 1.02-1.38 / from 1500 on 1.05-1.30, 768 and 900 0.96-1.00 / 0.94-0.96; to 384 from 4096 on 1.21-1.42 /
//                     1.15-1.27
//   128 columns       to 256 from 1500 on 1.02-1.36 / from 2048 on 1.02-1.28 (1500 and 1750 0.98-1.01); to 384 from 4096 on 1.17-1.39 / 1.09-1.31,
//                     below 0.65-1.31
//   104 to 120        to 256 from 1500 on 1.10-1.35 / 1.06-1.30; to 384 from 4096 on 1.28-1.50 / 1.23-1.33
// The folded forward has fewer instructions to a block, so that a shorter chain saves it less.
constexpr int fwd_quad_limit_64(int n, bool padded) {
  if (!padded) return n >= 3000 ? 768 : n >= 2048 ? 640 : 512;
  return n >= 3500 ? 768 : n >= 3000 ? 704 : n >= 2500 ? 640 : n >= 2048 ? 576 : 512;
}
inline bool fwd_quad(int dp, const FwdParams &p) {
  const int n = p.seqlen_q;
  const int64_t wgs = (int64_t)p.batch * p.nheads * ((n + 31) / 32);
  const bool padded = p.headdim != direct_columns(dp, p.headdim);
  if (dp == 32) return n > 512 && wgs <= (n >= 2048 ? 1024 : n >= 1024 ? 768 : 512);
  if (dp == 64) return n > (padded && wgs > 256 ? 600 : 512) && wgs <= fwd_quad_limit_64(n, padded);
  if (dp == 96 && !padded && p.folded) return n >= 4096 && wgs > 256 && wgs <= 384;
  const int shortest = dp == 96 ? (padded ? (p.folded ? 1500 : 1000) : 2048) : !padded && p.folded ? 2048 : 1500;
  return dp <= 128 && n >= shortest && wgs <= (n >= 4096 ? 384 : 256);
}
inline int fwd_key_groups(int dp, const FwdParams &p) {
  if (!fwd_direct_ok(dp, p)) return 1;
  const int64_t heads = (int64_t)p.batch * p.nheads;
  return fwd_quad(dp, p) ? 4 : key_groups(dp, direct_columns(dp, p.headdim), heads, p.seqlen_q, false);
}
// One and two key groups in one grid (fwd_mixed_kernel): how many pairs of 64-row tiles of a head one group takes, 0 where all tiles
// are of one kind.  Three eighths of the tiles, a little more on the larger grids, whose last round the smaller tiles would make
// longer.  Time of one group over it, bf16, by workgroups of 128 rows, the row a backward follows / the folded one (the sizes:
// profiles/forward_forms_sweep.txt); where two groups are the better ones (key_groups) it is 0.94-1.05 of theirs:
//   64 columns       of 1024 to 3000 tokens to 448 1.05-1.16 / 1.00-1.15; to 512 from 1700 on 1.00-1.10 / 0.99-1.10, below with an even number
//                    of heads 1.01-1.09 / 0.98-1.06, with an odd one 0.97-1.03 / 0.94-0.99; from 4096 on two groups are the better ones
//   80, 96 columns   to 456 from 1700 on 1.01-1.13 / 0.97-1.13, of 1300 and 1500 tokens with an even number of heads 1.02-1.12 / 0.99-1.16, an odd
//                    one 0.97-1.02 / 0.96-0.97, of 1024 and 1100 0.89-1.06 / 0.91-1.03; to 480 from 2048 on 1.00-1.07 / 0.97-1.09; to 520
//                    from 2500 on 0.98-1.12 / 0.98-1.07, of 2048 0.98-1.00; to 576 (13/32 of the tiles) from 4096 on 1.03-1.09 / 1.02-
//                    1.09, below 0.81-1.04
//   128 columns      to 520 from 4096 on 1.01-1.13 / 0.97-1.13; to 576 1.02-1.07; below 4096 0.78-1.10
// At 32 columns 0.85-1.07 with no rule to it.  Padded heads and 48 columns have no such kernel.
inline int fwd_mixed_pairs(int dp, const FwdParams &p) {
  const int n = p.seqlen_q;
  const int64_t heads = (int64_t)p.batch * p.nheads, wgs = heads * ((n + kFwdBlockQ - 1) / kFwdBlockQ);
  if (wgs <= 3 * kCUs / 2 || wgs > 576 || !fwd_direct_ok(dp, p) || fwd_key_groups(dp, p) != 1) return 0;
  bool mixed = false;
  if (p.headdim == 64)
    mixed = n >= 1024 && n <= 3000 && wgs <= (n >= 1700 || heads % 2 == 0 ? 512 : 448);
  else if (p.headdim == 80 || p.headdim == 96)
    mixed = n >= (wgs > 520 ? 4096 : wgs > 480 ? 2500 : wgs > 456 ? 2048 : heads % 2 == 0 ? 1300 : 1700);
  else if (p.headdim == 128)
    mixed = n >= 4096;
  return mixed ? (n + 63) / 64 * (wgs <= 520 ? 12 : 13) / 32 : 0;
}
inline bool dq_direct_ok(int dp, const BwdParams &p) {
  return p.vec && direct_headdim_wide(dp, p.headdim) && direct_stride_ok(p.k) && direct_stride_ok(p.v);
}
inline int dq_key_groups(int dp, const BwdParams &p) {
  return dq_direct_ok(dp, p) ? key_groups(dp, direct_columns(dp, p.headdim), (int64_t)p.batch * p.nheads, p.seqlen_q, true) : 1;
}
inline bool dkdv_direct_ok(int dp, const BwdParams &p) {
  return p.vec && direct_headdim(dp, p.headdim) && dp != 96 && direct_stride_ok(p.q) && direct_stride_ok(p.d_o) &&
         direct_stride_ok(p.k) && direct_stride_ok(p.v);
}
// Where the paired dK/dV kernel (fa2_bwd_dkdv_pair.hpp) is the better one.  Its workgroups are half as long
// and start faster; its loop reads every Q and dO tile for 64 keys instead of 128.  Time of the other
// kernel over its own, bf16, (batch, head) pairs x tokens:
//   192, 256 columns  2.7 at 256, 1.5 at 192 (16 x 4096): always (the other one is the generic kernel)
//   96 columns        1.02 (4 x 16384) to 1.6 (4 x 4096), 1.05-1.07 on large grids: always (likewise)
//   128 columns       1.59 (1 x 16384), 1.24 (4 x 8192), 1.10 (4 x 12288) below 512 workgroups of 128 keys;
//                     above, 1.05 (64 x 2048), 1.02 (256 x 4096), 0.99 (16 x 4096), but 0.95 (8 x 8192) and
//                     0.98 (16 x 16384): there its extra tile loads cost board power, and clock
//   64 columns        1.56 (4 x 4096), 1.31 (64 x 512), 1.13 (4 x 16384) while the other kernel's workgroups
//                     are all resident (512); 1.16 (256 x 512), 1.09 (256 x 1024), 1.06 (64 x 2048) while
//                     they are short or few; 0.97 (256 x 2048), 0.93 (64 x 4096) beyond
//   48 columns        (heads of 40 and 48 in rows of 64; the other kernel multiplies all 64) 1.78 (4 x 4096), 1.19
//                     (4 x 16384) while that is resident; 1.04-1.06 to 1024 tokens (4096 x 640, 2048 x 1024); beyond them
//                     1.02-1.12 up to 2.75 x 2^21 rows times workgroups (96 x 2048, 20 x 5000, 80 x 3000), 0.99 at 3 x 2^21
//                     (48 x 4096, 12 x 8192), 0.95-1.03 above (32 x 8192, 16 x 8192).  40 columns within 3 % of that
//   32 columns        1.72 (4 x 4096), 1.28 (16 x 4096), 1.03 (1024 x 512); 0.96 (256 x 1024), 0.92 beyond;
//                     of 128 tokens and fewer 1.05 to 1.3, but 0.92-1.0 at 640 to 768 workgroups (8 us kernels)
inline bool dkdv_pair_ok(int dp, const BwdParams &p) {
  if (!(p.vec && direct_headdim_wide(dp, p.headdim) && direct_stride_ok(p.q) && direct_stride_ok(p.d_o) &&
        direct_stride_ok(p.k) && direct_stride_ok(p.v)))
    return false;
  // Twice the workgroups: not where only tiles of 128 keys make a grid that can be launched (more than 8.4
  // million heads).
  if ((int64_t)((p.seqlen_k + kDkvPairBlockKV - 1) / kDkvPairBlockKV) * p.batch * p.nheads > kMaxWorkgroups) return false;
  if (dp > 128 || dp == 96) return true;
  const int64_t wgs = (int64_t)((p.seqlen_k + kDkvBlockKV - 1) / kDkvBlockKV) * p.batch * p.nheads;
  if (dp == 128) return wgs < 2 * kCUs || p.seqlen_q <= 4096;
  if (direct_columns(dp, p.headdim) == 48) return wgs <= 2 * kCUs || p.seqlen_q <= 1024 || wgs * p.seqlen_q < 3 << 21;
  return wgs <= 2 * kCUs || p.seqlen_q <= 512 || (dp == 64 && wgs * p.seqlen_q <= (1 << 21));
}
// Key rows per workgroup of the dK/dV kernel that launch_dkdv picks (p.n_tiles follows from it).
inline int dkdv_block_kv(int dp, const BwdParams &p) { return dkdv_pair_ok(dp, p) ? kDkvPairBlockKV : kDkvBlockKV; }
// The sequence-parallel (atomic dQ) kernels: the fast dK/dV kernel's conditions, a head dimension
// of exactly 32, 64 or 128 and 16-byte aligned dq rows.
inline bool seqpar_atomic_ok(int dp, const BwdParams &p) {
  return dkdv_direct_ok(dp, p) && p.headdim == dp && (dp == 32 || dp == 64 || dp == 128);
}

// Whether the dK/dV kernel behind a dQ kernel starts with the last heads (from_the_end).  Time of a backward with the heads from the front
// over that from the end, bf16, in turn in one process: 128 heads and more of 300 to 2048 tokens 1.00-1.07 (4096 x 512 D=64 1.012-1.016,
// 640 x 1024 D=96 1.014-1.023, 2048 x 300 D=48 1.04-1.08, 512 x 1024 D=128 1.015-1.022), beyond 1.00-1.01; fewer 0.986-1.007, in the
// geometric mean 0.998, since the heads that dQ works on at its end are then most of them; but at 128 columns from 64 heads on 1.002-
// 1.013 (64 x 4096 1.012).
inline bool dkdv_from_the_end(int dp, int64_t heads) { return heads >= (dp == 128 ? 64 : 128); }
// The order of a joint grid, in runs of 8 workgroups that keep heads on their XCDs: every joint_period-th run is of dQ.  A
// workgroup of dQ has twice the rows of one of dK/dV, or with two key groups as many.
__host__ __device__ constexpr int joint_period(int key_groups) { return key_groups == 1 ? 3 : 2; }
constexpr int64_t joint_workgroups(int64_t n_dq, int64_t n_dkdv, int period) {
  const int64_t rounds_dq = (n_dq + 7) / 8, rounds_dkdv = (n_dkdv + 8 * (period - 1) - 1) / (8 * (period - 1));
  return (rounds_dq > rounds_dkdv ? rounds_dq : rounds_dkdv) * 8 * period;
}
// Whether dQ and dK/dV run in one grid (fa2_bwd_joint.hpp) behind a launch that forms delta, and with how many key groups dQ: 0 where
// two launches are as fast, dQ forming delta for dK/dV.  Time of the two launches over that of delta and the joint grid,
// bf16, in turn in one process (7700 sizes: profiles/joint_backward_sweep.txt), as the middle nine tenths of the sizes that the lines take (beside
// them of those they leave), by workgroups of 128 query rows; keys as many as queries:
//   columns    to 128       to 160              to 208              to 256              to 352              to 512
//   32         1.30-1.48    1.13-1.53           1.09-1.43           1.01-1.40           1.08-1.25 (1.01)    - (0.86-1.15)
//   48, 64     1.30-1.62    1.21-1.47           1.12-1.43           1.05-1.31           1.06-1.16 (1.00)    1.02-1.13 (0.85-1.13)
//   80, 96     1.29-1.60    1.20-1.46           1.05-1.38           1.01-1.20 (0.94)    1.04-1.18 (1.01)    1.04-1.15 (0.91-1.07)
//   112, 128   1.22-1.65    1.14-1.41           1.00-1.36           1.01-1.26 (0.93)    1.00-1.26           0.94-1.17 (0.87-1.09)
//   160-224    1.05-1.58    1.03-1.37 (0.99)    0.97-1.20 (0.97)    0.97-1.05 (0.93)    0.98-1.20           0.99-1.08 (0.91-1.06)
//   256        1.08-1.70    1.09-1.36           1.04-1.23           0.98-1.08 (0.96)    1.03-1.27           1.01-1.12 (0.95-1.13)
// Sequences of up to 128 or 256 tokens beside the lines 0.8-1.2.  To 128 workgroups dQ has the key groups it takes in front of a dK/dV kernel,
// beyond one: 64 rows to a workgroup would load K and V twice as often, and two groups are 0.75-1.0 of its rate there (up to 1.1 times at
// 32 to 64 columns and 129 to 512 tokens).  Beyond 512 workgroups two launches fill the chip as well, and what is gained is the end of the
// first: inside the lines 0.97-1.16, in the geometric mean 1.05; padded heads, numbers of heads that do not divide by 8, 32 and 160 columns,
// more than 2000 or 3000 workgroups 0.82-1.09, below 1.0 on the average.
// Unlike lengths, by keys over queries: to 512 workgroups 0.1 to 4 inside the lines 0.93-1.66, in the geometric mean 1.2, and with a fifth of
// the keys and fewer (512 tokens and more) 1.0-1.3 beside them as well; to 128 workgroups from 160 columns on 0.79-0.95 where short sequences
// have more keys (64 x 256, 1024 keys 0.79).  With many more keys most workgroups of dK/dV see no query, and the grid, whose order takes the
// lengths to be alike, is padded with ones of dQ that do not exist: 32 x 512 D=192, 4096 keys 0.69.
inline int joint_key_groups_by_size(int dp, const BwdParams &p) {
  if (!dq_direct_ok(dp, p) || !dkdv_pair_ok(dp, p)) return 0;
  const int64_t heads = (int64_t)p.batch * p.nheads, wgs = heads * ((p.seqlen_q + kDqBlockQ - 1) / kDqBlockQ);
  const int64_t n = p.seqlen_q, nk = p.seqlen_k;
  const int cols = direct_columns(dp, p.headdim);
  const bool wide = dp > 128, padded = p.headdim != cols;
  if (wgs > 2 * kCUs) {
    if (padded || (heads % 8 != 0 && wgs > 4 * kCUs)) return 0;
    if (wgs <= 4 * kCUs ? nk > 4 * n : wgs <= 2000 ? nk > 4 * n || 2 * nk < n : nk < n || nk > n + n / 4) return 0;
    if (dp == 64) return wgs <= 576 && n >= 1500 && heads % 8 == 0;
    if (dp == 96) return wgs <= 800 && n > 160 && n <= 1100;
    if (dp == 128) return n >= 128 && n <= 2048 && (n == 128 || wgs <= (n <= 400 || n >= 1100 ? 3000 : 2000));
    if (cols == 256) return n >= 96 && n <= 1100 && (n <= 128 || wgs <= (n <= 192 ? 640 : 2000));
    return cols >= 192 && n >= 96 && n <= 1100 && (n <= 128 || (n > 200 && (wgs <= 576 || (wgs > 1100 && wgs <= 2000))));
  }
  if (wgs <= kCUs / 2) {
    if (nk > (!wide || wgs <= 64 || n > 512 ? 4 : wgs <= 96 || n > 256 ? 2 : 1) * n) return 0;
    return n > 128 || wgs <= (wide ? 64 : 96) ? dq_key_groups(dp, p) : 0;
  }
  if (nk > 4 * n) return 0;
  if (n >= 512 && 5 * nk <= n) return 1;
  if (wgs <= kCUs) {
    if (n <= 256) return wgs <= 160 && n > (wide ? 255 : 128);
    if (dp == 96 || (dp == 128 && padded) || cols == 256) return wgs <= 208 || n > 512;
    return !wide || wgs <= 176 || (n > 512 && (wgs <= 208 || n <= 3100));
  }
  if (dp <= 64) return n >= 1500 && wgs <= (dp == 32 ? 336 : heads % 8 ? 400 : 512);
  if (!wide) return dp == 96 ? n >= 768 : n > 256;
  if (cols == 256) return n >= 96 && wgs <= 384;
  return wgs <= 352 ? n >= 96 : wgs <= 384 && n >= 3000;
}
// Whether such a grid can be launched, and the one that forms delta in front of it: a joint grid has up to three times the workgroups
// of its larger kind.  Where not, two launches run, each with a limit of its own.
inline bool joint_fits(const BwdParams &p, int key_groups) {
  const int64_t heads = (int64_t)p.batch * p.nheads;
  const int64_t n_dq = heads * ((p.seqlen_q + kDqBlockQ / key_groups - 1) / (kDqBlockQ / key_groups));
  const int64_t n_dkdv = heads * ((p.seqlen_k + kDkvPairBlockKV - 1) / kDkvPairBlockKV);
  return joint_workgroups(n_dq, n_dkdv, joint_period(key_groups)) <= kMaxWorkgroups &&
         heads * (((int64_t)p.seqlen_q_rounded + 15) / 16) <= INT_MAX;
}
inline int joint_key_groups(int dp, const BwdParams &p) {
  const int groups = joint_key_groups_by_size(dp, p);
  return groups > 0 && joint_fits(p, groups) ? groups : 0;
}
// The key groups of dQ in a call of these sizes, whatever part of the gradient is asked for: so a call for a part gives the bits of a
// call for all of it.  (dQ by itself would rather have two where the joint grid has one: 8 x 4096 D=128 58.3 us with two, 74.2 with
// one, 32 x 1024 D=256 41.3 and 42.6; the whole backward 132 in two launches and 116 in
// the joint grid, 91.8 and 85.1.)
inline int dq_key_groups_of_call(int dp, const BwdParams &p) {
  const int joint = joint_key_groups(dp, p);
  return joint > 0 ? joint : dq_key_groups(dp, p);
}
// Workgroup i's place in the order of its own kind (which may lie beyond the end of that).
struct JointPlace {
  bool dq;
  int index;
};
__host__ __device__ constexpr JointPlace joint_place(int i, int period) {
  const int run = i / 8, turn = run % period, round = run / period;
  const bool dq = turn == period - 1;
  return {dq, (dq ? round : round * (period - 1) + turn) * 8 + i % 8};
}

// Size of the head groups map_workgroup is given, for `heads` (batch, head) pairs and a table group
// size `group`: the heads are split into floor(heads / group) groups of (nearly) equal size, each a
// multiple of 8 so that a head stays on one XCD.  Equal groups, because a small last group would start
// its heaviest tiles late and finish them alone (96 heads as 64 + 32 cost 5 % against one group of 96);
// fewer than two table groups' worth of heads form a single group, walked heaviest tile first over
// the whole grid.
inline int equal_head_groups(int group, int64_t heads) {
  const int64_t n_groups = heads / group > 0 ? heads / group : 1;
  const int64_t per_group = (heads + n_groups - 1) / n_groups;
  return (int)((per_group + 7) / 8 * 8);
}
// Whether the balanced walk (balanced_index) may reorder a grid that fits the chip at once, and in which head groups;
// `group` is the table's.  The walk pairs rounds of the grid as if the whole of it were ordered heaviest tile first.  Over
// several head groups it is not, and heavy tiles came to lie beside heavy ones.  Sharing in L2 does not need the groups
// there, since all tiles run at once, so all heads form one.  Time in the groups over that in one, bf16, forward / dQ:
//   walked      1.27 (232 x 384, 32 columns), 1.17 / 1.08 (184 x 256, 64 columns), 1.08 / 1.01 (64 x 512, 128 columns)
//   in order    1.16 / 1.11 (136 x 700, 32 columns), 1.04 / 1.04 (184 x 512, 64 columns), 1.16 / 1.05 (64 x 512)
// One group of heads that are no multiple of 8 spreads a head's tiles over the XCDs.  Up to twice the table's group
// that still pays on the whole (dK/dV, walked in the groups over one group: 1.0-1.13 on 34 to 123 heads, but 0.91 at
// 59 x 384 and 0.89 at 55 x 512, 128 columns).  Beyond, it is 0.9 to 1.3 with no rule to it, and walking over the groups
// 0.91 to 1.09 of going in order: these grids run in their groups, in order.
struct ResidentWalk {
  bool balanced;
  int head_group;
};
inline ResidentWalk resident_walk(int group, int64_t heads) {
  return {heads % 8 == 0 || heads < 2 * group, (int)((heads + 7) / 8 * 8)};
}

// bf16 != 0 selects the bf16 kernels, otherwise fp16.
// p.folded: the LDS-direct forward takes its exponents straight from the score MFMAs (Q fragments
// multiplied by scale * log2(e) and rounded once); the generic forward ignores it.
// F32: the variants that store the output in fp32 (p.o_f32), each a specialisation defined in an object of its own.
template <bool F32>
void launch_fwd(bool bf16, int dp, const FwdParams &p, dim3 grid, hipStream_t s);
template <>
void launch_fwd<false>(bool bf16, int dp, const FwdParams &p, dim3 grid, hipStream_t s);
template <>
void launch_fwd<true>(bool bf16, int dp, const FwdParams &p, dim3 grid, hipStream_t s);
// The LDS-direct forward kernels of 160 to 256 columns (dp is 192 or 256), instantiated apart from the others.
template <bool F32>
void launch_fwd_direct_wide(bool bf16, int dp, int key_groups, const FwdParams &p, dim3 grid, dim3 block, hipStream_t s);
template <>
void launch_fwd_direct_wide<false>(bool bf16, int dp, int key_groups, const FwdParams &p, dim3 grid, dim3 block, hipStream_t s);
template <>
void launch_fwd_direct_wide<true>(bool bf16, int dp, int key_groups, const FwdParams &p, dim3 grid, dim3 block, hipStream_t s);
// Rounds fp32 arrays to fp16 (fa2_cast.hpp); one launch for all of them.
void launch_cast(const CastParams &p, dim3 grid, hipStream_t s);
void launch_preprocess(bool bf16, const PreParams &p, dim3 grid, hipStream_t s);
// delta with the bits of the fast dQ kernel's own, for rows of whole chunks (p.vec); p.n_tiles is not read.
void launch_delta(bool bf16, const PreParams &p, dim3 grid, hipStream_t s);
// fuse_delta: the fast dQ kernel also forms delta from O and dO (dq_direct_ok must hold).
void launch_dq(bool bf16, int dp, const BwdParams &p, int key_groups, dim3 grid, bool fuse_delta, hipStream_t s);
// With p.dq_accum set the sequence-parallel kernel runs: dK, dV and atomic dQ contributions.
void launch_dkdv(bool bf16, int dp, const BwdParams &p, dim3 grid, hipStream_t s);
// dQ (of p.dq_tiles tiles) and dK/dV in one grid of joint_workgroups, both reading delta; a specialisation for each type.
template <typename T>
void launch_joint(int dp, const JointParams &p, int key_groups, dim3 grid, hipStream_t s);
template <>
void launch_joint<__bf16>(int dp, const JointParams &p, int key_groups, dim3 grid, hipStream_t s);
template <>
void launch_joint<_Float16>(int dp, const JointParams &p, int key_groups, dim3 grid, hipStream_t s);
void launch_dq_accum_zero(float *acc, int64_t floats, hipStream_t s);
void launch_dq_accum_convert(bool bf16, const BwdParams &p, hipStream_t s);

}  // namespace fa2
