// Kernel parameter blocks and tile constants shared by the host-side C ABI and the device code.
#pragma once

#include <stdint.h>

namespace fa2 {

constexpr float kLog2e = 1.4426950408889634f;
constexpr float kLn2 = 0.6931471805599453f;

constexpr int kCUs = 256;  // compute units of an MI355X
// Workgroups of 256 threads a launch may have: the hardware is handed the grid in threads, as a 32-bit number, and
// of a larger grid only what is left modulo 2^32 runs, without an error.
constexpr long long kMaxWorkgroups = 0xffffffffll / 256;

// One (batch, nheads, seqlen, headdim) tensor: base pointer and strides in elements.
struct Tensor4 {
  void *ptr;
  int64_t stride_batch, stride_head, stride_seq;
};
// Row offsets inside a 64-row tile of the tensor fit 32 bits.
constexpr bool direct_stride_ok(const Tensor4 &t) { return t.stride_seq < (int64_t(1) << 24); }

// Every MFMA kernel runs 4 waves per workgroup, each wave owning 32 rows of the operand that stays
// in registers: 128 query rows (forward, dQ) or 128 key rows (dK/dV) per workgroup.
constexpr int kFwdWaves = 4;
constexpr int kFwdBlockQ = 32 * kFwdWaves;
constexpr int kDqWaves = 4;
constexpr int kDqBlockQ = 32 * kDqWaves;
constexpr int kDkvWaves = 4;
constexpr int kDkvBlockKV = 32 * kDkvWaves;
constexpr int kDkvPairBlockKV = 64;  // key rows per workgroup of the paired dK/dV kernel (two waves share 32)
// Its workgroups per CU: registers and LDS leave room for three up to 64 columns, two up to 128.
constexpr int dkdv_pair_wg_per_cu(int dp) { return dp <= 64 ? 3 : dp <= 128 ? 2 : 1; }
// Workgroups per CU of the forward with four key groups, whose tiles of 128 keys take 80 KiB of LDS at 64 columns and all 160 at 96
// and 128.
constexpr int fwd_quad_wg_per_cu(int dp) { return dp <= 32 ? 4 : dp <= 64 ? 2 : 1; }
// Rows of the streamed operand per LDS tile.
constexpr int kFwdBlockKV = 64;
constexpr int kDqBlockKV = 64;
constexpr int kDkvBlockQ = 64;

struct FwdParams {
  Tensor4 q, k, v, o;
  float *lse;
  int batch, nheads, seqlen_q, seqlen_k, headdim, seqlen_q_rounded;
  int n_qtiles;
  int head_group;  // (batch, head) pairs whose tiles are dispatched together (multiple of 8)
  int resident_grid;  // number of workgroups when all of them fit the chip at once, else 0: see balanced_index
  float scale;       // softmax scale (natural units)
  float scale_log2;  // scale * log2(e)
  int vec;           // 16-byte global accesses are legal for every tensor
  int mixed_singles;  // fwd_mixed_kernel: tiles of 64 rows per head that it takes as they are (else 0); n_qtiles counts all of them
  int folded;        // a row with fwd_exp_folded, for the host: see launch_fwd (fa2_launch.hpp)
  float *o_f32;      // contiguous fp32 tensor that receives the output widened, or null; o.ptr may be null beside it
};

struct BwdParams {
  Tensor4 q, k, v, d_o, dq, dk, dv;
  Tensor4 o;         // only read by the dQ kernel when it also forms delta
  float *delta_out;  // where that kernel writes delta (the same buffer `delta` points to)
  // Sequence-parallel mode only: fp32 (batch * nheads, dq_accum_rows, headdim) accumulator the
  // key-tile kernel adds its dQ contributions to; dq_accum_rows is seqlen_q rounded up to the
  // kernel's 64-row query tile.
  float *dq_accum;
  int dq_accum_rows;
  const float *lse;
  const float *delta;
  int batch, nheads, seqlen_q, seqlen_k, headdim, seqlen_q_rounded;
  int n_tiles;  // key tiles (dK/dV kernel) or query tiles (dQ kernel)
  int head_group;  // (batch, head) pairs whose tiles are dispatched together (multiple of 8)
  int resident_grid;  // number of workgroups when all of them fit the chip at once, else 0: see balanced_index
  float scale, scale_log2;
  int vec;
  bool grads_f32;  // dq, dk and dv are fp32 tensors (strides in fp32 elements)
  bool last_heads_first;  // the dK/dV kernel takes the heads from the end: see from_the_end
};

// dQ and dK/dV in one grid: n_tiles and resident_grid of `both` are dK/dV's and the whole grid's.  (One record for both: a
// second one, 340 bytes more to hand over, showed in the host time of a launch.)
struct JointParams {
  BwdParams both;
  int dq_tiles;      // query tiles per (batch, head) pair
  int n_dq, n_dkdv;  // workgroups of each
};

struct PreParams {
  Tensor4 o, d_o;
  float *delta;
  int batch, nheads, seqlen_q, headdim, seqlen_q_rounded;
  unsigned n_tiles;  // tiles of 16 rows over all (batch, head) pairs
  int vec;
};

// Arrays of fp32 numbers to round to fp16, at most kCastJobs in one launch.
constexpr int kCastJobs = 3;
constexpr int kCastThreads = 256, kCastBlock = 16 * kCastThreads;  // elements per workgroup
struct CastParams {
  const float *src[kCastJobs];
  void *dst[kCastJobs];
  int64_t n[kCastJobs];
  unsigned first[kCastJobs];  // first workgroup of an array
};

}  // namespace fa2
