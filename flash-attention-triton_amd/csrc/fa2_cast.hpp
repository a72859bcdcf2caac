// fp32 arrays rounded to fp16: what q, k and v (in one launch) and dO of an fp32 model pass through in front of the
// attention kernels.  Memory bound: 6.7 TB/s on 32 x 20 x 1024 x 96 (four tensors in 226 us, 378 MB each; a device copy
// reaches 4.9).  Four loads per thread before its first store keep enough in flight; they go past the caches, which
// the rounded values should have.
#pragma once

#include "fa2_common.hpp"

namespace fa2 {

// A workgroup rounds kCastBlock consecutive elements; a thread's four 16-byte loads are in flight together.
__global__ __launch_bounds__(kCastThreads) void cast_f16_kernel(const CastParams p) {
  const unsigned wg = blockIdx.x;
  const int job = wg >= p.first[2] ? 2 : wg >= p.first[1] ? 1 : 0;
  const int64_t n = p.n[job];
  const int64_t at = (int64_t)(wg - p.first[job]) * kCastBlock;
  const float *src = p.src[job] + at;
  _Float16 *dst = (_Float16 *)p.dst[job] + at;
  const int left = (int)min(n - at, (int64_t)kCastBlock);  // elements of this workgroup, at least one
  constexpr int VECS = kCastBlock / (4 * kCastThreads);
  if (left == kCastBlock) {
    f32x4 x[VECS];
#pragma unroll
    for (int i = 0; i < VECS; i++)
      x[i] = __builtin_nontemporal_load(reinterpret_cast<const f32x4 *>(src + 4 * (threadIdx.x + i * kCastThreads)));
#pragma unroll
    for (int i = 0; i < VECS; i++)
      *reinterpret_cast<s16x4 *>(dst + 4 * (threadIdx.x + i * kCastThreads)) = Elem<_Float16>::pack4(x[i]);
    return;
  }
  for (int i = threadIdx.x; i < left; i += kCastThreads) dst[i] = (_Float16)src[i];
}

}  // namespace fa2
