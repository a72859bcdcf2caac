// dK/dV kernel with the two accumulators split over a pair of waves.
//
// In bwd_dkdv_direct_kernel a wave owns 32 keys and both of their accumulators.  Here two waves share the
// 32 keys: each forms S, P, dP and dS of one of the two 32-row blocks of a 64-row query tile, then one of
// them (role 0) accumulates dV over the whole tile, for which it needs the P of both blocks, and the other
// (role 1) dK, for which it needs the dS of both.  They hand each other the missing half (2 KiB per wave
// and tile) through LDS: role 0 gives its dS, role 1 its P, already packed to half precision in the
// register layout the receiver's MFMAs want, so an exchange is two 16-byte writes and two 16-byte reads
// per lane at the lane's own offset.  No product is formed twice, every output is still owned by one wave
// and accumulated in a fixed order.  A workgroup is two such pairs: 64 keys.
//
// Why: one accumulator per wave instead of two is what fits wide heads into the register file.  At 256
// columns K and V fragments take 128 registers and one accumulator another 128; both accumulators would
// need 384 before the first score.  The generic kernel covers 256 columns in two passes over the queries
// instead, forms S and dP twice and waits for its staging registers: B=2 H=8 N=4096 D=256, bf16,
// 756 -> 275 us (1000 TFLOP/s over the four products, 72 % of a large library matmul's rate on the same
// card); D=192 (in one pass) 337 -> 220 us.  What bounds it now: one wave per SIMD, whose exponentials,
// dS and exchange have only the wave's own MFMAs to hide under.  K and V fragments and the accumulator fill the
// accumulation registers (ResidentB in fa2_common.hpp); the loop copies nothing between the two halves of the register file
// (463 instructions for its 64 MFMAs at 256 columns).
//
// At 128 columns and below one accumulator per wave lets two (three at 64) workgroups share a CU, and
// workgroups of 64 keys fill the chip from fewer heads: dkdv_pair_ok (fa2_launch.hpp) says where that beats
// bwd_dkdv_direct_kernel and by how much.  The loop is the faster one per shader cycle (67 % of the matrix
// pipe's cycles busy against 60 % at 16 x 16384 tokens, D=128), but it moves twice the tile bytes, and on
// long sequences the board's power limit takes the clock down by what the cycles gained (1.69 GHz against
// 1.93).
//
// COLS (below): columns multiplied, as in the forward (fa2_fwd.hpp).
//
// The two roles are two instantiations of the loop selected once per wave.  With one loop and selects (or
// branches) on the role inside it the kernel was 2 to 5 % slower (or spilled).  The barriers of the two
// instantiations match one to one.
#pragma once

#include <type_traits>

#include "fa2_common.hpp"

namespace fa2 {

template <int DP>
struct DkvPairLayout {
  static constexpr int BQ = kDkvBlockQ, KEYS = kDkvPairBlockKV;
  static constexpr int LP = lds_pitch(DP);
  static constexpr int TILE_ELEMS = BQ * LP;
  static constexpr int STAGE_ELEMS = 2 * TILE_ELEMS;  // Q tile, dO tile
  static constexpr int STAGES = 2;
  // Per stage: lse * log2(e) and -delta of the tile's rows (floats, two shorts each).
  static constexpr int STAT_BASE = STAGES * STAGE_ELEMS;
  static constexpr int STAT_ELEMS = 4 * BQ;
  static constexpr int XCHG_BASE = STAT_BASE + STAGES * STAT_ELEMS;
  static constexpr int XCHG_WAVE = 2 * 64 * 8;  // two fragments of 16 bytes per lane
  // Two exchange buffers, used alternately, save a barrier per tile; at 96 and 128 columns the second one
  // would leave no room for two workgroups per CU.
  static constexpr int XBUFS = DP == 96 || DP == 128 ? 1 : 2;
  static constexpr int TOTAL_ELEMS = XCHG_BASE + XBUFS * kDkvWaves * XCHG_WAVE;
  static constexpr int PATCH_ELEMS = kDkvWaves * 32 * (DP + 8);
  static_assert(STAT_BASE >= PATCH_ELEMS, "the output patch overlays the stages");
};

// `place` gives the workgroup's place in the order of map_workgroup.
template <typename T, int DP, bool PAD, int role, int COLS, typename Place>
__device__ __forceinline__ void bwd_dkdv_pair(const BwdParams &p, short *smem, Place place) {
  using L = DkvPairLayout<DP>;
  constexpr int BQ = L::BQ, KS = COLS / 16, DB = (COLS + 31) / 32, R = 2 * DB, LP = L::LP;
  constexpr int NTHREADS = 64 * kDkvWaves;
  using Loader = TileLoader<DP, BQ, kDkvWaves, PAD>;
  constexpr int LOADS = Loader::LOADS;

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c = lane & 31, h = lane >> 5;
  const int i16 = lane & 15, g2 = (lane >> 4) & 1;

  const int BH = p.batch * p.nheads;
  int bh, kt;  // key tile 0 has the longest query range: rank == key tile
  map_workgroup(place(), BH, p.n_tiles, p.head_group, bh, kt);
  if (p.last_heads_first) bh = from_the_end(bh, BH);
  const int b = bh / p.nheads, hd = bh % p.nheads;
  const int kv0 = kt * L::KEYS;
  const int kv0w = kv0 + 32 * (wave >> 1);

  const short *Q = (const short *)p.q.ptr + b * p.q.stride_batch + hd * p.q.stride_head;
  const short *K = (const short *)p.k.ptr + b * p.k.stride_batch + hd * p.k.stride_head;
  const short *V = (const short *)p.v.ptr + b * p.v.stride_batch + hd * p.v.stride_head;
  const short *DO = (const short *)p.d_o.ptr + b * p.d_o.stride_batch + hd * p.d_o.stride_head;
  const float *LSE = p.lse + (int64_t)bh * p.seqlen_q_rounded;
  const float *DELTA = p.delta + (int64_t)bh * p.seqlen_q_rounded;

  const int hdim = PAD ? p.headdim : COLS;
  const Loader qload(uniform_ptr(Q), (int64_t)uniform64((uint64_t)p.q.stride_seq), hdim / 8),
      gload(uniform_ptr(DO), (int64_t)uniform64((uint64_t)p.d_o.stride_seq), hdim / 8);
  const int seqlen_q = p.seqlen_q;
  const float scale_log2 = p.scale_log2;

  const int q_begin = kv0;  // first query tile that can see these keys (kv0 is a multiple of BQ)
  const int n_tiles = (seqlen_q > q_begin) ? (seqlen_q - q_begin + BQ - 1) / BQ : 0;
  // Tiles are taken from the end of the sequence towards the diagonal: the workgroups of a head that run
  // at the same time then read the same Q and dO tiles at the same time, whatever their keys.
  const int q_top = q_begin + (n_tiles - 1) * BQ;         // first row of tile 0
  const bool ragged = n_tiles > 0 && q_top + BQ > seqlen_q;  // tile 0 holds rows beyond the sequence

  const unsigned lds_base = lds_u32(smem);
  if (PAD) {
    zero_lds<NTHREADS>(smem, L::STAT_BASE);
    __syncthreads();
  }
  auto issue_tile = [&](int t) {
    const unsigned dst = lds_base + 2u * (unsigned)((t & 1) * L::STAGE_ELEMS);
    const int row0 = q_top - t * BQ;
    if (t > 0 || !ragged) {
      qload.issue(row0, dst);
      gload.issue(row0, dst + 2u * L::TILE_ELEMS);
    } else {
      qload.issue_clamped(row0, seqlen_q, dst);
      gload.issue_clamped(row0, seqlen_q, dst + 2u * L::TILE_ELEMS);
    }
  };
  // lse and delta pass through registers a tile ahead, as in bwd_dkdv_direct_kernel.  (Rows clamped to
  // the sequence: the row mask zeroes what lies beyond.)
  float lse_reg = 0.f, delta_reg = 0.f;
  auto load_stats = [&](int t) {
    if (tid < BQ) {
      const int row = max(min(q_top - t * BQ + tid, seqlen_q - 1), 0);
      lse_reg = LSE[row];
      delta_reg = DELTA[row];
    }
  };
  auto store_stats = [&](int t) {
    float *sl = reinterpret_cast<float *>(smem + L::STAT_BASE + (t & 1) * L::STAT_ELEMS);
    if (tid < BQ) {
      sl[tid] = lse_reg * kLog2e;
      sl[BQ + tid] = -delta_reg;  // negated: it is the accumulator the dP MFMAs start from
    }
  };

  // Tile 0 into stage 0; the workgroup's K and V rows on their way into registers through stage 1.
  constexpr unsigned K_AT = 2u * (unsigned)L::STAGE_ELEMS, V_AT = K_AT + 2u * (unsigned)L::TILE_ELEMS;
  {
    const Loader kload(K + (int64_t)kv0 * p.k.stride_seq, p.k.stride_seq, hdim / 8),
        vload(V + (int64_t)kv0 * p.v.stride_seq, p.v.stride_seq, hdim / 8);
    const int k_rows = p.seqlen_k - kv0;  // key rows of this tile that exist (>= 1)
    if (n_tiles > 0) issue_tile(0);
    if (k_rows >= BQ) kload.issue(0, lds_base + K_AT); else kload.issue_clamped(0, k_rows, lds_base + K_AT);
    if (k_rows >= BQ) vload.issue(0, lds_base + V_AT); else vload.issue_clamped(0, k_rows, lds_base + V_AT);
  }
  load_stats(0);
  const float l0 = lse_reg, d0 = delta_reg;
  load_stats(1);

  // Swizzled fragment addresses.  qrow: rows of this wave's query block in the Q tile of the stage read
  // next (the dO tile sits TILE_ELEMS behind); tlo, thi: transposed fragments of the tile this wave
  // contracts with (dO for role 0, Q for role 1), the wave's own block first.
  const lds_cptr lds0 = to_lds(smem);
  constexpr int NK = kept_addresses(LP, KS, 2), ND = kept_addresses(LP, DB, 4);
  lds_cptr qrow[NK], tlo[ND], thi[ND];
#pragma unroll
  for (int ks = 0; ks < NK; ks++) qrow[ks] = lds0 + role * 32 * LP + swz_off<LP>(c, 2 * ks + h);
  {
    const int rowlo = 4 * h + (i16 >> 2);
    const int sub = (i16 & 1) * 4;
    const lds_cptr t0 = lds0 + (role ? 32 * LP : L::TILE_ELEMS);
#pragma unroll
    for (int db = 0; db < ND; db++) {
      const int chunk = 4 * db + 2 * g2 + ((i16 & 3) >> 1);
      tlo[db] = t0 + swz_off<LP>(rowlo, chunk) + sub;
      thi[db] = t0 + swz_off<LP>(rowlo + 8, chunk) + sub;
    }
  }
  constexpr int other_block = role ? -32 * LP : 32 * LP;  // from the own block to the partner's
  typedef const __attribute__((address_space(3))) float *stat_ptr;
  typedef const __attribute__((address_space(3))) f32x4 *stat4_ptr;
  stat_ptr stat = reinterpret_cast<stat_ptr>(lds0 + L::STAT_BASE) + 32 * role + 4 * h;
  // Exchange areas of the pair, role 0's and then role 1's, both at constant offsets from one address.  (With an
  // address for each the padded kernel at 256 columns was one register short: 20 bytes of scratch per lane.)
  short *xchg = smem + L::XCHG_BASE + (wave & ~1) * L::XCHG_WAVE + 8 * lane;
  constexpr int XPUT = role * L::XCHG_WAVE, XGET = (1 - role) * L::XCHG_WAVE;

  f32x16 acc[DB];
#pragma unroll
  for (int db = 0; db < DB; db++)
#pragma unroll
    for (int i = 0; i < 16; i++) acc[db][i] = 0.f;
  // Element i of a block that starts at query row qb is row qb + 4h + 8 (i / 4) + i % 4; it is kept
  // when key column <= row < seqlen_q, tested as one unsigned compare: (row - column) < (seqlen_q - column).
  const int kvcol = kv0w + c;
  const int row_shift = 4 * h - kvcol;
  const unsigned row_span = (unsigned)max(seqlen_q - kvcol, 0);

  {
    const float l1 = lse_reg, d1 = delta_reg;
    lse_reg = l0;
    delta_reg = d0;
    store_stats(0);
    lse_reg = l1;
    delta_reg = d1;
    store_stats(1);
  }
  wait_vmem_all();
  __syncthreads();
  // B operands: lane (c, h) holds row kv0w + c of K and of V, columns 16 ks + 8 h + j.
  s16x8 kf[KS], vf[KS];
  {
    const int r = 32 * (wave >> 1) + c;
#pragma unroll
    for (int ks = 0; ks < KS; ks++) {
      kf[ks] = lds_read_128(lds0 + (int)(K_AT / 2) + swz_off<LP>(r, 2 * ks + h));
      vf[ks] = lds_read_128(lds0 + (int)(V_AT / 2) + swz_off<LP>(r, 2 * ks + h));
    }
  }
  s16x8 ring[R];
#pragma unroll
  for (int ks = 0; ks < KS; ks++) ring[ks] = lds_read_128(qrow[ks % NK] + ks / NK * 128);
  // Every wave has its K and V fragments: stage 1 is free for its tile.
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  __syncthreads();
  if (n_tiles > 1) issue_tile(1);

  auto t_frag = [&](int f, int block) -> s16x8 {
    s16x4 a0 = lds_read_tr(tlo[f % DB % ND] + f % DB / ND * 128 + block + 16 * (f / DB) * LP);
    s16x4 a1 = lds_read_tr(thi[f % DB % ND] + f % DB / ND * 128 + block + 16 * (f / DB) * LP);
    return __builtin_shufflevector(a0, a1, 0, 1, 2, 3, 4, 5, 6, 7);
  };

  constexpr bool WIDE = DP > 128;  // one wave per SIMD: ResidentB
  // One 64-row query tile.  One barrier in its middle (two with a single exchange buffer):
  //     A: S = Q K^T of the own block         ring <- dO rows
  //     B: dP = dO V^T                        ring <- transposed fragments, own block; exponentials
  //     C: acc += own block                   ring <- transposed fragments, partner's block
  //        dS; what the partner needs goes to the exchange buffer
  //     -- barrier: both halves are in the exchange buffer, nobody reads this stage any more and the
  //        next tile has landed in the other one
  //     D: acc += partner's block             ring <- Q rows of the next tile; loads of tile t + 2
  auto tile = [&](int t, auto masked_tag, auto spread_tag) __attribute__((always_inline)) {
    constexpr bool MASKED = decltype(masked_tag)::value;
    constexpr bool SPREAD = decltype(spread_tag)::value;
    const int dstage = (t & 1) ? -L::STAGE_ELEMS : L::STAGE_ELEMS;
    f32x16 s, dp;
    f32x4 l4[4], d4[4];
#pragma unroll
    for (int i = 0; i < 16 && !WIDE; i++) s[i] = 0.f;
#pragma unroll
    for (int ks = 0; ks < KS; ks++) {
      if constexpr (WIDE) {
        if (ks == 0) ResidentB<T>::zero(s, ring[ks], kf[ks]);
        else if (SPREAD) ResidentB<T>::next_loaded(s, ring[ks], kf[ks]);
        else ResidentB<T>::next(s, ring[ks], kf[ks]);
      } else {
        s = Elem<T>::mfma(ring[ks], kf[ks], s);
      }
      ring[ks] = lds_read_128(qrow[ks % NK] + ks / NK * 128 + L::TILE_ELEMS);
#pragma unroll
      for (int g = part(4, KS, ks); g < part(4, KS, ks + 1); g++) {
        l4[g] = *reinterpret_cast<stat4_ptr>(stat + 8 * g);
        d4[g] = *reinterpret_cast<stat4_ptr>(stat + BQ + 8 * g);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    const int rel = q_top - t * BQ + 32 * role + row_shift;
    // The chain starts from -delta, so that dS = P * dP needs no subtraction.
    dp = __builtin_shufflevector(__builtin_shufflevector(d4[0], d4[1], 0, 1, 2, 3, 4, 5, 6, 7),
                                 __builtin_shufflevector(d4[2], d4[3], 0, 1, 2, 3, 4, 5, 6, 7), 0, 1, 2, 3, 4, 5,
                                 6, 7, 8, 9, 10, 11, 12, 13, 14, 15);
#pragma unroll
    for (int ks = 0; ks < KS; ks++) {
      if constexpr (WIDE) {
        if (SPREAD && ks > 0) ResidentB<T>::next_loaded(dp, ring[ks], vf[ks]);
        else ResidentB<T>::next(dp, ring[ks], vf[ks]);
      } else {
        dp = Elem<T>::mfma(ring[ks], vf[ks], dp);
      }
      ring[ks] = t_frag(ks, 0);
      if (KS < R && ks == 0) ring[R - 1] = t_frag(R - 1, 0);  // the slot no dO row was in
      if (WIDE && ks == 0) chain_end(s);
#pragma unroll
      for (int i = part(16, KS, ks); i < part(16, KS, ks + 1); i++) {
        float x = fast_exp2(s[i] * scale_log2 - l4[i >> 2][i & 3]);
        if (MASKED && (unsigned)(rel + (8 * (i >> 2) + (i & 3))) >= row_span) x = 0.f;
        s[i] = x;  // P takes the place of S
      }
      asm volatile("" : "+v"(s));
      __builtin_amdgcn_sched_barrier(0);
    }
    if (WIDE && role == 1) chain_end(dp);  // (role 0 takes dP up behind the first MFMA of its accumulator)
    // The own block is consumed; the row pointers move on to the next tile.
#pragma unroll
    for (int ks = 0; ks < NK; ks++) qrow[ks] += dstage;
    const s16x8 pf[2] = {Elem<T>::pack8(f32x8{s[0], s[1], s[2], s[3], s[4], s[5], s[6], s[7]}),
                         Elem<T>::pack8(f32x8{s[8], s[9], s[10], s[11], s[12], s[13], s[14], s[15]})};
    const int xoff = L::XBUFS == 2 ? (t & 1) * kDkvWaves * L::XCHG_WAVE : 0;
    // The partner has taken what it was given for the tile before.
    if (L::XBUFS == 1) tile_barrier();
    auto give = [&](const s16x8 (&x)[2]) {
      *reinterpret_cast<s16x8 *>(xchg + xoff + XPUT) = x[0];
      *reinterpret_cast<s16x8 *>(xchg + xoff + XPUT + 64 * 8) = x[1];
    };
    s16x8 df[2];
    auto pack_ds = [&]() {
      df[0] = Elem<T>::pack8(f32x8{dp[0], dp[1], dp[2], dp[3], dp[4], dp[5], dp[6], dp[7]});
      df[1] = Elem<T>::pack8(f32x8{dp[8], dp[9], dp[10], dp[11], dp[12], dp[13], dp[14], dp[15]});
    };
    // Role 0 has its P and forms dS beside the MFMAs; role 1 needs dS first.
    if (role == 1) {
      give(pf);
#pragma unroll
      for (int i = 0; i < 16; i++) dp[i] = s[i] * dp[i];
      pack_ds();
    }
#pragma unroll
    for (int f = 0; f < R; f++) {
      acc[f % DB] = Elem<T>::mfma(ring[f], role ? df[f / DB] : pf[f / DB], acc[f % DB]);
      ring[f] = t_frag(f, other_block);
      if (WIDE && role == 0 && f == 0) chain_end(dp);
      if (role == 0) {
#pragma unroll
        for (int i = part(16, R, f); i < part(16, R, f + 1); i++) dp[i] = s[i] * dp[i];
        asm volatile("" : "+v"(dp));
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    if (role == 0) {
      pack_ds();
      give(df);
    }
    if (t >= 1 && t + 1 < n_tiles) store_stats(t + 1);
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
    tile_barrier();
    const s16x8 got[2] = {*reinterpret_cast<const s16x8 *>(xchg + xoff + XGET),
                          *reinterpret_cast<const s16x8 *>(xchg + xoff + XGET + 64 * 8)};
    if (t + 2 < n_tiles) {
      load_stats(t + 2);
      if (!SPREAD) issue_tile(t + 2);
    }
    const unsigned ldst = lds_base + 2u * (unsigned)((t & 1) * L::STAGE_ELEMS);
    const int lrow0 = q_top - (t + 2) * BQ;
#pragma unroll
    for (int f = 0; f < R; f++) {
      acc[f % DB] = Elem<T>::mfma(ring[f], got[f / DB], acc[f % DB]);
      if (f < KS) ring[f] = lds_read_128(qrow[f % NK] + f / NK * 128);
      if (SPREAD) {
#pragma unroll
        for (int i = part(2 * LOADS, R, f); i < part(2 * LOADS, R, f + 1); i++) {
          if (i < LOADS) qload.issue_one(lrow0, ldst, i);
          else gload.issue_one(lrow0, ldst + 2u * L::TILE_ELEMS, i - LOADS);
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int db = 0; db < ND; db++) {
      tlo[db] += dstage;
      thi[db] += dstage;
    }
    stat += (t & 1) ? -(L::STAT_ELEMS / 2) : L::STAT_ELEMS / 2;
  };

  // Rows beyond the sequence lie in the first tile, the diagonal in the last.
  int t = 0;
  if (ragged || n_tiles == 1) tile(t++, std::true_type{}, std::false_type{});
  for (; t < n_tiles - 2; t++) tile(t, std::false_type{}, std::true_type{});
  for (; t < n_tiles - 1; t++) tile(t, std::false_type{}, std::false_type{});
  for (; t < n_tiles; t++) tile(t, std::true_type{}, std::false_type{});

  // The patch overlays the stages; reads of them that are still in flight fetch values nobody uses.
  const Tensor4 &out = role ? p.dk : p.dv;
  __syncthreads();
  short *patch = smem + wave * 32 * (DP + 8);
  store_transposed_acc<T, COLS, true>(acc, role ? p.scale : 1.0f, patch, grad_rows(p, out, b, hd, kv0w), out.stride_seq,
                              p.seqlen_k - kv0w, hdim, true, p.grads_f32);
}

template <typename T, int DP, bool PAD, int COLS = DP>
__global__ __launch_bounds__(64 * kDkvWaves, (dkdv_pair_wg_per_cu(DP))) void bwd_dkdv_pair_kernel(const BwdParams p) {
  __shared__ __attribute__((aligned(1024))) short smem[DkvPairLayout<DP>::TOTAL_ELEMS];
  const auto place = [&]() -> int { return p.resident_grid ? balanced_index(blockIdx.x, p.resident_grid) : blockIdx.x; };
  if (__builtin_amdgcn_readfirstlane(threadIdx.x >> 6) & 1)
    bwd_dkdv_pair<T, DP, PAD, 1, COLS>(p, smem, place);
  else
    bwd_dkdv_pair<T, DP, PAD, 0, COLS>(p, smem, place);
}

}  // namespace fa2
