// Host-side (run on the CPU by tests/test_joint_backward.py): reads "heads seqlen_q seqlen_k seqlen_q_rounded headdim" per line and
// writes, for contiguous aligned tensors of one batch, the key groups of dQ in a call for it alone, those of a joint grid (0: two
// launches), that grid's workgroups, and the key groups of dQ in front of a dK/dV kernel.
#include <cstdio>

#include "fa2_common.hpp"
#include "fa2_launch.hpp"

int main() {
  fa2::BwdParams p = {};
  while (std::scanf("%d %d %d %d %d", &p.nheads, &p.seqlen_q, &p.seqlen_k, &p.seqlen_q_rounded, &p.headdim) == 5) {
    p.batch = p.vec = 1;
    for (fa2::Tensor4 *t : {&p.q, &p.k, &p.v, &p.o, &p.d_o, &p.dq, &p.dk, &p.dv}) t->stride_seq = p.headdim;
    int dp = 0;
    for (int row : {256, 192, 128, 96, 64, 32}) dp = p.headdim <= row ? row : dp;
    const int groups = fa2::joint_key_groups(dp, p);
    const long long heads = p.nheads, rows = groups > 0 ? fa2::kDqBlockQ / groups : 1;
    const long long n_dq = (p.seqlen_q + rows - 1) / rows * heads;
    const long long n_dkdv = (p.seqlen_k + fa2::kDkvPairBlockKV - 1ll) / fa2::kDkvPairBlockKV * heads;
    std::printf("%d %d %lld %d\n", fa2::dq_key_groups_of_call(dp, p), groups,
                groups > 0 ? (long long)fa2::joint_workgroups(n_dq, n_dkdv, fa2::joint_period(groups)) : 0ll, fa2::dq_key_groups(dp, p));
  }
}
