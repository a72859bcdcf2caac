// Host-side check (run on the CPU by tests/test_joint_backward.py) of the order of a joint grid of dQ and dK/dV workgroups:
// each of either kind exactly once, behind balanced_index where the grid is resident, and no more workgroups than a round
// beyond those.
#include <cstdio>
#include <vector>

#include "fa2_common.hpp"
#include "fa2_launch.hpp"

int main() {
  int bad = 0;
  for (int groups = 1; groups <= 2; groups++) {
    const int period = fa2::joint_period(groups);
    for (int n_dq = 1; n_dq < 420; n_dq += 1 + n_dq / 16)
      for (int n_dkdv = 1; n_dkdv < 900; n_dkdv += 1 + n_dkdv / 16)
        for (int balanced = 0; balanced < 2; balanced++) {
          const int total = (int)fa2::joint_workgroups(n_dq, n_dkdv, period);
          std::vector<int> dq(n_dq, 0), dkdv(n_dkdv, 0);
          for (int i = 0; i < total; i++) {
            const fa2::JointPlace at = fa2::joint_place(balanced ? fa2::balanced_index(i, total) : i, period);
            if (at.index < 0) bad++;
            if (at.dq && at.index < n_dq) dq[at.index]++;
            if (!at.dq && at.index < n_dkdv) dkdv[at.index]++;
          }
          for (int x : dq) bad += x != 1;
          for (int x : dkdv) bad += x != 1;
          bad += total % (8 * period) != 0;
          const int smaller = total - 8 * period;  // one round less would not do
          bad += smaller / period >= n_dq && smaller / period * (period - 1) >= n_dkdv;
        }
  }
  std::printf("joint grid %s\n", bad ? "BAD" : "ok");
  return bad != 0;
}
