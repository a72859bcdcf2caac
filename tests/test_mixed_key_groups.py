"""One and two key groups in one forward grid (fwd_mixed_kernel in csrc/fa2_fwd.hpp): the order of its tiles and what the compiler
made of the kernel, on the CPU, and results at the edges of the rule that picks it (fwd_mixed_pairs in csrc/fa2_launch.hpp)."""

from __future__ import annotations

import math
import pathlib
import re
import subprocess

import pytest
import torch

from tests.test_code_objects import LDS_PER_CU, REGS_PER_LANE, records  # noqa: F401

ROOT = pathlib.Path(__file__).resolve().parent.parent
HIPCC = pathlib.Path("/opt/rocm/bin/hipcc")

ORDER = """
#include <algorithm>
#include <cstdio>
#include <vector>
#include "fa2_launch.hpp"
int main() {
  for (int tiles = 3; tiles < 300; tiles++)
    for (int pairs = 1; 2 * pairs < tiles; pairs++) {
      const int singles = tiles - 2 * pairs;
      std::vector<int> rows(tiles, 0);
      int next_single = 0, next_pair = 0;
      for (int pos = 0; pos < singles + pairs; pos++) {
        const fa2::MixedPlace at = fa2::mixed_place(pos, tiles, singles);
        int &next = at.single ? next_single : next_pair;
        if (at.rank != next++ || at.rank >= (at.single ? singles : pairs))
          return std::printf("%d tiles, %d pairs: place %d is %d of %d\\n", tiles, pairs, pos, at.rank, at.single), 1;
        if (at.single) rows[tiles - 1 - at.rank]++;
        else rows[2 * (pairs - 1 - at.rank)]++, rows[2 * (pairs - 1 - at.rank) + 1]++;
      }
      if (std::count(rows.begin(), rows.end(), 1) != tiles) return std::printf("%d tiles, %d pairs: not every row once\\n", tiles, pairs), 1;
    }
  // Whatever the rule picks leaves tiles of both kinds.
  int picked = 0;
  for (int d : {32, 48, 64, 72, 80, 96, 112, 128, 160})
    for (int heads = 1; heads < 140; heads++)
      for (int n = 1; n < 20000; n += 37) {
        fa2::FwdParams p = {};
        p.batch = 1, p.nheads = heads, p.seqlen_q = p.seqlen_k = n, p.headdim = d, p.vec = 1;
        p.q.stride_seq = p.k.stride_seq = p.v.stride_seq = d;
        const int dp = d <= 32 ? 32 : d <= 64 ? 64 : d <= 96 ? 96 : d <= 128 ? 128 : 192;
        const int pairs = fa2::fwd_mixed_pairs(dp, p);
        if (pairs == 0) continue;
        picked++;
        if (2 * pairs >= (n + 63) / 64 || (d != 64 && d != 80 && d != 96 && d != 128)) return std::printf("%d x %d, %d: %d pairs\\n", heads, n, d, pairs), 1;
      }
  if (picked == 0) return std::printf("never picked\\n"), 1;
  std::printf("ok\\n");
}
"""


def test_every_row_once_and_longest_first(tmp_path):
    if not HIPCC.exists():
        pytest.skip("hipcc not installed")
    src, exe = tmp_path / "order.hip", tmp_path / "order"
    src.write_text(ORDER.replace('#include "fa2_launch.hpp"', '#include "fa2_common.hpp"\n#include "fa2_launch.hpp"'))
    build = subprocess.run([str(HIPCC), "-x", "hip", "--cuda-host-only", "-O1", "-std=c++17", "-Wno-unused-command-line-argument",
                            f"-I{ROOT / 'flash-attention-triton_amd' / 'csrc'}", f"-I{ROOT / 'include'}", "-o", str(exe), str(src)],
                           capture_output=True, text=True, timeout=300)
    assert build.returncode == 0, build.stderr[-2000:]
    run = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert run.returncode == 0 and run.stdout == "ok\n", run.stdout + run.stderr


@pytest.mark.parametrize("heads,n,d,mixed", [
    (54, 1024, 64, True), (64, 1024, 64, True), (57, 1024, 64, False), (33, 1300, 64, False), (41, 1500, 64, False), (35, 1700, 64, True), (29, 2048, 64, True),
    (36, 1300, 80, True), (38, 1500, 96, True), (39, 1300, 80, False), (33, 1500, 96, False), (57, 1024, 80, False), (50, 1024, 96, False), (32, 1700, 96, True),
    (34, 1700, 80, False), (29, 2048, 80, True), (32, 2048, 96, False), (26, 2500, 80, True), (16, 4096, 96, True), (18, 4096, 80, True), (18, 4000, 80, False),
    (16, 4096, 128, True), (16, 4095, 128, False), (20, 3000, 128, False), (16, 4096, 104, False), (40, 1300, 48, False)])
def test_mixed_only_where_it_measured_faster(heads, n, d, mixed):
    """Both sides of the lines of fwd_mixed_pairs."""
    import importlib

    capi = importlib.import_module("flash-attention-triton_amd._capi")
    assert (capi.launch_info(1, heads, n, n, d)["fwd"]["form"] == "mixed") == mixed


def test_mixed_kernels_share_a_cu_like_their_parts(records):  # noqa: F811
    seen = set()
    for r in records:
        m = re.match(r"_ZN3fa216fwd_mixed_kernelI(DF16b|DF16_)Li(\d+)ELb([01])ELb([01])ELi(\d+)E", r["name"])
        if not m:
            continue
        dp, cols = int(m.group(2)), int(m.group(5))
        seen.add((m.group(1), dp, int(m.group(3)), int(m.group(4)), cols))
        waves = REGS_PER_LANE // ((int(r["vgpr_count"]) + 7) // 8 * 8)
        assert min(waves, LDS_PER_CU // int(r["group_segment_fixed_size"])) >= (3 if dp == 64 else 2), r["name"]
        assert int(r["private_segment_fixed_size"]) == 0, r["name"]
    assert seen == {(t, dp, pre, f32, cols) for t in ("DF16b", "DF16_") for pre in (0, 1) for f32 in (0, 1)
                    for dp, cols in ((64, 64), (96, 80), (96, 96), (128, 128))}


# bf16 rounds P to 8 bits (half a unit 2^-9 = 2.0e-3) and O likewise; fp16 2^-12 = 2.4e-4: of a row's largest probabilities the
# errors average, so the relative 2-norm stays below one unit, 4e-3 and 5e-4.  The folded forward rounds Q once more.
REL = {torch.bfloat16: 4e-3, torch.float16: 5e-4, torch.float32: 2e-3}


@pytest.mark.gpu
@pytest.mark.parametrize("heads,nq,nk,d,dtype", [
    (43, 1025, 1025, 64, torch.bfloat16), (64, 1024, 900, 64, torch.float16), (17, 2999, 3100, 64, torch.bfloat16),
    (49, 1024, 1024, 80, torch.float16), (10, 5001, 5001, 80, torch.bfloat16), (25, 2100, 700, 96, torch.bfloat16),
    (32, 2048, 2048, 96, torch.float32), (12, 6000, 64, 80, torch.bfloat16), (17, 4097, 4097, 96, torch.float16), (36, 1300, 1300, 80, torch.bfloat16), (26, 2500, 2500, 96, torch.float32),
    (12, 4097, 4000, 128, torch.bfloat16), (16, 4500, 4500, 128, torch.float16), (1, 65000, 130, 128, torch.bfloat16)],
    ids=lambda x: str(x).replace("torch.", ""))
@pytest.mark.parametrize("grad", (False, True))
def test_forward_matches_the_oracle(heads, nq, nk, d, dtype, grad):
    import flash_attention_triton_amd as fa

    gen = torch.Generator(device="cuda").manual_seed(nq)
    q, k, v = (torch.randn((1, heads, n, d), generator=gen, device="cuda").to(dtype) for n in (nq, nk, nk))
    q.requires_grad_(grad)
    with torch.set_grad_enabled(grad):
        out = fa.flash_attention_v2(q, k, v).detach()
    # Rows at the ends of the sequence and around the line between the two kinds, of the first and the last head.
    tiles = (nq + 63) // 64
    line = 64 * 2 * (tiles * 12 // 32)
    rows = torch.tensor(sorted({r for at in (0, nq // 2, line, 64 * 2 * (tiles * 13 // 32), nq - 80) for r in range(max(at - 40, 0), min(at + 90, nq))}),
                        device="cuda")
    for hd in (0, heads - 1):
        s = (q[0, hd, rows].detach().double() @ k[0, hd].double().T) / math.sqrt(d)
        s.masked_fill_(torch.arange(nk, device="cuda")[None] > rows[:, None], -math.inf)
        want = torch.softmax(s, -1) @ v[0, hd].double()
        err = (out[0, hd, rows].double() - want).norm() / want.norm()
        assert err < REL[dtype] * (1.5 if not grad else 1), (hd, err.item())
