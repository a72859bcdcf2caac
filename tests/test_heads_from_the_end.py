"""The order of heads that the dK/dV kernel takes behind the dQ kernel (from_the_end in csrc/fa2_common.hpp): every head once, and from the
end only where there are many."""

from __future__ import annotations

import pathlib
import subprocess

import pytest

ROOT = pathlib.Path(__file__).resolve().parent.parent
HIPCC = pathlib.Path("/opt/rocm/bin/hipcc")

SOURCE = """
#include <cstdio>
#include <vector>
#include "fa2_common.hpp"
#include "fa2_launch.hpp"
int main() {
  for (int dp : {32, 64, 96, 128, 192, 256})
    for (int heads : {1, 16, 63, 64, 127, 128, 4096})
      if (fa2::dkdv_from_the_end(dp, heads) != (heads >= (dp == 128 ? 64 : 128))) return std::printf("%d columns, %d heads\\n", dp, heads), 1;
  for (int heads : {1, 2, 7, 8, 9, 16, 17, 24, 640, 641, 4096}) {
    std::vector<int> seen(heads, 0);
    for (int i = 0; i < heads; i++) {
      const int bh = fa2::from_the_end(i, heads);
      if (bh < 0 || bh >= heads || seen[bh]++) return std::printf("heads %d: %d -> %d\\n", heads, i, bh), 1;
      if (heads % 8 == 0 && bh % 8 != i % 8) return std::printf("heads %d: %d leaves its XCD\\n", heads, i), 1;
    }
    if (fa2::from_the_end(0, heads) < heads - 8) return std::printf("heads %d: starts early\\n", heads), 1;
  }
  std::printf("ok\\n");
}
"""


def test_every_head_once(tmp_path):
    if not HIPCC.exists():
        pytest.skip("hipcc not installed")
    src, exe = tmp_path / "order.hip", tmp_path / "order"
    src.write_text(SOURCE)
    build = subprocess.run([str(HIPCC), "-x", "hip", "--cuda-host-only", "-O1", "-std=c++17", "-Wno-unused-command-line-argument",
                            f"-I{ROOT / 'flash-attention-triton_amd' / 'csrc'}", f"-I{ROOT / 'include'}", "-o", str(exe), str(src)],
                           capture_output=True, text=True, timeout=300)
    assert build.returncode == 0, build.stderr[-2000:]
    run = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert run.returncode == 0 and run.stdout == "ok\n", run.stdout + run.stderr
