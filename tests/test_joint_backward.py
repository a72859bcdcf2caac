"""dQ, dK and dV in one grid (csrc/fa2_bwd_joint.hpp): the order of its workgroups and what the compiler made of the kernel,
on the CPU, and gradients at the edges of the rule that picks it (joint_key_groups in csrc/fa2_launch.hpp)."""

from __future__ import annotations

import ctypes
import math
import pathlib
import re
import subprocess

import pytest
import torch

from oracle import naive_attention as oracle
from tests.test_code_objects import COLUMNS, LDS_PER_CU, REGS_PER_LANE, records  # noqa: F401

ROOT = pathlib.Path(__file__).resolve().parent.parent
HIPCC = pathlib.Path("/opt/rocm/bin/hipcc")
ATOL, RTOL = 2e-2, 1e-2


def _host_program(source: str, tmp_path) -> str:
    if not HIPCC.exists():
        pytest.skip("hipcc not installed")
    exe = tmp_path / source.partition(".")[0]
    build = subprocess.run(
        [str(HIPCC), "-x", "hip", "--cuda-host-only", "-O1", "-std=c++17", "-Wno-unused-command-line-argument",
         f"-I{ROOT / 'flash-attention-triton_amd' / 'csrc'}", f"-I{ROOT / 'include'}",
         "-o", str(exe), str(ROOT / "tests" / source)], capture_output=True, text=True, timeout=300)
    assert build.returncode == 0, build.stderr[-2000:]
    return str(exe)


def test_every_workgroup_of_either_kind_once(tmp_path):
    run = subprocess.run([_host_program("joint_grid_check.hip", tmp_path)], capture_output=True, text=True, timeout=60)
    assert run.returncode == 0 and run.stdout.endswith("ok\n"), run.stdout + run.stderr


@pytest.fixture(scope="module")
def rule(tmp_path_factory):
    """(heads, seqlen_q, seqlen_k, headdim[, seqlen_q_rounded]) ... -> (key groups of dQ in a call for it alone, of the joint grid, its
    workgroups, key groups of dQ in front of dK/dV) ..."""
    program = _host_program("joint_rule.hip", tmp_path_factory.mktemp("rule"))

    def of(sizes):
        lines = "".join(f"{h} {nq} {nk} {rest[0] if rest else nq} {d}\n" for h, nq, nk, d, *rest in sizes)
        out = subprocess.run([program], input=lines, check=True, capture_output=True, text=True, timeout=60).stdout
        return [tuple(map(int, line.split())) for line in out.splitlines()]

    return of


def test_a_grid_too_large_to_launch_is_two_launches(rule):
    """Sizes whose dQ and dK/dV grids can each be launched (16.7 million workgroups), but not the joint one; and rows of delta
    beyond what the launch in front of it takes, where dQ can form delta by itself."""
    assert [groups for _, groups, _, _ in rule([
        (1, 100, 540_000_000, 8), (8_000_000, 128, 128, 128), (6_000_000, 128, 128, 256), (17, 1000, 1000, 64, 2**31 - 1)])] == [0] * 4
    for _, groups, workgroups, _ in rule([(h, n, nk, d) for h in (8, 1 << 16, 1 << 20, 3 << 20, 1 << 22, 8_000_000, 12_000_000)
                                          for n in (96, 128, 700) for nk in (1, 128, 700, 100_000) for d in (64, 96, 128, 256)]):
        assert workgroups <= 0xFFFFFFFF // 256


def test_a_call_for_dq_alone_takes_the_key_groups_of_the_whole_backward(rule):
    """Sums in the same order, so the same bits, whatever part of the gradient is asked for."""
    sizes = [(h, n, n, d) for d in (32, 40, 48, 64, 72, 80, 96, 104, 128, 160, 176, 192, 224, 256)
             for n in (64, 100, 129, 256, 333, 512, 640, 1000, 1500, 2048, 3000, 4096, 5000, 8192) for h in (*range(1, 70), 80, 96, 128, 200, 512, 1024)]
    got = rule(sizes)
    assert all(alone == (joint or two_launches) for alone, joint, _, two_launches in got)
    assert {(joint, two_launches) for _, joint, _, two_launches in got} == {(0, 1), (0, 2), (1, 1), (1, 2), (2, 2)}


def test_unlike_lengths(rule):
    """On both sides of each line of seqlen_k; what the sizes measured is at joint_key_groups."""
    sizes = [(32, 512, 2048, 64), (32, 512, 2049, 64), (32, 512, 1, 64), (32, 512, 1024, 192), (32, 512, 1025, 192), (64, 256, 257, 160), (64, 256, 256, 160),
             (48, 256, 512, 256), (48, 256, 513, 256), (3, 4096, 16384, 256),  # 128 workgroups of 128 rows
             (16, 2048, 8192, 128), (16, 2048, 8193, 128), (64, 512, 102, 96), (64, 512, 103, 96), (8, 4096, 819, 192), (8, 4096, 820, 192), (128, 256, 25, 160),  # 512
             (128, 1024, 2048, 128), (128, 1024, 300, 128), (128, 1024, 4097, 128), (256, 512, 2048, 256), (256, 1024, 4096, 256),  # 2000
             (160, 1024, 512, 128), (160, 1024, 511, 128), (264, 1100, 1300, 128), (264, 1100, 1400, 128), (2048, 128, 160, 128), (2048, 128, 161, 128), (2048, 128, 127, 128)]
    assert [groups for _, groups, _, _ in rule(sizes)] == [2, 0, 2, 2, 0, 0, 2, 2, 0, 2,
                                                           1, 0, 1, 0, 1, 0, 0, 1, 1, 0, 1, 0, 1, 0, 1, 0, 1, 0, 0]


@pytest.mark.parametrize("heads,n,d,groups", [
    (96, 128, 64, 2), (97, 64, 64, 0), (64, 128, 256, 2), (65, 64, 192, 0), (48, 129, 160, 2), (64, 200, 224, 2), (42, 300, 192, 2),  # 128
    (80, 192, 128, 1), (80, 192, 160, 0), (80, 256, 160, 1), (84, 256, 128, 0), (67, 300, 128, 1), (64, 512, 128, 1), (8, 4096, 128, 1),  # 256
    (64, 512, 96, 0), (52, 512, 96, 1), (56, 513, 80, 0), (48, 640, 80, 1), (64, 500, 112, 0), (48, 640, 112, 1), (44, 500, 192, 1), (48, 512, 192, 0),
    (40, 640, 192, 1), (8, 3100, 224, 1), (9, 3200, 224, 0), (52, 512, 256, 1), (56, 512, 256, 0), (48, 640, 256, 1), (16, 2048, 64, 1),
    (14, 3000, 32, 1), (15, 3000, 32, 0), (24, 2048, 64, 1), (33, 2048, 64, 0), (32, 2048, 64, 1), (24, 2048, 96, 1), (48, 767, 96, 0), (48, 768, 96, 1),  # 512
    (128, 512, 128, 1), (150, 256, 128, 0), (96, 320, 112, 1), (176, 192, 192, 1), (177, 192, 192, 0), (16, 3000, 160, 1), (17, 3000, 160, 0),
    (12, 4096, 192, 1), (384, 96, 256, 1), (385, 96, 256, 0),
    (576, 128, 224, 1), (600, 200, 224, 0), (72, 1000, 192, 1), (80, 1000, 192, 0), (288, 512, 224, 1), (256, 512, 224, 0), (1280, 192, 224, 0),  # beyond
    (1280, 256, 160, 0), (400, 160, 96, 0), (400, 161, 96, 1), (200, 512, 80, 1), (224, 512, 96, 0), (4096, 128, 128, 1), (1496, 256, 128, 1),
    (1504, 256, 128, 0), (256, 1024, 128, 0), (248, 1024, 128, 1), (256, 1100, 128, 1), (520, 192, 256, 0), (320, 192, 256, 1), (328, 192, 256, 0), (1024, 100, 256, 1),
    (1024, 512, 256, 0), (1024, 1024, 64, 0), (512, 2048, 32, 0), (640, 512, 112, 0), (36, 2048, 64, 0), (32, 2300, 64, 1)])
def test_joint_only_where_it_measured_faster(rule, heads, n, d, groups):
    """Both sides of the lines of joint_key_groups."""
    assert rule([(heads, n, n, d)])[0][1] == groups


def test_joint_kernels_share_a_cu_like_their_parts(records):  # noqa: F811
    """As many workgroups to a CU as the paired dK/dV kernel has, and no scratch memory but for the values kept across the
    choice of the kind."""
    seen = set()
    for r in records:
        m = re.match(r"_ZN3fa216bwd_joint_kernelI(DF16b|DF16_)Li(\d+)ELb([01])ELi([12])ELi(\d+)E", r["name"])
        if not m:
            continue
        dtype, dp, pad, groups, cols = m.group(1), *map(int, m.groups()[1:])
        seen.add((dtype, dp, pad, groups, cols))
        waves = REGS_PER_LANE // ((int(r["vgpr_count"]) + 7) // 8 * 8)
        assert min(waves, LDS_PER_CU // int(r["group_segment_fixed_size"])) >= (3 if dp <= 64 else 2 if dp <= 128 else 1), r["name"]
        assert int(r["private_segment_fixed_size"]) <= (20 if dp == 128 else 0), r["name"]
    assert seen == {(t, dp, pad, kg, cols) for t in ("DF16b", "DF16_") for dp, widths in COLUMNS.items() for cols in widths
                    for pad in (0, 1) for kg in (1, 2)}


@pytest.mark.gpu
@pytest.mark.parametrize("heads,n,d,dtype", [
    (8, 4096, 128, torch.bfloat16), (64, 512, 64, torch.float16), (16, 2048, 64, torch.bfloat16), (12, 2500, 120, torch.bfloat16),  # up to 256
    (24, 1024, 96, torch.bfloat16), (17, 1024, 192, torch.float16), (9, 2000, 224, torch.bfloat16), (32, 1024, 256, torch.bfloat16),
    (13, 3000, 32, torch.float16), (12, 4096, 128, torch.bfloat16), (50, 700, 48, torch.bfloat16),  # workgroups of 128 rows and beyond
    (33, 1000, 128, torch.bfloat16), (31, 2000, 128, torch.bfloat16), (33, 500, 128, torch.bfloat16), (61, 500, 128, torch.bfloat16),
    (56, 500, 128, torch.bfloat16), (9, 3700, 96, torch.bfloat16), (11, 1900, 96, torch.bfloat16)],  # (second rounds walked backwards)
    ids=lambda x: str(x).replace("torch.", ""))
def test_part_of_the_gradient_has_the_bits_of_all_of_it(capi, heads, n, d, dtype):
    """fa2_bwd with dq == NULL, or dk == dv == NULL, launches one of the two kernels by itself."""
    gen = torch.Generator(device="cuda").manual_seed(heads + d)
    q, k, v, d_o = (torch.randn((1, heads, n, d), generator=gen, device="cuda").to(dtype) for _ in range(4))
    lse = torch.logsumexp((q.float() @ k.float().transpose(-1, -2).contiguous() / math.sqrt(d)).masked_fill(
        ~torch.ones(n, n, dtype=torch.bool, device="cuda").tril(), -math.inf), -1) if n <= 1100 else torch.full((1, heads, n), 8.0, device="cuda")
    delta = torch.randn((1, heads, n), generator=gen, device="cuda")

    def run(*wanted):
        out = {name: torch.full_like(q, 7.0) for name in ("dq", "dk", "dv")}
        a = capi.BwdArgs(lse=lse.data_ptr(), delta=delta.data_ptr(), workspace=None, batch=1, nheads=heads, seqlen_q=n, seqlen_k=n, headdim=d,
                         seqlen_q_rounded=n, softmax_scale=1 / math.sqrt(d), deterministic=1, config_id=capi.FA2_CONFIG_AUTO,
                         dtype=capi.FA2_DTYPE_BF16 if dtype == torch.bfloat16 else capi.FA2_DTYPE_F16)
        for name, t in {"q": q, "k": k, "v": v, "d_o": d_o, **{x: out[x] for x in wanted}}.items():
            setattr(a, name, capi.Tensor(t.data_ptr(), *t.stride()[:3]))
        capi.check(capi.load().fa2_bwd_packed(ctypes.byref(a), torch.cuda.current_stream().cuda_stream), "fa2_bwd_packed")
        return out

    full, only_dq, only_dkdv = run("dq", "dk", "dv"), run("dq"), run("dk", "dv")
    assert torch.equal(only_dq["dq"], full["dq"]) and torch.equal(only_dkdv["dk"], full["dk"]) and torch.equal(only_dkdv["dv"], full["dv"])
    assert all((t == 7).all() for t in (only_dq["dk"], only_dq["dv"], only_dkdv["dq"]))


@pytest.mark.gpu
@pytest.mark.parametrize("heads,nq,nk,d,dtype", [
    (1, 1, 1, 64, torch.bfloat16), (96, 64, 64, 128, torch.float16), (97, 64, 64, 128, torch.bfloat16),  # one key group, 32 or fewer tokens
    (3, 129, 700, 40, torch.bfloat16), (3, 700, 129, 128, torch.bfloat16), (2, 65, 1, 256, torch.float16),  # kinds of unlike number
    (64, 192, 192, 48, torch.bfloat16), (65, 160, 160, 48, torch.bfloat16), (9, 1000, 1000, 104, torch.bfloat16),  # 128 workgroups and more
    (41, 300, 333, 32, torch.bfloat16), (32, 1024, 1024, 64, torch.float16), (27, 1153, 1100, 72, torch.bfloat16),
    (11, 3000, 3000, 96, torch.bfloat16), (43, 500, 500, 256, torch.bfloat16), (60, 200, 200, 176, torch.bfloat16),
    (136, 520, 520, 128, torch.bfloat16), (136, 520, 520, 120, torch.bfloat16), (200, 512, 500, 80, torch.bfloat16), (200, 512, 520, 80, torch.float16),  # more than 512
    (300, 100, 260, 160, torch.bfloat16), (520, 120, 120, 256, torch.bfloat16),
    (33, 500, 2000, 64, torch.bfloat16), (64, 512, 60, 96, torch.float16), (17, 2048, 300, 128, torch.bfloat16), (33, 512, 1000, 192, torch.float16),  # unlike lengths
    (176, 192, 192, 192, torch.bfloat16), (72, 1000, 1000, 192, torch.bfloat16), (576, 128, 128, 224, torch.float16)], ids=lambda x: str(x).replace("torch.", ""))
def test_gradients_at_the_edges_of_the_rule(fa, heads, nq, nk, d, dtype):
    gen = torch.Generator(device="cuda").manual_seed(nq + heads)
    q, d_o = (torch.randn(1, heads, nq, d, generator=gen, device="cuda").to(dtype) for _ in range(2))
    k, v = (torch.randn(1, heads, nk, d, generator=gen, device="cuda").to(dtype) for _ in range(2))
    leaves = [t.requires_grad_(True) for t in (q, k, v)]
    grads = torch.autograd.grad(fa.flash_attention_v2(*leaves), leaves, d_o)
    for at in {0, heads // 2, heads - 1}:
        one = [t.detach()[:, at : at + 1].float() for t in (q, k, v, d_o)]
        _, *want = oracle.naive_backward(*one, 1.0 / math.sqrt(d), torch.float32)
        for name, got, ref in zip(("dq", "dk", "dv"), grads, want):
            assert torch.isfinite(got).all(), name
            err = (got[:, at : at + 1].float() - ref).abs()
            assert (err <= ATOL + RTOL * ref.abs()).all(), f"{name}, head {at}: max abs err {err.max().item():.3e}"
