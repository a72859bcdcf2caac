"""The forward with four key groups (fwd_quad_kernel in csrc/fa2_fwd.hpp): where it is picked and what the compiler made of it, on
the CPU, and its results at the edges of its tiles."""

from __future__ import annotations

import math
import re

import pytest
import torch

from oracle import naive_attention as oracle
from tests.test_code_objects import COLUMNS, LDS_PER_CU, REGS_PER_LANE, records  # noqa: F401

ATOL, RTOL = 2e-2, 1e-2


@pytest.mark.parametrize("heads,n,d,groups", [
    (24, 640, 32, 4), (32, 513, 32, 2), (24, 1024, 32, 4), (32, 1024, 32, 2), (16, 2048, 32, 4), (17, 2048, 32, 2), (8, 512, 64, 2),
    (16, 1024, 64, 4), (17, 1024, 64, 2), (10, 2048, 48, 4), (11, 2048, 40, 2), (8, 3072, 64, 4), (8, 1024, 96, 2), (8, 1024, 80, 2),  # (0.95 of two groups' rate)
    (4, 2048, 80, 4), (4, 2047, 96, 2), (8, 1000, 72, 4), (8, 999, 88, 2), (15, 601, 40, 4), (16, 600, 56, 2), (8, 576, 40, 4), (9, 2048, 40, 4),
    (10, 2048, 56, 2), (8, 3000, 48, 4), (8, 3000, 40, 2), (9, 1024, 72, 2), (10, 767, 96, 2), (3, 4096, 96, 4), (5, 1500, 128, 4), (5, 1499, 128, 2), (3, 4096, 104, 4), (4, 4096, 128, 2),
    (1, 8192, 160, 2)])
def test_four_key_groups_only_where_they_measured_faster(capi, heads, n, d, groups):
    info = capi.launch_info(1, heads, n, n, d)["fwd"]
    assert info["key_groups"] == groups and info["block_rows"] == 128 // groups
    if groups == 4:
        assert info["workgroups"] == heads * math.ceil(n / 32) and info["wg_per_cu"] == {32: 4, 40: 2, 48: 2, 64: 2}.get(d, 1)


@pytest.mark.parametrize("heads,n,d,groups", [
    (5, 1500, 128, 2), (4, 2047, 128, 2), (4, 2048, 128, 4), (5, 1500, 104, 4), (4, 2048, 80, 2), (1, 8192, 96, 2), (3, 4096, 96, 4), (3, 4096, 80, 4),
    (3, 4000, 96, 2), (5, 1499, 72, 2), (5, 1500, 88, 4), (16, 1024, 64, 4), (16, 2048, 32, 4)])
def test_the_folded_row_has_lines_of_its_own(capi, heads, n, d, groups):
    row = capi.load().fa2_pick_config_forward_only(capi.FA2_DTYPE_BF16, d, n, n)
    assert capi.launch_info(1, heads, n, n, d, row)["fwd"]["key_groups"] == groups


def test_four_key_groups_fit_a_cu(records):  # noqa: F811
    seen = set()
    for r in records:
        m = re.match(r"_ZN3fa215fwd_quad_kernelI(DF16b|DF16_)Li(\d+)ELb([01])ELb([01])ELb([01])ELi(\d+)E", r["name"])
        if not m:
            continue
        seen.add((m.group(1), *map(int, m.groups()[1:])))
        dp = int(m.group(2))
        waves = REGS_PER_LANE // ((int(r["vgpr_count"]) + 7) // 8 * 8)
        assert min(waves, LDS_PER_CU // int(r["group_segment_fixed_size"])) >= {32: 4, 64: 2}.get(dp, 1), r["name"]
        assert int(r["private_segment_fixed_size"]) == int(r["vgpr_spill_count"]) == 0, r["name"]
    assert seen == {(t, dp, pad, pre, f32, cols) for t in ("DF16b", "DF16_") for dp in (32, 64, 96, 128) for cols in COLUMNS[dp]
                    for pad in (0, 1) for pre in (0, 1) for f32 in (0, 1)}


@pytest.mark.gpu
@pytest.mark.parametrize("d,dtype", [(32, torch.bfloat16), (24, torch.float16), (40, torch.bfloat16), (48, torch.float16), (64, torch.bfloat16),
                                     (72, torch.bfloat16), (80, torch.float16), (96, torch.float32), (104, torch.bfloat16), (128, torch.bfloat16)],
                         ids=lambda x: str(x).replace("torch.", ""))
@pytest.mark.parametrize("nq,nk", [(1500, 1500), (1537, 1), (1569, 33), (1600, 127), (1633, 129), (1568, 1631), (1665, 400), (1504, 3000)])
def test_four_key_groups_edges(fa, d, dtype, nq, nk):
    """Query tiles with one to four groups at work, one to thirteen tiles of 128 keys, ragged ends of both."""
    gen = torch.Generator(device="cuda").manual_seed(nq + d)
    q = torch.randn(1, 2, nq, d, generator=gen, device="cuda").mul_(1.5).to(dtype)
    k, v = (torch.randn(1, 2, nk, d, generator=gen, device="cuda").to(dtype) for _ in range(2))
    out = fa.flash_attention_v2(q.clone().requires_grad_(True), k, v).detach()
    with torch.no_grad():
        only = fa.flash_attention_v2(q, k, v)
    want = oracle.naive_causal_attention(q.float(), k.float(), v.float(), 1.0 / math.sqrt(d))
    for got in (out, only):
        assert torch.isfinite(got).all()
        err = (got.float() - want).abs()
        assert (err <= ATOL + RTOL * want.abs()).all(), f"max abs err {err.max().item():.3e}"


@pytest.mark.gpu
@pytest.mark.parametrize("bias", [-1e30, -3e38, float("-inf")])
@pytest.mark.parametrize("first,last", [(32, 64), (32, 128), (96, 300)])
def test_keys_hidden_from_a_group(fa, bias, first, last):
    """Keys that a bias column hides where they are all that a group's first block, or several groups' first blocks, hold."""
    gen = torch.Generator(device="cuda").manual_seed(first)
    q, k, v = (torch.randn(1, 2, 1600, 64, generator=gen, device="cuda").bfloat16() for _ in range(3))
    q[..., -1] = 1.0
    k[..., -1] = 0.0
    k[:, :, first:last, -1] = bias
    s = q.float() @ k.float().transpose(-1, -2).contiguous() / 8.0
    s = s.masked_fill(~torch.ones(1600, 1600, dtype=torch.bool, device="cuda").tril(), float("-inf"))
    want = torch.softmax(s, -1) @ v.float()
    with torch.no_grad():
        only = fa.flash_attention_v2(q, k, v)
    for got in (fa.flash_attention_v2(q.clone().requires_grad_(True), k, v).detach(), only):
        err = (got.float() - want).abs()
        assert (err <= ATOL + RTOL * want.abs()).all(), f"max abs err {err.max().item():.3e}"
