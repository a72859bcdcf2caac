"""The inline-assembly MFMAs of the kernels from 160 columns on (ResidentB in csrc/fa2_common.hpp), which the compiler's hazard
recogniser does not see: in the code it made, no MFMA reads a register that one of the two wait states before it wrote on the
vector unit, and no vector instruction reads a score chain's result before its wait states are over."""

from __future__ import annotations

import math
import pathlib
import re
import subprocess

import pytest
import torch

from tests.test_code_objects import LLVM, _kernel_records

OBJDUMP = LLVM / "llvm-objdump"
SOURCES = r"[va]\[?\d+(?::\d+)?\]?"


def _registers(operand: str) -> set:
    m = re.fullmatch(r"([va])(?:(\d+)|\[(\d+):(\d+)\])", operand)
    if not m:
        return set()
    first = int(m.group(2) or m.group(3))
    return {(m.group(1), i) for i in range(first, int(m.group(4) or first) + 1)}


def _operands(line: str) -> list[str]:
    return re.findall(SOURCES, line.split("//")[0].partition(" ")[2])


def _hazards(lines: list[str]) -> list[str]:
    """`lines`: one kernel's instructions in order.  Branches are not followed: what a block starts with has its s_nop."""
    found = []
    written: list[tuple[int, set]] = []  # (wait state, registers) of vector instructions
    chain: list = []  # [registers, wait state of issue] of the last result in vector registers
    now = 0
    for text in lines:
        op = text.split()[0]
        if op == "s_nop":
            now += int(text.split()[1], 0) + 1
            continue
        operands = _operands(text)
        if op.startswith("v_mfma_f32_32x32x16"):
            reads = set().union(*(_registers(o) for o in operands[1:]))
            if any(now - at <= 2 and regs & reads for at, regs in written[-3:]):
                found.append(f"written too late for: {text}")
            chain = [_registers(operands[0]), now] if operands[0].startswith("v") else []
        elif op.startswith("v_"):
            if chain and now - chain[1] <= 11 and set().union(set(), *(_registers(o) for o in operands)) & chain[0]:
                found.append(f"result not there yet: {text}")
            if operands:
                written.append((now, _registers(operands[0])))
        now += 1
    return found


def test_the_check_sees_both_mistakes():
    mfma = "v_mfma_f32_32x32x16_bf16 v[0:15], v[16:19], a[0:3], v[0:15]"
    assert _hazards(["v_accvgpr_write_b32 a3, v40", mfma]) and _hazards(["v_mov_b32_e32 v16, v40", "s_nop 0", mfma])
    assert not _hazards(["v_accvgpr_write_b32 a3, v40", "s_nop 1", mfma]) and not _hazards(["v_mov_b32_e32 v20, v40", mfma])
    assert _hazards([mfma, "s_nop 9", "v_exp_f32_e32 v50, v3"]) and not _hazards([mfma, "s_nop 11", "v_exp_f32_e32 v50, v3"])


def test_no_operand_is_written_too_late_and_no_result_read_too_early(tmp_path):
    import importlib

    capi = importlib.import_module("flash-attention-triton_amd._capi")
    if not capi.LIBRARY_PATH.exists() or not OBJDUMP.exists():
        pytest.skip("library not built, or no ROCm LLVM tools")
    _kernel_records(capi.LIBRARY_PATH, tmp_path)  # (unbundles the code objects)
    wide = re.compile(r"<(_ZN3fa2\d+\w*kernelI(?:DF16b|DF16_)Li(?:192|256)E\w*)>:")
    checked = 0
    for obj in sorted(tmp_path.glob("code*.o")):
        listing = subprocess.run([str(OBJDUMP), "-d", "--no-show-raw-insn", "--no-leading-addr", str(obj)], check=True,
                                 capture_output=True, text=True).stdout
        for part in re.split(r"\n(?=(?:[0-9a-f]+ )?<_ZN3fa2)", listing):
            name = wide.search(part[:400])
            if not name or not re.search(r"fwd_direct_kernel|dq_direct_kernel|pair_kernel|joint_kernel", name.group(1)):
                continue
            lines = [s for s in (line.strip() for line in part.split("\n")[1:]) if s and not s.startswith("<")]
            assert not (bad := _hazards(lines)), (name.group(1), bad[:3])
            checked += sum(s.startswith("v_mfma_f32_32x32x16") for s in lines) > 0
    assert checked >= 100


# fp16 rounds P and O to 11 bits, bf16 to 8: a relative 2-norm below one unit, 5e-4 and 4e-3; gradients, whose dS is a difference of
# rounded values, twice that.
@pytest.mark.gpu
@pytest.mark.parametrize("heads,nq,nk,d,dtype", [
    (300, 129, 129, 256, torch.bfloat16), (16, 333, 300, 256, torch.float16), (3, 65, 1, 256, torch.float32), (70, 512, 520, 256, torch.float16),
    (33, 1100, 1100, 224, torch.bfloat16), (16, 700, 650, 216, torch.float16), (40, 1025, 1025, 192, torch.bfloat16),
    (16, 2000, 129, 160, torch.float16)], ids=lambda x: str(x).replace("torch.", ""))
def test_wide_heads_match_64_bits(heads, nq, nk, d, dtype):
    import flash_attention_triton_amd as fa

    gen = torch.Generator(device="cuda").manual_seed(d + nq)
    q, k, v, g = (torch.randn((1, heads, n, d), generator=gen, device="cuda").to(dtype) for n in (nq, nk, nk, nq))
    for x in (q, k, v):
        x.requires_grad_(True)
    out = fa.flash_attention_v2(q, k, v)
    got = [out.detach(), *torch.autograd.grad(out, (q, k, v), g)]
    at = [0, heads - 1]
    qd, kd, vd = (x[0, at].detach().double().requires_grad_(True) for x in (q, k, v))
    s = qd @ kd.transpose(1, 2).contiguous() / math.sqrt(d)
    s = s.masked_fill(torch.arange(nk, device="cuda")[None] > torch.arange(nq, device="cuda")[:, None], -math.inf)
    o = torch.softmax(s, -1) @ vd
    want = [o.detach(), *torch.autograd.grad(o, (qd, kd, vd), g[0, at].double())]
    unit = 4e-3 if dtype == torch.bfloat16 else 5e-4
    for name, x, w in zip(("o", "dq", "dk", "dv"), got, want):
        if nk == 1 and name in ("dq", "dk"):  # a softmax of one key has no gradient: rounding against the size of its summands
            assert x[0, at].double().abs().max() < 1e-2
            continue
        err = (x[0, at].double() - w).norm() / w.norm()
        assert err < unit * (1 if name == "o" else 2), (name, err.item())
