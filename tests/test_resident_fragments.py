"""The inline-assembly MFMAs of the kernels from 160 columns on (ResidentB in csrc/fa2_common.hpp) and of the dK/dV kernel that
holds both accumulators (csrc/fa2_bwd_dkdv.hpp), which the compiler's hazard recogniser does not see: in the code it made, no MFMA
reads a register that one of the two wait states before it wrote on the vector unit, and nothing touches an MFMA's result before its
wait states are over, along every branch."""

from __future__ import annotations

import math
import pathlib
import re
import subprocess

import pytest
import torch

from tests.test_code_objects import COLUMNS, LLVM, PAIR_COLUMNS, _kernel_records

OBJDUMP = LLVM / "llvm-objdump"
REGISTERS = re.compile(r"\b([va])(?:(\d+)|\[(\d+):(\d+)\])")
RESULT_STATES = 12  # behind an 8-pass MFMA (32x32x16) on gfx950, what the compiler itself leaves there
OPERAND_STATES = 2  # between a vector instruction's result and an MFMA that reads it
READS_AND_WRITES = ("v_", "ds_", "global_", "buffer_", "scratch_", "flat_")


def _parse(listing: list[str]):
    """[op, registers of each operand, wait states, index of a branch's target, text] per instruction."""
    code, at = [], {}
    for line in listing:
        text, _, comment = line.partition("//")
        op, _, rest = text.strip().partition(" ")
        where = re.match(r"\s*([0-9A-F]+):", comment)
        if where:
            at[int(where.group(1), 16)] = len(code)
        operands = [frozenset((kind, i) for i in range(int(one or first), int(one or last) + 1))
                    for kind, one, first, last in REGISTERS.findall(rest)] if op.startswith(READS_AND_WRITES) else []
        states = int(rest.split()[0], 0) + 1 if op == "s_nop" else 1
        target = None
        if op.startswith(("s_cbranch", "s_branch")):
            jump = int(rest.split()[0]) & 0xFFFF
            target = (int(where.group(1), 16) if where else 4 * len(code)) + 4 + 4 * (jump - 0x10000 if jump >= 0x8000 else jump)
        code.append([op, operands, states, target, line.strip()])
    for c in code:
        if c[3] is not None:
            c[3] = at[c[3]] if at else c[3] // 4
    return code


def _hazards(listing: list[str]) -> list[str]:
    """`listing`: one kernel's instructions in order."""
    code = _parse(listing)
    found = []
    seen = set()

    def walk(i, now, results, written):
        """From instruction i on.  results: (registers, wait state of issue) of the MFMAs in flight; written: the same of vector
        instructions.  A walk that a branch began ends where nothing of what came before it is left."""
        began_at = now if results or written else None
        while i < len(code):
            op, operands, states, target, text = code[i]
            results = [r for r in results if now - r[1] <= RESULT_STATES]
            written = [w for w in written if now - w[1] <= OPERAND_STATES]
            if began_at is not None and i > 0 and all(at >= began_at for _, at in results + written):
                return
            if op.startswith("v_mfma"):
                chained = operands[3] if len(operands) > 3 else None
                if any(regs & o for regs, _ in written for o in operands[1:]):
                    found.append(f"written too late for: {text}")
                # (A product may add to the one before it in the same registers with no wait.)
                if any(regs & o for regs, _ in results for k, o in enumerate(operands) if k in (1, 2) or not regs == chained == operands[0]):
                    found.append(f"result not there yet: {text}")
                results = [r for r in results if r[0] != operands[0]] + [(operands[0], now)]
            elif op.startswith(READS_AND_WRITES):
                if any(regs & o for regs, _ in results for o in operands):
                    found.append(f"result not there yet: {text}")
                if op.startswith("v_") and operands:
                    written = written + [(operands[0], now)]
            now += states
            if target is not None:
                state = (target, tuple((r, now - at) for r, at in results), tuple((w, now - at) for w, at in written))
                if (results or written) and state not in seen:
                    seen.add(state)
                    walk(target, now, results, written)
            if op in ("s_branch", "s_endpgm"):
                if began_at is not None:
                    return
                results, written = [], []
            i += 1

    walk(0, 0, [], [])
    return found


def test_the_check_sees_every_mistake():
    mfma = "v_mfma_f32_32x32x16_bf16 v[0:15], v[16:19], a[0:3], v[0:15]"
    other = "v_mfma_f32_32x32x16_bf16 a[16:31], v[20:23], v[24:27], a[16:31]"
    second = "v_mfma_f32_32x32x16_bf16 v[32:47], v[20:23], a[4:7], 0"
    read = "v_exp_f32_e32 v50, v3"
    assert _hazards(["v_accvgpr_write_b32 a3, v40", mfma]) and _hazards(["v_mov_b32_e32 v16, v40", "s_nop 0", mfma])
    assert not _hazards(["v_accvgpr_write_b32 a3, v40", "s_nop 1", mfma]) and not _hazards(["v_mov_b32_e32 v20, v40", mfma])
    assert _hazards([mfma, "s_nop 10", read]) and not _hazards([mfma, "s_nop 11", read]) and not _hazards([mfma, mfma])
    for between in (other, second):  # another product does not end the wait
        assert _hazards([mfma, between, read]) and _hazards([mfma, between, "s_nop 9", read]) and not _hazards([mfma, between, "s_nop 10", read])
    assert not _hazards([other, mfma, second])
    for use in ("ds_write_b128 v60, v[0:3]", "global_store_dwordx4 v[60:61], v[12:15], off", "scratch_store_dword off, v7, s0",
                "v_mov_b32_e32 v4, 0", "v_mfma_f32_32x32x16_bf16 v[32:47], v[12:15], a[0:3], 0", "v_mfma_f32_32x32x16_bf16 v[8:23], v[60:63], a[0:3], 0"):
        assert _hazards([mfma, use]) and not _hazards([mfma, "s_nop 11", use]), use
    # Along the branch (two instructions on; two back: the loop's end meets its start), not along what it jumps over.
    assert _hazards([mfma, "s_cbranch_scc1 1", "s_nop 11", read]) and not _hazards([mfma, "s_nop 11", "s_cbranch_scc1 1", "s_nop 0", read])
    assert _hazards([read, "s_nop 3", mfma, "s_cbranch_scc1 65532", "s_endpgm"]) and not _hazards([read, mfma, "s_nop 11", "s_cbranch_scc1 65532", "s_endpgm"])
    assert not _hazards([mfma, "s_branch 1", read, "s_nop 11", read])


def test_no_operand_is_written_too_late_and_no_result_read_too_early(tmp_path):
    import importlib

    capi = importlib.import_module("flash-attention-triton_amd._capi")
    if not capi.LIBRARY_PATH.exists() or not OBJDUMP.exists():
        pytest.skip("library not built, or no ROCm LLVM tools")
    built = {r["name"] for r in _kernel_records(capi.LIBRARY_PATH, tmp_path)}  # (unbundles the code objects)
    inline = re.compile(r"_ZN3fa2\d+(?:(?:fwd_direct|bwd_dq_direct|bwd_dkdv_pair|bwd_joint)_kernelI(?:DF16b|DF16_)Li(?:192|256)E"
                        r"|bwd_dkdv_direct_kernelI)")
    want = {name for name in built if inline.match(name)}
    checked = set()
    for obj in sorted(tmp_path.glob("code*.o")):
        listing = subprocess.run([str(OBJDUMP), "-d", "--no-show-raw-insn", str(obj)], check=True, capture_output=True, text=True).stdout
        for part in re.split(r"\n(?=[0-9a-f]+ <)", listing):
            name = re.match(r"[0-9a-f]+ <(\w+)>:\n", part)
            if not name or name.group(1) not in want:
                continue
            lines = [s for s in (line.strip() for line in part.split("\n")[1:]) if re.match(r"[a-z]\w+", s)]
            assert sum(s.startswith("v_mfma_f32_32x32x16") for s in lines) > 0
            assert not (bad := _hazards(lines)), (name.group(1), bad[:3])
            checked.add(name.group(1))
    assert checked == want
    wide = [dp for dp in COLUMNS if dp > 128]
    forms = 2 * 2 * sum(len(COLUMNS[dp]) for dp in wide)  # of either type, padded and not
    count = {k: sum(k in name for name in want) for k in ("fwd_direct", "dq_direct", "dkdv_pair", "joint", "dkdv_direct")}
    assert set(wide) <= set(PAIR_COLUMNS)
    # Key groups, and fp32 output or delta formed on the way; the dK/dV kernel at 32, 64 and 128 columns, padded or not or with atomics.
    assert count == {"fwd_direct": forms * 4, "dq_direct": forms * 4, "dkdv_pair": forms, "joint": forms * 2, "dkdv_direct": 2 * 3 * 3}


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
