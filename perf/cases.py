"""Performance cases of the causal attention path: what its users have it do, with how each is made,
run, priced and compared.

``flash_attention_v2`` is called in two ways: in training (forward, then the gradients of q, k and v
through autograd) and in inference (forward alone under ``torch.no_grad()``).  The ranges are those of the
package's workloads, of its test shapes and of plain transformer layers: 64 to 16384 tokens, head
dimensions 32 to 256 (multiples of 16, the widths models use), one (batch, head) pair per GPU up to
thousands of them, bf16, fp16 and fp32 inputs, both backward modes, tensors that are contiguous in
(batch, head, token, column) order or views of a projection's (batch, token, head, column) output.
"""

from __future__ import annotations

import math

import torch

import flash_attention_triton_amd as fa

_DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}


def _case(name, kind, batch, heads, seqlen, headdim, dtype, layout="bhnd", deterministic=False, qk_std=1.0,
          seqlen_k=None):
    case = {"kind": kind, "batch": batch, "heads": heads, "seqlen_q": seqlen,
            "seqlen_k": seqlen if seqlen_k is None else seqlen_k, "headdim": headdim, "dtype": dtype,
            "layout": layout, "deterministic": deterministic, "qk_std": qk_std}
    return dict(case, name=name) if name else case


def listed():
    return [
        # The smallest training step (the package's first workload): launches and host time count.
        _case("small-train-f16-d64", "train", 2, 4, 512, 64, "f16"),
        # One user's short, ragged prompt: a prefill of a few hundred tokens, latency bound.
        _case("short-prompt-bf16-d128", "infer", 1, 16, 333, 128, "bf16"),
        # A layer trained at moderate length with reproducible gradients.
        _case("train-det-bf16-d64", "train", 4, 16, 2048, 64, "bf16", deterministic=True),
        # The 7B-style layer everything else is compared with: training step ...
        _case("train-bf16-d128", "train", 2, 32, 4096, 128, "bf16"),
        # ... and the same layer evaluated or prefilled, where nothing will be differentiated.
        _case("prefill-bf16-d128", "infer", 2, 32, 4096, 128, "bf16"),
        # Long context, few heads: the largest pass.
        _case("long-train-det-bf16-d128", "train", 1, 16, 16384, 128, "bf16", deterministic=True),
        # Ragged length, fp16, peaked softmax.
        _case("ragged-train-f16-d64", "train", 8, 12, 3000, 64, "f16", qk_std=3.0),
        # fp32 model without autocast: inputs are cast to fp16 and results back, as the reference does.
        _case("train-f32-d96", "train", 32, 20, 1024, 96, "f32"),
        # Many short sequences (BERT-style batches) in the layout a fused projection produces.
        _case("short-seqs-train-bf16-d64-bnhd", "train", 256, 16, 512, 64, "bf16", layout="bnhd"),
        # Wide heads.
        _case("train-bf16-d256", "train", 2, 8, 4096, 256, "bf16"),
        # Fine-tuning one sequence on a shard of a model's heads: few (batch, head) pairs for the chip.
        _case("one-seq-train-bf16-d128-bnhd", "train", 1, 8, 4096, 128, "bf16", layout="bnhd"),
        # Prefill of one odd-sized prompt in fp16 on few heads, tensors as the projections leave them.
        _case("prompt-f16-d80-bnhd", "infer", 1, 12, 5001, 80, "f16", layout="bnhd"),
    ]


# Time of a FLOP at a head dimension, relative to 128 columns (wide heads and narrow ones run slower).
def _weight(headdim):
    return 1.0 if 96 <= headdim <= 128 else 2.0 if 64 <= headdim < 96 else 4.0


def draw(rng):
    """One more case of the ranges above: lengths over their logarithm, every second one odd-sized."""
    limit = 3.0e12  # weighted FLOPs: below the largest listed case
    headdim = rng.choice((32, 48, 64, 64, 80, 96, 128, 128, 128, 160, 192, 256))
    heads = rng.choice((1, 2, 4, 8, 12, 16, 20, 32))
    seqlen = round(math.exp(rng.uniform(math.log(64), math.log(16384))))
    if rng.random() < 0.5:
        seqlen = max(64, round(seqlen / 64) * 64)
    kind = rng.choice(("train", "train", "infer"))
    per_pair = _weight(headdim) * (3.5 if kind == "train" else 1.0) * 2.0 * seqlen * seqlen * headdim
    while heads > 1 and heads * per_pair > limit:
        heads //= 2
    most = min(256.0, limit / (heads * per_pair), 1.2e8 / (heads * seqlen * headdim))
    batch = max(1, int(math.exp(rng.uniform(0.0, math.log(max(1.0, most))))))
    dtype = rng.choice(("bf16", "bf16", "bf16", "f16", "f16", "f32"))
    seqlen_k = seqlen if rng.random() < 0.9 else max(64, int(seqlen * rng.uniform(0.5, 1.5)))
    return _case(None, kind, batch, heads, seqlen, headdim, dtype, rng.choice(("bhnd", "bnhd")),
                 rng.random() < 0.3, rng.choice((1.0, 1.0, 1.0, 3.0 if dtype == "f16" else 1.0)), seqlen_k)


def prepare(case, seed):
    """q, k, v and, for training, the output's gradient, drawn on the GPU.  With layout "bnhd" the tensors
    are stored (batch, token, head, column), as a projection's output reshaped to heads is, and the attention
    is handed transposed views of them; the output's gradient then arrives in that order as well."""
    device = torch.device("cuda")
    gen = torch.Generator(device=device).manual_seed(seed)
    train = case["kind"] == "train"
    bnhd = case["layout"] == "bnhd"

    def tensor(seqlen, std):
        b, h, d = case["batch"], case["heads"], case["headdim"]
        shape = (b, seqlen, h, d) if bnhd else (b, h, seqlen, d)
        x = torch.randn(shape, generator=gen, device=device, dtype=torch.float32)
        return x.mul_(std).to(_DTYPES[case["dtype"]])

    q = tensor(case["seqlen_q"], case["qk_std"])
    k = tensor(case["seqlen_k"], case["qk_std"])
    v = tensor(case["seqlen_k"], 1.0)
    d_o = tensor(case["seqlen_q"], 1.0) if train else None
    for x in (q, k, v):
        x.requires_grad_(train)
    return {"q": q, "k": k, "v": v, "d_o": d_o, "bnhd": bnhd, "deterministic": case["deterministic"]}


def run(state):
    """Training: the output and the gradients of q, k and v.  Inference: the output."""
    q, k, v = inputs = (state["q"], state["k"], state["v"])
    if state["bnhd"]:
        q, k, v = q.transpose(1, 2), k.transpose(1, 2), v.transpose(1, 2)
    if state["d_o"] is None:
        with torch.no_grad():
            out = fa.flash_attention_v2(q, k, v, None, state["deterministic"])
            return out.transpose(1, 2) if state["bnhd"] else out
    out = fa.flash_attention_v2(q, k, v, None, state["deterministic"])
    if state["bnhd"]:
        out = out.transpose(1, 2)
    return [out.detach(), *torch.autograd.grad(out, inputs, state["d_o"])]


def work(case):
    """Each input read once, each output written once; two products per (query, key) pair under the
    diagonal in the forward and five in the backward."""
    nq, nk = case["seqlen_q"], case["seqlen_k"]
    heads, d = case["batch"] * case["heads"], case["headdim"]
    full = min(nq, nk)
    pairs = full * (full + 1) // 2 + (nq - full) * nk
    train = case["kind"] == "train"
    size = 4 if case["dtype"] == "f32" else 2
    elements = (3 * nq + 2 * nk + nq + 2 * nk if train else 2 * nq + 2 * nk) * d
    return {"bytes": heads * elements * size, "flops": heads * pairs * d * (4 + 10 if train else 4)}


def tolerance(case):
    """About four times the largest error of O, dQ, dK and dV against the same attention evaluated in 64
    bits (333 and 2048 tokens, head dimensions 48 to 256): 2.6e-3 in bf16, 3.1e-4 in fp16 (7.4e-4 with
    peaked scores), 5.7e-4 for fp32 tensors computed in fp16."""
    if case["dtype"] == "bf16":
        return {"rel": 1e-2}
    if case["qk_std"] > 1.0:
        return {"rel": 3e-3}
    return {"rel": 2.3e-3 if case["dtype"] == "f32" else 1.3e-3}
