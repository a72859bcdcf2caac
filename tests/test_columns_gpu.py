"""GPU tests of the kernels whose column count is below their LDS pitch (48, 80, 160 and 224 columns in rows of 64,
128 and 256): exact, padded and neighbouring head dimensions, small grids (two key groups) and large ones.  The
tensors are slices of wider ones whose other columns are NaN, so a value read past a row's end would show.  Same oracle
and tolerance as tests/test_parity_gpu.py."""

from __future__ import annotations

import math

import pytest
import torch

from oracle import naive_attention as oracle

pytestmark = pytest.mark.gpu

ATOL, RTOL = 2e-2, 1e-2


def _sliced(shape, dtype, gen):
    b, h, n, d = shape
    wide = torch.full((b, h, n, d + 16), float("nan"), dtype=dtype, device="cuda")
    wide[..., 8 : 8 + d] = torch.randn(shape, generator=gen, device="cuda").to(dtype)
    return wide[..., 8 : 8 + d]


@pytest.mark.parametrize("heads", [2, 300], ids=["few", "many"])
@pytest.mark.parametrize("d,dtype", [(40, torch.bfloat16), (48, torch.bfloat16), (48, torch.float16), (72, torch.float16),
                                     (80, torch.float16), (80, torch.bfloat16), (88, torch.bfloat16), (136, torch.bfloat16),
                                     (160, torch.bfloat16), (160, torch.float16), (168, torch.float16), (216, torch.float16),
                                     (224, torch.bfloat16), (232, torch.bfloat16)])
@pytest.mark.parametrize("nq,nk", [(129, 129), (193, 260)])
def test_column_counts_below_the_pitch(fa, heads, d, dtype, nq, nk):
    gen = torch.Generator(device="cuda").manual_seed(d)
    q, d_o = _sliced((1, heads, nq, d), dtype, gen), _sliced((1, heads, nq, d), dtype, gen)
    k, v = _sliced((1, heads, nk, d), dtype, gen), _sliced((1, heads, nk, d), dtype, gen)
    leaves = [t.detach().requires_grad_(True) for t in (q, k, v)]
    out = fa.flash_attention_v2(*leaves)
    grads = torch.autograd.grad(out, leaves, d_o)
    with torch.no_grad():
        only = fa.flash_attention_v2(q, k, v)
    last = [t[:, heads - 1 :].float() for t in (q, k, v, d_o)]
    o, *want = oracle.naive_backward(*last, 1.0 / math.sqrt(d), torch.float32)
    for name, got, ref in (("o", out, o), ("o, forward only", only, o), *zip(("dq", "dk", "dv"), grads, want)):
        assert torch.isfinite(got).all(), name
        got = got[:, heads - 1 :].float()
        err = (got - ref).abs()
        assert (err <= ATOL + RTOL * ref.abs()).all(), f"{name}: max abs err {err.max().item():.3e}"
