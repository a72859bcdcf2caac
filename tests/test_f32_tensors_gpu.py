"""fp32 tensors: rounded in one launch, results stored widened by the kernels.

An fp32 call has to give the bits of the same call on the tensors torch rounds to fp16, widened."""

from __future__ import annotations

import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu

# 4096 elements are one workgroup of the cast: (1, 1, 64, 64) is exactly one, (1, 1, 65, 63) one element less.
SHAPES = [(1, 1, 64, 64), (1, 1, 65, 63), (1, 1, 1, 8), (2, 3, 333, 64), (1, 8, 640, 128), (3, 5, 129, 80), (2, 2, 200, 72),
          (1, 3, 257, 96), (2, 20, 700, 96), (1, 2, 300, 256), (1, 2, 150, 200), (1, 3, 77, 33)]


def _inputs(shape, layout):
    gen = torch.Generator().manual_seed(sum(shape))
    b, h, n, d = shape
    out = []
    for _ in range(4):
        t = torch.randn((b, h, n, d), generator=gen).cuda()
        if layout == "bnhd":
            t = t.transpose(1, 2).contiguous().transpose(1, 2)
        elif layout == "gaps":
            t = torch.cat([t, t], -1)[..., :d]
        elif layout == "unaligned":
            t = torch.cat([t.new_zeros(1), t.flatten()])[1:].view(shape)
        out.append(t)
    return out


def _pass(fa, q, k, v, d_o):
    q, k, v = (t.detach().requires_grad_() for t in (q, k, v))
    o = fa.flash_attention_v2(q, k, v)
    return (o, *torch.autograd.grad(o, (q, k, v), d_o))


@pytest.mark.parametrize("layout", ["bhnd", "bnhd", "gaps", "unaligned"])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_f32_call_is_the_f16_call_widened(fa2_module, shape, layout):
    q, k, v, d_o = _inputs(shape, layout)
    got = _pass(fa2_module, q, k, v, d_o)
    want = _pass(fa2_module, *(t.half() for t in (q, k, v, d_o)))
    with torch.no_grad():
        got += (fa2_module.flash_attention_v2(q, k, v),)
        want += (fa2_module.flash_attention_v2(*(t.half() for t in (q, k, v))),)
    for name, g, w in zip(("o", "dq", "dk", "dv", "o under no_grad"), got, want):
        assert g.dtype == torch.float32 and torch.equal(g, w.float()), name
    assert got[0].is_contiguous()


def test_output_may_change_before_the_backward(fa2_module):
    """The backward reads the node's own fp16 output, not the tensor the caller got."""
    q, k, v, d_o = _inputs((2, 3, 200, 64), "bhnd")
    want = _pass(fa2_module, q, k, v, d_o)
    q, k, v = (t.requires_grad_() for t in (q, k, v))
    o = fa2_module.flash_attention_v2(q, k, v)
    o.detach().zero_()
    for g, w in zip(torch.autograd.grad(o, (q, k, v), d_o), want[1:]):
        assert torch.equal(g, w)


def test_lazily_cloned_inputs_stay_shared(fa2_module):
    """Rounding only reads: a copy-on-write clone is not copied for it."""
    tensors = _inputs((1, 2, 130, 64), "bhnd")
    clones = [torch._lazy_clone(t) for t in tensors[:3]]
    assert all(torch._C._is_cow_tensor(t) for t in clones)
    with torch.no_grad():
        got = fa2_module.flash_attention_v2(*clones)
    assert all(torch._C._is_cow_tensor(t) for t in clones)
    assert torch.equal(got, _pass(fa2_module, *tensors)[0])


@pytest.mark.parametrize("sizes", [(1,), (4096,), (4095, 4097), (5, 8192, 12289), (4096, 3, 20000)], ids=str)
def test_cast_rounds_as_torch_does(capi, sizes):
    lib = capi.load()
    special = torch.tensor([0.0, -0.0, float("inf"), float("-inf"), 65504.0, 65519.99, 65520.0, 1e30, 5.96e-8, 2.98e-8,
                            2.9802322e-8, 6.1e-5, 1.00048828125, 1.00146484375, 1e-42])
    gen = torch.Generator().manual_seed(len(sizes))
    src = []
    for n in sizes:
        t = torch.randn(n, generator=gen) * torch.exp2(torch.randint(-30, 17, (n,), generator=gen).float())
        t[max(0, n - len(special)):] = special[:n]
        src.append(t.cuda())
    dst = [torch.full((t.numel() + 8,), 7.0, dtype=torch.float16, device="cuda") for t in src]
    jobs = (capi.Cast * len(sizes))(*(capi.Cast(s.data_ptr(), d.data_ptr(), s.numel()) for s, d in zip(src, dst)))
    capi.check(lib.fa2_cast_f32_to_f16(jobs, len(sizes), torch.cuda.current_stream().cuda_stream), "fa2_cast_f32_to_f16")
    torch.cuda.synchronize()
    for s, d in zip(src, dst):
        assert torch.equal(d[:-8], s.half()) and (d[-8:] == 7).all()
    assert lib.fa2_cast_f32_to_f16(jobs, 4, ctypes.c_void_p(0)) != 0
    assert lib.fa2_cast_f32_to_f16(jobs, 0, ctypes.c_void_p(0)) != 0


@pytest.mark.parametrize("shape", [(2, 3, 333, 64), (1, 8, 130, 128), (1, 2, 200, 224), (1, 3, 77, 33)], ids=lambda s: "x".join(map(str, s)))
def test_f32_output_at_any_float_address(fa2_module, capi, shape):
    """fa2_fwd_packed_f32_out where o_f32 is 16-byte aligned and where it is not (the generic kernel), with o and without
    it.  The values are those of o, and the two kernels' differ by no more than a rounding or two of fp16."""
    lib = capi.load()
    b, h, n, d = shape
    q, k, v = (t.half() for t in _inputs(shape, "bhnd")[:3])
    stream = torch.cuda.current_stream().cuda_stream

    def arg(t):
        return capi.Tensor(t.data_ptr(), *fa2_module._strides3(t)) if t is not None else capi.Tensor(None, 0, 0, 0)

    def forward(floats_off, want_o):
        o = torch.empty_like(q) if want_o else None
        lse = torch.empty((b, h, 512), device="cuda")
        buf = torch.full((q.numel() + 8,), 7.0, device="cuda")
        args = capi.FwdArgs(arg(q), arg(k), arg(v), arg(o), lse.data_ptr(), b, h, n, n, d, 512, d**-0.5,
                            capi.FA2_DTYPE_F16, capi.FA2_CONFIG_AUTO)
        capi.check(lib.fa2_fwd_packed_f32_out(ctypes.byref(args), buf.data_ptr() + 4 * floats_off, stream), "fa2_fwd_packed_f32_out")
        torch.cuda.synchronize()
        out = buf[floats_off : floats_off + q.numel()].view(shape)
        assert (buf[:floats_off] == 7).all() and (buf[floats_off + q.numel() :] == 7).all()
        return out, o, lse

    aligned, o, lse = forward(0, True)
    assert torch.equal(aligned, o.float())
    for off in (0, 1, 2, 4):
        out, o2, lse2 = forward(off, True)
        assert torch.equal(out, o2.float())
        assert torch.equal(out, forward(off, False)[0])
        # One rounding of P per product differs between the kernels (2^-11 of values of order 1), one of the result.
        torch.testing.assert_close(out, aligned, atol=2e-3, rtol=2e-3)
        torch.testing.assert_close(lse2, lse, atol=1e-4, rtol=1e-5)
    assert lib.fa2_status_string(lib.fa2_fwd_packed_f32_out(None, 16, stream)).decode() == "FA2_ERR_NULL_POINTER"
