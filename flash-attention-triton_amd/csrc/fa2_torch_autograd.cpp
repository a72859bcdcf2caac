// Autograd boundary in C++: FlashAttentionV2Function of the reference
// (src/flash_attention_triton/flash_attention_2.py:280-384) as a torch::autograd::Function whose
// forward and backward call the C ABI of libfa2_gfx950.so directly.
//
// Why it exists: with the autograd function written in Python, PyTorch's backward engine has to
// hand the backward to its device thread and that thread has to take the interpreter lock; at
// the smallest workloads that hand-over and the interpreter's own overhead cost more than the
// kernels take (B=2 H=4 N=512 D=64, fp16: 27 us of kernels; a forward + backward step took 110 us and
// takes 70 with this node, 34 where the engine stays on the calling thread).  A C++ node needs no
// interpreter lock.  The Python module keeps the reference-shaped class as well and uses
// this one when it is built.
//
// Host code only: tensors come in validated (CUDA device, all fp16, bf16 or fp32, equal dtypes and consistent
// shapes) from the Python wrapper, which also owns the reference's assertions and exception types.
#include <torch/extension.h>

#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>

#include <array>
#include <cmath>
#include <stdexcept>
#include <string>

#include "fa2_gfx950.h"

namespace {

fa2_tensor as_arg(const at::Tensor &t) {
  return fa2_tensor{t.data_ptr(), t.stride(0), t.stride(1), t.stride(2)};
}

void check(int status, const char *what) {
  if (status == FA2_OK) return;
  throw std::runtime_error(std::string(what) + " failed: " + fa2_status_string(status) + ": " +
                           fa2_last_error_string());
}

void *current_stream(const at::Tensor &t) {
  return static_cast<void *>(c10::hip::getCurrentHIPStream(t.device().index()).stream());
}

int dtype_code(const at::Tensor &t) { return t.scalar_type() == at::kBFloat16 ? FA2_DTYPE_BF16 : FA2_DTYPE_F16; }

// The tensor as the kernels can read it.  They take any batch, head and row stride, so a view such as
// (batch, token, head, column) memory transposed to (batch, head, token, column) goes in as it is,
// provided it meets what the LDS-direct kernels ask of their operands: whole 16-byte chunks, aligned
// rows and a row stride below 2^24 elements (fa2_launch.hpp).  Any other strided view is copied: one with
// whole chunks but odd alignment because a copy is cheaper than the generic kernels, one without (head
// dimension not a multiple of 8) so that those kernels, which run either way, read rows that lie together.
// A contiguous tensor goes in as it is; the generic kernels run where its base is not 16-byte aligned.
// B=256 H=16 N=512 D=64, bf16 views, forward + backward: 1661 us with the four copies (568 us of them),
// 1205 us without.
at::Tensor readable(const at::Tensor &t) {
  if (t.is_contiguous()) return t;
  const bool direct = t.stride(3) == 1 && t.size(3) % 8 == 0 && t.stride(0) % 8 == 0 && t.stride(1) % 8 == 0 &&
                      t.stride(2) % 8 == 0 && t.stride(2) < (int64_t(1) << 24) &&
                      reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0;
  return direct ? t : t.contiguous();
}

// fp32 tensors rounded to fp16, at most three in one launch, with the strides t.to(at::kHalf) would give.  Tensors
// without gaps are arrays to the kernel whatever the order of their dimensions; any other is torch's.
template <size_t N>
std::array<at::Tensor, N> rounded_to_half(const std::array<at::Tensor, N> &in) {
  std::array<at::Tensor, N> out;
  std::array<fa2_cast, N> jobs;
  int count = 0;
  for (size_t i = 0; i < N; i++) {
    const at::Tensor &t = in[i];
    if (t.numel() > 0 && t.is_non_overlapping_and_dense() && !t.is_neg() && !t._is_zerotensor() &&
        reinterpret_cast<uintptr_t>(t.const_data_ptr()) % 16 == 0) {
      out[i] = at::empty_like(t, t.options().dtype(at::kHalf));
      // (A const pointer: asked for a writable one, a lazily cloned tensor would copy itself first.)
      jobs[count++] = fa2_cast{t.const_data_ptr<float>(), out[i].data_ptr(), t.numel()};
    } else {
      out[i] = t.to(at::kHalf);
    }
  }
  if (count > 0) check(fa2_cast_f32_to_f16(jobs.data(), count, current_stream(in[0])), "fa2_cast_f32_to_f16");
  return out;
}

int64_t rounded(int64_t seqlen_q, int64_t max_headdim) {
  return (seqlen_q + max_headdim - 1) / max_headdim * max_headdim;
}

struct FlashAttentionV2 : public torch::autograd::Function<FlashAttentionV2> {
  // softmax_scale > 0 (the wrapper folds a negative scale into the sign of q).
  static at::Tensor forward(torch::autograd::AutogradContext *ctx, const at::Tensor &q_in, const at::Tensor &k_in,
                            const at::Tensor &v_in, double softmax_scale, bool deterministic,
                            int64_t max_headdim, bool forward_only) {
    const c10::DeviceGuard guard(q_in.device());
    // fp32 tensors are computed in fp16, as the reference does.  The casts are the node's and not the
    // graph's so that the backward can hand out fp32 gradients: the kernels store them widened, which saves
    // a pass over each.  B=32 H=20 N=1024 D=96, forward + backward: 1205 us, with casts in the graph 1339 us.
    // The kernel stores the output in fp32 as well (1138 us with torch's pass over it, 1113 so), and q, k and v are rounded
    // in one launch (1141 us with torch's casts, 1123 so).
    const bool f32 = q_in.scalar_type() == at::kFloat;
    std::array<at::Tensor, 3> half;
    if (f32) half = rounded_to_half(std::array<at::Tensor, 3>{q_in, k_in, v_in});
    const at::Tensor q = readable(f32 ? half[0] : q_in), k = readable(f32 ? half[1] : k_in),
                     v = readable(f32 ? half[2] : v_in);
    const int64_t batch = q.size(0), nheads = q.size(1), seqlen_q = q.size(2), headdim = q.size(3);
    const int64_t seqlen_k = k.size(2);
    const int64_t seqlen_q_rounded = rounded(seqlen_q, max_headdim);
    // Contiguous whatever the strides of q.  With fp32 tensors the kernel stores the result in fp32, and in
    // fp16 only where a backward will read that.
    at::Tensor o, o_f32;
    if (!f32 || !forward_only) o = at::empty(q.sizes(), q.options());
    if (f32) o_f32 = at::empty(q.sizes(), q_in.options());
    at::Tensor lse = at::empty({batch, nheads, seqlen_q_rounded}, q.options().dtype(at::kFloat));

    fa2_fwd_args a;
    a.q = as_arg(q);
    a.k = as_arg(k);
    a.v = as_arg(v);
    a.o = o.defined() ? as_arg(o) : fa2_tensor{nullptr, 0, 0, 0};
    a.lse = lse.data_ptr<float>();
    a.batch = (int)batch;
    a.nheads = (int)nheads;
    a.seqlen_q = (int)seqlen_q;
    a.seqlen_k = (int)seqlen_k;
    a.headdim = (int)headdim;
    a.seqlen_q_rounded = (int)seqlen_q_rounded;
    a.softmax_scale = (float)softmax_scale;
    a.dtype = dtype_code(q);
    // forward_only: the caller knows that nothing will be differentiated, so no backward reads lse.
    a.config_id = forward_only ? fa2_pick_config_forward_only(a.dtype, a.headdim, a.seqlen_q, a.seqlen_k)
                               : FA2_CONFIG_AUTO;
    if (forward_only && a.config_id < 0) check(-a.config_id, "fa2_pick_config_forward_only");
    check(f32 ? fa2_fwd_packed_f32_out(&a, o_f32.data_ptr<float>(), current_stream(q))
              : fa2_fwd_packed(&a, current_stream(q)), "fa2_fwd");

    ctx->save_for_backward({q, k, v, o, lse});
    ctx->saved_data["softmax_scale"] = softmax_scale;
    ctx->saved_data["deterministic"] = deterministic;
    ctx->saved_data["f32"] = f32;
    return f32 ? o_f32 : o;
  }

  static torch::autograd::variable_list backward(torch::autograd::AutogradContext *ctx,
                                                 torch::autograd::variable_list grads) {
    const auto saved = ctx->get_saved_variables();
    const at::Tensor &q = saved[0], &k = saved[1], &v = saved[2], &o = saved[3], &lse = saved[4];
    const c10::DeviceGuard guard(q.device());
    // Like the reference (flash_attention_2.py:364) the backward is not differentiable.
    const at::NoGradGuard no_grad;
    at::Tensor d_o = grads[0];
    if (d_o.scalar_type() == at::kFloat && q.scalar_type() == at::kHalf && d_o.is_cuda()) {
      d_o = rounded_to_half(std::array<at::Tensor, 1>{d_o})[0];
    } else if (d_o.scalar_type() != q.scalar_type()) {
      d_o = d_o.to(q.scalar_type());
    }
    d_o = readable(d_o);
    // (empty_like keeps the order of a dense view's dimensions: the gradients of transposed projections come
    // out in the projections' own order.)
    const bool f32 = ctx->saved_data["f32"].toBool();
    const at::TensorOptions like = q.options().dtype(f32 ? at::kFloat : q.scalar_type());
    at::Tensor dq = at::empty_like(q, like), dk = at::empty_like(k, like), dv = at::empty_like(v, like);
    at::Tensor delta = at::empty_like(lse);

    // Both launches of the reference launcher (preprocess, then the main kernel) in one call:
    // with `o` in the record the library forms delta on the way.
    fa2_bwd_args a;
    a.q = as_arg(q);
    a.k = as_arg(k);
    a.v = as_arg(v);
    a.o = as_arg(o);
    a.d_o = as_arg(d_o);
    a.dq = as_arg(dq);  // (fp32 with f32)
    a.dk = as_arg(dk);
    a.dv = as_arg(dv);
    a.lse = lse.data_ptr<float>();
    a.delta = delta.data_ptr<float>();
    a.workspace = nullptr;  // fa2_bwd_workspace_bytes is 0: dQ is written directly
    a.batch = (int)q.size(0);
    a.nheads = (int)q.size(1);
    a.seqlen_q = (int)q.size(2);
    a.seqlen_k = (int)k.size(2);
    a.headdim = (int)q.size(3);
    a.seqlen_q_rounded = (int)lse.size(2);
    a.softmax_scale = (float)ctx->saved_data["softmax_scale"].toDouble();
    a.dtype = dtype_code(q);
    a.deterministic = ctx->saved_data["deterministic"].toBool() ? 1 : 0;
    a.config_id = FA2_CONFIG_AUTO;
    check((f32 ? fa2_bwd_packed_f32_grads : fa2_bwd_packed)(&a, current_stream(q)), "fa2_bwd");
    return {dq, dk, dv, at::Tensor(), at::Tensor(), at::Tensor(), at::Tensor()};
  }
};

// A tensor the node may save.  Autograd refuses to save a tensor made in inference mode; a strided view of
// one goes in as a copy, which is an ordinary tensor.
at::Tensor savable(const at::Tensor &t) { return t.is_inference() && !t.is_contiguous() ? t.contiguous() : t; }

at::Tensor flash_attention_v2(const at::Tensor &q, const at::Tensor &k, const at::Tensor &v,
                              double softmax_scale, bool deterministic, int64_t max_headdim, bool forward_only) {
  if (at::GradMode::is_enabled() && (q.requires_grad() || k.requires_grad() || v.requires_grad()))
    return FlashAttentionV2::apply(savable(q), savable(k), savable(v), softmax_scale, deterministic, max_headdim,
                                   forward_only);
  return FlashAttentionV2::apply(q, k, v, softmax_scale, deterministic, max_headdim, forward_only);
}

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  m.doc() = "C++ autograd node over the C ABI of libfa2_gfx950.so";
  m.def("flash_attention_v2", &flash_attention_v2,
        "q, k, v: CUDA fp16/bf16/fp32 (B, H, N, D), any strides; softmax_scale > 0; returns o in their type",
        py::arg("q"), py::arg("k"), py::arg("v"), py::arg("softmax_scale"), py::arg("deterministic"),
        py::arg("max_headdim"), py::arg("forward_only") = false);
  m.def("abi_version", []() { return FA2_ABI_VERSION; });  // of the header this node was compiled with
}
