// PyTorch-ROCm extension `flash_attn_v100_cuda`: validation, allocation, device
// guard and stream lookup around the C launchers declared in fused_mha.h.
//
// Mirrors the reference extension kernel/fused_mha_api.cpp (mha_fwd :13-72,
// mha_bwd :74-162, pybind :164-168): same module name, same function names
// (`fwd`, `bwd`), same argument meaning and the same error convention
// (TORCH_CHECK -> RuntimeError).  Differences:
//   * fwd returns [out, lse] (one logsumexp) instead of [out, max, sum];
//   * bwd takes lse instead of (D, sum, max); delta is computed on the device
//     in fp32 inside the launcher;
//   * head size 64 is accepted as well as 128; any seqlen > 0 is accepted (the
//     reference assumes a multiple of 32, README.md:3, without checking);
//   * inputs that are not dense (B, N, H, D) are read through their strides
//     (or copied dense when the strides do not qualify) instead of being read
//     with wrong strides;
//   * the arch gate asks for gfx950 instead of sm_70 (:21-23).
#include <torch/extension.h>
#include <ATen/hip/EmptyTensor.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPCachingAllocator.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPGraphsC10Utils.h>
#include <c10/hip/HIPStream.h>
#include <hip/hip_runtime_api.h>
#include <torch/csrc/jit/frontend/tracer.h>

#include <algorithm>
#include <atomic>
#include <cmath>
#include <cstring>
#include <vector>

#include "fused_mha.h"
#include "fmha_internal.h"

#define CHECK_DEVICE(x) TORCH_CHECK(x.is_cuda(), #x " must be on the GPU")
#define CHECK_SHAPE(x, ...) \
  TORCH_CHECK(x.sizes() == torch::IntArrayRef({__VA_ARGS__}), #x " must have shape (" #__VA_ARGS__ ")")

namespace {

void check_arch(int device) {
  // The property query copies a structure of more than a kilobyte; the answer never changes.
  static std::atomic<bool> known_gfx950[64];
  if (device >= 0 && device < 64 && known_gfx950[device].load(std::memory_order_relaxed)) return;
  hipDeviceProp_t prop;
  TORCH_CHECK(hipGetDeviceProperties(&prop, device) == hipSuccess, "hipGetDeviceProperties failed");
  TORCH_CHECK(std::strncmp(prop.gcnArchName, "gfx950", 6) == 0, "This repo only supports gfx950 (MI355X) GPUs, got ",
              prop.gcnArchName);
  if (device >= 0 && device < 64) known_gfx950[device].store(true, std::memory_order_relaxed);
}

void check_rc(int rc, const char* what) {
  TORCH_CHECK(rc == FUSED_MHA_OK, what, " failed: ", fused_mha_error_string(rc));
}

// torch.empty without the dispatcher, which costs more than the allocation itself.
at::Tensor gpu_empty(at::IntArrayRef size, at::ScalarType dtype, const at::Tensor& like) {
  return at::Tensor(at::detail::empty_cuda(size, dtype, like.device(), std::nullopt));
}

at::Tensor dense(const at::Tensor& x) { return x.is_contiguous() ? x : x.contiguous(); }

// A (batch, seqlen, heads, head_size) input as the kernels take it: the tensor
// itself with its strides when they qualify (last dimension contiguous, rows on
// 16-byte boundaries; e.g. a slice of a packed QKV projection or a
// (batch, heads, seqlen, head_size)-backed view), otherwise a dense copy.  The
// reference copies (flash_attn_interface.py:14-15) or mis-reads such inputs.
struct Operand {
  const void* ptr;
  fused_mha_strides st;
  at::Tensor copy;  // undefined where the tensor itself is read
  explicit Operand(const at::Tensor& x) : ptr(x.data_ptr()), st{x.stride(0), x.stride(1), x.stride(2)} {
    const int64_t sb = st.batch, sn = st.seq, sh = st.head;
    const bool ok = x.stride(3) == 1 && sb >= 0 && sn >= 0 && sh >= 0 && ((sb | sn | sh) & 7) == 0 &&
                    sn < (int64_t(1) << 24) && sh < (int64_t(1) << 31) && (reinterpret_cast<uintptr_t>(ptr) & 15u) == 0;
    if (ok) return;
    copy = x.contiguous();
    ptr = copy.data_ptr();
    st = {copy.stride(0), copy.stride(1), copy.stride(2)};
  }
};

// Makes the device of a tensor the current one, which it nearly always is: asking is cheaper than setting it and back.
struct OnDeviceOf {
  c10::OptionalDeviceGuard guard;
  explicit OnDeviceOf(const at::Tensor& x) {
    if (c10::hip::current_device() != x.get_device()) guard.reset_device(x.device());
  }
};

// From this size on (where the backward takes about a millisecond) it is worth asking what memory there is.
constexpr size_t kLargeWorkspace = (size_t)1 << 30;

// How much of `wanted` bytes torch's allocator can hand out without giving back what it has cached: its largest free
// block, or half of what the device has left of this process's share.  Half, because whatever is allocated next needs
// its memory more than the backward, which only gets slower without it.  A free block of another stream counts too:
// then, and where nothing can be said (a graph capture has a pool of its own, other allocators may not answer), the
// allocation is tried and the caller handles its failure.  The current device must be `device`.
size_t workspace_room(c10::DeviceIndex device, size_t wanted) {
  namespace caching = c10::hip::HIPCachingAllocator;
  if (c10::hip::currentStreamCaptureStatusMayInitCtx() != c10::hip::CaptureStatus::None || caching::name() != "native")
    return wanted;
  size_t block = 1;  // with 0 the answer would take in what the device has left
  caching::cacheInfo(device, &block);
  if (block >= wanted) return wanted;
  size_t left = 0, total = 0;
  if (hipMemGetInfo(&left, &total) != hipSuccess) return block;
  constexpr auto kAll = static_cast<size_t>(c10::CachingAllocator::StatType::AGGREGATE);
  const double share = caching::getMemoryFraction(device) * (double)total;
  const double used = (double)caching::getDeviceStats(device).reserved_bytes[kAll].current;
  left = std::min(left, (size_t)std::max(share - used, 0.0));
  return std::min(wanted, std::max(block, left / 2));
}

}  // namespace

namespace {

// The forward; lse (batch x heads x seqlen, fp32) is not produced if nullptr.
at::Tensor forward(const at::Tensor& q,  // batch x seqlen x heads x head_size
                   const at::Tensor& k,  // batch x seqlen x heads x head_size
                   const at::Tensor& v,  // batch x seqlen x heads x head_size
                   const c10::optional<at::Tensor>& out_, at::Tensor* lse, const float softmax_scale, bool is_causal) {
  auto q_dtype = q.dtype();
  TORCH_CHECK(q_dtype == torch::kFloat16, "This repo only supports fp16 data type");
  TORCH_CHECK(k.dtype() == q_dtype, "query and key must have the same dtype");
  TORCH_CHECK(v.dtype() == q_dtype, "query and value must have the same dtype");

  TORCH_CHECK(q.dim() == 4, "query must have 4 dimensions (batch, seqlen, heads, head_size)");
  TORCH_CHECK(k.dim() == 4 && v.dim() == 4, "key and value must have 4 dimensions");
  TORCH_CHECK(q.stride(-1) == 1, "Input tensor must have contiguous last dimension");
  TORCH_CHECK(k.stride(-1) == 1, "Input tensor must have contiguous last dimension");
  TORCH_CHECK(v.stride(-1) == 1, "Input tensor must have contiguous last dimension");

  const auto sizes = q.sizes();
  const int batch_size = sizes[0];
  const int seqlen_q = sizes[1];
  const int num_heads = sizes[2];
  const int head_size = sizes[3];
  TORCH_CHECK(batch_size > 0, "batch size must be postive");
  TORCH_CHECK(head_size == 64 || head_size == 128, "current repo only supports head dimension 64 or 128");
  TORCH_CHECK(seqlen_q > 0, "seqlen must be positive");
  CHECK_SHAPE(q, batch_size, seqlen_q, num_heads, head_size);
  CHECK_SHAPE(k, batch_size, seqlen_q, num_heads, head_size);
  CHECK_SHAPE(v, batch_size, seqlen_q, num_heads, head_size);

  CHECK_DEVICE(q); CHECK_DEVICE(k); CHECK_DEVICE(v);
  check_arch(q.get_device());

  at::Tensor out;
  if (out_.has_value()) {
    out = out_.value();
    TORCH_CHECK(out.dtype() == q_dtype, "Output must have the same dtype as inputs");
    CHECK_DEVICE(out);
    TORCH_CHECK(out.is_contiguous(), "Output tensor must be contiguous");
    CHECK_SHAPE(out, batch_size, seqlen_q, num_heads, head_size);
  } else {
    out = gpu_empty({batch_size, seqlen_q, num_heads, head_size}, at::kHalf, q);
  }

  const OnDeviceOf device_guard(q);
  const Operand qo(q), ko(k), vo(v);
  hipStream_t stream = c10::hip::getCurrentHIPStream().stream();
  if (lse) {
    *lse = gpu_empty({batch_size, num_heads, seqlen_q}, at::kFloat, q);
    check_rc(fused_mha_forward_strided(qo.ptr, &qo.st, ko.ptr, &ko.st, vo.ptr, &vo.st,
                                       out.data_ptr(), lse->data_ptr(), batch_size, num_heads, seqlen_q, head_size,
                                       softmax_scale, is_causal ? 1 : 0, stream),
             "fused_mha_forward");
  } else {
    check_rc(fmha_forward_without_lse(qo.ptr, &qo.st, ko.ptr, &ko.st, vo.ptr, &vo.st,
                                      out.data_ptr(), batch_size, num_heads, seqlen_q, head_size, softmax_scale,
                                      is_causal ? 1 : 0, stream),
             "fused_mha_forward");
  }
  return out;
}

}  // namespace

std::vector<at::Tensor> mha_fwd(const at::Tensor& q, const at::Tensor& k, const at::Tensor& v,
                                const c10::optional<at::Tensor>& out_, const float softmax_scale, bool is_causal) {
  at::Tensor lse;
  at::Tensor out = forward(q, k, v, out_, &lse, softmax_scale, is_causal);
  return {out, lse};
}

std::vector<at::Tensor> mha_bwd(const at::Tensor& dout,  // batch x seqlen x heads x head_size
                                const at::Tensor& q, const at::Tensor& k, const at::Tensor& v,
                                const at::Tensor& out,   // batch x seqlen x heads x head_size
                                const at::Tensor& lse,   // batch x heads x seqlen, fp32
                                c10::optional<at::Tensor>& dq_, c10::optional<at::Tensor>& dk_,
                                c10::optional<at::Tensor>& dv_, const float softmax_scale, const bool is_causal) {
  auto q_dtype = q.dtype();
  TORCH_CHECK(q_dtype == torch::kFloat16, "This repo only supports fp16 data type");
  TORCH_CHECK(k.dtype() == q_dtype, "query and key must have the same dtype");
  TORCH_CHECK(v.dtype() == q_dtype, "query and value must have the same dtype");
  TORCH_CHECK(out.dtype() == q_dtype, "query and out must have the same dtype");
  TORCH_CHECK(dout.dtype() == q_dtype, "query and dout must have the same dtype");
  TORCH_CHECK(lse.dtype() == torch::kFloat32, "lse must be fp32");

  TORCH_CHECK(q.dim() == 4, "query must have 4 dimensions (batch, seqlen, heads, head_size)");
  TORCH_CHECK(k.dim() == 4 && v.dim() == 4, "key and value must have 4 dimensions");
  TORCH_CHECK(out.dim() == 4 && dout.dim() == 4, "out and dout must have 4 dimensions");
  TORCH_CHECK(q.stride(-1) == 1, "Input tensor must have contiguous last dimension");
  TORCH_CHECK(k.stride(-1) == 1, "Input tensor must have contiguous last dimension");
  TORCH_CHECK(v.stride(-1) == 1, "Input tensor must have contiguous last dimension");
  TORCH_CHECK(dout.stride(-1) == 1, "Input tensor must have contiguous last dimension");

  const auto sizes = q.sizes();
  const int batch_size = sizes[0];
  const int seqlen_q = sizes[1];
  const int num_heads = sizes[2];
  const int head_size = sizes[3];
  TORCH_CHECK(batch_size > 0, "batch size must be postive");
  TORCH_CHECK(head_size == 64 || head_size == 128, "current repo only supports head dimension 64 or 128");
  TORCH_CHECK(seqlen_q > 0, "seqlen must be positive");
  CHECK_SHAPE(q, batch_size, seqlen_q, num_heads, head_size);
  CHECK_SHAPE(k, batch_size, seqlen_q, num_heads, head_size);
  CHECK_SHAPE(v, batch_size, seqlen_q, num_heads, head_size);
  CHECK_SHAPE(out, batch_size, seqlen_q, num_heads, head_size);
  CHECK_SHAPE(dout, batch_size, seqlen_q, num_heads, head_size);
  CHECK_SHAPE(lse, batch_size, num_heads, seqlen_q);

  CHECK_DEVICE(q); CHECK_DEVICE(k); CHECK_DEVICE(v);
  CHECK_DEVICE(out); CHECK_DEVICE(dout); CHECK_DEVICE(lse);
  check_arch(q.get_device());

  const OnDeviceOf device_guard(q);
  auto grad_like = [&](c10::optional<at::Tensor>& g, const char* name) {
    if (g.has_value()) {
      at::Tensor t = g.value();
      TORCH_CHECK(t.dtype() == q_dtype, name, " must have the same dtype as q");
      TORCH_CHECK(t.is_cuda(), name, " must be on the GPU");
      TORCH_CHECK(t.is_contiguous(), name, " must be contiguous");
      TORCH_CHECK(t.sizes() == q.sizes(), name, " must have the shape of q");
      return t;
    }
    return gpu_empty({batch_size, seqlen_q, num_heads, head_size}, at::kHalf, q);
  };
  at::Tensor dq = grad_like(dq_, "dq"), dk = grad_like(dk_, "dk"), dv = grad_like(dv_, "dv");

  const Operand qo(q), ko(k), vo(v), go(dout);
  at::Tensor od = dense(out), ld = dense(lse);
  // Statistics, and at head size 128 room for dS; a large one only as far as it is there for the taking.
  const size_t min_bytes = fused_mha_backward_min_workspace_bytes(batch_size, num_heads, seqlen_q, head_size);
  const size_t wanted = fmha_backward_workspace_for(batch_size, num_heads, seqlen_q, head_size, is_causal ? 1 : 0);
  size_t ws_bytes = wanted;
  if (ws_bytes >= kLargeWorkspace)
    ws_bytes = fmha_backward_workspace_within(batch_size, num_heads, seqlen_q, head_size,
                                              workspace_room(q.get_device(), ws_bytes));
  if (ws_bytes == wanted)
    ws_bytes += fmha_backward_count_bytes(batch_size, num_heads, seqlen_q, head_size, is_causal ? 1 : 0);
  at::Tensor workspace;
  try {
    workspace = gpu_empty({(int64_t)ws_bytes}, at::kByte, q);
  } catch (const c10::OutOfMemoryError&) {
    if (ws_bytes == min_bytes) throw;
    ws_bytes = min_bytes;
    workspace = gpu_empty({(int64_t)ws_bytes}, at::kByte, q);
  }
  hipStream_t stream = c10::hip::getCurrentHIPStream().stream();
  check_rc(fused_mha_backward_strided(qo.ptr, &qo.st, ko.ptr, &ko.st, vo.ptr, &vo.st,
                                      od.data_ptr(), go.ptr, &go.st, ld.data_ptr(), workspace.data_ptr(),
                                      ws_bytes, dq.data_ptr(), dk.data_ptr(), dv.data_ptr(), batch_size, num_heads,
                                      seqlen_q, head_size, softmax_scale, is_causal ? 1 : 0, stream),
           "fused_mha_backward");
  return {dq, dk, dv};
}

namespace {

c10::MaybeOwned<at::Tensor> last_dim_contiguous(const at::Tensor& x) {
  return x.stride(-1) == 1 ? c10::MaybeOwned<at::Tensor>::borrowed(x) : c10::MaybeOwned<at::Tensor>::owned(x.contiguous());
}

// The autograd node of flash_attn_func.  Native on purpose: a torch.autograd.Function written in Python
// costs about 60 us per forward and backward, most of it in handing the interpreter lock to the engine's
// device thread and back, which is more than the kernels of a small problem take.
class AttentionNode : public torch::autograd::Function<AttentionNode> {
 public:
  static at::Tensor forward(torch::autograd::AutogradContext* ctx, const at::Tensor& q_in, const at::Tensor& k_in,
                            const at::Tensor& v_in, double softmax_scale, bool is_causal) {
    const auto q = last_dim_contiguous(q_in), k = last_dim_contiguous(k_in), v = last_dim_contiguous(v_in);
    at::Tensor lse;
    at::Tensor out = ::forward(*q, *k, *v, c10::nullopt, &lse, (float)softmax_scale, is_causal);
    ctx->save_for_backward(torch::autograd::variable_list{*q, *k, *v, out, lse});
    ctx->saved_data["softmax_scale"] = softmax_scale;
    ctx->saved_data["causal"] = is_causal;
    return out;
  }

  static torch::autograd::variable_list backward(torch::autograd::AutogradContext* ctx,
                                                 torch::autograd::variable_list grad_out) {
    const auto saved = ctx->get_saved_variables();
    c10::optional<at::Tensor> none_q, none_k, none_v;
    auto grads = mha_bwd(*last_dim_contiguous(grad_out[0]), saved[0], saved[1], saved[2], saved[3], saved[4], none_q,
                         none_k, none_v, (float)ctx->saved_data["softmax_scale"].toDouble(),
                         ctx->saved_data["causal"].toBool());
    return {grads[0], grads[1], grads[2], at::Tensor(), at::Tensor()};
  }
};

}  // namespace

// flash_attn_func: attention with its gradient.  softmax_scale defaults to head_size ** -0.5.
at::Tensor attention(const at::Tensor& q, const at::Tensor& k, const at::Tensor& v,
                     c10::optional<double> softmax_scale, bool is_causal) {
  const double scale = softmax_scale.has_value() ? *softmax_scale : std::pow((double)q.size(-1), -0.5);
  // A tangent (forward-mode differentiation) goes to the node too, whatever the grad mode: it refuses it.
  const auto has_tangent = [](const at::Tensor& x) { return x._fw_grad(/*level=*/0).defined(); };
  if ((at::GradMode::is_enabled() && (q.requires_grad() || k.requires_grad() || v.requires_grad())) ||
      has_tangent(q) || has_tangent(k) || has_tangent(v))
    return AttentionNode::apply(q, k, v, scale, is_causal);
  return forward(*last_dim_contiguous(q), *last_dim_contiguous(k), *last_dim_contiguous(v), c10::nullopt, nullptr,
                 (float)scale, is_causal);
}

// An argument and what the caller gave for it.  While torch.jit.trace records a tensor is not converted: a scale that is one is an
// input of the recorded node then, and its value at that time would be a constant of the graph.  Plain values, which are the
// rule, are converted without asking (small calls wait for the host: asking for each option costs 0.05 of their 4.6 us).
template <typename T>
struct __attribute__((visibility("hidden"))) Given {  // as pybind11's handles are
  py::handle object;
  T value{};
};
namespace pybind11::detail {
template <typename T>
struct type_caster<Given<T>> {
  PYBIND11_TYPE_CASTER(Given<T>, make_caster<T>::name);
  bool load(handle src, bool convert) {
    value.object = src;
    const bool plain = src.is_none() || PyBool_Check(src.ptr()) || PyFloat_CheckExact(src.ptr());
    if (!plain && torch::jit::tracer::isTracing()) return true;
    make_caster<T> caster;
    if (!caster.load(src, convert)) return false;
    value.value = cast_op<T>(std::move(caster));
    return true;
  }
};
}  // namespace pybind11::detail

// What flash_attn_func calls.  torch.jit.trace records a Python autograd function as a node, and would keep what this module
// returns as a constant: under it the call goes to the function in Python, with the options as they were given.
py::object flash_attn(const at::Tensor& q, const at::Tensor& k, const at::Tensor& v,
                      const Given<c10::optional<double>>& softmax_scale, const Given<bool>& is_causal) {
  if (torch::jit::tracer::isTracing())
    return py::module_::import("flash_attn_v100.flash_attn_interface")
        .attr("FlashAttnFunc").attr("apply")(q, k, v, softmax_scale.object, is_causal.object);
  return py::cast(attention(q, k, v, softmax_scale.value, is_causal.value));
}

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  m.doc() = "FlashAttention forward/backward for gfx950";
  m.def("attention", &flash_attn, "Attention, differentiable in q, k and v, also under torch.jit.trace");
  m.def("fwd", &mha_fwd, "Forward pass");
  m.def("bwd", &mha_bwd, "Backward pass");
}
