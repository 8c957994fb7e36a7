// Native kernels of the torch operators (namespace wan_hip) that ops.py defines, for the calls a
// program makes over and over: plain CUDA (HIP) tensors in the layout the kernels take.
//
// ops.py's Python functions stay the definition of every operator: they hold the checks and
// their error messages.  What is registered here for the CUDA key checks the same conditions,
// allocates the outputs and calls the C ABI; a call that does not meet them goes on to the Python
// function.  Nothing is launched in that case.  For the AutogradCUDA key, a call that needs no
// gradient goes straight to the kernels below autograd; any other goes through the operator's
// Python autograd kernel, as without this file.
//
// Why: a call took 20 us of host time (operator wrapper in Python 12, checks, ctypes and
// allocation 8) where the small kernels take 4; with these 6-8.
#include <ATen/ATen.h>
#include <ATen/core/dispatch/Dispatcher.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/GradMode.h>
#include <torch/library.h>

#include <limits>

#include "../../include/wan_attn.h"

namespace {

using at::Tensor;
using c10::DispatchKeySet;
using c10::IValue;
using c10::OperatorHandle;
using torch::jit::Stack;

// The operator's kernels for another backend than CUDA are the Python functions (the autograd
// kernel among them), which take tensors of any device.
void to_python(const OperatorHandle& op, DispatchKeySet ks, Stack* stack) {
  op.redispatchBoxed(ks.remove_backend(c10::BackendComponent::CUDABit) |
                         DispatchKeySet(c10::BackendComponent::CPUBit),
                     stack);
}

void autograd(const OperatorHandle& op, DispatchKeySet ks, Stack* stack) {
  if (c10::GradMode::is_enabled()) {
    const size_t n = op.schema().arguments().size();
    for (size_t i = stack->size() - n; i < stack->size(); ++i) {
      const IValue& v = (*stack)[i];
      if (v.isTensor() && v.toTensor().defined() && v.toTensor().requires_grad()) return to_python(op, ks, stack);
    }
  }
  op.redispatchBoxed(ks & c10::after_ADInplaceOrView_keyset, stack);
}

// The arguments of one call, and what the checks need of them.
struct Call {
  Stack* stack;
  size_t n, base;
  Call(const OperatorHandle& op, Stack* s)
      : stack(s), n(op.schema().arguments().size()), base(s->size() - n) {}

  const IValue& operator[](size_t i) const { return (*stack)[base + i]; }
  const Tensor& tensor(size_t i) const { return (*this)[i].toTensor(); }
  bool has(size_t i) const { return !(*this)[i].isNone(); }
  float real(size_t i) const { return static_cast<float>((*this)[i].toDouble()); }
  int64_t integer(size_t i) const { return (*this)[i].toInt(); }
  void* ptr(size_t i) const { return has(i) ? tensor(i).data_ptr() : nullptr; }

  void give(IValue a) {
    stack->resize(base);
    stack->push_back(std::move(a));
  }
  void give(IValue a, IValue b) {
    give(std::move(a));
    stack->push_back(std::move(b));
  }
};

// A kernel behind the check that every tensor is one: None for a tensor that is not optional arrives
// as an undefined one, and the Python function says so.
template <void (*kernel)(const OperatorHandle&, DispatchKeySet, Stack*)>
void defined(const OperatorHandle& op, DispatchKeySet ks, Stack* stack) {
  for (size_t i = stack->size() - op.schema().arguments().size(); i < stack->size(); ++i) {
    const IValue& v = (*stack)[i];
    if (v.isTensor() && !v.toTensor().defined()) return to_python(op, ks, stack);
  }
  kernel(op, ks, stack);
}

bool plain(const Tensor& t, at::ScalarType type, c10::Device dev) {
  return t.layout() == at::kStrided && t.scalar_type() == type && t.device() == dev;
}

bool aligned(const Tensor& t) { return reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0; }

// [B, L, H, 128], the channels contiguous
bool rows4(const Tensor& t, c10::Device dev) {
  return plain(t, at::kBFloat16, dev) && t.dim() == 4 && t.size(3) == 128 && t.numel() > 0 &&
         t.size(0) <= std::numeric_limits<int>::max() && t.size(1) <= std::numeric_limits<int>::max() &&
         t.stride(3) == 1 && t.stride(0) % 8 == 0 && t.stride(1) % 8 == 0 && t.stride(2) % 8 == 0 && aligned(t);
}

bool vec(const Tensor& t, int64_t n, at::ScalarType type, c10::Device dev) {
  return plain(t, type, dev) && t.numel() == n && t.is_contiguous();
}

// a contiguous, aligned bf16 tensor of these sizes
bool block(const Tensor& t, at::IntArrayRef sizes, c10::Device dev) {
  return plain(t, at::kBFloat16, dev) && t.sizes() == sizes && t.is_contiguous() && t.numel() > 0 && aligned(t);
}

bool small_int(int64_t v) { return v >= std::numeric_limits<int>::min() && v <= std::numeric_limits<int>::max(); }

bool qkv(const Call& c) {
  const Tensor &q = c.tensor(0), &k = c.tensor(1), &v = c.tensor(2);
  const auto dev = q.device();
  return dev.is_cuda() && rows4(q, dev) && rows4(k, dev) && rows4(v, dev) && k.sizes() == v.sizes() &&
         q.size(0) == k.size(0) && q.size(2) == k.size(2);
}

// cos / sin [L, 64] at arguments i and i + 1, both there or (where allowed) neither
bool rope(const Call& c, size_t i, int64_t L, c10::Device dev, bool optional = false) {
  if (optional && !c.has(i) && !c.has(i + 1)) return true;
  return c.has(i) && c.has(i + 1) && vec(c.tensor(i), L * 64, at::kFloat, dev) &&
         vec(c.tensor(i + 1), L * 64, at::kFloat, dev);
}

bool lengths(const Call& c, size_t i, int64_t B, c10::Device dev) {
  return !c.has(i) || vec(c.tensor(i), B, at::kInt, dev);
}

wan_tensor t4(const Tensor& t) { return wan_tensor{t.data_ptr(), t.stride(0), t.stride(1), t.stride(2)}; }

// The launch's device, its current stream, and allocation on it.
struct Site {
  at::AutoDispatchBelowADInplaceOrView below;
  c10::DeviceGuard guard;
  at::TensorOptions bf16;
  explicit Site(const Tensor& t) : guard(t.device()), bf16(t.options()) {}
  void* stream() const {
    return c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(guard.current_device().index()).stream();
  }
  Tensor rows(const Tensor& like) const { return at::empty(like.sizes(), bf16); }
  Tensor floats(at::IntArrayRef sizes) const { return at::empty(sizes, bf16.dtype(at::kFloat)); }
  Tensor bytes(size_t n) const { return at::empty({static_cast<int64_t>(n)}, bf16.dtype(at::kByte)); }
};

// Scratch that a call may do without: undefined for 0 bytes.
struct Scratch {
  Tensor t;
  size_t n;
  Scratch(const Site& s, size_t bytes) : n(bytes) {
    if (n != 0) t = s.bytes(n);
  }
  void* ptr() const { return n != 0 ? t.data_ptr() : nullptr; }
};

void check(const char* fn, int rc) {
  TORCH_CHECK(rc == 0, fn, " failed (code ", rc, "): ", wan_attn_last_error());
}

struct Dims {
  int B, Lq, H, Lk;
  Dims(const Tensor& q, const Tensor& k)
      : B((int)q.size(0)), Lq((int)q.size(1)), H((int)q.size(2)), Lk((int)k.size(1)) {}
};

// flash_self_attn(q, k, v, softmax_scale, actual_seqlen_k)
void flash_self_attn(const OperatorHandle& op, DispatchKeySet ks, Stack* stack) {
  Call c(op, stack);
  if (!qkv(c) || c.integer(4) > c.tensor(1).size(1) || !small_int(c.integer(4))) return to_python(op, ks, stack);
  const Tensor &q = c.tensor(0), &k = c.tensor(1), &v = c.tensor(2);
  const Dims d(q, k);
  const Site s(q);
  Tensor out = s.rows(q);
  const Scratch ws(s, wan_flash_attn_workspace(d.B, d.H, d.Lq, d.Lk));
  check("wan_flash_self_attn", wan_flash_self_attn_ws(t4(q), t4(k), t4(v), t4(out), d.B, d.H, d.Lq, d.Lk, 128, c.real(3),
                                                      (int)c.integer(4), ws.ptr(), ws.n, s.stream()));
  c.give(std::move(out));
}

// cross_attn(q, k, v, seqlen_k?, softmax_scale)
void cross_attn(const OperatorHandle& op, DispatchKeySet ks, Stack* stack) {
  Call c(op, stack);
  if (!qkv(c) || !lengths(c, 3, c.tensor(0).size(0), c.tensor(0).device())) return to_python(op, ks, stack);
  const Tensor &q = c.tensor(0), &k = c.tensor(1), &v = c.tensor(2);
  const Dims d(q, k);
  const Site s(q);
  Tensor out = s.rows(q);
  const Scratch ws(s, wan_flash_attn_workspace(d.B, d.H, d.Lq, d.Lk));
  check("wan_cross_attn", wan_cross_attn_ws(t4(q), t4(k), t4(v), t4(out), d.B, d.H, d.Lq, d.Lk, 128, c.real(4),
                                            static_cast<const int32_t*>(c.ptr(3)), ws.ptr(), ws.n, s.stream()));
  c.give(std::move(out));
}

// self_attn_fused(q, k, v, gamma_q, gamma_k, eps, cos, sin, softmax_scale)
void self_attn_fused(const OperatorHandle& op, DispatchKeySet ks, Stack* stack) {
  Call c(op, stack);
  const Tensor &q = c.tensor(0), &k = c.tensor(1), &v = c.tensor(2);
  const auto dev = q.device();
  if (!qkv(c) || k.size(1) != q.size(1) || !vec(c.tensor(3), q.size(2) * 128, at::kBFloat16, dev) ||
      !vec(c.tensor(4), q.size(2) * 128, at::kBFloat16, dev) || !rope(c, 6, q.size(1), dev))
    return to_python(op, ks, stack);
  const Dims d(q, k);
  const Site s(q);
  Tensor out = s.rows(q);
  const Scratch ws(s, wan_self_attn_fused_workspace(d.B, d.H, d.Lq));
  check("wan_self_attn_fused", wan_self_attn_fused(t4(q), t4(k), t4(v), t4(out), d.B, d.H, d.Lq, 128, c.ptr(3), c.ptr(4),
                                                   c.real(5), static_cast<const float*>(c.ptr(6)),
                                                   static_cast<const float*>(c.ptr(7)), c.real(8), ws.ptr(), ws.n,
                                                   s.stream()));
  c.give(std::move(out));
}

// self_attn_fused_sumsq(q, k, v, sumsq, gamma_q, gamma_k, eps, cos, sin, softmax_scale)
void self_attn_fused_sumsq(const OperatorHandle& op, DispatchKeySet ks, Stack* stack) {
  Call c(op, stack);
  const Tensor &q = c.tensor(0), &k = c.tensor(1), &v = c.tensor(2);
  const auto dev = q.device();
  if (!qkv(c) || k.size(1) != q.size(1) ||
      !vec(c.tensor(3), 4 * q.size(2) * q.size(0) * q.size(1), at::kFloat, dev) ||
      !vec(c.tensor(4), q.size(2) * 128, at::kBFloat16, dev) ||
      !vec(c.tensor(5), q.size(2) * 128, at::kBFloat16, dev) || !rope(c, 7, q.size(1), dev))
    return to_python(op, ks, stack);
  const Dims d(q, k);
  const Site s(q);
  const Tensor inv = s.floats({(int64_t)d.B * d.Lq}), khat = s.rows(q);
  Tensor out = s.rows(q);
  const Scratch ws(s, wan_flash_attn_workspace(d.B, d.H, d.Lq, d.Lq));
  const auto *cos = static_cast<const float*>(c.ptr(7)), *sin = static_cast<const float*>(c.ptr(8));
  float* inv_q = static_cast<float*>(inv.data_ptr());
  void* stream = s.stream();
  check("wan_rms_norm_qk_sumsq",
        wan_rms_norm_qk_sumsq(t4(k), khat.data_ptr(), d.B, d.Lq, d.H, 128, c.ptr(5), c.real(6), cos, sin,
                              static_cast<const float*>(c.ptr(3)), inv_q, stream));
  check("wan_flash_attn_qnorm",
        wan_flash_attn_qnorm_ws(t4(q), t4(khat), t4(v), t4(out), d.B, d.H, d.Lq, d.Lq, 128, inv_q, c.ptr(4), cos, sin,
                                c.real(9), nullptr, ws.ptr(), ws.n, stream));
  c.give(std::move(out));
}

// cross_attn_fused(q, k, v, gamma_q, eps, seqlen_k?, softmax_scale)
void cross_attn_fused(const OperatorHandle& op, DispatchKeySet ks, Stack* stack) {
  Call c(op, stack);
  const Tensor &q = c.tensor(0), &k = c.tensor(1), &v = c.tensor(2);
  const auto dev = q.device();
  if (!qkv(c) || !vec(c.tensor(3), q.size(2) * 128, at::kBFloat16, dev) || !lengths(c, 5, q.size(0), dev))
    return to_python(op, ks, stack);
  const Dims d(q, k);
  const Site s(q);
  const Scratch ws(s, wan_cross_attn_fused_workspace(d.B, d.H, d.Lq));
  Tensor out = s.rows(q);
  check("wan_cross_attn_fused",
        wan_cross_attn_fused(t4(q), t4(k), t4(v), t4(out), d.B, d.H, d.Lq, d.Lk, 128, c.ptr(3), c.real(4), c.real(6),
                             static_cast<const int32_t*>(c.ptr(5)), ws.ptr(), ws.n, s.stream()));
  c.give(std::move(out));
}

// flash_attn_qnorm(q, k, v, inv_rms_q, gamma_q, cos?, sin?, seqlen_k?, softmax_scale)
void flash_attn_qnorm(const OperatorHandle& op, DispatchKeySet ks, Stack* stack) {
  Call c(op, stack);
  const Tensor &q = c.tensor(0), &k = c.tensor(1), &v = c.tensor(2);
  const auto dev = q.device();
  if (!qkv(c) || !vec(c.tensor(3), q.size(0) * q.size(1), at::kFloat, dev) ||
      !vec(c.tensor(4), q.size(2) * 128, at::kBFloat16, dev) || !rope(c, 5, q.size(1), dev, true) ||
      !lengths(c, 7, q.size(0), dev))
    return to_python(op, ks, stack);
  const Dims d(q, k);
  const Site s(q);
  Tensor out = s.rows(q);
  const Scratch ws(s, wan_flash_attn_workspace(d.B, d.H, d.Lq, d.Lk));
  check("wan_flash_attn_qnorm",
        wan_flash_attn_qnorm_ws(t4(q), t4(k), t4(v), t4(out), d.B, d.H, d.Lq, d.Lk, 128,
                                static_cast<const float*>(c.ptr(3)), c.ptr(4), static_cast<const float*>(c.ptr(5)),
                                static_cast<const float*>(c.ptr(6)), c.real(8),
                                static_cast<const int32_t*>(c.ptr(7)), ws.ptr(), ws.n, s.stream()));
  c.give(std::move(out));
}

// rope(x, cos, sin)
void rope_op(const OperatorHandle& op, DispatchKeySet ks, Stack* stack) {
  Call c(op, stack);
  const Tensor& x = c.tensor(0);
  if (!x.device().is_cuda() || !rows4(x, x.device()) || !rope(c, 1, x.size(1), x.device()))
    return to_python(op, ks, stack);
  const Dims d(x, x);
  const Site s(x);
  Tensor out = s.rows(x);
  check("wan_rope", wan_rope(t4(x), out.data_ptr(), d.B, d.Lq, d.H, 128, static_cast<const float*>(c.ptr(1)),
                             static_cast<const float*>(c.ptr(2)), s.stream()));
  c.give(std::move(out));
}

// rms_norm(x, gamma, eps, cos?, sin?)
void rms_norm(const OperatorHandle& op, DispatchKeySet ks, Stack* stack) {
  Call c(op, stack);
  const Tensor& x = c.tensor(0);
  const auto dev = x.device();
  if (!dev.is_cuda() || !rows4(x, dev) || !vec(c.tensor(1), x.size(2) * 128, at::kBFloat16, dev) ||
      !rope(c, 3, x.size(1), dev, true))
    return to_python(op, ks, stack);
  const Dims d(x, x);
  const Site s(x);
  Tensor out = s.rows(x);
  check("wan_rms_norm", wan_rms_norm(t4(x), out.data_ptr(), d.B, d.Lq, d.H, 128, c.ptr(1), c.real(2),
                                     static_cast<const float*>(c.ptr(3)), static_cast<const float*>(c.ptr(4)), nullptr,
                                     s.stream()));
  c.give(std::move(out));
}

// rms_inv(x, eps)
void rms_inv(const OperatorHandle& op, DispatchKeySet ks, Stack* stack) {
  Call c(op, stack);
  const Tensor& x = c.tensor(0);
  if (!x.device().is_cuda() || !rows4(x, x.device())) return to_python(op, ks, stack);
  const Dims d(x, x);
  const Site s(x);
  Tensor inv = s.floats({d.B, d.Lq});
  check("wan_rms_norm", wan_rms_norm(t4(x), nullptr, d.B, d.Lq, d.H, 128, nullptr, c.real(1), nullptr, nullptr,
                                     static_cast<float*>(inv.data_ptr()), s.stream()));
  c.give(std::move(inv));
}

// adaln(x, y?, e?, frames, gate_idx, shift_idx, scale_idx, ln_weight?, ln_bias?, eps, norm, e_mod?)
void adaln(const OperatorHandle& op, DispatchKeySet ks, Stack* stack) {
  Call c(op, stack);
  const Tensor& x = c.tensor(0);
  const auto dev = x.device();
  if (!dev.is_cuda() || x.dim() != 3 || !block(x, x.sizes(), dev) || x.size(0) > std::numeric_limits<int>::max() ||
      x.size(1) > std::numeric_limits<int>::max() || x.size(2) > std::numeric_limits<int>::max())
    return to_python(op, ks, stack);
  const int64_t C = x.size(2), frames = c.integer(3);
  int mod_rows = 6;
  bool ok = small_int(frames) && (!c.has(1) || block(c.tensor(1), x.sizes(), dev)) &&
            (!c.has(2) || block(c.tensor(2), {frames, 6, C}, dev)) && c.has(7) == c.has(8) &&
            (!c.has(7) || (block(c.tensor(7), {C}, dev) && block(c.tensor(8), {C}, dev)));
  for (size_t i = 4; i <= 6; ++i) ok = ok && small_int(c.integer(i));
  if (ok && c.has(11)) {
    const Tensor& m = c.tensor(11);
    ok = m.dim() == 3 && m.size(1) >= 1 && m.size(1) <= 6 && block(m, {frames, m.size(1), C}, dev);
    if (ok) mod_rows = (int)m.size(1);
  }
  if (!ok) return to_python(op, ks, stack);
  const bool norm = c[10].toBool();
  const Site s(x);
  Tensor r = c.has(1) ? s.rows(x) : at::empty({0}, s.bf16), h = norm ? s.rows(x) : at::empty({0}, s.bf16);
  check("wan_adaln_ex",
        wan_adaln_ex(x.data_ptr(), c.ptr(1), c.has(1) ? r.data_ptr() : nullptr, norm ? h.data_ptr() : nullptr,
                     (int)x.size(0), (int)x.size(1), (int)C, c.ptr(2), (int)frames, (int)c.integer(4), c.ptr(11),
                     mod_rows, (int)c.integer(5), (int)c.integer(6), c.ptr(7), c.ptr(8), c.real(9), s.stream()));
  c.give(std::move(r), std::move(h));
}

// qkv_proj_sumsq(x, weight, bias, sq_cols)
void qkv_proj_sumsq(const OperatorHandle& op, DispatchKeySet ks, Stack* stack) {
  Call c(op, stack);
  const Tensor &x = c.tensor(0), &w = c.tensor(1), &b = c.tensor(2);
  const auto dev = x.device();
  const int64_t sq = c.integer(3);
  if (!dev.is_cuda() || x.dim() != 3 || w.dim() != 2 || !block(x, x.sizes(), dev) ||
      !block(w, {w.size(0), x.size(2)}, dev) || !block(b, {w.size(0)}, dev) || !small_int(sq) || sq < 0 ||
      !small_int(x.size(0) * x.size(1)) || !small_int(x.size(2)) || !small_int(w.size(0)))
    return to_python(op, ks, stack);
  const int M = (int)(x.size(0) * x.size(1)), N = (int)w.size(0), K = (int)x.size(2);
  const Site s(x);
  Tensor out = at::empty({x.size(0), x.size(1), N}, s.bf16);
  Tensor sumsq = s.floats({std::max<int64_t>(sq / 64, 1), M});
  const Scratch ws(s, wan_qkv_proj_workspace(M, N, K));
  check("wan_qkv_proj_sumsq",
        wan_qkv_proj_sumsq_ws(x.data_ptr(), w.data_ptr(), b.data_ptr(), out.data_ptr(),
                              static_cast<float*>(sumsq.data_ptr()), M, N, K, K, K, N, (int)sq, ws.ptr(), ws.n,
                              s.stream()));
  c.give(std::move(out), std::move(sumsq));
}

// linear(x, weight, bias): what the kernel does not take (a misaligned weight among it) is torch's, in
// the Python function
void linear(const OperatorHandle& op, DispatchKeySet ks, Stack* stack) {
  Call c(op, stack);
  const Tensor &x = c.tensor(0), &w = c.tensor(1), &b = c.tensor(2);
  const auto dev = x.device();
  if (!dev.is_cuda() || x.dim() != 3 || w.dim() != 2 || !block(x, x.sizes(), dev) ||
      !block(w, {w.size(0), x.size(2)}, dev) || !block(b, {w.size(0)}, dev) || w.size(0) % 256 != 0 ||
      x.size(2) % 64 != 0 || x.size(2) >= int64_t(1) << 23 || !small_int(x.size(0) * x.size(1)) ||
      !small_int(w.size(0)))
    return to_python(op, ks, stack);
  const int M = (int)(x.size(0) * x.size(1)), N = (int)w.size(0), K = (int)x.size(2);
  const Site s(x);
  Tensor out = at::empty({x.size(0), x.size(1), N}, s.bf16);
  const Scratch ws(s, wan_qkv_proj_workspace(M, N, K));
  check("wan_qkv_proj_sumsq",
        wan_qkv_proj_sumsq_ws(x.data_ptr(), w.data_ptr(), b.data_ptr(), out.data_ptr(), nullptr, M, N, K, K, K, N, 0,
                              ws.ptr(), ws.n, s.stream()));
  c.give(std::move(out));
}

}  // namespace

#define WAN_OPS(X)                                                                                  \
  X("flash_self_attn", flash_self_attn) X("cross_attn", cross_attn) X("self_attn_fused", self_attn_fused) \
  X("self_attn_fused_sumsq", self_attn_fused_sumsq) X("cross_attn_fused", cross_attn_fused)         \
  X("flash_attn_qnorm", flash_attn_qnorm) X("rope", rope_op) X("rms_norm", rms_norm) X("rms_inv", rms_inv) \
  X("adaln", adaln) X("qkv_proj_sumsq", qkv_proj_sumsq) X("linear", linear)

TORCH_LIBRARY_IMPL(wan_hip, CUDA, m) {
#define WAN_IMPL(name, fn) m.impl(name, torch::CppFunction::makeFromBoxedFunction<&defined<&fn>>());
  WAN_OPS(WAN_IMPL)
#undef WAN_IMPL
}

TORCH_LIBRARY_IMPL(wan_hip, AutogradCUDA, m) {
#define WAN_IMPL(name, fn) m.impl(name, torch::CppFunction::makeFromBoxedFunction<&autograd>());
  WAN_OPS(WAN_IMPL)
#undef WAN_IMPL
}
