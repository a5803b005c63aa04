// The Monarch layer's differentiable op as a native torch operator: mmuon::butterfly_linear
// (x2, w1, w2) -> (out, out1) and mmuon::butterfly_linear_bwd, over the C ABI's
// mmuon_butterfly_linear_fwd / _bwd.
//
// Why native: at 1000 tokens of the toy model the kernels of a forward and backward take
// 57 us, but the Python form of the op (argument checks, allocations, two custom-op
// dispatches, ctypes calls) took 190 us of host time, so the GPU waited for the host up
// to about 4000 tokens of the 1.3B layers.
//
// The library's functions are bound at the first launch (loader, mmuon_torch_bind) to the
// ones that monarch_muon_amd/_abi.py loads, so MMUON_LIB selects them here too; a library of
// another ABI than this file was compiled with is refused.
#include <ATen/ATen.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/library.h>

#include <algorithm>
#include <atomic>
#include <mutex>
#include <string>
#include <tuple>

#include "../../include/mmuon.h"

namespace {

using at::Tensor;
using Pair = std::tuple<Tensor, Tensor>;
using Triple = std::tuple<Tensor, Tensor, Tensor>;

struct Abi {
  int (*fwd)(const mmuon_butterfly_args*, void*) = nullptr;
  int (*bwd)(const mmuon_butterfly_args*, void*) = nullptr;
  size_t (*workspace)(const mmuon_butterfly_args*) = nullptr;
  const char* (*last_error)() = nullptr;
} abi;
std::atomic<bool> bound{false};
int (*loader)() = nullptr;         // loads the library and binds it; 0 where it did
thread_local std::string refusal;  // why it did not

void bind_library() {
  if (bound.load(std::memory_order_acquire)) return;
  refusal = "libmmuon.so is not loaded";
  TORCH_CHECK(loader != nullptr && loader() == 0, refusal);
}

void check_rc(int rc, const char* what) {
  TORCH_CHECK(rc == 0, what, " failed (code ", rc, "): ", abi.last_error());
}

void require_cuda(const Tensor& t) {
  TORCH_CHECK(t.is_cuda(), "libmmuon kernels need tensors on a ROCm GPU (no CPU path)");
}

mmuon_butterfly_args make_args(const Tensor& x2, const Tensor& w1, const Tensor& w2) {
  for (const Tensor* t : {&x2, &w1, &w2}) require_cuda(*t);
  const char* names[3] = {"x", "w1", "w2"};
  const Tensor* ts[3] = {&x2, &w1, &w2};
  for (int i = 0; i < 3; ++i)
    TORCH_CHECK_TYPE(ts[i]->scalar_type() == at::kBFloat16, "the MI355X butterfly computes in bfloat16; ", names[i],
                     " is torch.", c10::getDtypeNames(ts[i]->scalar_type()).first,
                     " (run under torch.autocast(dtype=torch.bfloat16) or pass bf16 tensors)");
  TORCH_CHECK_VALUE(w1.dim() == 3 && w2.dim() == 3 && x2.dim() == 2,
                    "expected x2 (B, n), w1 (k, q, p), w2 (l, s, r)");
  TORCH_CHECK_VALUE(w1.size(0) == w2.size(0) && w1.size(1) == w2.size(2) && x2.size(1) == w1.size(0) * w1.size(2),
                    "butterfly shapes do not chain: x2 ", x2.sizes(), ", w1 ", w1.sizes(), ", w2 ", w2.sizes(),
                    " (need k == l, q == r, n == k p)");
  // 32-bit sides in the C struct; the library checks their ranges
  TORCH_CHECK_VALUE(std::max({w1.size(0), w1.size(1), w1.size(2), w2.size(1)}) <= INT32_MAX,
                    "butterfly: block sides beyond 32 bits");
  bind_library();
  mmuon_butterfly_args a{};
  a.tokens = x2.size(0);
  a.nblocks = int32_t(w1.size(0));
  a.q = int32_t(w1.size(1));
  a.p = int32_t(w1.size(2));
  a.s = int32_t(w2.size(1));
  a.dtype = MMUON_BF16;
  a.x = x2.data_ptr();
  a.w1 = w1.data_ptr();
  a.w2 = w2.data_ptr();
  return a;
}

// The kernels read rows of 16-B chunks.  A gradient may be a contiguous view at any element
// (one of the parts that torch.cat's backward hands out): such a one is copied.
Tensor dense_aligned(const Tensor& t) {
  const Tensor c = t.contiguous();
  return reinterpret_cast<uintptr_t>(c.const_data_ptr()) % 16 == 0 ? c : c.clone();
}

void* stream_of(const Tensor& t) { return c10::hip::getCurrentHIPStream(t.device().index()).stream(); }

Pair linear_impl(const Tensor& x, const Tensor& w1_, const Tensor& w2_) {
  const Tensor x2 = x.contiguous(), w1 = w1_.contiguous(), w2 = w2_.contiguous();
  mmuon_butterfly_args a = make_args(x2, w1, w2);
  const c10::DeviceGuard guard(x2.device());
  Tensor out = at::empty({x2.size(0), w2.size(1) * w2.size(0)}, x2.options());
  Tensor out1 = at::empty({w2.size(0), x2.size(0), w2.size(2)}, x2.options());
  a.out = out.data_ptr();
  a.out1 = out1.data_ptr();
  check_rc(abi.fwd(&a, stream_of(x2)), "mmuon_butterfly_fwd");
  return {out, out1};
}

Triple linear_bwd_impl(const Tensor& x, const Tensor& w1_, const Tensor& w2_, const Tensor& out1_,
                       const Tensor& dout_) {
  const Tensor x2 = x.contiguous(), w1 = w1_.contiguous(), w2 = w2_.contiguous();
  const Tensor out1 = out1_.contiguous(), dout = dense_aligned(dout_);
  mmuon_butterfly_args a = make_args(x2, w1, w2);
  TORCH_CHECK_VALUE(out1.dim() == 3 && out1.size(0) == w2.size(0) && out1.size(1) == x2.size(0) &&
                        out1.size(2) == w2.size(2) && dout.dim() == 2 && dout.size(0) == x2.size(0) &&
                        dout.size(1) == w2.size(0) * w2.size(1),
                    "out1 ", out1.sizes(), " / dout ", dout.sizes(), " do not match the forward");
  TORCH_CHECK_TYPE(out1.scalar_type() == at::kBFloat16 && dout.scalar_type() == at::kBFloat16,
                   "out1 and dout must be bfloat16");
  require_cuda(out1);
  require_cuda(dout);
  const c10::DeviceGuard guard(x2.device());
  Tensor dx = at::empty(x2.sizes(), x2.options()), dw1 = at::empty(w1.sizes(), w1.options()),
         dw2 = at::empty(w2.sizes(), w2.options());
  a.out1 = out1.data_ptr();
  a.dout = dout.data_ptr();
  a.dx = dx.data_ptr();
  a.dw1 = dw1.data_ptr();
  a.dw2 = dw2.data_ptr();
  Tensor ws = at::empty({std::max<int64_t>(int64_t(abi.workspace(&a)), 256)}, x2.options().dtype(at::kByte));
  a.workspace = ws.data_ptr();
  a.workspace_bytes = size_t(ws.numel());
  check_rc(abi.bwd(&a, stream_of(x2)), "mmuon_butterfly_bwd");
  return {dx, dw1, dw2};
}

Pair call_linear(const Tensor& x2, const Tensor& w1, const Tensor& w2) {
  static auto op = c10::Dispatcher::singleton()
                       .findSchemaOrThrow("mmuon::butterfly_linear", "")
                       .typed<Pair(const Tensor&, const Tensor&, const Tensor&)>();
  return op.call(x2, w1, w2);
}
Triple call_linear_bwd(const Tensor& x2, const Tensor& w1, const Tensor& w2, const Tensor& out1, const Tensor& dout) {
  static auto op = c10::Dispatcher::singleton()
                       .findSchemaOrThrow("mmuon::butterfly_linear_bwd", "")
                       .typed<Triple(const Tensor&, const Tensor&, const Tensor&, const Tensor&, const Tensor&)>();
  return op.call(x2, w1, w2, out1, dout);
}

using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

struct LinearFn : torch::autograd::Function<LinearFn> {
  static variable_list forward(AutogradContext* ctx, const Tensor& x2, const Tensor& w1, const Tensor& w2) {
    at::AutoDispatchBelowADInplaceOrView below;
    auto [out, out1] = call_linear(x2, w1, w2);
    ctx->save_for_backward({x2, w1, w2, out1});
    // out1 is saved for the backward and has no gradient of its own: no zeros are made for it
    ctx->set_materialize_grads(false);
    return {out, out1};
  }
  static variable_list backward(AutogradContext* ctx, const variable_list& grads) {
    const variable_list saved = ctx->get_saved_variables();
    const Tensor &x2 = saved[0], &w1 = saved[1], &w2 = saved[2], &out1 = saved[3];
    Tensor dout = grads[0];
    if (!dout.defined()) dout = x2.new_zeros_symint({x2.sym_size(0), w2.sym_size(0) * w2.sym_size(1)});
    auto [dx, dw1, dw2] = call_linear_bwd(x2, w1, w2, out1, dout);
    return {dx, dw1, dw2};
  }
};

// The backward op has no derivative of its own.
struct LinearBwdFn : torch::autograd::Function<LinearBwdFn> {
  static variable_list forward(AutogradContext*, const Tensor& x2, const Tensor& w1, const Tensor& w2,
                               const Tensor& out1, const Tensor& dout) {
    at::AutoDispatchBelowADInplaceOrView below;
    auto [dx, dw1, dw2] = call_linear_bwd(x2, w1, w2, out1, dout);
    return {dx, dw1, dw2};
  }
  static variable_list backward(AutogradContext*, const variable_list&) {
    TORCH_CHECK(false, "Trying to backward through mmuon.butterfly_linear_bwd.default but no autograd formula was "
                       "registered.");
  }
};

bool any_requires_grad(std::initializer_list<const Tensor*> ts) {
  if (!at::GradMode::is_enabled()) return false;
  return std::any_of(ts.begin(), ts.end(), [](const Tensor* t) { return t->requires_grad(); });
}
Pair linear_autograd(const Tensor& x2, const Tensor& w1, const Tensor& w2) {
  if (any_requires_grad({&x2, &w1, &w2})) {
    const variable_list r = LinearFn::apply(x2, w1, w2);
    return {r[0], r[1]};
  }
  at::AutoDispatchBelowADInplaceOrView below;
  return call_linear(x2, w1, w2);
}

Triple linear_bwd_autograd(const Tensor& x2, const Tensor& w1, const Tensor& w2, const Tensor& out1,
                           const Tensor& dout) {
  if (any_requires_grad({&x2, &w1, &w2, &out1, &dout})) {
    const variable_list r = LinearBwdFn::apply(x2, w1, w2, out1, dout);
    return {r[0], r[1], r[2]};
  }
  at::AutoDispatchBelowADInplaceOrView below;
  return call_linear_bwd(x2, w1, w2, out1, dout);
}

}  // namespace

TORCH_LIBRARY_FRAGMENT(mmuon, m) {
  m.def("butterfly_linear(Tensor x2, Tensor w1, Tensor w2) -> (Tensor, Tensor)", {at::Tag::pt2_compliant_tag});
  m.def("butterfly_linear_bwd(Tensor x2, Tensor w1, Tensor w2, Tensor out1, Tensor dout) -> (Tensor, Tensor, Tensor)",
        {at::Tag::pt2_compliant_tag});
}
TORCH_LIBRARY_IMPL(mmuon, CompositeExplicitAutograd, m) {
  m.impl("butterfly_linear", linear_impl);
  m.impl("butterfly_linear_bwd", linear_bwd_impl);
}
TORCH_LIBRARY_IMPL(mmuon, Autograd, m) {
  m.impl("butterfly_linear", linear_autograd);
  m.impl("butterfly_linear_bwd", linear_bwd_autograd);
}

extern "C" {

void mmuon_torch_set_loader(int (*fn)()) { loader = fn; }

void mmuon_torch_refuse(const char* why) { refusal = why; }

int mmuon_torch_bind(int version, void* fwd, void* bwd, void* workspace, void* last_error) {
  if (version != MMUON_ABI_VERSION) {
    refusal = "the layer's operator was built for ABI " + std::to_string(MMUON_ABI_VERSION) + ", libmmuon.so has ABI " +
              std::to_string(version) + ": build both again with `python -m monarch_muon_amd.build`";
    return -1;
  }
  static std::mutex mutex;
  const std::lock_guard<std::mutex> lock(mutex);
  if (bound) return 0;  // by another thread's first call
  abi.fwd = reinterpret_cast<decltype(abi.fwd)>(fwd);
  abi.bwd = reinterpret_cast<decltype(abi.bwd)>(bwd);
  abi.workspace = reinterpret_cast<decltype(abi.workspace)>(workspace);
  abi.last_error = reinterpret_cast<decltype(abi.last_error)>(last_error);
  bound.store(true, std::memory_order_release);
  return 0;
}

}  // extern "C"
