// Products around a short batch of tokens (gemm/narrow_gemm.hip), for the modules that have them.
#pragma once
#include <torch/extension.h>
#include <ATen/autocast_mode.h>
#include <ATen/hip/HIPContext.h>
#include <hip/hip_runtime_api.h>

#include <initializer_list>

extern "C" {
int ds_narrow_gemm_ok(int64_t, int64_t, int64_t, int64_t, int64_t, int, int);
int64_t ds_narrow_gemm_scratch(int64_t, int64_t, int64_t, int, int);
int ds_narrow_gemm_pays(int64_t, int64_t, int64_t, int, int);
int ds_narrow_gemm(const void*, const void*, void*, int64_t, int64_t, int64_t, int64_t, int64_t, int, int, void*, hipStream_t);
void ds_narrow_gemm_tune(int, int);
int ds_wide_gemm_pays(int64_t, int64_t, int64_t, int, int);
void ds_wide_gemm_tune(int, int);
void ds_wide_plan(int64_t, int64_t, int64_t, int, int64_t*);
int ds_wide_gated_pays(int64_t, int64_t, int64_t);
int ds_wide_gated(const void*, const void*, void*, int64_t, int64_t, int64_t, int64_t, hipStream_t);
}

namespace {
using torch::Tensor;

// No transform, dispatch mode, tracer or autocast has to see what becomes of these tensors, and none carries a tangent or a lazy bit or is
// anything but strided (asked first: such tensors may have no sizes)
bool unseen(std::initializer_list<const Tensor*> ts) {
  using K = c10::DispatchKey;
  static const c10::DispatchKeySet special({K::Python, K::PythonTLSSnapshot, K::FuncTorchBatched, K::FuncTorchGradWrapper, K::Batched,
                                            K::Functionalize, K::Conjugate, K::Negative, K::ZeroTensor});
  if (!(c10::impl::tls_local_dispatch_key_set().included_ - c10::default_included_set).empty() || at::autocast::is_autocast_enabled(at::kCUDA))
    return false;
  for (const Tensor* t : ts)
    if (t->defined() && (t->key_set().has_any(special) || t->layout() != at::kStrided || t->is_nested() || t->_fw_grad(0).defined())) return false;
  return true;
}
// ... nor autograd
bool unwatched(const Tensor& a, const Tensor& b) {
  return !(at::GradMode::is_enabled() && (a.requires_grad() || b.requires_grad())) && unseen({&a, &b});
}

// A B^T over the inner dimension: a [M, K], or [K, M] if not a_along; b [N, K], or [K, N]. Whether the kernels take it as it lies.
bool narrow_sizes(const Tensor& a, const Tensor& b, bool a_along, bool b_along, int64_t& M, int64_t& N, int64_t& K, int64_t& lda, int64_t& ldb) {
  if (!a.is_cuda() || a.device() != b.device() || a.scalar_type() != at::kBFloat16 || b.scalar_type() != at::kBFloat16 || a.dim() != 2 || b.dim() != 2 ||
      a.stride(1) != 1 || b.stride(1) != 1)
    return false;
  M = a.size(a_along ? 0 : 1), K = a.size(a_along ? 1 : 0), N = b.size(b_along ? 0 : 1);
  lda = a.size(0) > 1 ? a.stride(0) : a.size(1), ldb = b.size(0) > 1 ? b.stride(0) : b.size(1);
  return b.size(b_along ? 1 : 0) == K && ds_narrow_gemm_ok(M, N, K, lda, ldb, a_along, b_along) &&
         !((uintptr_t)a.const_data_ptr() % 16 || (uintptr_t)b.const_data_ptr() % 16);
}

// The product. Undefined where the kernels do not take it or (unless asked to take what they can) the library's is faster. sizes: the result's where it
// is no matrix (a view of one, made in an autograd function, could not be changed in place).
Tensor narrow_product(const Tensor& a, const Tensor& b, bool a_along, bool b_along, bool any, at::OptionalIntArrayRef sizes = c10::nullopt) {
  int64_t M, N, K, lda, ldb;
  if (!narrow_sizes(a, b, a_along, b_along, M, N, K, lda, ldb) || (!any && !ds_narrow_gemm_pays(M, N, K, a_along, b_along))) return Tensor();
  const char *pa = (const char*)a.const_data_ptr(), *pb = (const char*)b.const_data_ptr();
  const c10::DeviceGuard guard(a.device());  // (the stream below is the tensors' device's, whichever is current)
  Tensor c = torch::empty(sizes ? *sizes : at::IntArrayRef{M, N}, a.options());
  const int64_t scratch = ds_narrow_gemm_scratch(M, N, K, a_along, b_along);
  const Tensor part = scratch ? torch::empty({scratch}, a.options().dtype(at::kByte)) : Tensor();
  const int rc = ds_narrow_gemm(pa, pb, c.data_ptr(), M, N, K, lda, ldb, a_along, b_along, scratch ? part.data_ptr() : nullptr,
                                at::hip::getCurrentHIPStream().stream());
  TORCH_CHECK(rc == 0, "narrow_gemm failed: ", hipGetErrorString((hipError_t)rc));
  return c;
}

// x [.., I] W [O, I]^T
Tensor linear_product(Tensor x, Tensor w) {
  if (unwatched(x, w) && x.dim() >= 2 && x.is_contiguous() && w.dim() == 2 && x.size(-1) == w.size(1) && x.numel()) {
    auto sizes = x.sizes().vec();
    sizes.back() = w.size(0);
    const Tensor y = narrow_product(x.view({-1, x.size(-1)}), w, true, true, false, sizes);
    if (y.defined()) return y;
  }
  return at::linear(x, w);
}
}  // namespace
