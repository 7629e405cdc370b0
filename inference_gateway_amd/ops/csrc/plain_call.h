// Whether a product may go to a kernel here in place of the library's, which
// autograd, vmap, a trace, a dispatch mode and autocast see.
#pragma once
#include <ATen/autocast_mode.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <torch/extension.h>

namespace igw {

inline bool call_is_plain() {
  using K = c10::DispatchKey;
  const auto seen = c10::impl::tls_local_dispatch_key_set().included_;
  return !seen.has_any(c10::DispatchKeySet(
             {K::Python, K::PythonTLSSnapshot, K::FuncTorchVmapMode,
              K::FuncTorchDynamicLayerFrontMode, K::FuncTorchBatched,
              K::Functionalize, K::Tracer})) &&
         !at::autocast::is_autocast_enabled(at::kCUDA);
}

inline bool plain_bf16(const torch::Tensor& t, c10::Device where) {
  using K = c10::DispatchKey;
  return t.defined() && t.scalar_type() == torch::kBFloat16 &&
         t.layout() == torch::kStrided && t.device() == where &&
         !t.key_set().has_any(c10::DispatchKeySet(
             {K::Python, K::FuncTorchBatched, K::FuncTorchGradWrapper,
              K::Functionalize, K::ZeroTensor, K::NestedTensor})) &&
         !(at::GradMode::is_enabled() && t.requires_grad()) &&
         !t._fw_grad(0).defined();
}

}  // namespace igw
