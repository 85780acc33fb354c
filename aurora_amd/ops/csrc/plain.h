// Which tensors a kernel may stand in for library operations on.
#pragma once
#include <c10/core/GradMode.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <torch/extension.h>

// True where nobody follows what is done with ``t``: no gradient is recorded, backward or
// forward, no transform (vmap, grad) or subclass wraps it, no trace or mode sees operations.
inline bool plain(const torch::Tensor& t) {
  using c10::DispatchKey;
  return !(c10::GradMode::is_enabled() && t.requires_grad()) &&
         !t.key_set().has_any(c10::DispatchKeySet(
             {DispatchKey::Python, DispatchKey::FuncTorchBatched,
              DispatchKey::FuncTorchGradWrapper, DispatchKey::Functionalize})) &&
         !c10::impl::tls_is_dispatch_key_included(DispatchKey::Tracer) &&
         !c10::impl::TorchDispatchModeTLS::any_modes_set() && !t._fw_grad(0).defined();
}
