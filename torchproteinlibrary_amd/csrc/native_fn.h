// native_fn.h -- what the layers' native autograd functions share.
//
// The Python autograd functions of the layers spend most of a small call in
// the interpreter, and more in the backward, which the engine runs on a thread
// of its own: RMSD of 8 structures, forward and backward, 131 us as a Python
// function and 95 as a native one, of which the kernels take 20.  So a plain
// eager call goes through a torch::autograd::Function here, and whatever is
// not plain (a tracer, a transform, a mode, a tensor subclass, a tangent) goes
// through the Python function as before.
#pragma once

#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/TracerMode.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <hip/hip_runtime.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/functions/basic_ops.h>
#include <torch/extension.h>

#include <cstdlib>
#include <cstring>
#include <initializer_list>
#include <memory>
#include <utility>

#include "host_flags.h"

namespace native_fn {

using torch::Tensor;
using torch::autograd::variable_list;

// Whether a call with these tensors (the first is the one that may need a
// gradient) is a plain eager one.
inline bool plain(std::initializer_list<const Tensor*> tensors) {
    if (at::tracer::impl::is_dispatch_enabled() || at::impl::torch_function_mode_enabled() ||
        c10::impl::TorchDispatchModeTLS::any_modes_set() ||
        c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::FuncTorchDynamicLayerFrontMode) ||
        c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::Functionalize))
        return false;
    const c10::DispatchKeySet special({c10::DispatchKey::Python, c10::DispatchKey::PythonTLSSnapshot,
                                       c10::DispatchKey::FuncTorchBatched, c10::DispatchKey::FuncTorchGradWrapper,
                                       c10::DispatchKey::Batched, c10::DispatchKey::Functionalize,
                                       c10::DispatchKey::ZeroTensor, c10::DispatchKey::Negative,
                                       c10::DispatchKey::Conjugate});
    bool first = true;
    for (const Tensor* t : tensors) {
        if (!t->defined() || !t->is_cuda() || t->layout() != torch::kStrided || t->is_nested() ||
            t->key_set().has_any(special) || t->_fw_grad(0).defined())
            return false;
        if (!first && t->requires_grad()) return false;
        first = false;
    }
    return true;
}

inline bool needs_grad(const Tensor& t) { return torch::GradMode::is_enabled() && t.requires_grad(); }

// Checks are on unless the environment turns them off or `stream` captures.
inline bool checks(hipStream_t stream) {
    const char* e = std::getenv("TPL_A2B_CHECKS");
    if (e && std::strcmp(e, "0") == 0) return false;
    hipStreamCaptureStatus s = hipStreamCaptureStatusNone;
    return hipStreamIsCapturing(stream, &s) == hipSuccess && s == hipStreamCaptureStatusNone;
}

// The status bits of launch(flags): 0 where checks are off.
template <typename Launch>
uint32_t run(hipStream_t stream, Launch launch) {
    if (checks(stream)) return host_flags::run(stream, launch);
    launch(nullptr);
    return 0;
}

// Lets the layer's Python code speak: module.function(args...), which raises
// or warns.
template <typename... Args>
void python(const char* module, const char* function, Args&&... args) {
    pybind11::gil_scoped_acquire gil;
    pybind11::module_::import(module).attr(function)(std::forward<Args>(args)...);
}

// The body of a backward.  It records nothing, an exception out of Python
// leaves it in the form that the engine hands to the calling thread, and
// gradients of its gradients are refused, as by once_differentiable.
template <typename Body>
variable_list backward(const variable_list& grads, Body body) {
    bool again = false;
    if (torch::GradMode::is_enabled())
        for (const Tensor& g : grads) again = again || (g.defined() && g.requires_grad());
    variable_list out;
    try {
        at::AutoGradMode off(false);
        out = body();
    } catch (pybind11::error_already_set& e) {
        pybind11::gil_scoped_acquire gil;
        e.restore();
        python_error err;
        err.persist();
        throw err;
    }
    if (!again) return out;
    variable_list some;
    for (Tensor& t : out)
        if (t.defined()) some.push_back(t.detach().set_requires_grad(true));
    const auto refuse = std::make_shared<torch::autograd::DelayedError>(
        "trying to differentiate twice a function that was marked with @once_differentiable", (int64_t)some.size());
    some = (*refuse)(std::move(some));
    size_t k = 0;
    for (Tensor& t : out)
        if (t.defined()) t = some[k++];
    return out;
}

inline Tensor like_dtype(const Tensor& grad, const Tensor& t) {
    const Tensor g = grad.contiguous();
    return g.scalar_type() == t.scalar_type() ? g : g.to(t.scalar_type());
}

}  // namespace native_fn
