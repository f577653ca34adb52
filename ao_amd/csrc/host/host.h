// Native host path of the eager operators: argument checks, output and workspace allocation and the launch in one call
// from Python, without the torch.library dispatcher and the per-operator Python checks behind it.
//
// What bounds it: a quantized linear of a few rows runs 5-20 us on the GPU, and the same call through
// torch.ops -> Python implementation -> ctypes took 18-26 us of host time, so a program that launches linears one after
// the other ran at the host's pace (4096 -> 1024, one row: 21.8 us a call for a 5.2 us kernel).
//
// Contract of every function here: it serves the plain case (exact torch.Tensor or Parameter arguments on one GPU, dtypes, shapes
// and strides as the kernels take them, no gradient or tangent to record, no mode, transform or trace active) and returns
// NotImplemented for everything else *before* it launches anything; only a pass of the model may find a shape that a kernel refuses
// later, and is then run again from its start by another route.  The caller takes the torch.library route, which reports errors,
// records for torch.compile, and covers the rare layouts.  Nothing is raised here.
#pragma once
#include <Python.h>

#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/hip/EmptyTensor.h>
#include <ATen/hip/HIPContext.h>
#include <ATen/core/grad_mode.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/hip/HIPFunctions.h>
#include <torch/csrc/autograd/python_variable.h>

#include "ao_amd.h"

namespace ao_host {

using at::Tensor;

inline PyObject* not_implemented() {
    Py_INCREF(Py_NotImplemented);
    return Py_NotImplemented;
}

inline bool only(c10::DispatchKeySet keys, c10::DispatchKeySet of) { return (keys.raw_repr() & ~of.raw_repr()) == 0; }

// Nothing may want to see this call: no torch function mode, and no dispatch key forced by a mode, transform or tracer.
inline bool nothing_watches() {
    static const c10::DispatchKeySet usual = c10::DispatchKeySet(c10::DispatchKey::BackendSelect) |
                                             c10::DispatchKeySet(c10::DispatchKey::ADInplaceOrView);
    return !at::impl::torch_function_mode_enabled() && only(c10::impl::tls_local_dispatch_key_set().included_, usual);
}

// The arguments of one call: every tensor() checks one argument, ok() is the conjunction.
struct Args {
    PyObject* const* v;
    bool ok = true;
    c10::DeviceIndex device = -1;
    bool grad = at::GradMode::is_enabled();

    // A dense GPU tensor of `dtype`, on the device of the others.  `optional`: None gives an undefined tensor.
    const Tensor& tensor(int i, at::ScalarType dtype, bool optional = false) { return tensor_of(v[i], dtype, optional); }
    const Tensor& tensor_of(PyObject* obj, at::ScalarType dtype, bool optional = false) {
        static const Tensor none;
        static const c10::DispatchKeySet plain = c10::DispatchKeySet(c10::DispatchKey::CUDA) |
                                                 c10::DispatchKeySet(c10::DispatchKey::AutogradCUDA) |
                                                 c10::DispatchKeySet(c10::DispatchKey::AutocastCUDA) |
                                                 c10::DispatchKeySet(c10::DispatchKey::ADInplaceOrView);
        if (optional && obj == Py_None) return none;
        if (!THPVariable_CheckExact(obj)) return fail(none);
        const Tensor& t = THPVariable_Unpack(obj);
        if (!t.defined() || t.scalar_type() != dtype || !only(t.key_set(), plain) || !t.is_cuda()) return fail(none);
        if (device < 0) device = t.get_device();
        // a tangent of forward-mode differentiation is recorded whatever the gradient mode
        if (t.get_device() != device || (grad && t.requires_grad()) || t._fw_grad(0).defined()) return fail(none);
        return t;
    }
    // Tensor of one of two 16-bit types
    const Tensor& tensor16(int i, at::ScalarType& dtype) {
        dtype = THPVariable_CheckExact(v[i]) && THPVariable_Unpack(v[i]).defined() &&
                        THPVariable_Unpack(v[i]).scalar_type() == at::kHalf ? at::kHalf : at::kBFloat16;
        return tensor(i, dtype);
    }
    int64_t integer(int i) { return integer_of(v[i]); }
    int64_t integer_of(PyObject* obj) {
        const int64_t r = PyLong_Check(obj) ? PyLong_AsLongLong(obj) : -1;
        if (r < 0) {
            PyErr_Clear();
            ok = false;
        }
        return r;
    }
    double real_of(PyObject* obj) {
        const double r = PyFloat_AsDouble(obj);
        if (r == -1.0 && PyErr_Occurred()) {
            PyErr_Clear();
            ok = false;
        }
        return r;
    }
    bool truth(int i) { return truth_of(v[i]); }
    bool truth_of(PyObject* obj) {
        if (obj != Py_True && obj != Py_False) ok = false;
        return obj == Py_True;
    }

 private:
    const Tensor& fail(const Tensor& none) {
        ok = false;
        return none;
    }
};

// Rows of activations: the last dimension contiguous, the leading ones collapsible to one row stride.
struct Rows {
    int64_t M = 0, K = 0, ld = 0;
    bool ok = false;
    explicit Rows(const Tensor& x) {
        const int64_t dim = x.dim();
        if (dim < 1) return;
        K = x.size(dim - 1);
        if (K < 1 || x.numel() < 1) return;
        M = x.numel() / K;
        if (x.is_contiguous())
            ld = K;
        else if (dim == 2 && x.stride(1) == 1)
            ld = x.stride(0);
        else
            return;
        ok = true;
    }
};

inline Tensor empty(at::IntArrayRef sizes, at::ScalarType dtype, c10::DeviceIndex device) {
    return Tensor(at::detail::empty_cuda(sizes, dtype, c10::Device(c10::kCUDA, device), std::nullopt));
}
// x's sizes with the last one replaced
inline Tensor empty_rows(const Tensor& x, int64_t n, at::ScalarType dtype) {
    c10::SmallVector<int64_t, 5> sizes(x.sizes().begin(), x.sizes().end());
    sizes.back() = n;
    return empty(sizes, dtype, x.get_device());
}
inline Tensor workspace(int64_t bytes, c10::DeviceIndex device) { return empty({(bytes + 3) / 4}, at::kFloat, device); }

inline hipStream_t stream_of(c10::DeviceIndex device) { return c10::hip::getCurrentHIPStream(device).stream(); }

// Launches go to the current device's context: a tensor of another device takes the guarded torch.library route.
inline bool current(c10::DeviceIndex device) { return device >= 0 && c10::hip::current_device() == device; }

inline const void* ptr(const Tensor& t) { return t.defined() ? t.const_data_ptr() : nullptr; }

template <typename F>
PyObject* guarded(F&& f) {
    try {
        return f();
    } catch (...) {  // an allocation that failed, for instance: the other route reports it
        PyErr_Clear();
        return not_implemented();
    }
}

#define AO_NEED(n)                                             \
    if (nargs != (n) || !nothing_watches()) return not_implemented(); \
    Args a{v}
#define AO_WANT(cond)                           \
    do {                                        \
        if (!(cond)) return not_implemented();  \
    } while (0)
#define AO_CALL(call) AO_WANT((call) == 0)

inline bool int4_weight_ok(const Tensor& packed, const Tensor& qparams, int64_t N, int64_t K, int64_t g) {
    if (!(g == 32 || g == 64 || g == 128 || g == 256) || N < 1 || K < 1) return false;
    const int64_t q = g > 128 ? g : 128, Kp = (K + q - 1) / q * q, rb = (N + 15) / 16;
    return packed.dim() == 4 && packed.size(0) == rb && packed.size(1) == Kp / 128 && packed.size(2) == 64 && packed.size(3) == 4 &&
           packed.is_contiguous() && qparams.dim() == 3 && qparams.size(0) == rb && qparams.size(1) == Kp / g &&
           qparams.size(2) == 16 && qparams.is_contiguous();
}

inline int64_t fp6_native_words(int64_t N, int64_t K) { return N / 16 * ((K + 127) / 128) * 384; }

// llama.cpp
PyObject* llama_forward(PyObject*, PyObject* const* v, Py_ssize_t nargs);

}  // namespace ao_host
