// Native host path of the eager operators: argument checks, output and workspace allocation and the launch in one call
// from Python, without the torch.library dispatcher and the per-operator Python checks behind it.
//
// What bounds it: a quantized linear of a few rows runs 5-20 us on the GPU, and the same call through
// torch.ops -> Python implementation -> ctypes took 18-26 us of host time, so a program that launches linears one after
// the other ran at the host's pace (4096 -> 1024, one row: 21.8 us a call for a 5.2 us kernel).
//
// Contract of every function here: it serves the plain case (exact torch.Tensor or Parameter arguments on one GPU,
// dtypes, shapes and strides as the kernels take them, no gradient to record, no mode, transform or trace active) and
// returns NotImplemented for everything else *before* it does anything.  The caller then takes the torch.library route,
// which reports errors, records for torch.compile, and covers the rare layouts.  Nothing is raised here.
#include <Python.h>

#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/hip/EmptyTensor.h>
#include <ATen/hip/HIPContext.h>
#include <ATen/core/grad_mode.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/hip/HIPFunctions.h>
#include <torch/csrc/autograd/python_variable.h>

#include "ao_amd.h"

namespace {

using at::Tensor;

PyObject* not_implemented() {
    Py_INCREF(Py_NotImplemented);
    return Py_NotImplemented;
}

bool only(c10::DispatchKeySet keys, c10::DispatchKeySet of) { return (keys.raw_repr() & ~of.raw_repr()) == 0; }

// Nothing may want to see this call: no torch function mode, and no dispatch key forced by a mode, transform or tracer.
bool nothing_watches() {
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
    const Tensor& tensor(int i, at::ScalarType dtype, bool optional = false) {
        static const Tensor none;
        static const c10::DispatchKeySet plain = c10::DispatchKeySet(c10::DispatchKey::CUDA) |
                                                 c10::DispatchKeySet(c10::DispatchKey::AutogradCUDA) |
                                                 c10::DispatchKeySet(c10::DispatchKey::AutocastCUDA) |
                                                 c10::DispatchKeySet(c10::DispatchKey::ADInplaceOrView);
        if (optional && v[i] == Py_None) return none;
        if (!THPVariable_CheckExact(v[i])) return fail(none);
        const Tensor& t = THPVariable_Unpack(v[i]);
        if (!t.defined() || t.scalar_type() != dtype || !only(t.key_set(), plain) || !t.is_cuda()) return fail(none);
        if (device < 0) device = t.get_device();
        if (t.get_device() != device || (grad && t.requires_grad())) return fail(none);
        return t;
    }
    // Tensor of one of two 16-bit types
    const Tensor& tensor16(int i, at::ScalarType& dtype) {
        dtype = THPVariable_CheckExact(v[i]) && THPVariable_Unpack(v[i]).defined() &&
                        THPVariable_Unpack(v[i]).scalar_type() == at::kHalf ? at::kHalf : at::kBFloat16;
        return tensor(i, dtype);
    }
    int64_t integer(int i) {
        const int64_t r = PyLong_Check(v[i]) ? PyLong_AsLongLong(v[i]) : -1;
        if (r < 0) {
            PyErr_Clear();
            ok = false;
        }
        return r;
    }
    double real(int i) {
        const double r = PyFloat_AsDouble(v[i]);
        if (r == -1.0 && PyErr_Occurred()) {
            PyErr_Clear();
            ok = false;
        }
        return r;
    }
    bool truth(int i) { return v[i] == Py_True; }

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

Tensor empty(at::IntArrayRef sizes, at::ScalarType dtype, c10::DeviceIndex device) {
    return Tensor(at::detail::empty_cuda(sizes, dtype, c10::Device(c10::kCUDA, device), std::nullopt));
}
// x's sizes with the last one replaced
Tensor empty_rows(const Tensor& x, int64_t n, at::ScalarType dtype) {
    c10::SmallVector<int64_t, 5> sizes(x.sizes().begin(), x.sizes().end());
    sizes.back() = n;
    return empty(sizes, dtype, x.get_device());
}
Tensor workspace(int64_t bytes, c10::DeviceIndex device) { return empty({(bytes + 3) / 4}, at::kFloat, device); }

hipStream_t stream_of(c10::DeviceIndex device) { return c10::hip::getCurrentHIPStream(device).stream(); }

// Launches go to the current device's context: a tensor of another device takes the guarded torch.library route.
bool current(c10::DeviceIndex device) { return device >= 0 && c10::hip::current_device() == device; }

const void* ptr(const Tensor& t) { return t.defined() ? t.const_data_ptr() : nullptr; }

bool bias_ok(const Tensor& bias, int64_t N) { return !bias.defined() || (bias.numel() == N && bias.is_contiguous()); }

bool int4_weight_ok(const Tensor& packed, const Tensor& qparams, int64_t N, int64_t K, int64_t g) {
    if (!(g == 32 || g == 64 || g == 128 || g == 256) || N < 1 || K < 1) return false;
    const int64_t q = g > 128 ? g : 128, Kp = (K + q - 1) / q * q, rb = (N + 15) / 16;
    return packed.dim() == 4 && packed.size(0) == rb && packed.size(1) == Kp / 128 && packed.size(2) == 64 && packed.size(3) == 4 &&
           packed.is_contiguous() && qparams.dim() == 3 && qparams.size(0) == rb && qparams.size(1) == Kp / g &&
           qparams.size(2) == 16 && qparams.is_contiguous();
}

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
#define AO_WANT(cond) \
    if (!(cond)) return not_implemented()
#define AO_CALL(call) \
    if ((call) != 0) return not_implemented()

// The weight a linear stands for: a bf16 matrix as the model sees it.  Read off the tensor itself, whatever its Python
// class; None where the caller passes the kernel's operands directly.
bool stands_for_bf16_matrix(PyObject* weight, int64_t N, int64_t K) {
    if (weight == Py_None) return true;
    if (!THPVariable_Check(weight)) return false;
    const Tensor& w = THPVariable_Unpack(weight);
    return w.defined() && w.scalar_type() == at::kBFloat16 && w.dim() == 2 && w.size(0) == N && w.size(1) == K &&
           !(at::GradMode::is_enabled() && w.requires_grad());
}

// (x, packed, qparams, group_size, N, K, bias, weight or None): x bf16 [..., K] -> bf16 [..., N]
PyObject* int4wo_linear(PyObject*, PyObject* const* v, Py_ssize_t nargs) {
    AO_NEED(8);
    const Tensor &x = a.tensor(0, at::kBFloat16), &packed = a.tensor(1, at::kInt), &qparams = a.tensor(2, at::kInt);
    const int64_t g = a.integer(3), N = a.integer(4), K = a.integer(5);
    const Tensor& bias = a.tensor(6, at::kBFloat16, true);
    AO_WANT(a.ok && current(a.device) && stands_for_bf16_matrix(v[7], N, K));
    const Rows r(x);
    AO_WANT(r.ok && r.K == K && int4_weight_ok(packed, qparams, N, K, g) && bias_ok(bias, N));
    return guarded([&]() -> PyObject* {
        Tensor y = empty_rows(x, N, at::kBFloat16), ws;
        int64_t need = 0;
        if (r.M >= 16 && r.M <= 256) {
            AO_CALL(ao_amd_int4wo_linear_ws_bytes(r.M, K, N, g, &need));
            if (need) ws = workspace(need, a.device);
        }
        hipStream_t st = stream_of(a.device);
        if (need) {
            AO_CALL(ao_amd_int4wo_linear_ws(ptr(x), r.M, K, r.ld, ptr(packed), ptr(qparams), N, g, ptr(bias), y.data_ptr(), AO_BF16,
                                            N, ws.data_ptr(), need, st));
        } else {
            AO_CALL(ao_amd_int4wo_linear(ptr(x), r.M, K, r.ld, ptr(packed), ptr(qparams), N, g, ptr(bias), y.data_ptr(), AO_BF16, N, st));
        }
        return THPVariable_Wrap(std::move(y));
    });
}

// (x, w_int8, scale, bias, weight or None): bf16(bf16(x @ w^T) * scale) (+ bias) on the streaming kernels
PyObject* int8wo_linear(PyObject*, PyObject* const* v, Py_ssize_t nargs) {
    AO_NEED(5);
    const Tensor &x = a.tensor(0, at::kBFloat16), &w = a.tensor(1, at::kChar), &scale = a.tensor(2, at::kBFloat16);
    const Tensor& bias = a.tensor(3, at::kBFloat16, true);
    AO_WANT(a.ok && current(a.device));
    const Rows r(x);
    AO_WANT(r.ok && w.dim() == 2 && w.size(1) == r.K && w.stride(1) == 1 && w.stride(0) % 16 == 0 && r.K % 128 == 0);
    const int64_t N = w.size(0);
    AO_WANT(stands_for_bf16_matrix(v[4], N, r.K) && scale.numel() == N && scale.is_contiguous() && bias_ok(bias, N));
    return guarded([&]() -> PyObject* {
        Tensor y = empty_rows(x, N, at::kBFloat16);
        AO_CALL(ao_amd_int8wo_linear(ptr(x), r.M, r.K, r.ld, ptr(w), w.stride(0), ptr(scale), N, ptr(bias), y.data_ptr(), AO_BF16, N,
                                     stream_of(a.device)));
        return THPVariable_Wrap(std::move(y));
    });
}

int64_t fp6_native_words(int64_t N, int64_t K) { return N / 16 * ((K + 127) / 128) * 384; }

// (ebits, mbits, x, native, scale): x fp16 [..., K] -> fp16 [..., N]
PyObject* fp6_linear(PyObject*, PyObject* const* v, Py_ssize_t nargs) {
    AO_NEED(5);
    const int64_t e = a.integer(0), m = a.integer(1);
    const Tensor &x = a.tensor(2, at::kHalf), &native = a.tensor(3, at::kInt), &scale = a.tensor(4, at::kHalf);
    AO_WANT(a.ok && current(a.device));
    const Rows r(x);
    AO_WANT(r.ok && r.ld == r.K && scale.dim() == 1 && scale.is_contiguous() && native.is_contiguous());
    const int64_t N = scale.size(0);
    AO_WANT(native.numel() == fp6_native_words(N, r.K));
    return guarded([&]() -> PyObject* {
        Tensor y = empty_rows(x, N, at::kHalf), ws;
        int64_t need = 0;
        if (r.M >= 16 && r.M <= 256) {
            AO_CALL(ao_amd_fp6_linear_ws_bytes(r.M, r.K, N, &need));
            if (need) ws = workspace(need, a.device);
        }
        hipStream_t st = stream_of(a.device);
        if (need) {
            AO_CALL(ao_amd_fp6_linear_ws(ptr(x), r.M, r.K, ptr(native), ptr(scale), N, (int)e, (int)m, y.data_ptr(), ws.data_ptr(), need, st));
        } else {
            AO_CALL(ao_amd_fp6_linear(ptr(x), r.M, r.K, ptr(native), ptr(scale), N, (int)e, (int)m, y.data_ptr(), st));
        }
        return THPVariable_Wrap(std::move(y));
    });
}

// (a, codes, scales, zeros, group_size, transposed): the fused matrix-core product over HQQ codes
PyObject* hqq_mixed_mm(PyObject*, PyObject* const* v, Py_ssize_t nargs) {
    AO_NEED(6);
    at::ScalarType dtype;
    const Tensor& x = a.tensor16(0, dtype);
    const bool is_signed = THPVariable_CheckExact(v[1]) && THPVariable_Unpack(v[1]).defined() && THPVariable_Unpack(v[1]).scalar_type() == at::kChar;
    const Tensor& b = a.tensor(1, is_signed ? at::kChar : at::kByte);
    const Tensor &scales = a.tensor(2, dtype), &zeros = a.tensor(3, dtype);
    const int64_t g = a.integer(4);
    const bool transposed = a.truth(5);
    AO_WANT(a.ok && current(a.device));
    AO_WANT(g > 0 && x.dim() == 2 && b.dim() == 2 && b.is_contiguous() && scales.dim() == 2 && scales.is_contiguous() && zeros.is_contiguous() &&
            scales.sizes() == zeros.sizes());
    const int64_t M = x.size(0), K = 2 * b.size(0), N = b.size(1), R = transposed ? N : K;
    AO_WANT(x.size(1) == R && x.stride(1) == 1 && x.stride(0) % 8 == 0 && (uintptr_t)ptr(x) % 16 == 0 && M >= 1 && M <= 64 &&
            scales.size(0) * g == K && scales.size(1) == N);
    AO_WANT(transposed ? N % 16 == 0 && g % 2 == 0 : K % 8 == 0 && g % 8 == 0 && N % 4 == 0);
    return guarded([&]() -> PyObject* {
        int64_t need = 0;
        AO_CALL(ao_amd_hqq_mixed_mm_mfma_workspace(M, K, N, transposed, &need));
        Tensor y = empty({M, transposed ? K : N}, dtype, a.device), ws = workspace(need, a.device);
        AO_CALL(ao_amd_hqq_mixed_mm_mfma(ptr(x), M, x.stride(0), ptr(b), is_signed, K, N, ptr(scales), ptr(zeros), g,
                                         dtype == at::kBFloat16 ? AO_BF16 : AO_F16, transposed, ws.data_ptr(), need, y.data_ptr(),
                                         stream_of(a.device)));
        return THPVariable_Wrap(std::move(y));
    });
}

#define AO_METHOD(f) {#f, (PyCFunction)(void (*)(void))f, METH_FASTCALL, nullptr}
PyMethodDef methods[] = {
    AO_METHOD(int4wo_linear),
    AO_METHOD(int8wo_linear),
    AO_METHOD(fp6_linear),
    AO_METHOD(hqq_mixed_mm),
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "ao_amd_host", "Native host path of the ao_amd operators.", -1, methods};

}  // namespace

PyMODINIT_FUNC PyInit_ao_amd_host() { return PyModule_Create(&module); }
