// The quantized linears and the HQQ product on the native host path (contract and reasons: host.h).
#include <ATen/autocast_mode.h>

#include "host.h"

using namespace ao_host;

namespace {

bool bias_ok(const Tensor& bias, int64_t N) { return !bias.defined() || (bias.numel() == N && bias.is_contiguous()); }

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
        AO_CALL(ao_amd_int4wo_linear_auto_bytes(ptr(x), r.M, K, r.ld, N, g, AO_BF16, &need));
        if (need) ws = workspace(need, a.device);
        AO_CALL(ao_amd_int4wo_linear_auto(ptr(x), r.M, K, r.ld, ptr(packed), ptr(qparams), N, g, ptr(bias), y.data_ptr(), AO_BF16, N,
                                          need ? ws.data_ptr() : nullptr, need, stream_of(a.device)));
        return THPVariable_Wrap(std::move(y));
    });
}

// (x, w_int8, scale, bias, weight or None): bf16(bf16(x @ w^T) * scale) (+ bias)
PyObject* int8wo_linear(PyObject*, PyObject* const* v, Py_ssize_t nargs) {
    AO_NEED(5);
    const Tensor &x = a.tensor(0, at::kBFloat16), &w = a.tensor(1, at::kChar), &scale = a.tensor(2, at::kBFloat16);
    const Tensor& bias = a.tensor(3, at::kBFloat16, true);
    AO_WANT(a.ok && current(a.device));
    const Rows r(x);
    AO_WANT(r.ok && w.dim() == 2 && w.size(1) == r.K && w.stride(1) == 1 && w.stride(0) % 16 == 0 && r.K % 64 == 0);
    const int64_t N = w.size(0);
    // without the kernel an odd multiple of 64 runs torch.mm, which autocast casts; the operator of the others it leaves alone
    AO_WANT(r.K % 128 == 0 || !at::autocast::is_autocast_enabled(at::kCUDA));
    AO_WANT(stands_for_bf16_matrix(v[4], N, r.K) && scale.numel() == N && scale.is_contiguous() && bias_ok(bias, N));
    return guarded([&]() -> PyObject* {
        Tensor y = empty_rows(x, N, at::kBFloat16), ws;
        int64_t need = 0;
        AO_CALL(ao_amd_int8wo_linear_ws_bytes(r.M, r.K, N, &need));
        if (need) ws = workspace(need, a.device);
        AO_CALL(ao_amd_int8wo_linear_ws(ptr(x), r.M, r.K, r.ld, ptr(w), w.stride(0), ptr(scale), N, ptr(bias), y.data_ptr(), AO_BF16, N,
                                        need ? ws.data_ptr() : nullptr, need, stream_of(a.device)));
        return THPVariable_Wrap(std::move(y));
    });
}

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
        AO_CALL(ao_amd_fp6_linear_auto_bytes(r.M, r.K, N, &need));
        if (need) ws = workspace(need, a.device);
        AO_CALL(ao_amd_fp6_linear_auto(ptr(x), r.M, r.K, ptr(native), ptr(scale), N, (int)e, (int)m, y.data_ptr(),
                                       need ? ws.data_ptr() : nullptr, need, stream_of(a.device)));
        return THPVariable_Wrap(std::move(y));
    });
}

// (a, codes, scales, zeros, group_size, transposed): the fused products over HQQ codes, of up to 64 rows or, MANY, of more by its tiles where
// they are faster than the dequantized weight and torch.matmul, which autocast casts
template <bool MANY>
PyObject* hqq_product(PyObject* const* v, Py_ssize_t nargs) {
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
    AO_WANT(x.size(1) == R && x.stride(1) == 1 && x.stride(0) % 8 == 0 && (uintptr_t)ptr(x) % 16 == 0 && M >= 1 && MANY == (M > 64) &&
            scales.size(0) * g == K && scales.size(1) == N);
    AO_WANT(transposed ? N % 16 == 0 && g % 2 == 0 : K % 8 == 0 && g % 8 == 0 && N % 4 == 0);
    const int code = dtype == at::kBFloat16 ? AO_BF16 : AO_F16;
    if (MANY) {
        AO_WANT(!at::autocast::is_autocast_enabled(at::kCUDA) && x.stride(0) < ((int64_t)1 << 24));
        int64_t need = -1;
        AO_CALL(ao_amd_hqq_mixed_mm_tiled_bytes(M, K, N, g, code, transposed, &need));
        AO_WANT(need >= 0);
        return guarded([&]() -> PyObject* {
            Tensor y = empty({M, transposed ? K : N}, dtype, a.device), ws;
            if (need) ws = workspace(need, a.device);
            AO_CALL(ao_amd_hqq_mixed_mm_tiled(ptr(x), M, x.stride(0), ptr(b), is_signed, K, N, ptr(scales), ptr(zeros), g, code, transposed,
                                              need ? ws.data_ptr() : nullptr, need, y.data_ptr(), stream_of(a.device)));
            return THPVariable_Wrap(std::move(y));
        });
    }
    return guarded([&]() -> PyObject* {
        int64_t need = 0;
        AO_CALL(ao_amd_hqq_mixed_mm_mfma_workspace(M, K, N, transposed, &need));
        Tensor y = empty({M, transposed ? K : N}, dtype, a.device), ws = workspace(need, a.device);
        AO_CALL(ao_amd_hqq_mixed_mm_mfma(ptr(x), M, x.stride(0), ptr(b), is_signed, K, N, ptr(scales), ptr(zeros), g, code,
                                         transposed, ws.data_ptr(), need, y.data_ptr(), stream_of(a.device)));
        return THPVariable_Wrap(std::move(y));
    });
}

PyObject* hqq_mixed_mm(PyObject*, PyObject* const* v, Py_ssize_t nargs) { return hqq_product<false>(v, nargs); }
PyObject* hqq_mixed_mm_many(PyObject*, PyObject* const* v, Py_ssize_t nargs) { return hqq_product<true>(v, nargs); }

#define AO_METHOD(f) {#f, (PyCFunction)(void (*)(void))f, METH_FASTCALL, nullptr}
PyMethodDef methods[] = {
    AO_METHOD(int4wo_linear),
    AO_METHOD(int8wo_linear),
    AO_METHOD(fp6_linear),
    AO_METHOD(hqq_mixed_mm),
    AO_METHOD(hqq_mixed_mm_many),
    {"llama_forward", (PyCFunction)(void (*)(void))llama_forward, METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "ao_amd_host", "Native host path of the ao_amd operators.", -1, methods};

}  // namespace

PyMODINIT_FUNC PyInit_ao_amd_host() { return PyModule_Create(&module); }
