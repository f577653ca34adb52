// One pass of the Llama-architecture model (batch 1) on the native host path: every launch of a decode step or of a prompt
// issued from one call.  A decode step is 5 launches a layer of 5-20 us each; issued operator by operator from Python they
// came 15 us apart, so a step that was not captured in a graph ran at the host's pace.
//
// The caller describes the model as nested tuples of tensors and numbers (Transformer._host_plan); they are checked
// completely before the first launch.
#include <ATen/autocast_mode.h>
#include <ATen/core/LegacyTypeDispatch.h>
#include <ATen/ops/embedding.h>
#include <ATen/ops/index.h>
#include <ATen/ops/linear.h>
#include <ATen/ops/mul.h>

#include <vector>

#include "host.h"

namespace ao_host {
namespace {

enum Kind { INT4 = 0, INT8 = 1, FP6 = 2 };

// (codes, scales, N, K, two_pass): packed + qparams, int8 + scale, or native + scale
struct Linear {
    Tensor codes, scales;
    int64_t N = 0, K = 0;
    bool two_pass = false;
};

struct Layer {
    Tensor attn_norm, ffn_norm, k_cache, v_cache;
    double attn_eps = 0, ffn_eps = 0;
    Linear wqkv, wo, w1, w3, w2;
    Tensor pair, pair_q;   // w1 and w3 interleaved (int4 decode)
};

struct Model {
    int kind = INT4, ebits = 0, mbits = 0;
    int64_t group = 0, n_head = 0, n_kv = 0, dim = 0, max_seq = 0, ksplit = 1;
    at::ScalarType dtype = at::kBFloat16;
    Tensor freqs, norm, cache_rows;
    double eps = 0;
    Linear output;
    std::vector<Layer> layers;
};

#define AO_TRY(call)                   \
    do {                               \
        if ((call) != 0) return false; \
    } while (0)

struct Reader {
    Args& a;
    PyObject* const* items = nullptr;
    Py_ssize_t n = 0, at = 0;
    Reader(Args& args, PyObject* tuple) : a(args) {
        if (PyTuple_Check(tuple)) {
            items = ((PyTupleObject*)tuple)->ob_item;
            n = PyTuple_GET_SIZE(tuple);
        } else {
            a.ok = false;
        }
    }
    PyObject* next() {
        if (at < n) return items[at++];
        a.ok = false;
        return Py_None;
    }
    Tensor tensor(at::ScalarType t, bool optional = false) { return a.tensor_of(next(), t, optional); }
    int64_t integer() { return a.integer_of(next()); }
    double real() { return a.real_of(next()); }
    bool truth() { return a.truth_of(next()); }
};

Linear read_linear(const Model& m, Args& a, PyObject* tuple) {
    Reader r(a, tuple);
    Linear l;
    l.codes = r.tensor(m.kind == INT8 ? at::kChar : at::kInt);
    l.scales = r.tensor(m.kind == INT4 ? at::kInt : m.kind == INT8 ? at::kBFloat16 : at::kHalf);
    l.N = r.integer();
    l.K = r.integer();
    l.two_pass = r.truth();
    if (!a.ok) return l;
    if (m.kind == INT4)
        a.ok = int4_weight_ok(l.codes, l.scales, l.N, l.K, m.group);
    else if (m.kind == INT8)
        a.ok = l.codes.dim() == 2 && l.codes.size(0) == l.N && l.codes.size(1) == l.K && l.codes.is_contiguous() && l.K % 128 == 0 &&
               l.scales.numel() == l.N && l.scales.is_contiguous();
    else
        a.ok = l.codes.numel() == fp6_native_words(l.N, l.K) && l.codes.is_contiguous() && l.scales.dim() == 1 && l.scales.numel() == l.N &&
               l.scales.is_contiguous();
    return l;
}

bool is_row(const Tensor& t, int64_t n) { return t.numel() == n && t.is_contiguous(); }

Layer read_layer(const Model& m, Args& a, PyObject* tuple) {
    Reader r(a, tuple);
    Layer l;
    l.attn_norm = r.tensor(m.dtype);
    l.attn_eps = r.real();
    l.wqkv = read_linear(m, a, r.next());
    l.wo = read_linear(m, a, r.next());
    l.k_cache = r.tensor(m.dtype);
    l.v_cache = r.tensor(m.dtype);
    l.ffn_norm = r.tensor(m.dtype);
    l.ffn_eps = r.real();
    l.w1 = read_linear(m, a, r.next());
    l.w3 = read_linear(m, a, r.next());
    l.w2 = read_linear(m, a, r.next());
    l.pair = r.tensor(at::kInt, true);
    l.pair_q = r.tensor(at::kInt, true);
    if (!a.ok) return l;
    const int64_t qkv = (m.n_head + 2 * m.n_kv) * 128, q = m.n_head * 128, ff = l.w1.N;
    auto cache_ok = [&](const Tensor& t) {
        return t.dim() == 4 && t.size(0) == 1 && t.size(1) == m.n_kv && t.size(2) == m.max_seq && t.size(3) == 128 && t.is_contiguous();
    };
    a.ok = is_row(l.attn_norm, m.dim) && is_row(l.ffn_norm, m.dim) && cache_ok(l.k_cache) && cache_ok(l.v_cache) && l.wqkv.N == qkv &&
           l.wqkv.K == m.dim && l.wo.N == m.dim && l.wo.K == q && l.w1.K == m.dim && l.w3.N == ff && l.w3.K == m.dim && l.w2.N == m.dim &&
           l.w2.K == ff && (!l.pair.defined() || int4_weight_ok(l.pair, l.pair_q, 2 * ff, m.dim, m.group));
    return l;
}

Model read_model(Args& a, PyObject* tuple) {
    Reader r(a, tuple);
    Model m;
    m.kind = (int)r.integer();
    m.ebits = (int)r.integer();
    m.mbits = (int)r.integer();
    m.group = r.integer();
    m.n_head = r.integer();
    m.n_kv = r.integer();
    m.ksplit = r.integer();
    if (m.kind == FP6) m.dtype = at::kHalf;
    m.freqs = r.tensor(m.dtype);
    PyObject* layers = r.next();
    m.norm = r.tensor(m.dtype);
    m.eps = r.real();
    PyObject* output = r.next();
    m.max_seq = r.integer();
    m.cache_rows = r.tensor(at::kInt);
    if (!a.ok || m.kind > FP6 || m.n_kv < 1 || m.n_head % m.n_kv || m.freqs.dim() != 3 || m.freqs.size(0) < m.max_seq ||
        m.freqs.size(1) != 64 || m.freqs.size(2) != 2 || !m.freqs.is_contiguous() || m.cache_rows.dim() != 1 ||
        m.cache_rows.size(0) != m.max_seq) {
        a.ok = false;
        return m;
    }
    m.output = read_linear(m, a, output);
    m.dim = m.output.K;
    Reader ls(a, layers);
    m.layers.reserve(ls.n);
    for (Py_ssize_t i = 0; i < ls.n && a.ok; ++i) m.layers.push_back(read_layer(m, a, ls.next()));
    a.ok = a.ok && m.dim % 8 == 0 && m.dim <= 8192 && is_row(m.norm, m.dim);
    return m;
}

// The launches of one pass.  Every method returns false where a kernel does not take the shape: the caller then runs its
// other route from the start (cache rows are written again with the same values).
struct Pass {
    const Model& m;
    c10::DeviceIndex device;
    hipStream_t st;
    bool f16 = m.kind == FP6;

    Tensor alloc(int64_t rows, int64_t cols) { return empty({rows, cols}, m.dtype, device); }

    bool linear(const Linear& l, const Tensor& x, int64_t M, Tensor& y) {
        if (l.two_pass) {
            // prefill-sized batches beyond the fused kernels: the weight once in 16 bits, then the library GEMM
            Tensor w = alloc(l.N, l.K);
            if (m.kind == INT4)
                AO_TRY(ao_amd_int4wo_dequantize(ptr(l.codes), ptr(l.scales), l.N, l.K, m.group, w.data_ptr(), st));
            else if (m.kind == INT8)
                AO_TRY(ao_amd_int8_to_bf16(ptr(l.codes), l.N, l.K, l.K, w.data_ptr(), st));
            else
                AO_TRY(ao_amd_fp6_native_to_f16(ptr(l.codes), ptr(l.scales), l.N, l.K, m.ebits, m.mbits, w.data_ptr(), st));
            y = at::linear(x, w);
            if (m.kind == INT8) y = at::mul(y, l.scales.view({l.N}));
            return true;
        }
        y = alloc(M, l.N);
        int64_t need = 0;
        if (m.kind == INT4)
            AO_TRY(ao_amd_int4wo_linear_auto_bytes(ptr(x), M, l.K, l.K, l.N, m.group, AO_BF16, &need));
        else if (m.kind == INT8)
            AO_TRY(ao_amd_int8wo_linear_ws_bytes(M, l.K, l.N, &need));
        else
            AO_TRY(ao_amd_fp6_linear_auto_bytes(M, l.K, l.N, &need));
        Tensor ws;
        if (need) ws = workspace(need, device);
        void* w = need ? ws.data_ptr() : nullptr;
        if (m.kind == INT4)
            return ao_amd_int4wo_linear_auto(ptr(x), M, l.K, l.K, ptr(l.codes), ptr(l.scales), l.N, m.group, nullptr, y.data_ptr(), AO_BF16,
                                             l.N, w, need, st) == 0;
        if (m.kind == INT8)
            return ao_amd_int8wo_linear_ws(ptr(x), M, l.K, l.K, ptr(l.codes), l.K, ptr(l.scales), l.N, nullptr, y.data_ptr(), AO_BF16, l.N, w,
                                           need, st) == 0;
        return ao_amd_fp6_linear_auto(ptr(x), M, l.K, ptr(l.codes), ptr(l.scales), l.N, m.ebits, m.mbits, y.data_ptr(), w, need, st) == 0;
    }

    // ---- one row: the norm, the residual and the gated product ride in the linears
    bool norm_linear(const Linear& l, const Tensor& x, const Tensor& w, double eps, Tensor& y) {
        y = alloc(1, l.N);
        if (m.kind == INT4)
            return ao_amd_int4wo_rmsnorm_linear(ptr(x), 1, l.K, l.K, ptr(w), (float)eps, ptr(l.codes), ptr(l.scales), l.N, m.group, nullptr,
                                                y.data_ptr(), AO_BF16, l.N, st) == 0;
        if (m.kind == INT8)
            return ao_amd_int8wo_rmsnorm_linear(ptr(x), 1, l.K, l.K, ptr(w), (float)eps, ptr(l.codes), l.K, ptr(l.scales), l.N, nullptr, l.N,
                                                y.data_ptr(), l.N, st) == 0;
        return ao_amd_fp6_rmsnorm_linear(ptr(x), 1, l.K, ptr(w), (float)eps, ptr(l.codes), ptr(l.scales), l.N, m.ebits, m.mbits, y.data_ptr(),
                                         st) == 0;
    }
    bool linear_add(const Linear& l, const Tensor& x, const Tensor& res, Tensor& y) {
        y = alloc(1, l.N);
        if (m.kind == INT4)
            return ao_amd_int4wo_linear_residual(ptr(x), 1, l.K, l.K, ptr(l.codes), ptr(l.scales), l.N, m.group, nullptr, ptr(res), l.N,
                                                 y.data_ptr(), l.N, st) == 0;
        if (m.kind == INT8)
            return ao_amd_int8wo_linear_residual(ptr(x), 1, l.K, l.K, ptr(l.codes), l.K, ptr(l.scales), l.N, ptr(res), l.N, y.data_ptr(),
                                                 l.N, st) == 0;
        return ao_amd_fp6_linear_fused(ptr(x), 1, l.K, ptr(l.codes), ptr(l.scales), l.N, m.ebits, m.mbits, ptr(res), nullptr, y.data_ptr(),
                                       st) == 0;
    }
    bool swiglu(const Layer& l, const Tensor& x, Tensor& y) {
        y = alloc(1, l.w1.N);
        const int64_t K = l.w1.K, N = l.w1.N;
        if (m.kind == INT4)
            return l.pair.defined() && ao_amd_int4wo_swiglu_interleaved(ptr(x), 1, K, K, ptr(l.ffn_norm), (float)l.ffn_eps, ptr(l.pair),
                                                                        ptr(l.pair_q), N, m.group, y.data_ptr(), N, st) == 0;
        if (m.kind == INT8)
            return ao_amd_int8wo_swiglu(ptr(x), 1, K, K, ptr(l.ffn_norm), (float)l.ffn_eps, ptr(l.w1.codes), ptr(l.w1.scales),
                                        ptr(l.w3.codes), ptr(l.w3.scales), K, N, y.data_ptr(), N, st) == 0;
        return ao_amd_fp6_swiglu(ptr(x), 1, K, ptr(l.ffn_norm), (float)l.ffn_eps, ptr(l.w1.codes), ptr(l.w1.scales), ptr(l.w3.codes),
                                 ptr(l.w3.scales), N, m.ebits, m.mbits, y.data_ptr(), st) == 0;
    }
    bool attend(const Tensor& qkv, int nparts, const Layer& l, const Tensor& pos, Tensor& y) {
        // workgroups per head: follows the cache length, since a graph freezes the launch (ops.decode_attention_splits)
        const int nsplit = m.max_seq <= 1024 ? 1 : m.max_seq <= 4096 ? 4 : m.max_seq <= 8192 ? 8 : 16;
        y = alloc(1, m.n_head * 128);
        Tensor ws;
        if (nsplit > 1) ws = workspace(m.n_head * nsplit * 130 * 4, device);
        void* w = nsplit > 1 ? ws.data_ptr() : nullptr;
        const int32_t* p = (const int32_t*)ptr(pos);
        if (f16)
            return ao_amd_llama_decode_attention_f16(ptr(qkv), ptr(m.freqs), p, l.k_cache.data_ptr(), l.v_cache.data_ptr(), (int)m.n_head,
                                                     (int)m.n_kv, 128, m.max_seq, nsplit, w, y.data_ptr(), st) == 0;
        return ao_amd_llama_decode_attention_split(nparts ? nullptr : ptr(qkv), nparts ? ptr(qkv) : nullptr, nparts, ptr(m.freqs), p,
                                                   l.k_cache.data_ptr(), l.v_cache.data_ptr(), (int)m.n_head, (int)m.n_kv, 128, m.max_seq,
                                                   nsplit, w, y.data_ptr(), st) == 0;
    }
    bool decode(Tensor x, const Tensor& pos, Tensor& logits) {
        for (const Layer& l : m.layers) {
            Tensor qkv, y, h, act;
            int nparts = 0;
            if (m.kind == INT4 && m.ksplit > 1) {
                nparts = (int)m.ksplit;
                qkv = empty({nparts, 1, l.wqkv.N}, at::kFloat, device);
                AO_TRY(ao_amd_int4wo_linear_partials(ptr(x), 1, l.wqkv.K, l.wqkv.K, ptr(l.attn_norm), (float)l.attn_eps, ptr(l.wqkv.codes),
                                                     ptr(l.wqkv.scales), l.wqkv.N, m.group, nparts, qkv.data_ptr(), l.wqkv.N, st));
            } else if (!norm_linear(l.wqkv, x, l.attn_norm, l.attn_eps, qkv)) {
                return false;
            }
            if (!attend(qkv, nparts, l, pos, y) || !linear_add(l.wo, y, x, h) || !swiglu(l, h, act) || !linear_add(l.w2, act, h, x)) return false;
        }
        return norm_linear(m.output, x, m.norm, m.eps, logits);
    }

    // ---- several rows
    bool prefill(Tensor x, const Tensor& pos, int64_t T, Tensor& logits) {
        // torch's indexing, as in the module chain, for its refusal of a position outside the cache (and the rotary table, which is no
        // shorter).  The attention finds the rows of the others itself: negative ones count from the end, as they do there.
        (void)at::index(m.cache_rows, {std::optional<Tensor>(pos)});
        Tensor n = alloc(T, m.dim);
        const Layer* first = m.layers.empty() ? nullptr : &m.layers[0];
        const Tensor& w0 = first ? first->attn_norm : m.norm;
        const float eps0 = (float)(first ? first->attn_eps : m.eps);
        AO_TRY(f16 ? ao_amd_rmsnorm_f16(ptr(x), ptr(w0), T, m.dim, eps0, n.data_ptr(), st)
                   : ao_amd_rmsnorm_bf16(ptr(x), ptr(w0), T, m.dim, eps0, n.data_ptr(), st));
        for (size_t i = 0; i < m.layers.size(); ++i) {
            const Layer& l = m.layers[i];
            const bool end = i + 1 == m.layers.size();
            const Tensor& next_w = end ? m.norm : m.layers[i + 1].attn_norm;
            const float next_eps = (float)(end ? m.eps : m.layers[i + 1].attn_eps);
            Tensor qkv, y = alloc(T, m.n_head * 128), o, gate, up, down;
            if (!linear(l.wqkv, n, T, qkv)) return false;
            AO_TRY(ao_amd_llama_prefill_attention_wrap(ptr(qkv), f16, ptr(m.freqs), m.freqs.size(0), ptr(pos), pos.scalar_type() == at::kLong, T,
                                                       l.k_cache.data_ptr(), l.v_cache.data_ptr(), (int)m.n_head, (int)m.n_kv, 128, m.max_seq,
                                                       y.data_ptr(), st));
            if (!linear(l.wo, y, T, o)) return false;
            Tensor h = alloc(T, m.dim), hn = alloc(T, m.dim);
            AO_TRY(ao_amd_add_rmsnorm(ptr(x), ptr(o), ptr(l.ffn_norm), f16, T, m.dim, (float)l.ffn_eps, h.data_ptr(), hn.data_ptr(), st));
            if (!linear(l.w1, hn, T, gate) || !linear(l.w3, hn, T, up)) return false;
            AO_TRY(ao_amd_silu_mul(ptr(gate), ptr(up), f16, T * l.w1.N, gate.data_ptr(), st));
            if (!linear(l.w2, gate, T, down)) return false;
            x = alloc(T, m.dim);
            n = alloc(T, m.dim);
            AO_TRY(ao_amd_add_rmsnorm(ptr(h), ptr(down), ptr(next_w), f16, T, m.dim, next_eps, x.data_ptr(), n.data_ptr(), st));
        }
        return linear(m.output, n, T, logits);
    }
};

}  // namespace

// (plan, tokens int32 or int64 [1, T] and the embedding table, or embedded tokens [1, T, dim] and None, positions [T]: int32 for T = 1,
// else int32 or int64) -> logits [1, T, vocab].  Tokens are looked up by torch's embedding, which refuses one outside the table; the
// caller calls an embedding module that does more itself.
PyObject* llama_forward(PyObject*, PyObject* const* v, Py_ssize_t nargs) {
    AO_NEED(4);
    auto index = [&](int i) -> const Tensor& {
        const bool is_long = THPVariable_CheckExact(v[i]) && THPVariable_Unpack(v[i]).defined() && THPVariable_Unpack(v[i]).scalar_type() == at::kLong;
        return a.tensor(i, is_long ? at::kLong : at::kInt);
    };
    at::ScalarType dtype;
    const bool embedded = v[2] == Py_None;
    const Tensor &rows = embedded ? a.tensor16(1, dtype) : index(1), &pos = index(3);
    const Tensor* table = embedded ? nullptr : &a.tensor16(2, dtype);
    AO_WANT(a.ok && current(a.device) && rows.dim() == (embedded ? 3 : 2) && rows.size(0) == 1 && (embedded || table->dim() == 2));
    const int64_t T = rows.size(1);
    AO_WANT(T >= 1 && pos.dim() == 1 && pos.numel() == T && pos.is_contiguous() && (T > 1 || pos.scalar_type() == at::kInt));
    // Autocast changes the types between the modules of a prompt (it clears a key that is excluded otherwise, so nothing_watches()
    // does not see it); a decode step is made of operators that it leaves alone.
    AO_WANT(T == 1 || !at::autocast::is_autocast_enabled(at::kCUDA));
    return guarded([&]() -> PyObject* {
        const Model m = read_model(a, v[0]);
        at::AutoDispatchBelowADInplaceOrView below;   // no gradient is recorded here: the arguments were looked at for one
        AO_WANT(a.ok && dtype == m.dtype && (embedded ? rows.size(2) : table->size(1)) == m.dim);
        const Tensor x = embedded ? rows : at::embedding(*table, rows);
        AO_WANT(x.is_contiguous() && (uintptr_t)ptr(x) % 16 == 0);
        Pass p{m, a.device, stream_of(a.device)};
        Tensor logits;
        AO_WANT(T == 1 ? p.decode(x, pos, logits) : p.prefill(x, pos, T, logits));
        return THPVariable_Wrap(logits.view({1, T, m.output.N}));
    });
}

}  // namespace ao_host
