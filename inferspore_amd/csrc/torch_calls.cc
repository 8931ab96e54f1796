// The calls of inferspore_amd/ops.py on plain operands, from torch's tensors to the C ABI without Python in between: a module of functions
// that look at every operand, launch on torch's current stream and return the C ABI's status, or None for whatever is not
// plain -- another tensor class, a wrong type, extent, layout or device -- which ops.py then takes or refuses as ever.  Nothing is
// kept between calls.
// The four calls around a decode step's GEMMs took their thread 24 us through Python's checks and ctypes, more than their kernels (11 us);
// from here they take 15, most of it the launches.  The first pass of a two-layer decode step on a new state: 382 and 337 us.
#include <torch/csrc/autograd/python_variable.h>

#include <ATen/ATen.h>
#include <ATen/autocast_mode.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPStream.h>

#include <algorithm>
#include <initializer_list>

#include "inferspore_amd.h"

namespace {

using at::Tensor;

// An operand as a call sees it: `t` is null for None.  Extents and memory are what the checks have seen: once the interpreter's lock is
// given up, another thread may change the tensor.
struct Operand {
    const Tensor* t = nullptr;
    void* memory = nullptr;
    int64_t dims = 0, count = 0, extent[5] = {};
    Operand() = default;
    explicit Operand(const Tensor& of) : t(&of), memory(of.mutable_data_ptr()), dims(of.dim()), count(of.numel()) {
        for (int d = 0; d < 5 && d < dims; d++) extent[d] = of.size(d);
    }
    int64_t size(int d) const { return extent[d]; }
    int64_t dim() const { return dims; }
    int64_t numel() const { return count; }
    void* data() const { return memory; }
    bool is(std::initializer_list<int64_t> shape) const {
        return dims == (int64_t)shape.size() && std::equal(shape.begin(), shape.end(), extent);
    }
    bool same_shape(const Operand& o) const { return dims <= 5 && dims == o.dims && std::equal(extent, extent + dims, o.extent); }
};

// A call that meets something else than plain operands notes it here and ends with None.
struct Call {
    PyObject* const* args;
    Py_ssize_t count;
    bool plain = true;

    Call(PyObject* const* a, Py_ssize_t n, Py_ssize_t expected) : args(a), count(n) {
        plain = n == expected && !at::impl::torch_function_mode_enabled();
    }
    // contiguous memory on the GPU of a tensor that is nothing but that
    Operand tensor(Py_ssize_t i, at::ScalarType type, bool optional = false) {
        Operand o;
        if (!plain) return o;
        if (args[i] == Py_None) {
            plain = optional;
            return o;
        }
        plain = THPVariable_CheckExact(args[i]);
        if (!plain) return o;
        static const c10::DispatchKeySet ordinary = c10::DispatchKeySet(c10::DispatchKey::CUDA) |
                                                    c10::getAutogradRelatedKeySetFromBackend(c10::BackendComponent::CUDABit) |
                                                    c10::getAutocastRelatedKeySetFromBackend(c10::BackendComponent::CUDABit) |
                                                    c10::DispatchKeySet(c10::DispatchKey::ADInplaceOrView);
        const Tensor& t = THPVariable_Unpack(args[i]);
        plain = t.is_cuda() && t.scalar_type() == type && (t.key_set().raw_repr() & ~ordinary.raw_repr()) == 0 && t.has_storage() && t.is_contiguous();
        for (int64_t d = 0; plain && d < t.dim(); d++) plain = t.size(d) <= INT32_MAX;
        return plain ? Operand(t) : o;
    }
    at::ScalarType float_type(Py_ssize_t i) {  // float16 or float32
        if (!plain) return at::kHalf;
        plain = THPVariable_CheckExact(args[i]);
        if (!plain) return at::kHalf;
        const at::ScalarType type = THPVariable_Unpack(args[i]).scalar_type();
        plain = type == at::kHalf || type == at::kFloat;
        return type;
    }
    int integer(Py_ssize_t i) {
        if (!plain) return 0;
        int overflow = 0;
        const long long v = PyLong_CheckExact(args[i]) ? PyLong_AsLongLongAndOverflow(args[i], &overflow) : 0;
        plain = PyLong_CheckExact(args[i]) && !overflow && v >= INT32_MIN && v <= INT32_MAX;
        return (int)v;
    }
    float number(Py_ssize_t i) {
        if (!plain) return 0.0f;
        if (PyLong_CheckExact(args[i])) return (float)integer(i);
        plain = PyFloat_CheckExact(args[i]);
        return plain ? (float)PyFloat_AS_DOUBLE(args[i]) : 0.0f;
    }
    void need(bool ok) { plain = plain && ok; }
};

isp_stream_t stream() { return c10::hip::getCurrentHIPStream().stream(); }

// Other threads may run while a call launches, as through ctypes.
struct InterpreterFree {
    PyThreadState* state = PyEval_SaveThread();
    ~InterpreterFree() { PyEval_RestoreThread(state); }
};

template <typename F>
PyObject* launched(const Call& call, F&& f) {
    if (!call.plain) Py_RETURN_NONE;
    int status;
    {
        InterpreterFree free;
        status = f();
    }
    return PyLong_FromLong(status);
}

// torch's accessors and allocator throw where a tensor has no memory or the device none left: the general path meets the same and
// reports it.
using Method = PyObject* (*)(PyObject*, PyObject* const*, Py_ssize_t);
template <Method F>
PyObject* guarded(PyObject* self, PyObject* const* args, Py_ssize_t n) {
    try {
        return F(self, args, n);
    } catch (...) {
        Py_RETURN_NONE;
    }
}

#define ISP_BY_TYPE(type, name) ((type) == at::kHalf ? name##_f16 : name##_f32)
#define ISP_BY_TYPE_WITH(type, name, suffix) ((type) == at::kHalf ? name##_f16##suffix : name##_f32##suffix)
#define ISP_METHOD(name) PyObject* name(PyObject*, PyObject* const* args, Py_ssize_t n)

ISP_METHOD(input_embedding) {  // ids, output, table, check_bounds
    Call c(args, n, 4);
    const auto type = c.float_type(1);
    const Operand ids = c.tensor(0, at::kInt), out = c.tensor(1, type), table = c.tensor(2, type);
    c.need(c.plain && ids.dim() == 1 && out.dim() == 2 && table.dim() == 2 && out.size(0) == ids.size(0) && table.size(1) == out.size(1) &&
           (args[3] == Py_True || args[3] == Py_False));
    return launched(c, [&] {
        return ISP_BY_TYPE(type, isp_embedding)(static_cast<const int32_t*>(ids.data()), out.data(), table.data(), (int)out.size(0),
                                                (int)out.size(1), args[3] == Py_True ? (int)table.size(0) : 0, stream());
    });
}

ISP_METHOD(cal_padding_offset) {  // padding_offset, cum_seqlens, lengths
    Call c(args, n, 3);
    const Operand offset = c.tensor(0, at::kInt), cum = c.tensor(1, at::kInt), lens = c.tensor(2, at::kInt);
    c.need(c.plain && offset.dim() == 2 && cum.dim() == 1 && lens.dim() == 1 && offset.size(0) == lens.size(0) &&
           offset.size(0) == cum.size(0) - 1);
    return launched(c, [&] {
        return isp_cal_padding_offset(static_cast<int32_t*>(offset.data()), static_cast<int32_t*>(cum.data()),
                                      static_cast<const int32_t*>(lens.data()), (int)offset.size(0), (int)offset.size(1), stream());
    });
}

ISP_METHOD(rmsnorm) {  // x, gamma, eps
    Call c(args, n, 3);
    const auto type = c.float_type(0);
    const Operand x = c.tensor(0, type), gamma = c.tensor(1, type);
    const float eps = c.number(2);
    c.need(c.plain && x.dim() == 2 && gamma.numel() == x.size(1));
    return launched(c, [&] { return ISP_BY_TYPE(type, isp_rmsnorm)(x.data(), gamma.data(), eps, (int)x.size(0), (int)x.size(1), stream()); });
}

ISP_METHOD(fused_add_bias_residual_rmsnorm) {  // residual, decoder_out, bias, gamma, eps, flags
    Call c(args, n, 6);
    const auto type = c.float_type(1);
    const Operand residual = c.tensor(0, type, true), x = c.tensor(1, type), bias = c.tensor(2, type, true), gamma = c.tensor(3, type);
    const float eps = c.number(4);
    const int flags = c.integer(5);
    c.need(c.plain && x.dim() == 2 && (!residual.t || (residual.same_shape(x) && residual.data() != x.data())) &&
           gamma.numel() == x.size(1) && (!bias.t || bias.numel() == x.size(1)));
    return launched(c, [&] {
        return ISP_BY_TYPE(type, isp_fused_add_bias_residual_rmsnorm)(residual.data(), x.data(), bias.data(), gamma.data(), eps,
                                                                      (int)x.size(0), (int)x.size(1), (unsigned)flags, stream());
    });
}

ISP_METHOD(act) {  // input, out
    Call c(args, n, 2);
    const auto type = c.float_type(0);
    const Operand in = c.tensor(0, type), out = c.tensor(1, type);
    c.need(c.plain && in.dim() == 3 && in.size(1) == 2 && out.is({in.size(0), in.size(2)}));
    return launched(c, [&] { return ISP_BY_TYPE(type, isp_swiglu)(in.data(), out.data(), (int)in.size(0), (int)in.size(2), stream()); });
}

// caches [layers, batch, kv_heads, max_seq_len, head_size] and a layer among theirs
bool caches_fit(const Operand& k, const Operand& v, int layer, int64_t batch, int64_t kv_heads, int64_t head_size) {
    return k.dim() == 5 && k.same_shape(v) && k.size(1) == batch && k.size(2) == kv_heads && k.size(4) == head_size &&
           layer >= 0 && layer < k.size(0);
}

// What the calls on packed qkv rows share: q_buf [batch, heads, seq, head_size], k_buf and v_buf likewise or absent.
bool qkv_fits(const Operand& q, const Operand& k, const Operand& v, const Operand& qkv, const Operand& bias, const Operand& offset,
              const Operand& history, const Operand& lengths) {
    if (qkv.dim() != 3 || q.dim() != 4) return false;
    const int64_t extra = qkv.size(1) - q.size(1);
    if (extra < 0 || extra % 2 != 0 || q.size(3) != qkv.size(2) || (k.t == nullptr) != (v.t == nullptr)) return false;
    for (const Operand* o : {&k, &v})
        if (o->t && !o->is({q.size(0), extra / 2, q.size(2), qkv.size(2)})) return false;
    return (!bias.t || bias.numel() == qkv.size(1) * qkv.size(2)) && offset.numel() >= qkv.size(0) && history.numel() >= q.size(0) &&
           (!lengths.t || lengths.numel() >= q.size(0));
}

ISP_METHOD(qkv_bias_rope_transpose) {  // q, k, v, qkv, bias, padding_offset, history, lengths, rotary_dim, base, max_position, ntk
    Call c(args, n, 12);
    const auto type = c.float_type(3);
    const Operand q = c.tensor(0, type), k = c.tensor(1, type), v = c.tensor(2, type), qkv = c.tensor(3, type), bias = c.tensor(4, type, true),
                  offset = c.tensor(5, at::kInt), history = c.tensor(6, at::kInt), lengths = c.tensor(7, at::kInt, true);
    const int rotary = c.integer(8), positions = c.integer(10);
    const float base = c.number(9);
    c.need(c.plain && qkv_fits(q, k, v, qkv, bias, offset, history, lengths) && (args[11] == Py_True || args[11] == Py_False));
    return launched(c, [&] {
        return ISP_BY_TYPE(type, isp_qkv_bias_rope_transpose)(
            q.data(), k.data(), v.data(), qkv.data(), bias.data(), static_cast<const int32_t*>(offset.data()),
            static_cast<const int32_t*>(history.data()), static_cast<const int32_t*>(lengths.data()), (int)q.size(0), (int)q.size(2),
            (int)qkv.size(0), (int)q.size(1), (int)((qkv.size(1) - q.size(1)) / 2), (int)qkv.size(2), rotary, base, positions,
            args[11] == Py_True, stream());
    });
}

ISP_METHOD(qkv_bias_rope_transpose_append) {  // q, k, v, k_cache, v_cache, layer, qkv, bias, padding_offset, history, lengths, rotary_dim, base
    Call c(args, n, 13);
    const auto type = c.float_type(6);
    const Operand q = c.tensor(0, type), k = c.tensor(1, type, true), v = c.tensor(2, type, true), k_cache = c.tensor(3, type),
                  v_cache = c.tensor(4, type), qkv = c.tensor(6, type), bias = c.tensor(7, type, true), offset = c.tensor(8, at::kInt),
                  history = c.tensor(9, at::kInt), lengths = c.tensor(10, at::kInt);
    const int layer = c.integer(5), rotary = c.integer(11);
    const float base = c.number(12);
    c.need(c.plain && qkv_fits(q, k, v, qkv, bias, offset, history, lengths) &&
           caches_fit(k_cache, v_cache, layer, q.size(0), (qkv.size(1) - q.size(1)) / 2, qkv.size(2)));
    return launched(c, [&] {
        return ISP_BY_TYPE(type, isp_qkv_bias_rope_transpose_append)(
            q.data(), k.data(), v.data(), k_cache.data(), v_cache.data(), layer, (int)k_cache.size(3), qkv.data(), bias.data(),
            static_cast<const int32_t*>(offset.data()), static_cast<const int32_t*>(history.data()),
            static_cast<const int32_t*>(lengths.data()), (int)q.size(0), (int)q.size(2), (int)qkv.size(0), (int)q.size(1),
            (int)((qkv.size(1) - q.size(1)) / 2), (int)qkv.size(2), rotary, base, stream());
    });
}

ISP_METHOD(rope_decode_append) {  // qkv, bias, k_cache, v_cache, layer, history, step, head_num, rotary_dim, base
    Call c(args, n, 10);
    const auto type = c.float_type(0);
    const Operand qkv = c.tensor(0, type), bias = c.tensor(1, type, true), k_cache = c.tensor(2, type), v_cache = c.tensor(3, type),
                  history = c.tensor(5, at::kInt);
    const int layer = c.integer(4), step = c.integer(6), heads = c.integer(7), rotary = c.integer(8);
    const float base = c.number(9);
    c.need(c.plain && qkv.dim() == 3 && qkv.size(1) >= heads && (qkv.size(1) - heads) % 2 == 0 &&
           (!bias.t || bias.numel() == qkv.size(1) * qkv.size(2)) && history.numel() >= qkv.size(0) &&
           caches_fit(k_cache, v_cache, layer, qkv.size(0), (qkv.size(1) - heads) / 2, qkv.size(2)));
    return launched(c, [&] {
        return ISP_BY_TYPE(type, isp_rope_decode_append)(qkv.data(), bias.data(), k_cache.data(), v_cache.data(), layer, (int)k_cache.size(3),
                                                         static_cast<const int32_t*>(history.data()), (int)qkv.size(0), heads,
                                                         (int)((qkv.size(1) - heads) / 2), (int)qkv.size(2), step, rotary, base, stream());
    });
}

ISP_METHOD(transpose_out_remove_padding) {  // padded, padding_offset, packed
    Call c(args, n, 3);
    const auto type = c.float_type(0);
    const Operand padded = c.tensor(0, type), offset = c.tensor(1, at::kInt), packed = c.tensor(2, type);
    c.need(c.plain && padded.dim() == 4 && packed.dim() == 3 && packed.size(1) == padded.size(1) && packed.size(2) == padded.size(3) &&
           offset.numel() >= packed.size(0));
    return launched(c, [&] {
        return ISP_BY_TYPE(type, isp_transpose_remove_padding)(padded.data(), static_cast<const int32_t*>(offset.data()), packed.data(),
                                                               (int)padded.size(0), (int)padded.size(1), (int)padded.size(2),
                                                               (int)padded.size(3), (int)packed.size(0), stream());
    });
}

ISP_METHOD(concat_kv_cache) {  // k_src, v_src, layer, query_length, history, k_dst, v_dst
    Call c(args, n, 7);
    const auto type = c.float_type(0);
    const Operand k = c.tensor(0, type), v = c.tensor(1, type), lengths = c.tensor(3, at::kInt), history = c.tensor(4, at::kInt),
                  k_cache = c.tensor(5, type), v_cache = c.tensor(6, type);
    const int layer = c.integer(2);
    c.need(c.plain && k.dim() == 4 && k.same_shape(v) &&
           caches_fit(k_cache, v_cache, layer, k.size(0), k.size(1), k.size(3)) && lengths.numel() >= k.size(0) &&
           history.numel() >= k.size(0));
    return launched(c, [&] {
        return ISP_BY_TYPE(type, isp_concat_kv_cache)(k.data(), v.data(), k_cache.data(), v_cache.data(), layer,
                                                      static_cast<const int32_t*>(lengths.data()), static_cast<const int32_t*>(history.data()),
                                                      (int)k.size(0), (int)k.size(1), (int)k.size(2), (int)k_cache.size(3), (int)k.size(3),
                                                      stream());
    });
}

ISP_METHOD(repeat_kv_cache) {  // k_cache, v_cache, context_length, layer, k_dst, v_dst
    Call c(args, n, 6);
    const auto type = c.float_type(0);
    const Operand k_cache = c.tensor(0, type), v_cache = c.tensor(1, type), context = c.tensor(2, at::kInt), k = c.tensor(4, type),
                  v = c.tensor(5, type);
    const int layer = c.integer(3);
    c.need(c.plain && k_cache.dim() == 5 && k.dim() == 4 && k.same_shape(v) && context.dim() >= 1 &&
           caches_fit(k_cache, v_cache, layer, context.size(0), k_cache.size(2), k.size(3)) && k.size(0) == context.size(0) &&
           k_cache.size(2) > 0 && k.size(1) % k_cache.size(2) == 0);
    return launched(c, [&] {
        return ISP_BY_TYPE(type, isp_repeat_kv_cache)(k_cache.data(), v_cache.data(), k.data(), v.data(), layer,
                                                      static_cast<const int32_t*>(context.data()), (int)k.size(0), (int)k.size(1),
                                                      (int)k_cache.size(2), (int)k_cache.size(3), (int)k.size(2), (int)k.size(3), stream());
    });
}

// float16 layers that are faster step by step, with the library's product for what is wide: 17 to 64 rows where a product has more than 32768
// columns; 65 to 128 rows of more than 8192 columns where gate and up projections have 400 to 650 million weights, 129 to 192 rows of more
// than 9216 where they have more than 400 million.  us a layer, steps and one call: 48 rows x 6144, inter 24576 278, 295; 40 x 10240, 27648,
// 8 key heads 411, 464; 96 x 9216, 24704 541, 625; 144 x 12288, 43008 1142, 1421.  Next to the lines: 17 x 6144, 24576 262, 236; 40 x 5120,
// 13824 162, 159; 112 x 8192, 28672 580, 576; 80 x 10240, 35840 925, 807; 144 x 9216, 32256 729, 685; 200 x 12288, 43008 1480, 1308.  The library's times jump from one number of rows
// to the next: 96 x 8192, 28672 takes 495 there and 554 here, 640 rows 1349 and 1437, the worst found on this side of the lines.
bool steps_are_faster(int rows, int64_t hidden, int64_t width, int64_t inter) {
    if (rows <= 64) return rows > 16 && (2 * inter > 32768 || width > 32768);
    const int64_t weights = 2 * inter * hidden;
    if (rows <= 128) return hidden > 8192 && weights > 400000000 && weights <= 650000000;
    return rows <= 192 && hidden > 9216 && weights > 400000000;
}

// A whole layer: its output, a status that is not 0, or None.  normed, residual, qkv, qkv_bias, o, gate_up, down, ffn_norm, next_norm, q,
// k_cache, v_cache, packed context, act, padding_offset, history, lengths, context lengths; layer, tokens, heads, kv_heads, head_size,
// longest context, rotary_dim; base, eps.
ISP_METHOD(context_layer) {
    Call c(args, n, 27);
    const auto type = c.float_type(0);
    Operand f[14];
    for (int i = 0; i < 14; i++) f[i] = c.tensor(i, type, i == 3);
    Operand lens[4];
    for (int i = 0; i < 4; i++) lens[i] = c.tensor(14 + i, at::kInt);
    const int layer = c.integer(18), tokens = c.integer(19), heads = c.integer(20), kv = c.integer(21), hs = c.integer(22),
              longest = c.integer(23), rotary = c.integer(24);
    const float base = c.number(25), eps = c.number(26);
    // a dispatch mode (a counter of operations, a tracer) sees the products of the steps
    c.need(c.plain && !c10::impl::dispatch_mode_enabled() && f[0].dim() == 2 && f[9].dim() == 4 && f[10].dim() == 5 && f[13].dim() == 2 && heads > 0 && kv > 0 && hs > 0);
    if (!c.plain) Py_RETURN_NONE;
    const int64_t hidden = f[0].size(1), batch = f[9].size(0), max_q = f[9].size(2), max_seq = f[10].size(3), inter = f[13].size(1),
                  width = ((int64_t)heads + 2ll * kv) * hs, context = (int64_t)heads * hs;
    c.need(tokens > 0 && batch > 0 && f[0].is({tokens, hidden}) && f[1].is({tokens, hidden}) && f[2].is({hidden, width}) &&
           (!f[3].t || f[3].is({width})) && f[4].is({context, hidden}) && f[5].is({hidden, 2 * inter}) && f[6].is({inter, hidden}) &&
           f[7].is({hidden}) && f[8].is({hidden}) && f[9].is({batch, heads, max_q, hs}) && caches_fit(f[10], f[11], layer, batch, kv, hs) &&
           f[12].is({tokens, heads, hs}) && f[13].is({tokens, inter}) && lens[0].numel() >= tokens && lens[1].numel() >= batch &&
           lens[2].numel() >= batch && lens[3].dim() >= 1 && lens[3].size(0) == batch && rotary >= 0 && rotary <= hs && rotary % 2 == 0 &&
           !at::autocast::is_autocast_enabled(at::kCUDA));
    const bool grad = at::GradMode::is_enabled();
    for (int i = 0; c.plain && i < 18; i++) {
        const Operand& o = i < 14 ? f[i] : lens[i - 14];
        if (o.t) c.need(o.t->device() == f[0].t->device() && (i >= 14 || ((uintptr_t)o.data() % 16 == 0 && !(grad && o.t->requires_grad()))));
    }
    if (!c.plain || f[0].data() == f[1].data() || (type == at::kHalf && steps_are_faster(tokens, hidden, width, inter))) Py_RETURN_NONE;
    const char *q = static_cast<const char*>(f[9].data()), *packed = static_cast<const char*>(f[12].data());
    if (packed >= q ? (size_t)(packed - q) < f[9].t->nbytes() : (size_t)(q - packed) < f[12].t->nbytes()) Py_RETURN_NONE;
    const size_t need = ISP_BY_TYPE_WITH(type, isp_context_layer_rows, _workspace)((int)batch, tokens, (int)hidden, heads, kv, hs, (int)max_q,
                                                                                   longest, (int)max_seq, (int)inter);
    if (need == 0) Py_RETURN_NONE;
    const Tensor workspace = at::empty({(int64_t)need}, f[0].t->options().dtype(at::kByte));
    Tensor out = at::empty_like(*f[0].t);
    int status;
    {
        InterpreterFree free;
        const auto ints = [&](int i) { return static_cast<const int32_t*>(lens[i].data()); };
        status = ISP_BY_TYPE(type, isp_context_layer_rows)(
            f[0].data(), f[1].data(), out.mutable_data_ptr(), f[2].data(), f[3].data(), f[4].data(), f[5].data(), f[6].data(), f[7].data(),
            f[8].data(), f[9].data(), f[10].data(), f[11].data(), f[12].data(), f[13].data(), ints(0), ints(1), ints(2), ints(3),
            workspace.mutable_data_ptr(), layer, (int)batch, tokens, (int)hidden, heads, kv, hs, (int)max_q, longest, (int)max_seq,
            (int)inter, rotary, base, eps, stream());
    }
    return status != ISP_OK ? PyLong_FromLong(status) : THPVariable_Wrap(std::move(out));
}

PyMethodDef methods[] = {
#define ISP_ENTRY(name) {#name, (PyCFunction)(void (*)(void))guarded<name>, METH_FASTCALL, nullptr}
    ISP_ENTRY(input_embedding), ISP_ENTRY(cal_padding_offset), ISP_ENTRY(rmsnorm), ISP_ENTRY(fused_add_bias_residual_rmsnorm),
    ISP_ENTRY(act), ISP_ENTRY(qkv_bias_rope_transpose), ISP_ENTRY(qkv_bias_rope_transpose_append), ISP_ENTRY(rope_decode_append),
    ISP_ENTRY(transpose_out_remove_padding), ISP_ENTRY(concat_kv_cache), ISP_ENTRY(repeat_kv_cache), ISP_ENTRY(context_layer),
#undef ISP_ENTRY
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_torch_calls", nullptr, -1, methods};

}  // namespace

// `built_for`: the torch and the Python whose headers this was compiled with; the loader takes no other.
PyMODINIT_FUNC PyInit__torch_calls() {
    PyObject* m = PyModule_Create(&module);
    if (m && PyModule_AddObject(m, "built_for", Py_BuildValue("(sii)", ISP_TORCH_VERSION, PY_MAJOR_VERSION, PY_MINOR_VERSION)) != 0) {
        Py_DECREF(m);
        return nullptr;
    }
    return m;
}
