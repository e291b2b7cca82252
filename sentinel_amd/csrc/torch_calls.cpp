// The Python entry points' way into the C ABI (sentinel_hip_attn.h) for the calls a program makes over and over: tensors that
// are what the call expects, outputs and workspace given, the current stream.  Checking a call's tensors and passing two
// dozen arguments through ctypes costs 10 - 20 us of Python, more than the small kernels take; here both are
// a few hundred nanoseconds.
//
// Every function returns True when it has made the call, and False, having done nothing, whenever anything is not
// as expected or the library refused the arguments: the Python code then makes the same call itself, allocates what is
// missing and raises what there is to raise.  That includes tensors whose methods throw (a tensor without storage, as tracing and
// vmap hand them in): no C++ exception leaves a function.  A runtime error is raised here and the call never made again: it may
// come from after the launch (or be an earlier, unrelated one), and the calls that work in place must not run twice.
#include <torch/csrc/autograd/python_variable.h>

#include <ATen/core/Tensor.h>
#include <c10/core/impl/VirtualGuardImpl.h>

#include "../../include/sentinel_hip_attn.h"

namespace {

// the library's functions, bound at load time by address: another build of the library can stand in for the usual one
struct Library {
    decltype(&sentinel_hip_flash_fwd) flash_fwd;
    decltype(&sentinel_hip_flash_bwd) flash_bwd;
    decltype(&sentinel_hip_flash_fwd_rope) flash_fwd_rope;
    decltype(&sentinel_hip_flash_bwd_rope) flash_bwd_rope;
    decltype(&sentinel_hip_flash_fwd_sparse) flash_fwd_sparse;
    decltype(&sentinel_hip_flash_bwd_sparse) flash_bwd_sparse;
    decltype(&sentinel_hip_flash_workspace_bytes) flash_workspace_bytes;
    decltype(&sentinel_hip_decode_attention) decode_attention;
    decltype(&sentinel_hip_decode_workspace_bytes) decode_workspace_bytes;
    decltype(&sentinel_hip_dense_softmax_fwd) dense_softmax_fwd;
    decltype(&sentinel_hip_dense_softmax_bwd) dense_softmax_bwd;
    decltype(&sentinel_hip_rope_rotate) rope_rotate;
    decltype(&sentinel_hip_last_error) last_error;
};
Library lib = {};
PyObject* current_raw_stream = nullptr;  // torch._C._cuda_getCurrentRawStream

// Arguments of one call; anything unexpected clears `ok`, after which nothing is touched any more.
#ifdef SENTINEL_CALLS_HOST_TENSORS  // the argument checks on host tensors, for tests without a GPU
constexpr c10::DeviceType kDevice = c10::DeviceType::CPU;
#else
constexpr c10::DeviceType kDevice = c10::DeviceType::CUDA;
#endif

struct Call {
    PyObject* const* args;
    Py_ssize_t count;
    bool ok = true;
    c10::Device device{kDevice};
    bool device_known = false;

    Call(PyObject* const* args_, Py_ssize_t count_, Py_ssize_t expected) : args(args_), count(count_) { ok = count == expected; }

    long long integer(int i) {
        if (!ok || !PyLong_Check(args[i])) return fail();
        int overflow = 0;
        const long long x = PyLong_AsLongLongAndOverflow(args[i], &overflow);
        if (overflow || x > 0x7fffffffLL || x < -0x7fffffffLL) return fail();
        return x;
    }
    int int32(int i) { return (int)integer(i); }
    float number(int i) {
        if (!ok || !PyFloat_Check(args[i])) return (float)fail();
        return (float)PyFloat_AS_DOUBLE(args[i]);
    }
    // a contiguous tensor of this type on the GPU of the call's other tensors
    const at::Tensor* any_tensor(PyObject* object) {
        if (!ok || !THPVariable_CheckExact(object)) return fail(), nullptr;
        const at::Tensor& t = THPVariable_Unpack(object);
        if (t.device().type() != kDevice || !t.is_contiguous()) return fail(), nullptr;
        if (!device_known) device = t.device();
        device_known = true;
        if (t.device() != device) return fail(), nullptr;
        return &t;
    }
    const at::Tensor* tensor(int i, c10::ScalarType type, int64_t dims) {
        const at::Tensor* t = ok ? any_tensor(args[i]) : nullptr;
        if (t && (t->scalar_type() != type || t->dim() != dims || t->numel() == 0)) fail();
        return ok ? t : nullptr;
    }
    // fp32 matrix [rows, cols]
    float* matrix(int i, int64_t rows, int64_t cols) {
        const at::Tensor* t = tensor(i, at::kFloat, 2);
        if (t && (t->size(0) != rows || t->size(1) != cols)) fail();
        return ok ? static_cast<float*>(t->data_ptr()) : nullptr;
    }
    void* same_shape(int i, const at::Tensor& like) {
        const at::Tensor* t = tensor(i, like.scalar_type(), like.dim());
        if (t && t->sizes() != like.sizes()) fail();
        return ok ? t->data_ptr() : nullptr;
    }
    // the optional workspace: none needed, or the caller's where it is large enough
    void* workspace(int i, size_t need, size_t* bytes) {
        *bytes = 0;
        if (!ok || need == 0) return nullptr;
        const at::Tensor* t = args[i] == Py_None ? nullptr : any_tensor(args[i]);
        if (!t || t->nbytes() < need) return fail(), nullptr;
        *bytes = t->nbytes();
        return t->data_ptr();
    }
    struct Rope {
        const float *cos = nullptr, *sin = nullptr;
        int positions = 0, offset = 0;
    };
    Rope rope(int i, int head_dim) {
        Rope r;
        if (!ok || args[i] == Py_None) return r;
        if (!PyTuple_CheckExact(args[i]) || PyTuple_GET_SIZE(args[i]) < 2 || PyTuple_GET_SIZE(args[i]) > 3) return fail(), r;
        const at::Tensor* cos = any_tensor(PyTuple_GET_ITEM(args[i], 0));
        const at::Tensor* sin = ok ? any_tensor(PyTuple_GET_ITEM(args[i], 1)) : nullptr;
        if (!ok) return r;
        if (cos->scalar_type() != at::kFloat || sin->scalar_type() != at::kFloat || cos->dim() != 2 || cos->sizes() != sin->sizes() ||
            cos->size(1) * 2 != head_dim || cos->size(0) > 0x7fffffff)
            return fail(), r;
        if (PyTuple_GET_SIZE(args[i]) == 3) {
            PyObject* offset = PyTuple_GET_ITEM(args[i], 2);
            if (!PyLong_Check(offset)) return fail(), r;
            int overflow = 0;
            const long long x = PyLong_AsLongLongAndOverflow(offset, &overflow);
            if (overflow || x < 0 || x > 0x7fffffffLL) return fail(), r;
            r.offset = (int)x;
        }
        r.cos = static_cast<const float*>(cos->data_ptr());
        r.sin = static_cast<const float*>(sin->data_ptr());
        r.positions = (int)cos->size(0);
        return r;
    }
    // the current stream, if the tensors are on the current device
    void* stream() {
        if (!ok) return nullptr;
        if (kDevice == c10::DeviceType::CPU) return nullptr;
        const c10::impl::VirtualGuardImpl guard(kDevice);
        if (guard.getDevice() != device) return fail(), nullptr;
        PyObject* index = PyLong_FromLong(device.index());
        PyObject* raw = index ? PyObject_CallOneArg(current_raw_stream, index) : nullptr;
        Py_XDECREF(index);
        if (!raw) {
            PyErr_Clear();
            return fail(), nullptr;
        }
        void* s = PyLong_AsVoidPtr(raw);
        Py_DECREF(raw);
        if (!s && PyErr_Occurred()) PyErr_Clear(), fail();
        return s;
    }
    long long fail() {
        ok = false;
        return 0;
    }
};

int truth(Call& c, int i) { return c.ok ? c.args[i] == Py_True ? 1 : c.args[i] == Py_False ? 0 : (int)c.fail() : 0; }

// other Python threads run meanwhile
struct WithoutGil {
    PyThreadState* state = PyEval_SaveThread();
    ~WithoutGil() { PyEval_RestoreThread(state); }
};
template <typename Function>
PyObject* made(const Call& call, Function&& function) {
    if (!call.ok) Py_RETURN_FALSE;
    int code;
    {
        const WithoutGil released;
        code = function();
    }
    if (code == SENTINEL_HIP_OK) Py_RETURN_TRUE;
    if (code == SENTINEL_HIP_INVALID_ARGUMENT || code == SENTINEL_HIP_UNSUPPORTED) Py_RETURN_FALSE;  // (found before any launch)
    PyErr_SetString(PyExc_RuntimeError, lib.last_error());
    return nullptr;
}

typedef PyObject* (*Entry)(PyObject*, PyObject* const*, Py_ssize_t);
template <Entry ENTRY>
PyObject* guarded(PyObject* self, PyObject* const* args, Py_ssize_t count) {
    try {
        return ENTRY(self, args, count);
    } catch (...) {
        if (PyErr_Occurred()) PyErr_Clear();
        Py_RETURN_FALSE;
    }
}

struct Pointers {
    const void *q = nullptr, *k = nullptr, *v = nullptr;
    Pointers(const Call& c, const at::Tensor* q_, const at::Tensor* k_, const at::Tensor* v_) {
        if (!c.ok) return;
        q = q_->data_ptr();
        k = k_->data_ptr();
        v = v_->data_ptr();
    }
};

// Geometry of a column-layout call: arguments first .. first + 7 (head_count, head_dim, scale, causal, column_start,
// column_count, pack_count, kv_heads)
struct Columns {
    int hq, d, causal, start, count, packs, hkv;
    float scale;
    int64_t cols = 0;
    const at::Tensor *q = nullptr, *k = nullptr, *v = nullptr;
    Columns(Call& c, int first) {
        hq = c.int32(first);
        d = c.int32(first + 1);
        scale = c.number(first + 2);
        causal = truth(c, first + 3);
        start = c.int32(first + 4);
        count = c.int32(first + 5);
        packs = c.int32(first + 6);
        hkv = c.int32(first + 7);
        q = c.tensor(0, at::kFloat, 2);
        k = c.tensor(1, at::kFloat, 2);
        v = c.tensor(2, at::kFloat, 2);
        if (!c.ok) return;
        cols = q->size(1);
        if (hq <= 0 || d <= 0 || d > 128 || hkv <= 0 || hq % hkv != 0 || q->size(0) != (int64_t)hq * d || k->size(0) != (int64_t)hkv * d ||
            v->size(0) != k->size(0) || k->size(1) != cols || v->size(1) != cols || cols > 0x7fffffff)
            c.fail();
    }
    int seq() const {
        const int64_t s = count > 0 ? count : cols - start;
        return s > 1 ? (int)s : 1;
    }
    int pack_count() const { return packs > 1 ? packs : 1; }
};

// (query, key, value, out, lse, head_count, head_dim, scale, causal, column_start, column_count, pack_count, kv_heads,
//  compute, workspace, rope, window, global_tokens, keep)
PyObject* columns_forward(PyObject*, PyObject* const* args, Py_ssize_t count) {
    Call c(args, count, 19);
    const Columns g(c, 5);
    const int compute = c.int32(13);
    const Call::Rope rope = c.rope(15, g.d);
    const int window = c.int32(16), global_tokens = c.int32(17);
    const bool keep = truth(c, 18);
    float* out = c.ok ? c.matrix(3, g.q->size(0), g.cols) : nullptr;
    float* lse = c.matrix(4, g.hq, g.cols);
    const size_t need = c.ok ? lib.flash_workspace_bytes(SENTINEL_HIP_F32, compute, SENTINEL_HIP_LAYOUT_COLUMNS, g.hq, g.hkv, g.d, g.seq(), g.pack_count(), keep) : 0;
    size_t bytes = 0;
    void* ws = c.workspace(14, need, &bytes);
    void* stream = c.stream();
    const Pointers in(c, g.q, g.k, g.v);
    return made(c, [&, q = in.q, k = in.k, v = in.v] {
        const int layout = SENTINEL_HIP_LAYOUT_COLUMNS | (keep ? SENTINEL_HIP_WORKSPACE_KEEP : 0);
        if (window > 0 || global_tokens != 0)
            return lib.flash_fwd_sparse(q, k, v, out, lse, rope.cos, rope.sin, rope.positions, rope.offset, window, global_tokens,
                                        SENTINEL_HIP_F32, compute, layout, g.hq, g.hkv, g.d, (int)g.cols, g.start, g.count, g.packs,
                                        g.scale, g.causal, ws, bytes, stream);
        if (!rope.cos)
            return lib.flash_fwd(q, k, v, out, lse, SENTINEL_HIP_F32, compute, layout, g.hq, g.hkv, g.d, (int)g.cols, g.start,
                                 g.count, g.packs, g.scale, g.causal, ws, bytes, stream);
        return lib.flash_fwd_rope(q, k, v, out, lse, rope.cos, rope.sin, rope.positions, rope.offset, SENTINEL_HIP_F32, compute,
                                  layout, g.hq, g.hkv, g.d, (int)g.cols, g.start, g.count, g.packs, g.scale, g.causal, ws, bytes,
                                  stream);
    });
}

// (query, key, value, out, lse, d_out, dq, dk, dv, delta, head_count, head_dim, scale, causal, column_start, column_count,
//  pack_count, kv_heads, compute, workspace, rope, window, global_tokens, reuse)
PyObject* columns_backward(PyObject*, PyObject* const* args, Py_ssize_t count) {
    Call c(args, count, 24);
    const Columns g(c, 10);
    const int compute = c.int32(18);
    const Call::Rope rope = c.rope(20, g.d);
    const int window = c.int32(21), global_tokens = c.int32(22);
    const bool reuse = truth(c, 23);
    const int64_t q_rows = c.ok ? g.q->size(0) : 0, kv_rows = c.ok ? g.k->size(0) : 0;
    const float* out = c.matrix(3, q_rows, g.cols);
    const float* lse = c.matrix(4, g.hq, g.cols);
    const float* d_out = c.matrix(5, q_rows, g.cols);
    float* dq = c.matrix(6, q_rows, g.cols);
    float* dk = c.matrix(7, kv_rows, g.cols);
    float* dv = c.matrix(8, kv_rows, g.cols);
    float* delta = c.ok ? c.matrix(9, g.hq, (int64_t)g.pack_count() * g.seq()) : nullptr;
    const size_t need = c.ok ? lib.flash_workspace_bytes(SENTINEL_HIP_F32, compute, SENTINEL_HIP_LAYOUT_COLUMNS, g.hq, g.hkv, g.d, g.seq(), g.pack_count(), 1) : 0;
    size_t bytes = 0;
    void* ws = c.workspace(19, need, &bytes);
    void* stream = c.stream();
    const Pointers in(c, g.q, g.k, g.v);
    return made(c, [&, q = in.q, k = in.k, v = in.v] {
        const int layout = SENTINEL_HIP_LAYOUT_COLUMNS | (reuse ? SENTINEL_HIP_WORKSPACE_REUSE : 0);
        if (window > 0 || global_tokens != 0)
            return lib.flash_bwd_sparse(q, k, v, out, lse, d_out, dq, dk, dv, delta, rope.cos, rope.sin, rope.positions, rope.offset,
                                        window, global_tokens, SENTINEL_HIP_F32, compute, layout, g.hq, g.hkv, g.d, (int)g.cols,
                                        g.start, g.count, g.packs, g.scale, g.causal, ws, bytes, stream);
        if (!rope.cos)
            return lib.flash_bwd(q, k, v, out, lse, d_out, dq, dk, dv, delta, SENTINEL_HIP_F32, compute, layout, g.hq, g.hkv, g.d,
                                 (int)g.cols, g.start, g.count, g.packs, g.scale, g.causal, ws, bytes, stream);
        return lib.flash_bwd_rope(q, k, v, out, lse, d_out, dq, dk, dv, delta, rope.cos, rope.sin, rope.positions, rope.offset,
                                  SENTINEL_HIP_F32, compute, layout, g.hq, g.hkv, g.d, (int)g.cols, g.start, g.count, g.packs,
                                  g.scale, g.causal, ws, bytes, stream);
    });
}

// [B, H, T, d] tensors of one type
struct Native {
    const at::Tensor *q = nullptr, *k = nullptr, *v = nullptr;
    int b = 0, hq = 0, hkv = 0, t = 0, d = 0, code = 0;
    explicit Native(Call& c) {
        q = c.ok ? c.any_tensor(c.args[0]) : nullptr;
        if (!c.ok) return;
        const c10::ScalarType type = q->scalar_type();
        code = type == at::kFloat ? SENTINEL_HIP_F32 : type == at::kBFloat16 ? SENTINEL_HIP_BF16 : type == at::kHalf ? SENTINEL_HIP_F16 : -1;
        if (code < 0 || q->dim() != 4 || q->numel() == 0) c.fail();
        k = c.tensor(1, type, 4);
        v = c.tensor(2, type, 4);
        if (!c.ok) return;
        for (int i = 0; i < 4; ++i)
            if (q->size(i) > 0x7fffffff || k->size(i) > 0x7fffffff) c.fail();
        if (v->sizes() != k->sizes() || k->size(0) != q->size(0) || k->size(2) != q->size(2) || k->size(3) != q->size(3)) c.fail();
        b = (int)q->size(0);
        hq = (int)q->size(1);
        hkv = (int)k->size(1);
        t = (int)q->size(2);
        d = (int)q->size(3);
    }
};

// an fp32 [B, H, T] tensor
float* row_values(Call& c, int i, const Native& g) {
    const at::Tensor* t = c.tensor(i, at::kFloat, 3);
    if (t && (t->size(0) != g.b || t->size(1) != g.hq || t->size(2) != g.t)) c.fail();
    return c.ok ? static_cast<float*>(t->data_ptr()) : nullptr;
}

// (q, k, v, out, lse, scale, causal, window, global_tokens)
PyObject* native_forward(PyObject*, PyObject* const* args, Py_ssize_t count) {
    Call c(args, count, 9);
    const Native g(c);
    void* out = c.ok ? c.same_shape(3, *g.q) : nullptr;
    float* lse = row_values(c, 4, g);
    const float scale = c.number(5);
    const int causal = truth(c, 6), window = c.int32(7), global_tokens = c.int32(8);
    void* stream = c.stream();
    const Pointers in(c, g.q, g.k, g.v);
    return made(c, [&, q = in.q, k = in.k, v = in.v] {
        if (window > 0 || global_tokens != 0)
            return lib.flash_fwd_sparse(q, k, v, out, lse, nullptr, nullptr, 0, 0, window, global_tokens, g.code, SENTINEL_HIP_COMPUTE_AUTO,
                                        SENTINEL_HIP_LAYOUT_BHTD, g.hq, g.hkv, g.d, 0, 0, g.t, g.b, scale, causal, nullptr, 0, stream);
        return lib.flash_fwd(q, k, v, out, lse, g.code, SENTINEL_HIP_COMPUTE_AUTO, SENTINEL_HIP_LAYOUT_BHTD, g.hq, g.hkv, g.d, 0, 0,
                             g.t, g.b, scale, causal, nullptr, 0, stream);
    });
}

// (q, k, v, out, lse, d_out, dq, dk, dv, delta, scale, causal, window, global_tokens)
PyObject* native_backward(PyObject*, PyObject* const* args, Py_ssize_t count) {
    Call c(args, count, 14);
    const Native g(c);
    const void* out = c.ok ? c.same_shape(3, *g.q) : nullptr;
    const float* lse = row_values(c, 4, g);
    const void* d_out = c.ok ? c.same_shape(5, *g.q) : nullptr;
    void* dq = c.ok ? c.same_shape(6, *g.q) : nullptr;
    void* dk = c.ok ? c.same_shape(7, *g.k) : nullptr;
    void* dv = c.ok ? c.same_shape(8, *g.k) : nullptr;
    const at::Tensor* delta = c.ok ? c.any_tensor(c.args[9]) : nullptr;
    if (delta && (delta->scalar_type() != at::kFloat || delta->numel() < (int64_t)g.hq * g.b * g.t)) c.fail();
    const float scale = c.number(10);
    const int causal = truth(c, 11), window = c.int32(12), global_tokens = c.int32(13);
    void* stream = c.stream();
    const Pointers in(c, g.q, g.k, g.v);
    float* dl = c.ok ? static_cast<float*>(delta->data_ptr()) : nullptr;
    return made(c, [&, q = in.q, k = in.k, v = in.v] {
        if (window > 0 || global_tokens != 0)
            return lib.flash_bwd_sparse(q, k, v, out, lse, d_out, dq, dk, dv, dl, nullptr, nullptr, 0, 0, window, global_tokens, g.code,
                                        SENTINEL_HIP_COMPUTE_AUTO, SENTINEL_HIP_LAYOUT_BHTD, g.hq, g.hkv, g.d, 0, 0, g.t, g.b, scale,
                                        causal, nullptr, 0, stream);
        return lib.flash_bwd(q, k, v, out, lse, d_out, dq, dk, dv, dl, g.code, SENTINEL_HIP_COMPUTE_AUTO, SENTINEL_HIP_LAYOUT_BHTD,
                             g.hq, g.hkv, g.d, 0, 0, g.t, g.b, scale, causal, nullptr, 0, stream);
    });
}

// (query, key_cache, value_cache, out, length, head_count, head_dim, kv_heads, scale, window, global_tokens, workspace)
PyObject* decode(PyObject*, PyObject* const* args, Py_ssize_t count) {
    Call c(args, count, 12);
    const int length = c.int32(4), hq = c.int32(5), d = c.int32(6), hkv = c.int32(7);
    const float scale = c.number(8);
    const int window = c.int32(9), global_tokens = c.int32(10);
    const at::Tensor* k = c.tensor(1, at::kFloat, 2);
    if (k && (k->size(0) != (int64_t)hkv * d || k->size(1) > 0x7fffffff || length <= 0)) c.fail();
    const float* q = c.matrix(0, (int64_t)hq * d, 1);
    const void* v = c.ok ? c.same_shape(2, *k) : nullptr;
    float* out = c.matrix(3, (int64_t)hq * d, 1);
    size_t bytes = 0;
    void* ws = c.ok ? c.workspace(11, lib.decode_workspace_bytes(hq, d, length), &bytes) : nullptr;
    void* stream = c.stream();
    const float* keys = c.ok ? static_cast<const float*>(k->data_ptr()) : nullptr;
    const int capacity = c.ok ? (int)k->size(1) : 0;
    return made(c, [&] {
        return lib.decode_attention(q, keys, static_cast<const float*>(v), out, hq, hkv, d, capacity, length, scale, window,
                                    global_tokens, ws, bytes, stream);
    });
}

// a [keys, queries] matrix or a [batch, keys, queries] stack
struct Scores {
    const at::Tensor* t = nullptr;
    float* data = nullptr;
    int batch = 0, keys = 0, queries = 0;
    Scores(Call& c, int i) {
        t = c.ok ? c.any_tensor(c.args[i]) : nullptr;
        if (!c.ok) return;
        const int64_t dims = t->dim();
        if (t->scalar_type() != at::kFloat || (dims != 2 && dims != 3) || t->numel() == 0) {
            c.fail();
            return;
        }
        for (int64_t j = 0; j < dims; ++j)
            if (t->size(j) > 0x7fffffff) c.fail();
        batch = dims == 3 ? (int)t->size(0) : 1;
        keys = (int)t->size(dims - 2);
        queries = (int)t->size(dims - 1);
        data = static_cast<float*>(t->data_ptr());
    }
};

// (scores, scale, window, global_tokens, query_position_start, segment_length)
PyObject* softmax_forward(PyObject*, PyObject* const* args, Py_ssize_t count) {
    Call c(args, count, 6);
    const Scores s(c, 0);
    const float scale = c.number(1);
    const int window = c.int32(2), global_tokens = c.int32(3), start = c.int32(4), segment = c.int32(5);
    void* stream = c.stream();
    return made(c, [&] {
        return lib.dense_softmax_fwd(s.data, s.batch, (long long)s.keys * s.queries, s.keys, s.queries,
                                     start, window, global_tokens, segment, scale, stream);
    });
}

// (probabilities, gradient, scale, window, global_tokens, query_position_start, segment_length)
PyObject* softmax_backward(PyObject*, PyObject* const* args, Py_ssize_t count) {
    Call c(args, count, 7);
    const Scores s(c, 0);
    void* gradient = c.ok ? c.same_shape(1, *s.t) : nullptr;
    const float scale = c.number(2);
    const int window = c.int32(3), global_tokens = c.int32(4), start = c.int32(5), segment = c.int32(6);
    void* stream = c.stream();
    return made(c, [&] {
        const long long stride = (long long)s.keys * s.queries;
        return lib.dense_softmax_bwd(s.data, stride, static_cast<float*>(gradient), stride, s.batch, s.keys, s.queries, start, window, global_tokens, segment, scale, stream);
    });
}

// (tensor, head_count, head_dim, pair_count, cos, sin, position_offset, segment_length, inverse)
PyObject* rotate(PyObject*, PyObject* const* args, Py_ssize_t count) {
    Call c(args, count, 9);
    const int heads = c.int32(1), d = c.int32(2), pairs = c.int32(3), offset = c.int32(6), segment = c.int32(7);
    const int inverse = truth(c, 8);
    const at::Tensor* t = c.tensor(0, at::kFloat, 2);
    const at::Tensor* cos = c.tensor(4, at::kFloat, 2);
    const void* sin = c.ok ? c.same_shape(5, *cos) : nullptr;
    if (c.ok && (heads <= 0 || pairs <= 0 || (int64_t)pairs * 2 != d || t->size(0) != (int64_t)heads * d || cos->size(1) != pairs ||
                 t->size(1) > 0x7fffffff || cos->size(0) > 0x7fffffff))
        c.fail();
    void* stream = c.stream();
    if (!c.ok) Py_RETURN_FALSE;
    float* data = static_cast<float*>(t->data_ptr());
    const float* cos_data = static_cast<const float*>(cos->data_ptr());
    const int cols = (int)t->size(1), positions = (int)cos->size(0);
    return made(c, [&] {
        return lib.rope_rotate(data, heads, d, cols, 0, cols, offset, segment, cos_data, static_cast<const float*>(sin), positions,
                               inverse, stream);
    });
}

// bind({function name: address}): the library the calls go to
PyObject* bind(PyObject*, PyObject* addresses) {
    if (!PyDict_Check(addresses)) {
        PyErr_SetString(PyExc_TypeError, "bind expects a dict of addresses");
        return nullptr;
    }
    Library bound = {};
    const auto take = [&](auto& slot, const char* name) {
        PyObject* address = PyDict_GetItemString(addresses, name);
        void* at = address ? PyLong_AsVoidPtr(address) : nullptr;
        if (!at) {
            if (!PyErr_Occurred()) PyErr_Format(PyExc_KeyError, "no address for %s", name);
            return false;
        }
        slot = reinterpret_cast<std::decay_t<decltype(slot)>>(at);
        return true;
    };
    if (!take(bound.flash_fwd, "sentinel_hip_flash_fwd") || !take(bound.flash_bwd, "sentinel_hip_flash_bwd") ||
        !take(bound.flash_fwd_rope, "sentinel_hip_flash_fwd_rope") || !take(bound.flash_bwd_rope, "sentinel_hip_flash_bwd_rope") ||
        !take(bound.flash_fwd_sparse, "sentinel_hip_flash_fwd_sparse") || !take(bound.flash_bwd_sparse, "sentinel_hip_flash_bwd_sparse") ||
        !take(bound.flash_workspace_bytes, "sentinel_hip_flash_workspace_bytes") ||
        !take(bound.decode_attention, "sentinel_hip_decode_attention") ||
        !take(bound.decode_workspace_bytes, "sentinel_hip_decode_workspace_bytes") ||
        !take(bound.dense_softmax_fwd, "sentinel_hip_dense_softmax_fwd") || !take(bound.dense_softmax_bwd, "sentinel_hip_dense_softmax_bwd") ||
        !take(bound.rope_rotate, "sentinel_hip_rope_rotate") || !take(bound.last_error, "sentinel_hip_last_error"))
        return nullptr;
    lib = bound;
    Py_RETURN_NONE;
}

#define SENTINEL_CALL(name) {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(guarded<name>)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {SENTINEL_CALL(columns_forward), SENTINEL_CALL(columns_backward), SENTINEL_CALL(native_forward),
                         SENTINEL_CALL(native_backward), SENTINEL_CALL(decode),           SENTINEL_CALL(softmax_forward),
                         SENTINEL_CALL(softmax_backward), SENTINEL_CALL(rotate),          {"bind", bind, METH_O, nullptr},
                         {nullptr, nullptr, 0, nullptr}};
#undef SENTINEL_CALL
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_torch_calls", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__torch_calls(void) {
    PyObject* torch_c = PyImport_ImportModule("torch._C");
    if (!torch_c) return nullptr;
    current_raw_stream = PyObject_GetAttrString(torch_c, "_cuda_getCurrentRawStream");
    Py_DECREF(torch_c);
    if (!current_raw_stream) return nullptr;
    return PyModule_Create(&module);
}
