// Host side of the Python mirror (cgpt_amd/ops.py): what every operator call checks about its tensors, done on the
// tensors themselves instead of through a dozen attribute lookups in Python, and the call of the library itself. A call of a small
// operator is bound by the host (about 2.6 us per kernel launch); the checks took longer than the launch (3 tensors: 1.3 us in
// Python, 0.15 us here; the 134 parameters of a 12-layer model's AdamW update: 300 us in Python, 25 us here), and so did the
// way through ctypes with ten to twenty arguments. us of host time a call, checks and call in Python and both here: add 4.5 -> 3.1,
// rmsnorm_backward 8.3 -> 5.9 (two launches), linear_backward 6.0 -> 3.6, attention 6.5 -> 3.2; a block of 128 tokens, forward and
// backward, 212.6 -> 169.7.
#include <Python.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cmath>
#include <exception>
#include <limits>

#include "cgptx.h"

namespace {

// The library's dtype code of a tensor, or -1.
int dtype_code(const at::Tensor& t) {
    switch (t.scalar_type()) {
        case at::ScalarType::Half: return CGPTX_F16;
        case at::ScalarType::BFloat16: return CGPTX_BF16;
        case at::ScalarType::Float: return CGPTX_F32;
        default: return -1;
    }
}

PyObject* none() { Py_RETURN_NONE; }

// A reference that is dropped on every way out, exceptions included.
struct Owned {
    PyObject* object = nullptr;
    Owned() = default;
    explicit Owned(PyObject* o) : object(o) {}
    Owned(Owned&& other) noexcept : object(other.release()) {}
    Owned(const Owned&) = delete;
    ~Owned() { Py_XDECREF(object); }
    PyObject* release() {
        PyObject* o = object;
        object = nullptr;
        return o;
    }
};

// tensors(*tensors) -> (dtype code, pointer of each), pointer 0 for None; None when one of them is no contiguous
// device tensor or they do not share one of the library's dtypes.
PyObject* tensors(PyObject*, PyObject* const* args, Py_ssize_t count) {
    Owned out(PyTuple_New(count + 1));
    if (out.object == nullptr) return nullptr;
    int code = -1;
    for (Py_ssize_t i = 0; i < count; ++i) {
        unsigned long long pointer = 0;
        if (args[i] != Py_None) {
            if (!THPVariable_Check(args[i])) return none();
            const at::Tensor& t = THPVariable_Unpack(args[i]);
            const int mine = dtype_code(t);
            if (code < 0) code = mine;
            if (mine < 0 || mine != code || !t.is_cuda() || t.layout() != at::kStrided || !t.is_contiguous())
                return none();
            pointer = reinterpret_cast<unsigned long long>(t.data_ptr());
        }
        PyTuple_SET_ITEM(out.object, i + 1, PyLong_FromUnsignedLongLong(pointer));
    }
    PyTuple_SET_ITEM(out.object, 0, PyLong_FromLong(code));
    return out.release();
}

// same_shape(*tensors) -> bool
PyObject* same_shape(PyObject*, PyObject* const* args, Py_ssize_t count) {
    for (Py_ssize_t i = 0; i < count; ++i) {
        if (!THPVariable_Check(args[i])) Py_RETURN_FALSE;
        if (i > 0 && THPVariable_Unpack(args[i]).sizes() != THPVariable_Unpack(args[0]).sizes()) Py_RETURN_FALSE;
    }
    Py_RETURN_TRUE;
}

struct Names {
    PyObject *parameter, *gradient, *state, *master, *first, *second;
};
Names names;

// A tensor attribute of an object. Null (no error set) if it is no tensor.
Owned tensor_attribute(PyObject* object, PyObject* name) {
    Owned value(PyObject_GetAttr(object, name));
    if (value.object == nullptr) PyErr_Clear();
    else if (!THPVariable_Check(value.object)) return Owned();
    return value;
}

// adamw_entries(entries, states or None, address of the cgptx_adamw_entry array, its length) -> bool. Fills the array when
// there are as many entries (looked at in a copy of the list, which other code may change meanwhile) and every entry is what the update takes: device tensors of one dtype and shape per entry, fp32 master copy and moments of that
// shape on the same device, and the states that the workspace was bound to. False otherwise (the caller says what is wrong).
PyObject* adamw_entries(PyObject*, PyObject* const* args, Py_ssize_t count) {
    if (count != 4 || !PyList_Check(args[0])) Py_RETURN_FALSE;
    const Owned entries(PyList_AsTuple(args[0]));
    if (entries.object == nullptr) return nullptr;
    const Py_ssize_t n = PyTuple_GET_SIZE(entries.object);
    PyObject* bound = args[1] == Py_None ? nullptr : args[1];
    if (bound != nullptr && (!PyList_Check(bound) || PyList_GET_SIZE(bound) != n)) Py_RETURN_FALSE;
    auto* out = reinterpret_cast<cgptx_adamw_entry*>(PyLong_AsUnsignedLongLong(args[2]));
    const Py_ssize_t length = PyLong_AsSsize_t(args[3]);
    if (PyErr_Occurred()) return nullptr;
    if (length != n) Py_RETURN_FALSE;
    for (Py_ssize_t i = 0; i < n; ++i) {
        PyObject* entry = PyTuple_GET_ITEM(entries.object, i);
        const Owned held_state(PyObject_GetAttr(entry, names.state));
        PyObject* state = held_state.object;
        if (state == nullptr) {
            PyErr_Clear();
            Py_RETURN_FALSE;
        }
        const Owned held[5] = {tensor_attribute(entry, names.parameter), tensor_attribute(entry, names.gradient),
                               tensor_attribute(state, names.master), tensor_attribute(state, names.first),
                               tensor_attribute(state, names.second)};
        bool fine = bound == nullptr || state == PyList_GET_ITEM(bound, i);
        for (const Owned& h : held) fine = fine && h.object != nullptr;
        if (fine) {
            const at::Tensor& p = THPVariable_Unpack(held[0].object);
            const at::Tensor& g = THPVariable_Unpack(held[1].object);
            const int code = dtype_code(p);
            fine = code >= 0 && p.is_cuda() && g.scalar_type() == p.scalar_type() && g.sizes() == p.sizes() && g.device() == p.device();
            for (int k = 2; k < 5; ++k) {
                const at::Tensor& t = THPVariable_Unpack(held[k].object);
                fine = fine && t.scalar_type() == at::ScalarType::Float && t.sizes() == p.sizes() && t.device() == p.device();
            }
            if (fine) {
                out[i].parameter = p.data_ptr();
                out[i].gradient = g.data_ptr();
                out[i].master_parameter = static_cast<float*>(THPVariable_Unpack(held[2].object).data_ptr());
                out[i].first_moment = static_cast<float*>(THPVariable_Unpack(held[3].object).data_ptr());
                out[i].second_moment = static_cast<float*>(THPVariable_Unpack(held[4].object).data_ptr());
                out[i].count = static_cast<size_t>(p.numel());
                out[i].dtype = code;
            }
        }
        if (!fine) Py_RETURN_FALSE;
    }
    Py_RETURN_TRUE;
}

// A tensor may refuse to say where or how large it is (fake tensors, symbolic sizes) with a C++ exception, which must not
// leave a C entry: it becomes the Python exception that the tensor's own method would raise.
template <PyObject* (*Function)(PyObject*, PyObject* const*, Py_ssize_t)>
PyObject* call(PyObject* self, PyObject* const* args, Py_ssize_t count) {
    try {
        return Function(self, args, count);
    } catch (const std::exception& error) {
        if (!PyErr_Occurred()) PyErr_SetString(PyExc_RuntimeError, error.what());
        return nullptr;
    }
}

// ---- whole operator calls ------------------------------------------------------------------------------------------------
// name(tensors ..., options ..., stream) -> the library's status (0: done), or None for a call that is not what it
// takes as a rule (a tensor of a subclass, a number of another kind, shapes that do not fit): the function of the same name in
// ops.py then looks at it closely, and either makes the call or says what is wrong. Nothing is refused here, and nothing is taken that
// is refused there.

// The arguments of a call; `ok` once false, the call is not taken.
struct Call {
    PyObject* const* args;
    bool ok = true;
    int code = -1;  // the dtype that the tensors share

    bool need(bool condition) { return ok = ok && condition; }
    // A contiguous device tensor of the call's dtype (null for None where `optional`).
    const at::Tensor* tensor(int i, bool optional = false) {
        if (!ok || (optional && args[i] == Py_None)) return nullptr;
        if (!need(THPVariable_CheckExact(args[i]))) return nullptr;
        const at::Tensor& t = THPVariable_Unpack(args[i]);
        const int mine = dtype_code(t);
        if (code < 0) code = mine;
        return need(mine >= 0 && mine == code && t.is_cuda() && t.layout() == at::kStrided && t.is_contiguous()) ? &t : nullptr;
    }
    // A contiguous device tensor of a type of its own.
    const at::Tensor* other(int i, at::ScalarType type, at::ScalarType or_type, bool contiguous = true) {
        if (!need(ok && THPVariable_CheckExact(args[i]))) return nullptr;
        const at::Tensor& t = THPVariable_Unpack(args[i]);
        return need((t.scalar_type() == type || t.scalar_type() == or_type) && t.is_cuda() && t.layout() == at::kStrided &&
                    (!contiguous || t.is_contiguous()))
                   ? &t : nullptr;
    }
    const at::Tensor* f32(int i) { return other(i, at::ScalarType::Float, at::ScalarType::Float); }
    const at::Tensor* ids(int i, size_t count) {
        const at::Tensor* t = other(i, at::ScalarType::Int, at::ScalarType::UInt32, false);
        need(ok && static_cast<size_t>(t->numel()) >= count);
        return t;
    }
    int flag(PyObject* o) {
        need(PyBool_Check(o));
        return o == Py_True ? 1 : 0;
    }
    int flag(int i) { return flag(args[i]); }
    size_t size(PyObject* o) {
        if (!need(ok && PyLong_CheckExact(o))) return 0;
        const size_t value = PyLong_AsSize_t(o);
        if (PyErr_Occurred()) {
            PyErr_Clear();
            ok = false;
        }
        return value;
    }
    size_t size(int i) { return size(args[i]); }
    float number(PyObject* o) {
        if (!need(ok && PyFloat_CheckExact(o) && std::fabs(PyFloat_AS_DOUBLE(o)) <= std::numeric_limits<float>::max())) return 0.0f;
        return static_cast<float>(PyFloat_AS_DOUBLE(o));
    }
    float positive(int i) {
        const float value = number(args[i]);
        need(ok && PyFloat_AS_DOUBLE(args[i]) > 0.0);
        return value;
    }
};

void* data(const at::Tensor* t) { return t != nullptr ? t->data_ptr() : nullptr; }
size_t at(const at::Tensor* t, int64_t i) { return static_cast<size_t>(t->size(i)); }
bool same(const at::Tensor* a, const at::Tensor* b) { return a->sizes() == b->sizes(); }

struct {
    PyObject *current_device, *current_raw_stream, *stream_type;                          // torch._C's, torch.cuda.Stream
    PyObject *cuda_stream, *query_heads, *kv_heads, *head_dim, *scale, *causal, *offset;  // attribute names
} python;

// The handle of a stream argument: of the current stream for None.
cgptx_stream stream_of(Call& c, int i) {
    PyObject* const given = c.args[i];
    Owned handle;
    if (!c.ok) return nullptr;
    if (given == Py_None) {
        const Owned device(PyObject_CallObject(python.current_device, nullptr));
        if (device.object != nullptr) handle.object = PyObject_CallFunctionObjArgs(python.current_raw_stream, device.object, nullptr);
    } else if (PyLong_CheckExact(given)) {
        Py_INCREF(given);
        handle.object = given;
    } else if (PyObject_IsInstance(given, python.stream_type) == 1) {
        handle.object = PyObject_GetAttr(given, python.cuda_stream);
    }
    void* value = nullptr;
    if (handle.object != nullptr && PyLong_CheckExact(handle.object)) value = PyLong_AsVoidPtr(handle.object);
    else c.ok = false;
    if (PyErr_Occurred()) {
        PyErr_Clear();
        c.ok = false;
    }
    return value;
}

// Other threads run during the library's call, as they do during one through ctypes.
struct WithoutLock {
    PyThreadState* state = PyEval_SaveThread();
    ~WithoutLock() { PyEval_RestoreThread(state); }
};
template <typename Launch>
PyObject* finish(const Call& c, Launch&& launch) {
    if (!c.ok) return none();
    int status = 0;
    {
        WithoutLock released;
        status = launch();
    }
    return PyLong_FromLong(status);
}

PyObject* rmsnorm_forward(Call c) {  // output, input, weight, epsilon, stream
    const at::Tensor *y = c.tensor(0), *x = c.tensor(1), *w = c.tensor(2);
    const float epsilon = c.positive(3);
    if (!c.need(c.ok && x->dim() == 2 && same(y, x) && w->dim() == 1 && at(w, 0) == at(x, 1))) return none();
    const auto stream = stream_of(c, 4);
    return finish(c, [&] { return cgptx_rmsnorm_forward(data(y), data(x), data(w), at(x, 0), at(x, 1), epsilon, c.code, stream); });
}

PyObject* rmsnorm_backward(Call c) {  // grad_input, grad_weight, grad_output, input, weight, epsilon, stream
    const at::Tensor *dx = c.tensor(0), *dw = c.tensor(1), *dy = c.tensor(2), *x = c.tensor(3), *w = c.tensor(4);
    const float epsilon = c.positive(5);
    if (!c.need(c.ok && x->dim() == 2 && same(x, dy) && same(x, dx) && w->dim() == 1 && dw->dim() == 1 && at(w, 0) == at(x, 1) &&
                at(dw, 0) == at(x, 1)))
        return none();
    const auto stream = stream_of(c, 6);
    return finish(c, [&] {
        return cgptx_rmsnorm_backward(data(dx), data(dw), data(dy), data(x), data(w), at(x, 0), at(x, 1), epsilon, c.code, stream);
    });
}

bool rotary_fits(const at::Tensor* q, const at::Tensor* k, const at::Tensor* cos, const at::Tensor* sin, size_t rotary_dim) {
    return q->dim() == 4 && k->dim() == 4 && at(q, 0) == at(k, 0) && at(q, 1) == at(k, 1) && at(q, 3) == at(k, 3) && cos->dim() == 2 &&
           same(cos, sin) && at(cos, 1) * 2 == (rotary_dim != 0 ? rotary_dim : at(q, 3));
}

PyObject* rope_forward(Call c) {  // query, key, cos, sin, rotary_dim, position_offset, stream
    const at::Tensor *q = c.tensor(0), *k = c.tensor(1), *cos = c.tensor(2), *sin = c.tensor(3);
    const size_t rotary_dim = c.size(4), offset = c.size(5);
    if (!c.need(c.ok && rotary_fits(q, k, cos, sin, rotary_dim))) return none();
    const auto stream = stream_of(c, 6);
    return finish(c, [&] {
        return cgptx_rope_forward(data(q), data(k), data(cos), data(sin), at(q, 0), at(q, 1), at(q, 2), at(k, 2), at(q, 3), rotary_dim,
                                  offset, at(cos, 0), c.code, stream);
    });
}

PyObject* rope_backward(Call c) {  // grad_query, grad_key, grad_rotated_query, grad_rotated_key, cos, sin, rotary_dim, position_offset, stream
    const at::Tensor *gq = c.tensor(0), *gk = c.tensor(1), *rq = c.tensor(2), *rk = c.tensor(3), *cos = c.tensor(4), *sin = c.tensor(5);
    const size_t rotary_dim = c.size(6), offset = c.size(7);
    if (!c.need(c.ok && same(gq, rq) && same(gk, rk) && rotary_fits(gq, gk, cos, sin, rotary_dim))) return none();
    const auto stream = stream_of(c, 8);
    return finish(c, [&] {
        return cgptx_rope_backward(data(gq), data(gk), data(rq), data(rk), data(cos), data(sin), at(gq, 0), at(gq, 1), at(gq, 2),
                                   at(gk, 2), at(gq, 3), rotary_dim, offset, at(cos, 0), c.code, stream);
    });
}

PyObject* swiglu_forward(Call c) {  // output, gate, up, stream
    const at::Tensor *y = c.tensor(0), *g = c.tensor(1), *u = c.tensor(2);
    if (!c.need(c.ok && same(g, y) && same(g, u))) return none();
    const auto stream = stream_of(c, 3);
    return finish(c, [&] { return cgptx_swiglu_forward(data(y), data(g), data(u), static_cast<size_t>(g->numel()), c.code, stream); });
}

PyObject* swiglu_backward(Call c) {  // grad_gate, grad_up, grad_output, gate, up, accumulate_gate, accumulate_up, stream
    const at::Tensor *dg = c.tensor(0), *du = c.tensor(1), *dy = c.tensor(2), *g = c.tensor(3), *u = c.tensor(4);
    const int accumulate_gate = c.flag(5), accumulate_up = c.flag(6);
    if (!c.need(c.ok && same(dy, dg) && same(dy, du) && same(dy, g) && same(dy, u))) return none();
    const auto stream = stream_of(c, 7);
    return finish(c, [&] {
        return cgptx_swiglu_backward(data(dg), data(du), data(dy), data(g), data(u), static_cast<size_t>(dy->numel()), accumulate_gate,
                                     accumulate_up, c.code, stream);
    });
}

// y[..., out] of x[..., in] and w[out, in], nothing empty.
bool projects(const at::Tensor* y, const at::Tensor* x, const at::Tensor* w) {
    const auto xs = x->sizes(), ys = y->sizes();
    return w->dim() == 2 && !xs.empty() && xs.size() == ys.size() && xs.back() == w->size(1) && ys.back() == w->size(0) && w->numel() > 0 &&
           xs.slice(0, xs.size() - 1) == ys.slice(0, ys.size() - 1);
}

PyObject* linear_forward(Call c) {  // output, input, weight, bias or None, stream
    const at::Tensor *y = c.tensor(0), *x = c.tensor(1), *w = c.tensor(2), *b = c.tensor(3, true);
    if (!c.need(c.ok && projects(y, x, w))) return none();
    const auto stream = stream_of(c, 4);
    return finish(c, [&] {
        return cgptx_linear_forward(data(y), data(x), data(w), data(b), static_cast<size_t>(x->numel()) / at(w, 1), at(w, 1), at(w, 0),
                                    c.code, stream);
    });
}

PyObject* linear_backward(Call c) {  // grad_input, grad_weight, grad_bias (or None each), grad_output, input, weight, three accumulate flags, stream
    const at::Tensor *dx = c.tensor(0, true), *dw = c.tensor(1, true), *db = c.tensor(2, true), *dy = c.tensor(3), *x = c.tensor(4), *w = c.tensor(5);
    const int input = c.flag(6), weight = c.flag(7), bias = c.flag(8);
    if (!c.need(c.ok && projects(dy, x, w) && (dx == nullptr || same(dx, x)) && (dw == nullptr || same(dw, w)) &&
                (db == nullptr || (db->dim() == 1 && at(db, 0) == at(w, 0)))))
        return none();
    const auto stream = stream_of(c, 9);
    return finish(c, [&] {
        return cgptx_linear_backward(data(dx), data(dw), data(db), data(dy), data(x), data(w), static_cast<size_t>(x->numel()) / at(w, 1),
                                     at(w, 1), at(w, 0), input, weight, bias, c.code, stream);
    });
}

PyObject* add(Call c) {  // output, a, b, stream
    const at::Tensor *y = c.tensor(0), *a = c.tensor(1), *b = c.tensor(2);
    if (!c.need(c.ok && same(a, y) && same(a, b))) return none();
    const auto stream = stream_of(c, 3);
    return finish(c, [&] { return cgptx_add(data(y), data(a), data(b), static_cast<size_t>(a->numel()), c.code, stream); });
}

// FlashAttentionOptions, and whether they fit the tensors.
struct Attention {
    size_t query_heads = 0, kv_heads = 0, head_dim = 0, offset = 0;
    float scale = 0.0f;
    int causal = 0;
    Attention(Call& c, PyObject* options) {
        auto get = [&](PyObject* name) {
            Owned value(PyObject_GetAttr(options, name));
            if (value.object == nullptr) PyErr_Clear();
            c.need(value.object != nullptr);
            return value;
        };
        if (const Owned v = get(python.query_heads); c.ok) query_heads = c.size(v.object);
        if (const Owned v = get(python.kv_heads); c.ok) kv_heads = c.size(v.object);
        if (const Owned v = get(python.head_dim); c.ok) head_dim = c.size(v.object);
        if (const Owned v = get(python.offset); c.ok) offset = c.size(v.object);
        if (const Owned v = get(python.scale); c.ok) scale = c.number(v.object);
        if (const Owned v = get(python.causal); c.ok) causal = c.flag(v.object);
    }
    bool fits(const at::Tensor* q, const at::Tensor* k, const at::Tensor* v) const {
        return q->dim() == 4 && k->dim() == 4 && same(v, k) && query_heads != 0 && kv_heads != 0 && head_dim != 0 && query_heads % kv_heads == 0 &&
               at(q, 0) == at(k, 0) && at(q, 2) == query_heads && at(k, 2) == kv_heads && at(q, 3) == head_dim && at(k, 3) == head_dim &&
               (!causal || (offset <= at(k, 1) && at(q, 1) <= at(k, 1) - offset));
    }
};
bool is_logsumexp(const at::Tensor* lse, const at::Tensor* q) { return lse->sizes() == q->sizes().slice(0, 3); }

PyObject* attention_forward(Call c) {  // output, logsumexp or None, query, key, value, options, stream
    const at::Tensor *o = c.tensor(0), *q = c.tensor(2), *k = c.tensor(3), *v = c.tensor(4);
    const at::Tensor* lse = c.args[1] != Py_None ? c.f32(1) : nullptr;
    if (!c.ok) return none();
    const Attention a(c, c.args[5]);
    if (!c.need(c.ok && a.fits(q, k, v) && same(o, q) && (lse == nullptr || is_logsumexp(lse, q)))) return none();
    const auto stream = stream_of(c, 6);
    return finish(c, [&] {
        return cgptx_flash_gqa_attention_forward(data(o), static_cast<float*>(data(lse)), data(q), data(k), data(v), at(q, 0), at(q, 1),
                                                 at(k, 1), a.query_heads, a.kv_heads, a.head_dim, a.scale, a.causal, a.offset, c.code, stream);
    });
}

PyObject* attention_backward_with_lse(Call c) {  // grad_query, grad_key, grad_value, grad_output, output, logsumexp, query, key, value, options, accumulate, stream
    const at::Tensor *dq = c.tensor(0), *dk = c.tensor(1), *dv = c.tensor(2), *d_o = c.tensor(3), *o = c.tensor(4), *q = c.tensor(6),
                     *k = c.tensor(7), *v = c.tensor(8), *lse = c.f32(5);
    if (!c.ok) return none();
    const Attention a(c, c.args[9]);
    const int accumulate = c.flag(10);
    if (!c.need(c.ok && a.fits(q, k, v) && same(q, d_o) && same(q, dq) && same(q, o) && same(k, dk) && same(k, dv) && is_logsumexp(lse, q)))
        return none();
    const auto stream = stream_of(c, 11);
    return finish(c, [&] {
        return cgptx_flash_gqa_attention_backward_with_lse(data(dq), data(dk), data(dv), data(d_o), data(o), static_cast<float*>(data(lse)),
                                                           data(q), data(k), data(v), at(q, 0), at(q, 1), at(k, 1), a.query_heads, a.kv_heads,
                                                           a.head_dim, a.scale, a.causal, a.offset, accumulate, c.code, stream);
    });
}

PyObject* attention_backward(Call c) {  // grad_query, grad_key, grad_value, grad_output, query, key, value, options, accumulate, stream
    const at::Tensor *dq = c.tensor(0), *dk = c.tensor(1), *dv = c.tensor(2), *d_o = c.tensor(3), *q = c.tensor(4), *k = c.tensor(5), *v = c.tensor(6);
    if (!c.ok) return none();
    const Attention a(c, c.args[7]);
    const int accumulate = c.flag(8);
    if (!c.need(c.ok && a.fits(q, k, v) && same(q, d_o) && same(q, dq) && same(k, dk) && same(k, dv))) return none();
    const auto stream = stream_of(c, 9);
    return finish(c, [&] {
        return cgptx_flash_gqa_attention_backward(data(dq), data(dk), data(dv), data(d_o), data(q), data(k), data(v), at(q, 0), at(q, 1), at(k, 1),
                                                  a.query_heads, a.kv_heads, a.head_dim, a.scale, a.causal, a.offset, accumulate, c.code, stream);
    });
}

PyObject* embedding_forward(Call c) {  // output, ids, count, weight, stream
    const at::Tensor *y = c.tensor(0), *w = c.tensor(3);
    const size_t count = c.size(2);
    const at::Tensor* ids = c.ids(1, count);
    if (!c.need(c.ok && count > 0 && w->dim() == 2 && static_cast<size_t>(y->numel()) == count * at(w, 1))) return none();
    const auto stream = stream_of(c, 4);
    return finish(c, [&] {
        return cgptx_embedding_forward(data(y), static_cast<const uint32_t*>(data(ids)), count, data(w), at(w, 0), at(w, 1), c.code, stream);
    });
}

PyObject* embedding_backward(Call c) {  // grad_weight, grad_output, ids, count, bounds_check, accumulate_weight, stream
    const at::Tensor *dw = c.tensor(0), *dy = c.tensor(1);
    const size_t count = c.size(3);
    const at::Tensor* ids = c.ids(2, count);
    const int bounds_check = c.flag(4), accumulate = c.flag(5);
    if (!c.need(c.ok && count > 0 && dw->dim() == 2 && dy->dim() >= 1 && dy->size(-1) == dw->size(1) &&
                static_cast<size_t>(dy->numel()) == count * at(dw, 1)))
        return none();
    const auto stream = stream_of(c, 6);
    return finish(c, [&] {
        return cgptx_embedding_backward(data(dw), data(dy), static_cast<const uint32_t*>(data(ids)), count, at(dw, 0), at(dw, 1), bounds_check,
                                        accumulate, c.code, stream);
    });
}

bool is_loss(const at::Tensor* loss) { return loss->numel() == 1; }

PyObject* cross_entropy_forward_backward(Call c) {  // loss, gradient, logits, targets, count, gradient_scale, stream
    const at::Tensor *g = c.tensor(1), *z = c.tensor(2), *loss = c.f32(0);
    const size_t count = c.size(4);
    const at::Tensor* targets = c.ids(3, count);
    const float scale = c.positive(5);
    if (!c.need(c.ok && count > 0 && z->dim() == 2 && at(z, 0) == count && at(z, 1) > 0 && is_loss(loss) && same(g, z))) return none();
    const auto stream = stream_of(c, 6);
    return finish(c, [&] {
        return cgptx_cross_entropy_forward_backward(static_cast<float*>(data(loss)), data(g), data(z), static_cast<const uint32_t*>(data(targets)),
                                                    count, at(z, 1), scale, c.code, stream);
    });
}

PyObject* cross_entropy_forward(Call c) {  // loss, logits, targets, count, stream
    const at::Tensor *z = c.tensor(1), *loss = c.f32(0);
    const size_t count = c.size(3);
    const at::Tensor* targets = c.ids(2, count);
    if (!c.need(c.ok && count > 0 && z->dim() == 2 && at(z, 0) == count && at(z, 1) > 0 && is_loss(loss))) return none();
    const auto stream = stream_of(c, 4);
    return finish(c, [&] {
        return cgptx_cross_entropy_forward(static_cast<float*>(data(loss)), data(z), static_cast<const uint32_t*>(data(targets)), count, at(z, 1),
                                           c.code, stream);
    });
}

PyObject* cut_cross_entropy_forward_backward(Call c) {  // loss, input_gradient, classifier_gradient, input, classifier, targets, count, scale, accumulate, stream
    const at::Tensor *dx = c.tensor(1), *dc = c.tensor(2), *x = c.tensor(3), *w = c.tensor(4), *loss = c.f32(0);
    const size_t count = c.size(6);
    const at::Tensor* targets = c.ids(5, count);
    const float scale = c.number(c.args[7]);
    const int accumulate = c.flag(8);
    if (!c.need(c.ok && count > 0 && x->dim() == 2 && w->dim() == 2 && at(x, 1) == at(w, 1) && at(x, 0) == count && same(dx, x) && same(dc, w) &&
                is_loss(loss)))
        return none();
    const auto stream = stream_of(c, 9);
    return finish(c, [&] {
        return cgptx_cut_cross_entropy_forward_backward(static_cast<float*>(data(loss)), data(dx), data(dc), data(x), data(w),
                                                        static_cast<const uint32_t*>(data(targets)), count, at(x, 1), at(w, 0), scale, accumulate,
                                                        c.code, stream);
    });
}

// A tensor that refuses to say what it is makes the call one that is not taken.
template <PyObject* (*Function)(Call), int COUNT>
PyObject* operation(PyObject*, PyObject* const* args, Py_ssize_t count) {
    if (count != COUNT) return none();
    try {
        return Function(Call{args});
    } catch (const std::exception&) {
        PyErr_Clear();
        return none();
    }
}
template <PyObject* (*Function)(Call), int COUNT>
PyMethodDef method(const char* name) {
    return {name, reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(operation<Function, COUNT>)), METH_FASTCALL, "the library's status, or None: not taken"};
}

PyMethodDef methods[] = {
    method<rmsnorm_forward, 5>("rmsnorm_forward"),
    method<rmsnorm_backward, 7>("rmsnorm_backward"),
    method<rope_forward, 7>("rope_forward"),
    method<rope_backward, 9>("rope_backward"),
    method<swiglu_forward, 4>("swiglu_forward"),
    method<swiglu_backward, 8>("swiglu_backward"),
    method<linear_forward, 5>("linear_forward"),
    method<linear_backward, 10>("linear_backward"),
    method<add, 4>("add"),
    method<attention_forward, 7>("attention_forward"),
    method<attention_backward_with_lse, 12>("attention_backward_with_lse"),
    method<attention_backward, 10>("attention_backward"),
    method<embedding_forward, 5>("embedding_forward"),
    method<embedding_backward, 7>("embedding_backward"),
    method<cross_entropy_forward_backward, 7>("cross_entropy_forward_backward"),
    method<cross_entropy_forward, 5>("cross_entropy_forward"),
    method<cut_cross_entropy_forward_backward, 10>("cut_cross_entropy_forward_backward"),
    {"tensors", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(call<tensors>)), METH_FASTCALL, "(dtype code, pointers) or None"},
    {"same_shape", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(call<same_shape>)), METH_FASTCALL, "whether all shapes are equal"},
    {"adamw_entries", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(call<adamw_entries>)), METH_FASTCALL, "fills an entry array"},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_dispatch", "Tensor checks of the operator mirror.", -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__dispatch() {
    names = {PyUnicode_InternFromString("parameter"), PyUnicode_InternFromString("gradient"), PyUnicode_InternFromString("state"),
             PyUnicode_InternFromString("master_parameter"), PyUnicode_InternFromString("first_moment"),
             PyUnicode_InternFromString("second_moment")};
    const Owned torch(PyImport_ImportModule("torch._C"));
    const Owned cuda(PyImport_ImportModule("torch.cuda"));
    if (torch.object == nullptr || cuda.object == nullptr) return nullptr;
    python = {PyObject_GetAttrString(torch.object, "_cuda_getDevice"), PyObject_GetAttrString(torch.object, "_cuda_getCurrentRawStream"),
              PyObject_GetAttrString(cuda.object, "Stream"),
              PyUnicode_InternFromString("cuda_stream"), PyUnicode_InternFromString("num_query_heads"), PyUnicode_InternFromString("num_kv_heads"),
              PyUnicode_InternFromString("head_dim"), PyUnicode_InternFromString("attention_scale"), PyUnicode_InternFromString("causal"),
              PyUnicode_InternFromString("query_position_offset")};
    if (python.current_device == nullptr || python.current_raw_stream == nullptr || python.stream_type == nullptr) return nullptr;
    return PyModule_Create(&module);
}
