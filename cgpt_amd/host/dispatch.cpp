// Host side of the Python mirror (cgpt_amd/ops.py): what every operator call checks about its tensors, done on the
// tensors themselves instead of through a dozen attribute lookups in Python. A call of a small operator is bound by the
// host (about 2.6 us per kernel launch); these checks took longer than the launch (3 tensors: 1.3 us in Python, 0.15 us
// here; the 134 parameters of a 12-layer model's AdamW update: 300 us in Python, 25 us here).
#include <Python.h>
#include <torch/csrc/autograd/python_variable.h>

#include <exception>

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

PyMethodDef methods[] = {
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
    return PyModule_Create(&module);
}
