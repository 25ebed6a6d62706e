// Host side of the Python mirror (cgpt_amd/ops.py): what every operator call checks about its tensors, done on the
// tensors themselves instead of through a dozen attribute lookups in Python. A call of a small operator is bound by the
// host (about 2.6 us per kernel launch); these checks took longer than the launch (3 tensors: 1.3 us in Python, 0.15 us
// here; the 134 parameters of a 12-layer model's AdamW update: 300 us in Python, 25 us here).
#include <Python.h>
#include <torch/csrc/autograd/python_variable.h>

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

// tensors(*tensors) -> (dtype code, pointer of each), pointer 0 for None; None when one of them is no contiguous
// device tensor or they do not share one of the library's dtypes.
PyObject* tensors(PyObject*, PyObject* const* args, Py_ssize_t count) {
    PyObject* out = PyTuple_New(count + 1);
    if (out == nullptr) return nullptr;
    int code = -1;
    for (Py_ssize_t i = 0; i < count; ++i) {
        unsigned long long pointer = 0;
        if (args[i] != Py_None) {
            if (!THPVariable_Check(args[i])) {
                Py_DECREF(out);
                return none();
            }
            const at::Tensor& t = THPVariable_Unpack(args[i]);
            const int mine = dtype_code(t);
            if (code < 0) code = mine;
            if (mine < 0 || mine != code || !t.is_cuda() || t.layout() != at::kStrided || !t.is_contiguous()) {
                Py_DECREF(out);
                return none();
            }
            pointer = reinterpret_cast<unsigned long long>(t.data_ptr());
        }
        PyTuple_SET_ITEM(out, i + 1, PyLong_FromUnsignedLongLong(pointer));
    }
    PyTuple_SET_ITEM(out, 0, PyLong_FromLong(code));
    return out;
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

// A tensor attribute of an object; the caller drops the reference it receives. Null (no error set) if it is no tensor.
PyObject* tensor_attribute(PyObject* object, PyObject* name) {
    PyObject* value = PyObject_GetAttr(object, name);
    if (value == nullptr) {
        PyErr_Clear();
        return nullptr;
    }
    if (!THPVariable_Check(value)) {
        Py_DECREF(value);
        return nullptr;
    }
    return value;
}

// adamw_entries(entries, states or None, address of the cgptx_adamw_entry array) -> bool. Fills the array when every
// entry is what the update takes: device tensors of one dtype and shape per entry, fp32 master copy and moments of that
// shape on the same device, and the states that the workspace was bound to. False otherwise (the caller says what is wrong).
PyObject* adamw_entries(PyObject*, PyObject* const* args, Py_ssize_t count) {
    if (count != 3 || !PyList_Check(args[0])) Py_RETURN_FALSE;
    const Py_ssize_t n = PyList_GET_SIZE(args[0]);
    PyObject* bound = args[1] == Py_None ? nullptr : args[1];
    if (bound != nullptr && (!PyList_Check(bound) || PyList_GET_SIZE(bound) != n)) Py_RETURN_FALSE;
    auto* out = reinterpret_cast<cgptx_adamw_entry*>(PyLong_AsUnsignedLongLong(args[2]));
    if (PyErr_Occurred()) return nullptr;
    for (Py_ssize_t i = 0; i < n; ++i) {
        PyObject* entry = PyList_GET_ITEM(args[0], i);
        PyObject* state = PyObject_GetAttr(entry, names.state);
        if (state == nullptr) {
            PyErr_Clear();
            Py_RETURN_FALSE;
        }
        PyObject* held[5] = {tensor_attribute(entry, names.parameter), tensor_attribute(entry, names.gradient),
                             tensor_attribute(state, names.master), tensor_attribute(state, names.first),
                             tensor_attribute(state, names.second)};
        bool fine = bound == nullptr || state == PyList_GET_ITEM(bound, i);
        for (PyObject* h : held) fine = fine && h != nullptr;
        if (fine) {
            const at::Tensor& p = THPVariable_Unpack(held[0]);
            const at::Tensor& g = THPVariable_Unpack(held[1]);
            const int code = dtype_code(p);
            fine = code >= 0 && p.is_cuda() && g.scalar_type() == p.scalar_type() && g.sizes() == p.sizes() && g.device() == p.device();
            for (int k = 2; k < 5; ++k) {
                const at::Tensor& t = THPVariable_Unpack(held[k]);
                fine = fine && t.scalar_type() == at::ScalarType::Float && t.sizes() == p.sizes() && t.device() == p.device();
            }
            if (fine) {
                out[i].parameter = p.data_ptr();
                out[i].gradient = g.data_ptr();
                out[i].master_parameter = static_cast<float*>(THPVariable_Unpack(held[2]).data_ptr());
                out[i].first_moment = static_cast<float*>(THPVariable_Unpack(held[3]).data_ptr());
                out[i].second_moment = static_cast<float*>(THPVariable_Unpack(held[4]).data_ptr());
                out[i].count = static_cast<size_t>(p.numel());
                out[i].dtype = code;
            }
        }
        for (PyObject* h : held) Py_XDECREF(h);
        Py_DECREF(state);
        if (!fine) Py_RETURN_FALSE;
    }
    Py_RETURN_TRUE;
}

PyMethodDef methods[] = {
    {"tensors", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(tensors)), METH_FASTCALL, "(dtype code, pointers) or None"},
    {"same_shape", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(same_shape)), METH_FASTCALL, "whether all shapes are equal"},
    {"adamw_entries", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(adamw_entries)), METH_FASTCALL, "fills an entry array"},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_dispatch", "Tensor checks of the operator mirror.", -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__dispatch() {
    names = {PyUnicode_InternFromString("parameter"), PyUnicode_InternFromString("gradient"), PyUnicode_InternFromString("state"),
             PyUnicode_InternFromString("master_parameter"), PyUnicode_InternFromString("first_moment"),
             PyUnicode_InternFromString("second_moment")};
    return PyModule_Create(&module);
}
