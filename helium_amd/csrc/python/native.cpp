// The parts of the Python mirror that a small execution spends its host time in, against the CPython API: tensor handles and
// execute_graph. Through ctypes a call on a 256 x 512 x 512 layer took 4.5 us on top of the library's 3.9 (argument arrays, a
// ctypes object and a Python destructor per tensor), and a training step with 53 results about 60 us.
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#include <structmember.h>

#include <vector>

#include "helium_hip.h"

namespace {

// The base of backend.Tensor: owns a he_tensor_t.
struct TensorObject {
    PyObject_HEAD
    he_tensor_t tensor;
};

void release(TensorObject* self) {
    he_tensor_t t = self->tensor;
    self->tensor = nullptr;
    if (!t) return;
    Py_BEGIN_ALLOW_THREADS  // (an upload that is still under way is waited for)
    he_tensor_free(t);
    Py_END_ALLOW_THREADS
}

// A handle as Python code has it: None, a number, or an object with a `value` (ctypes.c_void_p).
bool handle_from(PyObject* o, he_tensor_t* out) {
    *out = nullptr;
    if (o == Py_None) return true;
    PyObject* number = PyLong_Check(o) ? (Py_INCREF(o), o) : PyObject_GetAttrString(o, "value");
    if (!number) return false;
    bool ok = true;
    if (number != Py_None) {
        *out = (he_tensor_t)PyLong_AsVoidPtr(number);
        ok = !PyErr_Occurred();
    }
    Py_DECREF(number);
    return ok;
}

PyObject* tensor_new(PyTypeObject* type, PyObject*, PyObject*) {
    TensorObject* self = (TensorObject*)type->tp_alloc(type, 0);
    if (self) self->tensor = nullptr;
    return (PyObject*)self;
}
int tensor_init(PyObject* self, PyObject* args, PyObject* kwargs) {
    static const char* names[] = {"handle", nullptr};
    PyObject* handle = nullptr;
    he_tensor_t t = nullptr;
    if (!PyArg_ParseTupleAndKeywords(args, kwargs, "O", (char**)names, &handle) || !handle_from(handle, &t)) return -1;
    ((TensorObject*)self)->tensor = t;
    return 0;
}
void tensor_dealloc(PyObject* self) {
    release((TensorObject*)self);
    Py_TYPE(self)->tp_free(self);
}
PyObject* tensor_free(PyObject* self, PyObject*) {
    release((TensorObject*)self);
    Py_RETURN_NONE;
}
PyObject* get_handle(PyObject* self, void*) {
    he_tensor_t t = ((TensorObject*)self)->tensor;
    if (!t) Py_RETURN_NONE;
    return PyLong_FromVoidPtr(t);
}
int set_handle(PyObject* self, PyObject* value, void*) {
    he_tensor_t t = nullptr;
    if (!value || !handle_from(value, &t)) return -1;
    ((TensorObject*)self)->tensor = t;
    return 0;
}

PyGetSetDef tensor_getset[] = {{"_handle", get_handle, set_handle, "the he_tensor_t, as a number (None: freed)", nullptr}, {nullptr, nullptr, nullptr, nullptr, nullptr}};
PyMethodDef tensor_methods[] = {{"free", tensor_free, METH_NOARGS, "lets go of the storage"}, {nullptr, nullptr, 0, nullptr}};
PyTypeObject tensor_type = {PyVarObject_HEAD_INIT(nullptr, 0)};

// execute_graph(graph handle, {node: tensor}, most results, tensor class) -> {node: tensor}, or a status to raise.
PyObject* execute_graph(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
    if (nargs != 4 || !PyDict_Check(args[1]) || !PyType_Check(args[3]) || !PyType_IsSubtype((PyTypeObject*)args[3], &tensor_type)) {
        PyErr_SetString(PyExc_TypeError, "execute_graph takes a handle, a dict, a number and a tensor class");
        return nullptr;
    }
    void* graph = PyLong_AsVoidPtr(args[0]);
    const long most = PyLong_AsLong(args[2]);
    if (PyErr_Occurred()) return nullptr;
    std::vector<uint32_t> nodes, out_nodes((size_t)(most > 1 ? most : 1));
    std::vector<he_tensor_t> tensors, out_tensors(out_nodes.size());
    std::vector<PyObject*> held;  // (another thread may change the dict while the call runs)
    const size_t n = (size_t)PyDict_GET_SIZE(args[1]);
    nodes.reserve(n);
    tensors.reserve(n);
    held.reserve(n);
    PyObject *key, *value;
    bool ok = true;
    for (Py_ssize_t at = 0; ok && PyDict_Next(args[1], &at, &key, &value);) {
        he_tensor_t tensor = nullptr;
        if (PyObject_TypeCheck(value, &tensor_type)) {
            tensor = ((TensorObject*)value)->tensor;
        } else {  // (anything with a handle)
            PyObject* handle = PyObject_GetAttrString(value, "handle");
            ok = handle && handle_from(handle, &tensor);
            Py_XDECREF(handle);
            if (!ok) break;
        }
        PyObject* index = PyNumber_Index(key);  // (numpy's integers are fine)
        const unsigned long node = index ? PyLong_AsUnsignedLong(index) : (unsigned long)-1;
        Py_XDECREF(index);
        ok = !PyErr_Occurred();
        if (ok && node > 0xffffffffull) {
            PyErr_SetString(PyExc_OverflowError, "node id out of range");
            ok = false;
        }
        if (!ok) break;
        Py_INCREF(value);
        held.push_back(value);
        nodes.push_back((uint32_t)node);
        tensors.push_back(tensor);
    }
    int status = 0, count = 0;
    if (ok) {
        Py_BEGIN_ALLOW_THREADS
        status = he_execute_graph((he_graph_t)graph, nodes.data(), tensors.data(), (int)nodes.size(), out_nodes.data(), out_tensors.data(), (int)out_nodes.size(), &count);
        Py_END_ALLOW_THREADS
    }
    for (PyObject* v : held) Py_DECREF(v);
    if (!ok) return nullptr;
    if (status != 0) return PyLong_FromLong(status);
    PyTypeObject* type = (PyTypeObject*)args[3];
    PyObject* result = PyDict_New();
    for (int i = 0; i < count; i++) {
        TensorObject* t = result ? (TensorObject*)type->tp_alloc(type, 0) : nullptr;
        PyObject* node = t ? PyLong_FromUnsignedLong(out_nodes[i]) : nullptr;
        if (t) t->tensor = out_tensors[i];
        else he_tensor_free(out_tensors[i]);
        if (!node || PyDict_SetItem(result, node, (PyObject*)t) != 0) Py_CLEAR(result);
        Py_XDECREF(node);
        Py_XDECREF((PyObject*)t);
    }
    return result;
}

PyMethodDef functions[] = {{"execute_graph", (PyCFunction)(void*)execute_graph, METH_FASTCALL, "see backend.execute_graph"}, {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_native", nullptr, -1, functions, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__native() {
    tensor_type.tp_name = "helium_amd._native.Tensor";
    tensor_type.tp_basicsize = sizeof(TensorObject);
    tensor_type.tp_flags = Py_TPFLAGS_DEFAULT | Py_TPFLAGS_BASETYPE;
    tensor_type.tp_new = tensor_new;
    tensor_type.tp_init = tensor_init;
    tensor_type.tp_dealloc = tensor_dealloc;
    tensor_type.tp_getset = tensor_getset;
    tensor_type.tp_methods = tensor_methods;
    if (PyType_Ready(&tensor_type) < 0) return nullptr;
    PyObject* m = PyModule_Create(&module);
    if (!m) return nullptr;
    Py_INCREF(&tensor_type);
    if (PyModule_AddObject(m, "Tensor", (PyObject*)&tensor_type) < 0) return nullptr;
    return m;
}
