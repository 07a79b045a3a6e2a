// What an argument block of tensor addresses was made from, as bytes: one comparison tells whether it still holds.  A small
// Python extension and not part of the library's C ABI, since it reads torch's tensors where they are: four Python calls a
// tensor (data_ptr, stride, size, dtype) took 15 of the 60 us of a decode step.
#include <Python.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cstdint>
#include <vector>

namespace {

// tensor_key(list or tuple of tensors) -> bytes.  Read anew on every call; nothing of a tensor is kept.
PyObject *tensor_key(PyObject *, PyObject *tensors) {
    PyObject *seq = PySequence_Fast(tensors, "tensor_key: a list or tuple of tensors");
    if (!seq) return nullptr;
    PyObject *out = nullptr;
    try {
        std::vector<int64_t> key;
        const Py_ssize_t n = PySequence_Fast_GET_SIZE(seq);
        key.reserve(8 * n);
        for (Py_ssize_t i = 0; i < n; i++) {
            PyObject *item = PySequence_Fast_GET_ITEM(seq, i);
            if (!THPVariable_Check(item)) {
                PyErr_Format(PyExc_TypeError, "tensor_key: item %zd is a %s, not a tensor", i, Py_TYPE(item)->tp_name);
                Py_DECREF(seq);
                return nullptr;
            }
            const at::Tensor &t = THPVariable_Unpack(item);
            key.push_back((int64_t)(intptr_t)t.data_ptr());
            // a tensor without a device index has -1
            key.push_back((int64_t)t.scalar_type() | (int64_t)t.device().type() << 8 | (int64_t)(uint8_t)t.device().index() << 16 |
                          t.dim() << 32);
            for (const int64_t v : t.sizes()) key.push_back(v);
            for (const int64_t v : t.strides()) key.push_back(v);
        }
        out = PyBytes_FromStringAndSize((const char *)key.data(), (Py_ssize_t)(key.size() * sizeof(int64_t)));
    } catch (const std::exception &e) {   // a tensor without memory
        PyErr_SetString(PyExc_RuntimeError, e.what());
    }
    Py_DECREF(seq);
    return out;
}

PyMethodDef methods[] = {{"tensor_key", tensor_key, METH_O, "Address, type, device, sizes and strides of every tensor, as bytes."},
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "plan_key", nullptr, 0, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit_plan_key() { return PyModule_Create(&module); }
