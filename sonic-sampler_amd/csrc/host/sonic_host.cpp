// Native part of the eager call path: a Python extension (CPython API and torch's C++ tensors) that
// turns a call's tensors and scalars into the bytes of its argument struct and allocates its
// outputs. Both were most of a small call's host time in Python: about 25 attribute and method calls
// on tensors per argument struct and a keyword-parsed torch.empty per output.
//
//   make_layout(size, fields) -> capsule     fields: (code, offset, offset, offset, name) per argument
//   gather(capsule, *args) -> bytes          the struct, every other byte zero
//   unit_strides(names, *tensors)            ValueError naming the first tensor (None: skipped) that is not
//                                            contiguous along its last dimension
//   empty(device, dtype, *sizes) -> Tensor   torch.empty
//   entry(address, size) -> callable         the entry point at `address`, taking its struct's `size` bytes
//
// Argument codes: a scalar of the field's type ('i', 'I', 'q', 'Q'), or a tensor (None: zeros) whose
// address goes to the first offset ('T'), with its leading stride ('S'), or its leading and, of a
// three-dimensional one, its second stride ('U').
#include <Python.h>

#include <ATen/ATen.h>
#include <torch/csrc/Device.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/utils/device_lazy_init.h>

#include <cstring>
#include <memory>
#include <string>
#include <utility>
#include <vector>

namespace {

struct Field {
    char code;
    Py_ssize_t at[3];
    std::string name;
};

struct Layout {
    Py_ssize_t size;
    std::vector<Field> fields;
};

constexpr const char *CAPSULE = "sonic_sampler.layout";

void destroy(PyObject *capsule) { delete static_cast<Layout *>(PyCapsule_GetPointer(capsule, CAPSULE)); }

int field_bytes(char code) { return code == 'i' || code == 'I' ? 4 : 8; }

// Writes one argument of the struct; false with a Python error set.
bool put(const Field &f, PyObject *arg, char *out) {
    if (f.code == 'q' || f.code == 'i') {
        const long long v = PyLong_AsLongLong(arg);
        if (v == -1 && PyErr_Occurred()) return false;
        if (f.code == 'q') {
            std::memcpy(out + f.at[0], &v, 8);
            return true;
        }
        const int32_t w = (int32_t)v;
        if (w != v) {
            PyErr_Format(PyExc_OverflowError, "%s does not fit 32 bits", f.name.c_str());
            return false;
        }
        std::memcpy(out + f.at[0], &w, 4);
        return true;
    }
    if (f.code == 'Q' || f.code == 'I') {
        PyObject *index = PyNumber_Index(arg);  // integers of other types (numpy's) too
        if (!index) return false;
        const unsigned long long v = PyLong_AsUnsignedLongLong(index);
        Py_DECREF(index);
        if (v == (unsigned long long)-1 && PyErr_Occurred()) return false;
        if (f.code == 'Q') {
            std::memcpy(out + f.at[0], &v, 8);
            return true;
        }
        const uint32_t w = (uint32_t)v;
        if (w != v) {
            PyErr_Format(PyExc_OverflowError, "%s does not fit 32 bits", f.name.c_str());
            return false;
        }
        std::memcpy(out + f.at[0], &w, 4);
        return true;
    }
    if (arg == Py_None) return true;
    if (!THPVariable_Check(arg)) {
        PyErr_Format(PyExc_TypeError, "`%s` must be a tensor or None", f.name.c_str());
        return false;
    }
    const at::Tensor &t = THPVariable_Unpack(arg);
    const uint64_t p = (uint64_t)(uintptr_t)t.data_ptr();
    std::memcpy(out + f.at[0], &p, 8);
    if (f.code != 'T') {
        const int64_t s = t.stride(0);
        std::memcpy(out + f.at[1], &s, 8);
        if (f.code == 'U') {
            const int64_t step = t.dim() >= 3 ? t.stride(1) : 0;
            std::memcpy(out + f.at[2], &step, 8);
        }
    }
    return true;
}

// Runs fn, with a C++ exception as the Python one that torch's own bindings raise for it
// (torch.OutOfMemoryError, IndexError, NotImplementedError, ...).
template <class F>
PyObject *guarded(F fn) {
    HANDLE_TH_ERRORS
    return fn();
    END_HANDLE_TH_ERRORS
}

PyObject *make_layout(PyObject *, PyObject *args) {
    Py_ssize_t size = 0;
    PyObject *list = nullptr;
    if (!PyArg_ParseTuple(args, "nO!", &size, &PyList_Type, &list)) return nullptr;
    return guarded([&]() -> PyObject * {
        auto layout = std::make_unique<Layout>();
        layout->size = size;
        for (Py_ssize_t i = 0; i < PyList_GET_SIZE(list); ++i) {
            int code = 0;
            const char *name = nullptr;
            Field f;
            if (!PyArg_ParseTuple(PyList_GET_ITEM(list, i), "Cnnns", &code, &f.at[0], &f.at[1], &f.at[2], &name)) return nullptr;
            if (code <= 0 || code > 127 || !std::strchr("iIqQTSU", code)) {
                PyErr_Format(PyExc_ValueError, "unknown field code %d", code);
                return nullptr;
            }
            f.code = (char)code;
            f.name = name;
            const int used = f.code == 'S' ? 2 : f.code == 'U' ? 3 : 1;
            for (int k = 0; k < used; ++k) {
                if (f.at[k] < 0 || f.at[k] > size - field_bytes(f.code)) {
                    PyErr_Format(PyExc_ValueError, "field %s outside the struct", name);
                    return nullptr;
                }
            }
            layout->fields.push_back(std::move(f));
        }
        PyObject *capsule = PyCapsule_New(layout.get(), CAPSULE, destroy);
        if (capsule) layout.release();
        return capsule;
    });
}

// The GIL given up for a scope, as torch's own factories do: an allocation that misses the cache
// waits for the device, and other threads (a host callback that the wait depends on, too) go on.
struct ReleasedGil {
    PyThreadState *state = PyEval_SaveThread();
    ~ReleasedGil() { PyEval_RestoreThread(state); }
};

PyObject *gather(PyObject *, PyObject *const *args, Py_ssize_t n) {
    if (n < 1) {
        PyErr_SetString(PyExc_TypeError, "gather(layout, *args)");
        return nullptr;
    }
    const auto *layout = static_cast<Layout *>(PyCapsule_GetPointer(args[0], CAPSULE));
    if (!layout) return nullptr;
    if ((size_t)(n - 1) != layout->fields.size()) {
        PyErr_Format(PyExc_TypeError, "expected %zu arguments, got %zd", layout->fields.size(), n - 1);
        return nullptr;
    }
    PyObject *bytes = PyBytes_FromStringAndSize(nullptr, layout->size);
    if (!bytes) return nullptr;
    char *out = PyBytes_AS_STRING(bytes);
    std::memset(out, 0, (size_t)layout->size);
    PyObject *done = guarded([&]() -> PyObject * {
        for (size_t i = 0; i < layout->fields.size(); ++i)
            if (!put(layout->fields[i], args[i + 1], out)) return nullptr;
        return bytes;
    });
    if (!done) Py_DECREF(bytes);
    return done;
}

PyObject *unit_strides(PyObject *, PyObject *const *args, Py_ssize_t n) {
    if (n < 1 || !PyTuple_Check(args[0]) || PyTuple_GET_SIZE(args[0]) != n - 1) {
        PyErr_SetString(PyExc_TypeError, "unit_strides(names, *tensors) with a tuple of a name for each tensor");
        return nullptr;
    }
    return guarded([&]() -> PyObject * {
        for (Py_ssize_t i = 1; i < n; ++i) {
            if (args[i] == Py_None) continue;
            PyObject *name = PyTuple_GET_ITEM(args[0], i - 1);
            if (!THPVariable_Check(args[i])) {
                PyErr_Format(PyExc_TypeError, "`%S` must be a tensor or None", name);
                return nullptr;
            }
            const at::Tensor &t = THPVariable_Unpack(args[i]);
            if (t.dim() > 0 && t.stride(-1) != 1) {
                PyErr_Format(PyExc_ValueError, "`%S` must be contiguous along its last dimension", name);
                return nullptr;
            }
        }
        Py_RETURN_NONE;
    });
}

PyObject *empty(PyObject *, PyObject *const *args, Py_ssize_t n) {
    constexpr Py_ssize_t MAX_DIMS = 8;
    if (n < 2 || n > 2 + MAX_DIMS || !THPDevice_Check(args[0]) || !THPDtype_Check(args[1])) {
        PyErr_SetString(PyExc_TypeError, "empty(device, dtype, *sizes) with at most 8 sizes");
        return nullptr;
    }
    int64_t sizes[MAX_DIMS];
    for (Py_ssize_t i = 2; i < n; ++i) {
        sizes[i - 2] = PyLong_AsLongLong(args[i]);
        if (sizes[i - 2] == -1 && PyErr_Occurred()) return nullptr;
    }
    return guarded([&]() -> PyObject * {
        const auto options = at::TensorOptions()
                                 .device(reinterpret_cast<THPDevice *>(args[0])->device)
                                 .dtype(reinterpret_cast<THPDtype *>(args[1])->scalar_type);
        torch::utils::maybe_initialize_device(options);
        at::Tensor t;
        {
            const ReleasedGil released;
            t = at::empty(at::IntArrayRef(sizes, (size_t)(n - 2)), options);
        }
        return THPVariable_Wrap(std::move(t));
    });
}

// An entry point of the library called with the struct's bytes, the GIL released meanwhile. `self`
// is its (address, size of the struct): bytes of any other length are refused, the entry point would
// read past them.
PyObject *call_entry(PyObject *self, PyObject *bytes) {
    using Entry = int (*)(const void *);
    const auto fn = reinterpret_cast<Entry>(PyLong_AsVoidPtr(PyTuple_GET_ITEM(self, 0)));
    const Py_ssize_t size = PyLong_AsSsize_t(PyTuple_GET_ITEM(self, 1));
    if (PyErr_Occurred()) return nullptr;
    if (!PyBytes_Check(bytes)) {
        PyErr_SetString(PyExc_TypeError, "the argument struct's bytes are expected");
        return nullptr;
    }
    if (PyBytes_GET_SIZE(bytes) != size) {
        PyErr_Format(PyExc_ValueError, "an argument struct of %zd bytes is expected, got %zd", size, PyBytes_GET_SIZE(bytes));
        return nullptr;
    }
    return guarded([&]() -> PyObject * {
        // the argument structs hold 8-byte fields: a payload off an 8-byte boundary is copied
        const char *p = PyBytes_AS_STRING(bytes);
        std::vector<uint64_t> aligned;
        if ((uintptr_t)p % 8 != 0) {
            aligned.resize(((size_t)size + 7) / 8);
            std::memcpy(aligned.data(), p, (size_t)size);
            p = reinterpret_cast<const char *>(aligned.data());
        }
        int status = 0;
        {
            const ReleasedGil released;
            status = fn(p);
        }
        return PyLong_FromLong(status);
    });
}

PyMethodDef call_entry_def = {"call", (PyCFunction)call_entry, METH_O, nullptr};

PyObject *entry(PyObject *, PyObject *args) {
    PyObject *address = nullptr, *size = nullptr;
    if (!PyArg_ParseTuple(args, "O!O!", &PyLong_Type, &address, &PyLong_Type, &size)) return nullptr;
    if (!PyLong_AsVoidPtr(address)) {
        if (!PyErr_Occurred()) PyErr_SetString(PyExc_ValueError, "no entry point");
        return nullptr;
    }
    return PyCFunction_New(&call_entry_def, args);
}

PyMethodDef methods[] = {
    {"make_layout", (PyCFunction)make_layout, METH_VARARGS, nullptr},
    {"gather", (PyCFunction)(void (*)(void))gather, METH_FASTCALL, nullptr},
    {"unit_strides", (PyCFunction)(void (*)(void))unit_strides, METH_FASTCALL, nullptr},
    {"empty", (PyCFunction)(void (*)(void))empty, METH_FASTCALL, nullptr},
    {"entry", (PyCFunction)entry, METH_VARARGS, nullptr},
    {nullptr, nullptr, 0, nullptr},
};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_sonic_host", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__sonic_host() { return PyModule_Create(&module); }
