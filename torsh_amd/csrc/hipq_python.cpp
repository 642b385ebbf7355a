// The calls of torsh_amd/hipq.py into the C entry points, and its output tensors, without ctypes: a small call is its launches and
// what the host does around them.  One function per entry point, of the same name, its arguments converted by the entry point's
// own parameter types:
//   pointers  None, a dense torch tensor (its data), or an address as an int
//   numbers   int or float
// The first argument is the context's handle as an int.  A status other than 0 goes to the callable that set_error_handler was
// given.  As with ctypes, the interpreter lock is not held during the call.
//
// us a pass of small calls, which the host bounds or nearly does, ctypes / this: a quantize and a dequantize per channel with five
// outputs 21.0 / 17.5, per tensor with three 13.9 / 11.5, a convolution 11.75 / 9.9, a Linear of two launches into a given output 9.1 / 8.4
// (the two follow one another in 8).
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/ops/empty.h>
#include <torch/csrc/autograd/python_variable.h>

#include <exception>
#include <tuple>
#include <type_traits>
#include <utility>

#include "torsh_hipq.h"

namespace {

PyObject *g_error_handler = nullptr;

// Leaves the address of a tensor's data in `out`; false with an exception set.  Subclasses other than Parameter answer for themselves.
bool tensor_address(PyObject *o, bool dense, void **out) {
    if (THPVariable_CheckExact(o)) {
        const at::Tensor &t = THPVariable_Unpack(o);
        if (dense && !t.is_contiguous()) {
            PyErr_SetString(PyExc_ValueError, "hipq entry points take dense row-major tensors");
            return false;
        }
        *out = t.data_ptr();
        return true;
    }
    if (dense) {
        PyObject *c = PyObject_CallMethod(o, "is_contiguous", nullptr);
        if (!c) return false;
        const int yes = PyObject_IsTrue(c);
        Py_DECREF(c);
        if (yes < 0) return false;
        if (!yes) {
            PyErr_SetString(PyExc_ValueError, "hipq entry points take dense row-major tensors");
            return false;
        }
    }
    PyObject *a = PyObject_CallMethod(o, "data_ptr", nullptr);
    if (!a) return false;
    *out = PyLong_AsVoidPtr(a);
    Py_DECREF(a);
    return !PyErr_Occurred();
}

template <typename T>
bool convert(PyObject *o, T *out) {
    if constexpr (std::is_pointer_v<T>) {
        void *p = nullptr;
        if (o == Py_None) {
        } else if (PyLong_Check(o)) {
            p = PyLong_AsVoidPtr(o);
            if (PyErr_Occurred()) return false;
        } else if (!tensor_address(o, /*dense=*/true, &p)) {
            return false;
        }
        *out = static_cast<T>(p);
    } else if constexpr (std::is_floating_point_v<T>) {
        const double v = PyFloat_AsDouble(o);
        if (v == -1.0 && PyErr_Occurred()) return false;
        *out = static_cast<T>(v);
    } else {
        if (PyFloat_Check(o)) {
            PyErr_SetString(PyExc_TypeError, "an int is required, not float");
            return false;
        }
        const unsigned long long v = PyLong_AsUnsignedLongLongMask(o);  // (whatever has an __index__; two's complement, as ctypes)
        if (v == static_cast<unsigned long long>(-1) && PyErr_Occurred()) return false;
        *out = static_cast<T>(v);
    }
    return true;
}

PyObject *finish(int32_t status) {
    if (status != HIPQ_SUCCESS && g_error_handler) {
        PyObject *r = PyObject_CallFunction(g_error_handler, "i", static_cast<int>(status));
        if (!r) return nullptr;
        Py_DECREF(r);
    }
    Py_RETURN_NONE;
}

// A C++ exception (torch's, of a tensor without data) becomes a RuntimeError.
template <typename F>
PyObject *guarded(F f) {
    try {
        return f();
    } catch (const std::exception &e) {
        PyErr_SetString(PyExc_RuntimeError, e.what());
    } catch (...) {
        PyErr_SetString(PyExc_RuntimeError, "unknown C++ exception");
    }
    return nullptr;
}

template <auto F>
struct Entry;
template <typename... A, int32_t (*F)(A...)>
struct Entry<F> {
    static PyObject *call(PyObject *, PyObject *const *args, Py_ssize_t n) {
        return guarded([&]() -> PyObject * {
            if (n != static_cast<Py_ssize_t>(sizeof...(A))) {
                PyErr_Format(PyExc_TypeError, "%zd arguments are required, not %zd", static_cast<Py_ssize_t>(sizeof...(A)), n);
                return nullptr;
            }
            return with(args, std::index_sequence_for<A...>{});
        });
    }
    template <size_t... I>
    static PyObject *with(PyObject *const *args, std::index_sequence<I...>) {
        std::tuple<A...> values;
        if (!(convert(args[I], &std::get<I>(values)) && ...)) return nullptr;
        int32_t status;
        Py_BEGIN_ALLOW_THREADS;
        status = F(std::get<I>(values)...);
        Py_END_ALLOW_THREADS;
        return finish(status);
    }
};

// empty(sizes, dtype, device index): an uninitialized tensor on the GPU.  sizes: a tuple of ints (a torch.Size is one).
PyObject *empty(PyObject *, PyObject *const *args, Py_ssize_t n) {
    return guarded([&]() -> PyObject * {
        if (n != 3 || !PyTuple_Check(args[0]) || !THPDtype_Check(args[1]) || !PyLong_Check(args[2])) {
            PyErr_SetString(PyExc_TypeError, "empty(sizes as a tuple, dtype, device index)");
            return nullptr;
        }
        const Py_ssize_t rank = PyTuple_GET_SIZE(args[0]);
        c10::SmallVector<int64_t, 8> sizes;
        for (Py_ssize_t i = 0; i < rank; ++i) {
            const long long v = PyLong_AsLongLong(PyTuple_GET_ITEM(args[0], i));
            if (v == -1 && PyErr_Occurred()) return nullptr;
            sizes.push_back(v);
        }
        const long device = PyLong_AsLong(args[2]);
        if (device == -1 && PyErr_Occurred()) return nullptr;
        at::Tensor t;
        Py_BEGIN_ALLOW_THREADS;  // (an allocation may have to wait for the device)
        try {
            t = at::empty(sizes, at::TensorOptions()
                                     .dtype(reinterpret_cast<THPDtype *>(args[1])->scalar_type)
                                     .device(c10::Device(c10::kCUDA, static_cast<c10::DeviceIndex>(device))));
        } catch (...) {
            Py_BLOCK_THREADS;
            throw;
        }
        Py_END_ALLOW_THREADS;
        return THPVariable_Wrap(std::move(t));
    });
}

// pointers(blocks, names): the addresses of the named tensors of every dict, None and missing ones as 0, as one bytes object.
PyObject *pointers(PyObject *, PyObject *const *args, Py_ssize_t n) {
    return guarded([&]() -> PyObject * {
        if (n != 2 || !PyTuple_Check(args[1])) {
            PyErr_SetString(PyExc_TypeError, "pointers(sequence of dicts, tuple of names)");
            return nullptr;
        }
        PyObject *blocks = PySequence_Fast(args[0], "a sequence of blocks is required");
        if (!blocks) return nullptr;
        const Py_ssize_t count = PySequence_Fast_GET_SIZE(blocks), each = PyTuple_GET_SIZE(args[1]);
        PyObject *bytes = PyBytes_FromStringAndSize(nullptr, count * each * static_cast<Py_ssize_t>(sizeof(void *)));
        bool good = bytes != nullptr;
        try {
            void **to = good ? reinterpret_cast<void **>(PyBytes_AS_STRING(bytes)) : nullptr;
            for (Py_ssize_t b = 0; good && b < count; ++b)
                for (Py_ssize_t i = 0; good && i < each; ++i) {
                    PyObject *block = PySequence_Fast_GET_ITEM(blocks, b), *name = PyTuple_GET_ITEM(args[1], i), *t;
                    if (PyDict_CheckExact(block)) {
                        t = PyDict_GetItemWithError(block, name);
                        if (!t && PyErr_Occurred()) good = false;
                        Py_XINCREF(t);
                    } else {
                        t = PyObject_CallMethod(block, "get", "O", name);
                        if (!t) good = false;
                    }
                    *to = nullptr;
                    if (good && t && t != Py_None) good = tensor_address(t, /*dense=*/false, to);
                    ++to;
                    Py_XDECREF(t);
                }
        } catch (...) {
            Py_DECREF(blocks);
            Py_XDECREF(bytes);
            throw;
        }
        Py_DECREF(blocks);
        if (!good) {
            Py_XDECREF(bytes);
            return nullptr;
        }
        return bytes;
    });
}

PyObject *set_error_handler(PyObject *, PyObject *handler) {
    Py_XINCREF(handler);
    Py_XSETREF(g_error_handler, handler);
    Py_RETURN_NONE;
}

#define FAST(f) reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)(void)>(f))
#define ENTRY(name) {#name, FAST(&Entry<&name>::call), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {
    ENTRY(hipq_linear_dynamic_f32),
    ENTRY(hipq_linear_static_f32),
    ENTRY(hipq_linear_dynamic_packed_f32),
    ENTRY(hipq_linear_static_packed_f32),
    ENTRY(hipq_linear_dynamic_f32_noalloc),
    ENTRY(hipq_linear_i8_f32),
    ENTRY(hipq_linear_packed_i8_f32),
    ENTRY(hipq_quantize_dynamic_per_tensor_f32),
    ENTRY(hipq_quantize_per_tensor_f32_i8),
    ENTRY(hipq_quantize_per_tensor_f32_u8),
    ENTRY(hipq_quantize_per_row_f32_i8),
    ENTRY(hipq_quantize_per_channel_auto_f32_i8),
    ENTRY(hipq_quantize_per_channel_f32_i8),
    ENTRY(hipq_dequantize_with_params_i8_f32),
    ENTRY(hipq_dequantize_i8_f32),
    ENTRY(hipq_dequantize_per_channel_i8_f32),
    ENTRY(hipq_conv2d_u8i8_i8),
    ENTRY(hipq_conv2d_u8i8_i8_packed),
    ENTRY(hipq_conv2d_dynamic_f32_i8_packed),
    ENTRY(hipq_pack_rows_i8),
    {"empty", FAST(&empty), METH_FASTCALL, nullptr},
    {"pointers", FAST(&pointers), METH_FASTCALL, nullptr},
    {"set_error_handler", set_error_handler, METH_O, nullptr},
    {nullptr, nullptr, 0, nullptr},
};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_hipq_python", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__hipq_python(void) { return PyModule_Create(&module); }
