// bind.cpp -- the call path of the Python mirror (baloon_amd/__init__.py): a CPython extension that
// turns a call's arguments into the C ABI's (include/ix_gdn.h) and calls the library.
//
// The launches here take 1.4 to 5 us on the GPU at decode sizes, and a call through ctypes cost the
// host about 7 us (a tensor's device, layout and address each through Python, the stream through
// torch.cuda, a conversion object per argument): one token through the five drop-in launchers took
// 38 us for 16 us of kernels. Here an argument is read from the tensor's C++ object.
//
// Arguments are converted by the C parameter's type: pointers from tensors (on the GPU, contiguous)
// or None, descriptions from ctypes structures, the stream from None (torch's current one), a
// torch stream or an address. Anything but a plain torch.Tensor or Parameter goes through the
// mirror's own _ptr, which refuses or reads it as before. The library's functions are found by
// the mirror (lib()), which hands their addresses over.
#include <Python.h>

#include <cstring>
#include <tuple>
#include <utility>

#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/python_variable.h>

#include "ix_gdn.h"

namespace {

PyObject* g_load = nullptr;     // lib(): loads the library and binds the addresses below
PyObject* g_ptr = nullptr;      // _ptr()
PyObject* g_cdata = nullptr;    // the base of every ctypes type

// Every converter returns with a Python error set if the argument does not fit.
void* tensor_ptr(PyObject* o) {
    if (o == Py_None) return nullptr;
    if (THPVariable_CheckExact(o)) {
        const at::Tensor& t = THPVariable_Unpack(o);
        if (t.is_cuda() && t.layout() == c10::kStrided && t.is_contiguous()) return t.data_ptr();
    }
    PyObject* r = PyObject_CallOneArg(g_ptr, o);             // other objects, and the refusals
    if (!r) return nullptr;
    void* p = r == Py_None ? nullptr : PyLong_AsVoidPtr(r);
    Py_DECREF(r);
    return p;
}

long long integer(PyObject* o) {
    PyObject* i = PyNumber_Index(o);
    if (!i) return 0;
    const unsigned long long v = PyLong_AsUnsignedLongLongMask(i);
    Py_DECREF(i);
    return (long long)v;
}

// Any ctypes instance of the C structure's size or more (a program may declare its own mirror of it).
template <class T>
const T* structure(PyObject* o) {
    const int is = PyObject_IsInstance(o, g_cdata);
    if (is < 0) return nullptr;
    Py_buffer b;
    if (!is) {
        PyErr_Format(PyExc_TypeError, "expected a ctypes instance, got %R", (PyObject*)Py_TYPE(o));
        return nullptr;
    }
    if (PyObject_GetBuffer(o, &b, PyBUF_SIMPLE) != 0) return nullptr;
    const T* p = b.len >= (Py_ssize_t)sizeof(T) ? static_cast<const T*>(b.buf) : nullptr;
    PyBuffer_Release(&b);                                    // the caller holds the structure
    if (!p) PyErr_SetString(PyExc_TypeError, "structure too small");
    return p;
}

hipStream_t stream(PyObject* o) {
    if (o == Py_None) return c10::hip::getCurrentHIPStream().stream();
    if (PyLong_Check(o)) return static_cast<hipStream_t>(PyLong_AsVoidPtr(o));
    PyObject* v = PyObject_GetAttrString(o, "cuda_stream");
    if (!v) {                                                // a ctypes.c_void_p
        PyErr_Clear();
        v = PyObject_GetAttrString(o, "value");
        if (!v) return nullptr;
        if (v == Py_None) {
            Py_DECREF(v);
            return nullptr;
        }
    }
    hipStream_t s = static_cast<hipStream_t>(PyLong_AsVoidPtr(v));
    Py_DECREF(v);
    return s;
}

template <class T>
struct Arg {                                                 // pointers to device memory
    static T of(PyObject* o) { return static_cast<T>(tensor_ptr(o)); }
};
template <>
struct Arg<const ix_gdn_cfg*> {
    static const ix_gdn_cfg* of(PyObject* o) { return structure<ix_gdn_cfg>(o); }
};
template <>
struct Arg<const ix_gdn_out_gate*> {
    static const ix_gdn_out_gate* of(PyObject* o) {
        return o == Py_None ? nullptr : structure<ix_gdn_out_gate>(o);
    }
};
template <>
struct Arg<int> {
    static int of(PyObject* o) { return (int)integer(o); }
};
template <>
struct Arg<long long> {
    static long long of(PyObject* o) { return integer(o); }
};
template <>
struct Arg<size_t> {
    static size_t of(PyObject* o) { return (size_t)integer(o); }
};
template <>
struct Arg<float> {
    static float of(PyObject* o) { return (float)PyFloat_AsDouble(o); }
};
template <>
struct Arg<hipStream_t> {
    static hipStream_t of(PyObject* o) { return stream(o); }
};

template <class... A, size_t... I>
PyObject* invoke(hipError_t (*fn)(A...), PyObject* const* args, std::index_sequence<I...>) {
    // Braces: converted from left to right, up to the first error.
    const std::tuple<A...> v{(PyErr_Occurred() ? A{} : Arg<A>::of(args[I]))...};
    if (PyErr_Occurred()) return nullptr;
    hipError_t e;
    Py_BEGIN_ALLOW_THREADS
    e = fn(std::get<I>(v)...);
    Py_END_ALLOW_THREADS
    return PyLong_FromLong((long)e);
}

template <class... A>
PyObject* call(hipError_t (*&fn)(A...), const char* name, PyObject* const* args, Py_ssize_t n) {
    if (n != (Py_ssize_t)sizeof...(A)) {
        PyErr_Format(PyExc_TypeError, "%s takes %d arguments, got %d", name, (int)sizeof...(A), (int)n);
        return nullptr;
    }
    try {
        if (!fn) {
            PyObject* r = PyObject_CallNoArgs(g_load);
            if (!r) return nullptr;
            Py_DECREF(r);
            if (!fn) {
                PyErr_Format(PyExc_RuntimeError, "%s is not bound", name);
                return nullptr;
            }
        }
        return invoke(fn, args, std::index_sequence_for<A...>{});
    } catch (const std::exception& e) {                      // from torch's accessors
        if (!PyErr_Occurred()) PyErr_SetString(PyExc_RuntimeError, e.what());
        return nullptr;
    }
}

#define IX_CALLS(X)                                                                                              \
    X(ix_gdn_step) X(ix_gdn_conv_step) X(ix_gdn_l2_norm) X(ix_gdn_beta_gate) X(ix_gdn_out_norm) X(ix_gdn_decode) \
    X(ix_gdn_decode_noalloc) X(ix_gdn_decode_gated) X(ix_gdn_prefill) X(ix_gdn_prefill_gated)                    \
    X(ix_gdn_decode_window) X(ix_gdn_decode_window_mfma) X(ix_gdn_commit_window) X(ix_bf16_gemv)                 \
    X(ix_bf16_gemv_pair) X(ix_bf16_gemv_split) X(ix_mmvq_q8_0) X(ix_q8_1_quantize) X(ix_gdn_in_proj)

#define X(name)                                                                        \
    decltype(&::name) p_##name = nullptr;                                              \
    PyObject* w_##name(PyObject*, PyObject* const* a, Py_ssize_t n) { return call(p_##name, #name, a, n); }
IX_CALLS(X)
#undef X

// bind(name, address) for one of the calls above; other names are ignored.
PyObject* bind(PyObject*, PyObject* args) {
    const char* name;
    PyObject* at;
    if (!PyArg_ParseTuple(args, "sO", &name, &at)) return nullptr;
    void* p = PyLong_AsVoidPtr(at);
    if (PyErr_Occurred()) return nullptr;
#define X(f) \
    if (!strcmp(name, #f)) p_##f = reinterpret_cast<decltype(p_##f)>(p);
    IX_CALLS(X)
#undef X
    Py_RETURN_NONE;
}

// setup(lib, _ptr, ctypes' base type)
PyObject* setup(PyObject*, PyObject* args) {
    PyObject *l, *p, *c;
    if (!PyArg_ParseTuple(args, "OOO", &l, &p, &c)) return nullptr;
    Py_INCREF(l); Py_INCREF(p); Py_INCREF(c);
    g_load = l; g_ptr = p; g_cdata = c;
    Py_RETURN_NONE;
}

PyMethodDef methods[] = {
    {"setup", setup, METH_VARARGS, nullptr},
    {"bind", bind, METH_VARARGS, nullptr},
#define X(f) {#f, (PyCFunction)(void (*)(void))w_##f, METH_FASTCALL, nullptr},
    IX_CALLS(X)
#undef X
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_bind", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__bind(void) { return PyModule_Create(&module); }
