// bind.cpp -- the call path of the Python mirror (baloon_amd/__init__.py): a CPython extension that
// turns a call's arguments into the C ABI's (include/ix_gdn.h) and calls the library.
//
// The launches here take 1.4 to 5 us on the GPU at decode sizes, and a call through ctypes cost the
// host about 7 us (a tensor's device, layout and address each through Python, the stream through
// torch.cuda, a conversion object per argument): one token through the five drop-in launchers took
// 38 us for 16 us of kernels. Here an argument is read from the tensor's C++ object.
//
// Arguments are converted by the C parameter's type: pointers from tensors (plain torch.Tensor or
// Parameter, on the GPU, contiguous) or None, descriptions from ctypes structures, numbers from ints and
// floats, the stream from None (torch's current one), a torch stream or an address. A call with any other argument
// goes as a whole to the mirror's ctypes path, which reads or refuses it. The mirror hands over the addresses
// of the library's functions.
#include <Python.h>

#include <cstring>
#include <tuple>
#include <utility>

#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/utils/device_lazy_init.h>

#include "ix_gdn.h"

namespace {

PyObject* g_other = nullptr;    // the mirror's ctypes path: (name, arguments) -> code
PyObject* g_cdata = nullptr;    // the base of every ctypes type

// The converters set `other` for an argument that they leave to ctypes.
void* tensor_ptr(PyObject* o, bool& other) {
    if (o == Py_None) return nullptr;
    if (THPVariable_CheckExact(o)) {
        const at::Tensor& t = THPVariable_Unpack(o);
        if (t.is_cuda() && t.layout() == c10::kStrided && t.is_contiguous()) return t.data_ptr();
    }
    other = true;
    return nullptr;
}

long long integer(PyObject* o, bool& other) {
    if (PyLong_Check(o)) return (long long)PyLong_AsUnsignedLongLongMask(o);
    other = true;
    return 0;
}

float real(PyObject* o, bool& other) {
    if (PyFloat_Check(o)) return (float)PyFloat_AS_DOUBLE(o);
    other = true;
    return 0.0f;
}

// Any ctypes instance of the C structure's size or more (a program may declare its own mirror of it). The
// caller holds it.
template <class T>
const T* structure(PyObject* o, bool& other) {
    Py_buffer b;
    if (PyObject_IsInstance(o, g_cdata) == 1 && PyObject_GetBuffer(o, &b, PyBUF_SIMPLE) == 0) {
        const T* p = b.len >= (Py_ssize_t)sizeof(T) ? static_cast<const T*>(b.buf) : nullptr;
        PyBuffer_Release(&b);
        if (p) return p;
    }
    PyErr_Clear();
    other = true;
    return nullptr;
}

hipStream_t stream(PyObject* o, bool& other) {
    if (o == Py_None) {
        other = torch::utils::is_device_in_bad_fork(at::kCUDA);   // torch.cuda refuses such a process
        return other ? nullptr : c10::hip::getCurrentHIPStream().stream();
    }
    PyObject* v = PyLong_Check(o) ? Py_NewRef(o) : PyObject_GetAttrString(o, "cuda_stream");
    if (v && PyLong_Check(v)) {
        void* p = PyLong_AsVoidPtr(v);
        if (!PyErr_Occurred()) {
            Py_DECREF(v);
            return static_cast<hipStream_t>(p);
        }
    }
    Py_XDECREF(v);
    PyErr_Clear();
    other = true;
    return nullptr;
}

template <class T>
struct Arg {                                                 // pointers to device memory
    static T of(PyObject* o, bool& other) { return static_cast<T>(tensor_ptr(o, other)); }
};
template <>
struct Arg<const ix_gdn_cfg*> {
    static const ix_gdn_cfg* of(PyObject* o, bool& other) { return structure<ix_gdn_cfg>(o, other); }
};
template <>
struct Arg<const ix_gdn_out_gate*> {
    static const ix_gdn_out_gate* of(PyObject* o, bool& other) {
        return o == Py_None ? nullptr : structure<ix_gdn_out_gate>(o, other);
    }
};
template <>
struct Arg<int> {
    static int of(PyObject* o, bool& other) { return (int)integer(o, other); }
};
template <>
struct Arg<long long> {
    static long long of(PyObject* o, bool& other) { return integer(o, other); }
};
template <>
struct Arg<size_t> {
    static size_t of(PyObject* o, bool& other) { return (size_t)integer(o, other); }
};
template <>
struct Arg<float> {
    static float of(PyObject* o, bool& other) { return real(o, other); }
};
template <>
struct Arg<hipStream_t> {
    static hipStream_t of(PyObject* o, bool& other) { return stream(o, other); }
};

PyObject* through_ctypes(const char* name, PyObject* const* args, Py_ssize_t n) {
    PyObject* t = PyTuple_New(n);
    if (!t) return nullptr;
    for (Py_ssize_t i = 0; i < n; ++i) {
        Py_INCREF(args[i]);
        PyTuple_SET_ITEM(t, i, args[i]);
    }
    PyObject* r = PyObject_CallFunction(g_other, "sO", name, t);
    Py_DECREF(t);
    return r;
}

template <class... A, size_t... I>
PyObject* invoke(hipError_t (*fn)(A...), const char* name, PyObject* const* args, std::index_sequence<I...>) {
    bool other = false;
    // Braces: converted from left to right, up to the first that is left to ctypes.
    const std::tuple<A...> v{(other ? A{} : Arg<A>::of(args[I], other))...};
    if (other) return through_ctypes(name, args, (Py_ssize_t)sizeof...(A));
    hipError_t e;
    Py_BEGIN_ALLOW_THREADS
    e = fn(std::get<I>(v)...);
    Py_END_ALLOW_THREADS
    return PyLong_FromLong((long)e);
}

template <class... A>
PyObject* call(hipError_t (*fn)(A...), const char* name, PyObject* const* args, Py_ssize_t n) {
    if (n != (Py_ssize_t)sizeof...(A)) {
        PyErr_Format(PyExc_TypeError, "%s takes %d arguments, got %d", name, (int)sizeof...(A), (int)n);
        return nullptr;
    }
    if (!fn) {
        PyErr_Format(PyExc_RuntimeError, "%s is not bound", name);
        return nullptr;
    }
    try {
        return invoke(fn, name, args, std::index_sequence_for<A...>{});
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

// setup(the ctypes path, ctypes' base type)
PyObject* setup(PyObject*, PyObject* args) {
    PyObject *o, *c;
    if (!PyArg_ParseTuple(args, "OO", &o, &c)) return nullptr;
    Py_INCREF(o); Py_INCREF(c);
    g_other = o; g_cdata = c;
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
