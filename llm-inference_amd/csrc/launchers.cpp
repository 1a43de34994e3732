// The launchers of include/llm_amd/kernels.h as functions of a CPython module (_launchers), called
// with the arguments of the Python wrappers of the same names: torch tensors (or raw addresses, or
// None), numbers and a stream. A call checks and unwraps its arguments, takes the current stream,
// launches with the GIL released and raises LlmError if the library recorded an error.
//
// Most launchers run 2-10 us on the GPU, less than the Python bindings needed to prepare one call:
// several Python attribute calls per tensor, ctypes conversions, the stream object, two calls for the
// error. Host time of a call, launches included: rmsnorm_forward 9.6 -> 3.4 us; the four calls of an
// attention block (five launches) 47.0 -> 15.8 us, so that at Qwen3-0.6B's widths and 260 positions a
// block takes 16.8 us instead of 40.8 (15.3 on the GPU); a small LM head with its argmax 19.6 -> 8.8.
//
// A call takes only what it recognises: exact torch tensors (no subclass) on the GPU, contiguous, of
// a 16-bit type where bf16 is expected; exact ints and floats in range. For anything else it returns
// False without having launched, and the Python wrapper goes its general way, which converts what it
// accepts and reports what it refuses.
#include <Python.h>

#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/version.h>

#include <limits.h>
#include <stddef.h>

#include <type_traits>
#include <utility>

#include "llm_amd/kernels.h"

namespace {

PyObject *g_error = nullptr;  // LlmError, set by init

union Arg {
    void *p;
    int i;
    float f;
    size_t z;
};

// The device pointer of a tensor, a raw address or None.
bool take_pointer(PyObject *o, bool bits16, void *&out) {
    if (o == Py_None) {
        out = nullptr;
        return true;
    }
    if (PyLong_CheckExact(o)) {
        out = (void *)PyLong_AsUnsignedLongLongMask(o);
        return !PyErr_Occurred();
    }
    if (!THPVariable_CheckExact(o)) return false;
    const at::Tensor &t = THPVariable_Unpack(o);
    if (!t.defined() || !t.is_cuda() || t.layout() != at::kStrided || !t.is_contiguous()) return false;
    if (bits16 && t.scalar_type() != at::kBFloat16 && t.scalar_type() != at::kShort &&
        t.scalar_type() != at::kUInt16)
        return false;
    out = t.data_ptr();
    return true;
}

// A stream address, an object with one (torch.cuda.Stream), or None: torch's current stream.
bool take_stream(PyObject *o, void *&out) {
    if (o == Py_None) {
        out = c10::hip::getCurrentHIPStream().stream();
        return true;
    }
    if (PyLong_CheckExact(o)) {
        out = (void *)PyLong_AsUnsignedLongLongMask(o);
        return !PyErr_Occurred();
    }
    PyObject *address = PyObject_GetAttrString(o, "cuda_stream");
    if (!address) return false;
    const bool ok = PyLong_CheckExact(address);
    if (ok) out = (void *)PyLong_AsUnsignedLongLongMask(address);
    Py_DECREF(address);
    return ok && !PyErr_Occurred();
}

template <class T>
bool take(PyObject *o, Arg &a) {
    if constexpr (std::is_same_v<T, hipStream_t>) {
        return take_stream(o, a.p);
    } else if constexpr (std::is_pointer_v<T>) {
        return take_pointer(o, std::is_same_v<std::remove_cv_t<std::remove_pointer_t<T>>, bf16>, a.p);
    } else if constexpr (std::is_same_v<T, float>) {
        if (!PyFloat_CheckExact(o)) return false;
        a.f = (float)PyFloat_AS_DOUBLE(o);
        return true;
    } else {
        if (!PyLong_CheckExact(o)) return false;
        int overflow = 0;
        const long long v = PyLong_AsLongLongAndOverflow(o, &overflow);
        if (overflow) return false;
        if constexpr (std::is_same_v<T, size_t>) {
            a.z = (size_t)v;
            return v >= 0;
        } else {
            static_assert(std::is_same_v<T, int>, "argument type");
            a.i = (int)v;
            return v >= INT_MIN && v <= INT_MAX;
        }
    }
}

template <class T>
T value(const Arg &a) {
    if constexpr (std::is_pointer_v<T>)
        return (T)a.p;
    else if constexpr (std::is_same_v<T, float>)
        return a.f;
    else if constexpr (std::is_same_v<T, size_t>)
        return a.z;
    else
        return a.i;
}

// Workspace of the attention launchers: a tensor `att` holds the floats they need. (att is argument
// AT; the head count, head_dim and max_seq are arguments H, D and S.)
template <int AT, int H, int D, int S>
bool att_large_enough(PyObject *const *args, const Arg *v) {
    if (!THPVariable_CheckExact(args[AT])) return true;  // a raw address, checked by the library
    const at::Tensor &t = THPVariable_Unpack(args[AT]);
    return (size_t)t.numel() >= attention_workspace_floats(v[H].i, v[D].i, v[S].i);
}
bool no_check(PyObject *const *, const Arg *) { return true; }

template <class... T, size_t... I>
PyObject *launch(void (*fn)(T...), bool (*check)(PyObject *const *, const Arg *),
                 PyObject *const *args, Py_ssize_t n, std::index_sequence<I...>) {
    if (n != (Py_ssize_t)sizeof...(T)) Py_RETURN_FALSE;
    Arg v[sizeof...(T)];
    bool ok = false;
    try {
        ok = (take<T>(args[I], v[I]) && ...) && check(args, v);
    } catch (...) {  // the general way reports it
        ok = false;
    }
    if (!ok) {
        PyErr_Clear();
        Py_RETURN_FALSE;
    }
    Py_BEGIN_ALLOW_THREADS
    fn(value<T>(v[I])...);
    Py_END_ALLOW_THREADS
    if (const char *message = llm_last_error()) {
        PyErr_SetString(g_error, message);
        llm_clear_error();
        return nullptr;
    }
    Py_RETURN_TRUE;
}

template <auto FN, auto CHECK, class... T>
PyObject *call(void (*)(T...), PyObject *const *args, Py_ssize_t n) {
    return launch<T...>(FN, CHECK, args, n, std::index_sequence_for<T...>{});
}

template <auto FN, auto CHECK = no_check>
PyObject *entry(PyObject *, PyObject *const *args, Py_ssize_t n) {
    return call<FN, CHECK>(FN, args, n);
}

PyObject *init(PyObject *, PyObject *error) {
    Py_INCREF(error);
    Py_XSETREF(g_error, error);
    Py_RETURN_NONE;
}

#define LAUNCHER(NAME, ...) \
    {#NAME, (PyCFunction)(void *)entry<NAME, ##__VA_ARGS__>, METH_FASTCALL, nullptr}

PyMethodDef methods[] = {
    LAUNCHER(embedding_forward),
    LAUNCHER(rmsnorm_forward),
    LAUNCHER(gemv_forward),
    LAUNCHER(gemv_residual_forward),
    LAUNCHER(qkv_forward),
    LAUNCHER(gate_up_forward),
    LAUNCHER(rmsnorm_qkv_forward),
    LAUNCHER(rmsnorm_gemv_forward),
    LAUNCHER(rmsnorm_gate_up_forward),
    LAUNCHER(qk_norm_rope_forward),
    LAUNCHER(qk_norm_rope_rows),
    LAUNCHER(attention_forward, att_large_enough<4, 5, 7, 9>),
    LAUNCHER(attention_forward_noalloc),
    LAUNCHER(qk_norm_rope_attention_forward, att_large_enough<8, 10, 12, 15>),
    LAUNCHER(argmax_forward),
    LAUNCHER(sample_forward),
    LAUNCHER(swiglu_forward),
    {"init", init, METH_O, "The exception class of library errors."},
    {nullptr, nullptr, 0, nullptr},
};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_launchers", nullptr, -1, methods};

}  // namespace

PyMODINIT_FUNC PyInit__launchers(void) {
    PyObject *m = PyModule_Create(&module);
    // the torch whose tensors this reads: the package leaves the module alone under another
    if (m && PyModule_AddStringConstant(m, "TORCH_VERSION", TORCH_VERSION) < 0) Py_CLEAR(m);
    return m;
}
