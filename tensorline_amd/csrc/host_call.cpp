// Python's way into the kernel library's C entry points: `enter(address, *arguments)`, a Python module of its own, so that the library neither
// needs Python's headers to be built nor its symbols to be loaded.  Without this module ctypes does the same (kernels.py).
//
// What bounds a small eager step is the host: 11 to 18 us a launch, of which ctypes' conversions, with an object made around every pointer,
// stream, float and 64-bit number, took some 3.  Here an argument is converted where it stands: a tensor is its address, None
// a null pointer, an integer 64 bits of which a 32-bit parameter takes the low ones, a Python float a float, and a ctypes object its
// value, or its address where it is a structure.
//
// The call itself: under the System V calling convention of x86-64 integers and pointers fill the integer registers and then the stack in
// their own order, floats the vector registers in theirs, whatever the order between the two; and the caller clears the stack, so that
// what a callee does not have is not looked at.  So one type of function serves every entry point of up to HC_WORDS integers and
// HC_FLOATS floats that returns an int.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <stdint.h>

#if !defined(__x86_64__) || defined(_WIN32)
#error "the calls are made for the System V convention of x86-64"
#endif

#define HC_WORDS 56
#define HC_FLOATS 8

#define HC_8(X) X, X, X, X, X, X, X, X
typedef int (*HcEntry)(HC_8(long), HC_8(long), HC_8(long), HC_8(long), HC_8(long), HC_8(long), HC_8(long), HC_8(float));
#undef HC_8

static PyObject* hc_data_ptr;      // "data_ptr"

// One argument as a word or a float; false with an exception set.
static bool hc_take(PyObject* o, long* words, int* nwords, float* floats, int* nfloats) {
    long word = 0;
    float number = 0.f;
    bool is_float = false;
    if (o == Py_None) {
    } else if (PyLong_Check(o)) {
        word = (long)PyLong_AsUnsignedLongLongMask(o);
        if (word == -1 && PyErr_Occurred()) return false;
    } else if (PyFloat_Check(o)) {
        number = (float)PyFloat_AS_DOUBLE(o), is_float = true;
    } else if (PyObject_CheckBuffer(o)) {              // a ctypes object
        Py_buffer b;
        if (PyObject_GetBuffer(o, &b, PyBUF_FORMAT | PyBUF_SIMPLE) != 0) return false;
        const char kind = b.format && b.format[0] ? b.format[b.format[0] == '<' ? 1 : 0] : 0;
        bool known = b.ndim == 0;
        if (!known) {
        } else if (kind == 'T') {
            word = (long)(intptr_t)b.buf;              // (the caller holds the structure through the call)
        } else if (kind == 'f' && b.itemsize == 4) {
            number = *(const float*)b.buf, is_float = true;
        } else if (kind == 'd' || kind == 'f') {
            known = false;
        } else if (b.itemsize == 8) {
            word = *(const long*)b.buf;
        } else if (b.itemsize == 4) {
            word = kind == 'I' || kind == 'L' ? (long)*(const uint32_t*)b.buf : (long)*(const int32_t*)b.buf;
        } else {
            known = false;
        }
        PyBuffer_Release(&b);
        if (!known) {
            PyErr_Format(PyExc_TypeError, "a kernel takes no argument of type %s", Py_TYPE(o)->tp_name);
            return false;
        }
    } else {                                           // a tensor
        PyObject* at = PyObject_CallMethodNoArgs(o, hc_data_ptr);
        if (!at) return false;
        word = (long)PyLong_AsUnsignedLongLongMask(at);
        Py_DECREF(at);
        if (word == -1 && PyErr_Occurred()) return false;
    }
    if (is_float ? *nfloats >= HC_FLOATS : *nwords >= HC_WORDS) {
        PyErr_SetString(PyExc_TypeError, "more arguments than a call has room for");
        return false;
    }
    if (is_float) floats[(*nfloats)++] = number;
    else words[(*nwords)++] = word;
    return true;
}

static PyObject* hc_enter(PyObject*, PyObject* const* args, Py_ssize_t n) {
    if (n < 1 || !PyLong_Check(args[0])) {
        PyErr_SetString(PyExc_TypeError, "enter(address, *arguments)");
        return nullptr;
    }
    const HcEntry entry = (HcEntry)(uintptr_t)PyLong_AsUnsignedLongLongMask(args[0]);
    long w[HC_WORDS] = {};
    float f[HC_FLOATS] = {};
    int nw = 0, nf = 0;
    for (Py_ssize_t i = 1; i < n; ++i)
        if (!hc_take(args[i], w, &nw, f, &nf)) return nullptr;
    int status;
    Py_BEGIN_ALLOW_THREADS
#define HC_8(A, I) A[I], A[I + 1], A[I + 2], A[I + 3], A[I + 4], A[I + 5], A[I + 6], A[I + 7]
    status = entry(HC_8(w, 0), HC_8(w, 8), HC_8(w, 16), HC_8(w, 24), HC_8(w, 32), HC_8(w, 40), HC_8(w, 48), HC_8(f, 0));
#undef HC_8
    Py_END_ALLOW_THREADS
    return PyLong_FromLong(status);
}

static PyMethodDef hc_methods[] = {
    {"enter", (PyCFunction)(void (*)(void))hc_enter, METH_FASTCALL, "enter(address, *arguments): the status that a C entry point returns"},
    {nullptr, nullptr, 0, nullptr},
};
static PyModuleDef hc_module = {PyModuleDef_HEAD_INIT, "tensorline_call", nullptr, -1, hc_methods, nullptr, nullptr, nullptr, nullptr};

PyMODINIT_FUNC PyInit_tensorline_call(void) {
    hc_data_ptr = PyUnicode_InternFromString("data_ptr");
    return hc_data_ptr ? PyModule_Create(&hc_module) : nullptr;
}
