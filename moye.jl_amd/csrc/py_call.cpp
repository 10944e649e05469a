// moye_hip._call: the entry points a program calls in a loop, for CPython.  A call through ctypes converts seven to nine arguments
// and a descriptor per array, 3.5 us of a small gemm!'s 6.0; here the descriptors are put together on the stack.
// Every function returns the moye_status, or None where it does not know an argument (the caller then goes through ctypes, whose
// errors are the package's).  The library's functions come from bind(), as addresses: this module links to nothing.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <cstring>

#include "../../include/moye_hip.h"

static PyTypeObject *g_array, *g_tensor, *g_mma, *g_copy, *g_epilogue;  // MoYeArray and the ctypes structures
static PyObject* g_layout;                                              // Layout, where MoYeArray's module has it
static PyObject *s_ptr, *s_dtype, *s_memspace, *s_layout, *s_descriptor_, *s_descriptor;
static decltype(&moye_gemm) f_gemm;
static decltype(&moye_gemm_ex) f_gemm_ex;
static decltype(&moye_copy) f_copy;
static decltype(&moye_copy_if) f_copy_if;
static decltype(&moye_axpby) f_axpby;
static decltype(&moye_map) f_map;

// the memory of a ctypes structure of `type` (the argument keeps it alive during the call)
template <typename T>
static bool structure(PyObject* o, PyTypeObject* type, const T** out) {
    *out = nullptr;
    if (o == Py_None) return true;
    if (!PyObject_TypeCheck(o, type)) return false;
    Py_buffer view;
    if (PyObject_GetBuffer(o, &view, PyBUF_SIMPLE)) return false;
    const bool fits = view.len == (Py_ssize_t)sizeof(T);
    *out = static_cast<const T*>(view.buf);
    PyBuffer_Release(&view);
    return fits;
}

static bool integer(PyObject* o, PyObject* name, unsigned long long* out) {
    PyObject* v = PyObject_GetAttr(o, name);
    if (!v) return false;
    const bool is = PyLong_Check(v);
    *out = is ? PyLong_AsUnsignedLongLongMask(v) : 0;
    Py_DECREF(v);
    return is && !PyErr_Occurred();
}

// the descriptor of an array: a moye_tensor, a MoYeArray (its layout's flattened form with the pointer, element type and memory
// space filled in, as MoYeArray.tensor() does), or None.  A subclass of either class may have methods of its own: a MoYeArray's
// goes through ctypes, which asks tensor(), a Layout's is asked for its descriptor().
static bool tensor(PyObject* o, moye_tensor* store, const moye_tensor** out) {
    if (Py_TYPE(o) != g_array) return structure(o, g_tensor, out);
    unsigned long long ptr, dtype, memspace;
    if (!integer(o, s_ptr, &ptr) || !integer(o, s_dtype, &dtype) || !integer(o, s_memspace, &memspace)) return false;
    PyObject* layout = PyObject_GetAttr(o, s_layout);
    if (!layout) return false;
    PyObject* flat = reinterpret_cast<PyObject*>(Py_TYPE(layout)) == g_layout ? PyObject_GetAttr(layout, s_descriptor_) : nullptr;
    if (!flat || !PyBytes_CheckExact(flat)) {
        PyErr_Clear();
        Py_XDECREF(flat);
        flat = PyObject_CallMethodNoArgs(layout, s_descriptor);
    }
    Py_DECREF(layout);
    if (!flat) return false;
    const bool fits = PyBytes_CheckExact(flat) && PyBytes_GET_SIZE(flat) == (Py_ssize_t)sizeof(moye_tensor);
    if (fits) {
        memcpy(store, PyBytes_AS_STRING(flat), sizeof *store);
        store->ptr = reinterpret_cast<void*>(ptr);
        store->dtype = (int32_t)dtype;
        store->memspace = (int32_t)memspace;
        *out = store;
    }
    Py_DECREF(flat);
    return fits;
}

// one that has to be there
static bool given(PyObject* o, moye_tensor* store, const moye_tensor** out) { return o != Py_None && tensor(o, store, out); }

static bool number(PyObject* o, double* out) {
    *out = PyFloat_AsDouble(o);
    return !(*out == -1.0 && PyErr_Occurred());
}
static bool address(PyObject* o, void** out) {
    *out = nullptr;
    if (o == Py_None) return true;
    if (!PyLong_Check(o)) return false;
    *out = reinterpret_cast<void*>(PyLong_AsUnsignedLongLongMask(o));
    return !PyErr_Occurred();
}

static PyObject* unknown() {
    PyErr_Clear();
    Py_RETURN_NONE;
}
#define MOYE_CALL(EXPR)                \
    int32_t status;                    \
    Py_BEGIN_ALLOW_THREADS             \
    status = (EXPR);                   \
    Py_END_ALLOW_THREADS               \
    return PyLong_FromLong(status)

static PyObject* gemm(PyObject*, PyObject* const* a, Py_ssize_t n) {  // mma, D, A, B, C, alpha, stream
    const moye_tiled_mma* mma;
    moye_tensor s[4];
    const moye_tensor* t[4];
    double alpha;
    void* stream;
    if (!f_gemm || n != 7 || a[0] == Py_None || !structure(a[0], g_mma, &mma)) return unknown();
    for (int i = 0; i < 4; ++i)
        if (!(i < 3 ? given : tensor)(a[1 + i], &s[i], &t[i])) return unknown();
    if (!number(a[5], &alpha) || !address(a[6], &stream)) return unknown();
    MOYE_CALL(f_gemm(mma, t[0], t[1], t[2], t[3], (float)alpha, stream));
}

static PyObject* gemm_ex(PyObject*, PyObject* const* a, Py_ssize_t n) {  // mma, D, A, B, C, epilogue, workspace, bytes, stream
    const moye_tiled_mma* mma;
    const moye_gemm_epilogue* ep;
    moye_tensor s[4];
    const moye_tensor* t[4];
    void *ws, *stream;
    if (!f_gemm_ex || n != 9 || a[0] == Py_None || a[5] == Py_None || !structure(a[0], g_mma, &mma) || !structure(a[5], g_epilogue, &ep)) return unknown();
    for (int i = 0; i < 4; ++i)
        if (!(i < 3 ? given : tensor)(a[1 + i], &s[i], &t[i])) return unknown();
    const size_t bytes = PyLong_Check(a[7]) ? PyLong_AsSize_t(a[7]) : (size_t)-1;
    if (!PyLong_Check(a[7]) || PyErr_Occurred() || !address(a[6], &ws) || !address(a[8], &stream)) return unknown();
    MOYE_CALL(f_gemm_ex(mma, t[0], t[1], t[2], t[3], ep, ws, bytes, stream));
}

static PyObject* copy(PyObject*, PyObject* const* a, Py_ssize_t n) {  // tiled_copy, dst, src, stream
    const moye_tiled_copy* tc;
    moye_tensor s[2];
    const moye_tensor* t[2];
    void* stream;
    if (!f_copy || n != 4 || !structure(a[0], g_copy, &tc) || !given(a[1], &s[0], &t[0]) || !given(a[2], &s[1], &t[1]) || !address(a[3], &stream)) return unknown();
    MOYE_CALL(f_copy(tc, t[0], t[1], stream));
}

static PyObject* copy_if(PyObject*, PyObject* const* a, Py_ssize_t n) {  // dst, src, mask, stream
    moye_tensor s[3];
    const moye_tensor* t[3];
    void* stream;
    if (!f_copy_if || n != 4) return unknown();
    for (int i = 0; i < 3; ++i)
        if (!given(a[i], &s[i], &t[i])) return unknown();
    if (!address(a[3], &stream)) return unknown();
    MOYE_CALL(f_copy_if(t[0], t[1], t[2], stream));
}

static PyObject* axpby(PyObject*, PyObject* const* a, Py_ssize_t n) {  // a, X, b, Y, stream
    moye_tensor s[2];
    const moye_tensor* t[2];
    double x, y;
    void* stream;
    if (!f_axpby || n != 5 || !number(a[0], &x) || !given(a[1], &s[0], &t[0]) || !number(a[2], &y) || !given(a[3], &s[1], &t[1]) || !address(a[4], &stream)) return unknown();
    MOYE_CALL(f_axpby(x, t[0], y, t[1], stream));
}

static PyObject* map(PyObject*, PyObject* const* a, Py_ssize_t n) {  // op, dst, A, B, scalar, stream
    moye_tensor s[3];
    const moye_tensor* t[3];
    double scalar;
    void* stream;
    if (!f_map || n != 6 || !PyLong_Check(a[0])) return unknown();
    const long op = PyLong_AsLong(a[0]);
    if (PyErr_Occurred() || op != (long)(int32_t)op) return unknown();
    for (int i = 0; i < 3; ++i)
        if (!(i < 2 ? given : tensor)(a[1 + i], &s[i], &t[i])) return unknown();
    if (!number(a[4], &scalar) || !address(a[5], &stream)) return unknown();
    MOYE_CALL(f_map((int32_t)op, t[0], t[1], t[2], scalar, stream));
}

// bind(MoYeArray, Tensor, TiledMMA, TiledCopy, GemmEpilogue, addresses of moye_gemm, _gemm_ex, _copy, _copy_if, _axpby, _map)
static PyObject* bind(PyObject*, PyObject* args) {
    PyObject *ty[5];
    unsigned long long f[6];
    if (!PyArg_ParseTuple(args, "O!O!O!O!O!KKKKKK", &PyType_Type, &ty[0], &PyType_Type, &ty[1], &PyType_Type, &ty[2], &PyType_Type, &ty[3], &PyType_Type,
                          &ty[4], &f[0], &f[1], &f[2], &f[3], &f[4], &f[5]))
        return nullptr;
    PyTypeObject** slots[5] = {&g_array, &g_tensor, &g_mma, &g_copy, &g_epilogue};
    for (int i = 0; i < 5; ++i) {
        Py_INCREF(ty[i]);
        *slots[i] = reinterpret_cast<PyTypeObject*>(ty[i]);
    }
    Py_CLEAR(g_layout);
    if (PyObject* name = PyObject_GetAttrString(ty[0], "__module__")) {
        if (PyObject* module = PyImport_Import(name)) {
            g_layout = PyObject_GetAttrString(module, "Layout");
            Py_DECREF(module);
        }
        Py_DECREF(name);
    }
    PyErr_Clear();
    f_gemm = reinterpret_cast<decltype(f_gemm)>(f[0]);
    f_gemm_ex = reinterpret_cast<decltype(f_gemm_ex)>(f[1]);
    f_copy = reinterpret_cast<decltype(f_copy)>(f[2]);
    f_copy_if = reinterpret_cast<decltype(f_copy_if)>(f[3]);
    f_axpby = reinterpret_cast<decltype(f_axpby)>(f[4]);
    f_map = reinterpret_cast<decltype(f_map)>(f[5]);
    Py_RETURN_NONE;
}

#define MOYE_FAST(NAME) {#NAME, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(NAME)), METH_FASTCALL, nullptr}
static PyMethodDef methods[] = {MOYE_FAST(gemm), MOYE_FAST(gemm_ex), MOYE_FAST(copy), MOYE_FAST(copy_if), MOYE_FAST(axpby), MOYE_FAST(map),
                                {"bind", bind, METH_VARARGS, nullptr}, {nullptr, nullptr, 0, nullptr}};
static PyModuleDef module = {PyModuleDef_HEAD_INIT, "_call", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

PyMODINIT_FUNC PyInit__call() {
    s_ptr = PyUnicode_InternFromString("ptr");
    s_dtype = PyUnicode_InternFromString("dtype");
    s_memspace = PyUnicode_InternFromString("memspace");
    s_layout = PyUnicode_InternFromString("layout");
    s_descriptor_ = PyUnicode_InternFromString("_descriptor");
    s_descriptor = PyUnicode_InternFromString("descriptor");
    return PyModule_Create(&module);
}
