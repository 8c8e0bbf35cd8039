// warpdecode_amd._fast: capi.call for the stand-alone operators without ctypes' argument conversion.
//
// A dense block is nine calls of a few microseconds each, and the host is what they wait for: the operators' launches
// take 2.4 us of it each, ctypes' conversion of nine arguments another 0.7.  Through here a call costs 0.4 us less: the
// 216 calls of twenty-four Q8_0 blocks of hidden 2560 take 973 us instead of 1060, the 146 of the Q4_0 ones of hidden
// 1536 661 instead of 717, a 2048-row product with its quantisation 11.8 instead of 12.7 (in turn, in one process).
//
// Taken are calls whose arguments have the forms that programs use: None, int, float, ctypes.c_void_p or a ctypes array,
// each where ctypes takes it too.  Any other call goes to the ctypes path, so what is accepted and what is refused, and
// how, stay the same.  The interpreter's lock is released during a call, as ctypes does.  The library is not linked: its
// addresses come from ctypes once that has loaded it.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <cstring>
#include <tuple>
#include <type_traits>
#include <utility>

#include "../../include/warpdecode_amd.h"

namespace {

PyObject *g_slow = nullptr;   // call(name, *args) through ctypes
PyObject *g_check = nullptr;  // check(rc): raises for an error
PyTypeObject *g_void_p = nullptr, *g_array = nullptr;
PyObject *g_table = nullptr;  // name -> capsule of its Entry, of the loaded library

bool whole_number(PyObject *o, unsigned long long &v) {
    if (!PyLong_Check(o)) return false;
    v = PyLong_AsUnsignedLongLongMask(o);  // (as ctypes: the low bits, whatever the sign and size)
    return !PyErr_Occurred();
}
template <typename T>
bool from_python(PyObject *o, T *&p) {
    if (o == Py_None) {
        p = nullptr;
        return true;
    }
    if (PyLong_Check(o)) {
        unsigned long long v;
        if (!whole_number(o, v)) return false;
        p = reinterpret_cast<T *>(static_cast<uintptr_t>(v));
        return true;
    }
    const bool value = Py_TYPE(o) == g_void_p;
    if (!value && !PyObject_TypeCheck(o, g_array)) return false;
    Py_buffer view;  // (a c_void_p's memory is the pointer, an array's is what the pointer points at)
    if (PyObject_GetBuffer(o, &view, PyBUF_SIMPLE) != 0) return false;
    p = value ? *static_cast<T **>(view.buf) : static_cast<T *>(view.buf);
    PyBuffer_Release(&view);
    return true;
}
template <typename T>
bool whole(PyObject *o, T &v) {
    unsigned long long w;
    if (!whole_number(o, w)) return false;
    v = static_cast<T>(w);
    return true;
}
bool from_python(PyObject *o, int &v) { return whole(o, v); }
bool from_python(PyObject *o, size_t &v) { return whole(o, v); }
bool from_python(PyObject *o, float &v) {
    if (!PyFloat_Check(o)) return false;
    v = static_cast<float>(PyFloat_AS_DOUBLE(o));
    return true;
}

// Runs the call if its arguments are of the forms above; false: not run.
using Thunk = bool (*)(void *fn, PyObject *const *args, Py_ssize_t n, int &rc);

template <typename F>
struct Bound;
template <typename... P>
struct Bound<int(P...)> {
    template <size_t... I>
    static bool run_with(void *fn, PyObject *const *args, int &rc, std::index_sequence<I...>) {
        std::tuple<P...> v;
        if (!(from_python(args[I], std::get<I>(v)) && ...)) {
            PyErr_Clear();
            return false;
        }
        PyThreadState *const state = PyEval_SaveThread();
        rc = reinterpret_cast<int (*)(P...)>(fn)(std::get<I>(v)...);
        PyEval_RestoreThread(state);
        return true;
    }
    static bool run(void *fn, PyObject *const *args, Py_ssize_t n, int &rc) {
        return n == static_cast<Py_ssize_t>(sizeof...(P)) && run_with(fn, args, rc, std::index_sequence_for<P...>{});
    }
};

// A letter per argument, from which the caller tells whether the prototype is the one it would use.
template <typename T>
constexpr char code_of = std::is_pointer_v<T> ? 'p' : std::is_same_v<T, int> ? 'i' : std::is_same_v<T, float> ? 'f' : std::is_same_v<T, size_t> ? 'z' : '?';
template <typename F>
struct Codes;
template <typename... P>
struct Codes<int(P...)> {
    static constexpr char text[] = {code_of<P>..., 0};
};

struct Entry {
    const char *name;
    const char *codes;
    Thunk thunk;
    void *fn;
};
#define WD_BIND(f) {#f, Codes<decltype(f)>::text, Bound<decltype(f)>::run, nullptr}
Entry g_entries[] = {
    WD_BIND(wd_q8_k_quantize_f32),    WD_BIND(wd_q8_0_quantize_f32),   WD_BIND(wd_q8_0_quantize_f16),
    WD_BIND(wd_q8_1_quantize_f32),    WD_BIND(wd_gemv_q8_0_q8_1_f32),  WD_BIND(wd_gemv_q8_k_f32),
    WD_BIND(wd_gemv_q8_0_f32),        WD_BIND(wd_gemv_q6_k_q8_k_f32),  WD_BIND(wd_gemv_q8_0_batch_f32),
    WD_BIND(wd_silu_mul_experts_f32), WD_BIND(wd_add_shared_f32),      WD_BIND(wd_weighted_accum_experts_f32),
    WD_BIND(wd_router_gemv_f32),      WD_BIND(wd_topk_softmax),        WD_BIND(wd_convert_f16_to_f32),
    WD_BIND(wd_convert_f32_to_f16),   WD_BIND(wd_hc_combine_f32),
};
#undef WD_BIND

PyObject *call(PyObject *, PyObject *const *args, Py_ssize_t n, PyObject *keywords) {
    if (!g_slow) {
        PyErr_SetString(PyExc_RuntimeError, "warpdecode_amd._fast: prepare() comes first");
        return nullptr;
    }
    PyObject *const found = !keywords && n > 0 && PyUnicode_CheckExact(args[0]) ? PyDict_GetItemWithError(g_table, args[0]) : nullptr;
    if (found) {
        const Entry *const e = static_cast<const Entry *>(PyCapsule_GetPointer(found, nullptr));
        int rc = 0;
        if (e->thunk(e->fn, args + 1, n - 1, rc)) {
            if (rc != 0) return PyObject_CallFunction(g_check, "i", rc);
            Py_RETURN_NONE;
        }
    }
    if (PyErr_Occurred()) return nullptr;
    return PyObject_Vectorcall(g_slow, args, static_cast<size_t>(n), keywords);
}

// prepare(slow, check, c_void_p, Array): what call() needs; until bind() every call takes the slow path
PyObject *prepare(PyObject *, PyObject *args) {
    PyObject *slow, *check, *void_p, *array;
    if (!PyArg_ParseTuple(args, "OOO!O!", &slow, &check, &PyType_Type, &void_p, &PyType_Type, &array)) return nullptr;
    PyObject *const table = PyDict_New();
    if (!table) return nullptr;
    for (Entry &e : g_entries) e.fn = nullptr;
    Py_INCREF(slow);
    Py_INCREF(check);
    Py_INCREF(void_p);
    Py_INCREF(array);
    Py_XSETREF(g_table, table);
    Py_XSETREF(g_slow, slow);
    Py_XSETREF(g_check, check);
    Py_XSETREF(g_void_p, reinterpret_cast<PyTypeObject *>(void_p));
    Py_XSETREF(g_array, reinterpret_cast<PyTypeObject *>(array));
    Py_RETURN_NONE;
}
// names() -> the entry points that bind() takes
PyObject *names(PyObject *, PyObject *) {
    PyObject *const list = PyList_New(0);
    for (const Entry &e : g_entries) {
        PyObject *const name = list ? PyUnicode_FromString(e.name) : nullptr;
        if (!name || PyList_Append(list, name) != 0) {
            Py_XDECREF(name);
            Py_XDECREF(list);
            return nullptr;
        }
        Py_DECREF(name);
    }
    return list;
}
// signature(name) -> the arguments that bind() takes an entry point to have: p(ointer), i(nt), f(loat), z (size_t)
PyObject *signature(PyObject *, PyObject *args) {
    const char *name;
    if (!PyArg_ParseTuple(args, "s", &name)) return nullptr;
    for (const Entry &e : g_entries)
        if (std::strcmp(e.name, name) == 0) return PyUnicode_FromString(e.codes);
    PyErr_Format(PyExc_ValueError, "warpdecode_amd._fast: no %s here", name);
    return nullptr;
}
// bind(name, address): calls of this entry point go to the address from now on.  The same address may be bound again (a load that failed
// on the way is tried once more), another one may not.
PyObject *bind(PyObject *, PyObject *args) {
    const char *name;
    PyObject *address;
    if (!PyArg_ParseTuple(args, "sO!", &name, &PyLong_Type, &address)) return nullptr;
    void *const fn = PyLong_AsVoidPtr(address);
    if (PyErr_Occurred()) return nullptr;
    for (Entry &e : g_entries)
        if (g_table && fn && (!e.fn || e.fn == fn) && std::strcmp(e.name, name) == 0) {
            PyObject *const capsule = PyCapsule_New(&e, nullptr, nullptr);
            if (!capsule) return nullptr;
            e.fn = fn;
            const int rc = PyDict_SetItemString(g_table, name, capsule);
            Py_DECREF(capsule);
            if (rc != 0) return nullptr;
            Py_RETURN_NONE;
        }
    PyErr_Format(PyExc_ValueError, "warpdecode_amd._fast: %s cannot be bound", name);
    return nullptr;
}

PyMethodDef g_methods[] = {
    {"call", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(call)), METH_FASTCALL | METH_KEYWORDS,
     "call(name, *args): the entry point of that name; capi.check's error where it reports one"},
    {"prepare", prepare, METH_VARARGS, "prepare(slow, check, c_void_p, Array)"},
    {"names", names, METH_NOARGS, "the entry points that bind takes"},
    {"signature", signature, METH_VARARGS, "signature(name): a letter per argument, p, i, f or z"},
    {"bind", bind, METH_VARARGS, "bind(name, address)"},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef g_module = {PyModuleDef_HEAD_INIT, "_fast", "capi.call without ctypes' argument conversion", -1, g_methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__fast() { return PyModule_Create(&g_module); }
