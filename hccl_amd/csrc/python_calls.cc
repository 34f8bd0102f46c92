// CPython module _hccl_calls: calls of the C entry points without ctypes' conversions.
//
// A collective among n virtual ranks is n calls, and a small one is over before Python has made them.  8 ranks x 1001 fp32
// take 10.4 us through ctypes (a foreign-function call of seven converted arguments each time) and 6.3 through this, an
// AlltoAll among 32 ranks 40.9 and 22.2.
//
// Call(address, kinds, Array): one character of kinds per argument.  "i": an int (wraps like ctypes' integers); "p": an
// address, an int, None or a ctypes array; "l": a list or tuple of up to 64 ints or Nones (an array of addresses).  Given
// anything else it returns NotImplemented and the caller goes through ctypes, which converts or refuses it.  The GIL is
// released during the call, as ctypes does.  Every argument of the entry points is of INTEGER class (pointers, 32- and
// 64-bit integers), which the x86-64 System V calling convention passes in one 8-byte register or stack slot each whatever
// its width.
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#include <structmember.h>
#include <stdint.h>

namespace {

constexpr Py_ssize_t kMaxArgs = 12;
constexpr Py_ssize_t kMaxLists = 4;
constexpr Py_ssize_t kMaxPointers = 64;

struct Call {
    PyObject_HEAD
    void *fn;
    Py_ssize_t nargs;
    char kinds[kMaxArgs];
    PyObject *array_type;
    vectorcallfunc vectorcall;
};

typedef uint64_t W;

int invoke(void *f, Py_ssize_t n, const W *a)
{
    switch (n) {
        case 7: return reinterpret_cast<int (*)(W, W, W, W, W, W, W)>(f)(a[0], a[1], a[2], a[3], a[4], a[5], a[6]);
        case 6: return reinterpret_cast<int (*)(W, W, W, W, W, W)>(f)(a[0], a[1], a[2], a[3], a[4], a[5]);
        case 8: return reinterpret_cast<int (*)(W, W, W, W, W, W, W, W)>(f)(a[0], a[1], a[2], a[3], a[4], a[5], a[6], a[7]);
        case 9:
            return reinterpret_cast<int (*)(W, W, W, W, W, W, W, W, W)>(f)(a[0], a[1], a[2], a[3], a[4], a[5], a[6], a[7], a[8]);
        case 10:
            return reinterpret_cast<int (*)(W, W, W, W, W, W, W, W, W, W)>(f)(a[0], a[1], a[2], a[3], a[4], a[5], a[6], a[7], a[8],
                                                                              a[9]);
        case 11:
            return reinterpret_cast<int (*)(W, W, W, W, W, W, W, W, W, W, W)>(f)(a[0], a[1], a[2], a[3], a[4], a[5], a[6], a[7],
                                                                                 a[8], a[9], a[10]);
        default:
            return reinterpret_cast<int (*)(W, W, W, W, W, W, W, W, W, W, W, W)>(f)(a[0], a[1], a[2], a[3], a[4], a[5], a[6], a[7],
                                                                                    a[8], a[9], a[10], a[11]);
    }
}

// An int or None as a machine word; false (no exception set) for anything else.
inline bool word(PyObject *o, W *out)
{
    if (PyLong_Check(o)) {
        *out = PyLong_AsUnsignedLongLongMask(o);   // never fails on an int
        return true;
    }
    if (o == Py_None) {
        *out = 0;
        return true;
    }
    return false;
}

PyObject *call(PyObject *self, PyObject *const *args, size_t nargsf, PyObject *kwnames)
{
    const Call *c = reinterpret_cast<const Call *>(self);
    const Py_ssize_t n = PyVectorcall_NARGS(nargsf);
    if (n != c->nargs || (kwnames != nullptr && PyTuple_GET_SIZE(kwnames) != 0)) {
        PyErr_Format(PyExc_TypeError, "%zd positional arguments expected", c->nargs);
        return nullptr;
    }
    W a[kMaxArgs];
    W lists[kMaxLists][kMaxPointers];
    Py_ssize_t used = 0;
    for (Py_ssize_t k = 0; k < n; ++k) {
        PyObject *o = args[k];
        if (c->kinds[k] == 'i') {
            if (!PyLong_Check(o)) Py_RETURN_NOTIMPLEMENTED;
            a[k] = PyLong_AsUnsignedLongLongMask(o);
            continue;
        }
        if (c->kinds[k] == 'l') {
            if (!PyList_CheckExact(o) && !PyTuple_CheckExact(o)) Py_RETURN_NOTIMPLEMENTED;
            const Py_ssize_t len = PySequence_Fast_GET_SIZE(o);
            if (used == kMaxLists || len > kMaxPointers) Py_RETURN_NOTIMPLEMENTED;
            for (Py_ssize_t j = 0; j < kMaxPointers; ++j) lists[used][j] = 0;
            for (Py_ssize_t j = 0; j < len; ++j) {
                if (!word(PySequence_Fast_GET_ITEM(o, j), &lists[used][j])) Py_RETURN_NOTIMPLEMENTED;
            }
            a[k] = reinterpret_cast<W>(lists[used++]);
            continue;
        }
        if (word(o, &a[k])) continue;
        const int is_array = PyObject_IsInstance(o, c->array_type);
        if (is_array < 0) return nullptr;
        if (is_array == 0) Py_RETURN_NOTIMPLEMENTED;
        Py_buffer view;
        if (PyObject_GetBuffer(o, &view, PyBUF_SIMPLE) != 0) return nullptr;
        a[k] = reinterpret_cast<W>(view.buf);   // a ctypes array keeps its memory; the caller holds a reference to it
        PyBuffer_Release(&view);
    }
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = invoke(c->fn, n, a);
    Py_END_ALLOW_THREADS
    return PyLong_FromLong(rc);
}

PyObject *make(PyTypeObject *type, PyObject *args, PyObject *)
{
    unsigned long long address = 0;
    const char *kinds = nullptr;
    Py_ssize_t nargs = 0;
    PyObject *array_type = nullptr;
    if (!PyArg_ParseTuple(args, "Ks#O", &address, &kinds, &nargs, &array_type)) return nullptr;
    bool known = address != 0 && nargs >= 6 && nargs <= kMaxArgs;
    for (Py_ssize_t k = 0; known && k < nargs; ++k) known = kinds[k] == 'i' || kinds[k] == 'p' || kinds[k] == 'l';
    if (!known) {
        PyErr_SetString(PyExc_ValueError, "an address and 6 to 12 argument kinds of i, p, l expected");
        return nullptr;
    }
    Call *c = reinterpret_cast<Call *>(type->tp_alloc(type, 0));
    if (c == nullptr) return nullptr;
    c->fn = reinterpret_cast<void *>(address);
    c->nargs = nargs;
    for (Py_ssize_t k = 0; k < nargs; ++k) c->kinds[k] = kinds[k];
    Py_INCREF(array_type);
    c->array_type = array_type;
    c->vectorcall = call;
    return reinterpret_cast<PyObject *>(c);
}

void drop(PyObject *self)
{
    Py_XDECREF(reinterpret_cast<Call *>(self)->array_type);
    Py_TYPE(self)->tp_free(self);
}

PyTypeObject g_call_type = {PyVarObject_HEAD_INIT(nullptr, 0)};

PyModuleDef g_module = {PyModuleDef_HEAD_INIT, "_hccl_calls", nullptr, -1, nullptr, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__hccl_calls(void)
{
    g_call_type.tp_name = "_hccl_calls.Call";
    g_call_type.tp_basicsize = sizeof(Call);
    g_call_type.tp_flags = Py_TPFLAGS_DEFAULT | Py_TPFLAGS_HAVE_VECTORCALL;
    g_call_type.tp_vectorcall_offset = offsetof(Call, vectorcall);
    g_call_type.tp_call = PyVectorcall_Call;
    g_call_type.tp_new = make;
    g_call_type.tp_dealloc = drop;
    if (PyType_Ready(&g_call_type) < 0) return nullptr;
    PyObject *m = PyModule_Create(&g_module);
    if (m == nullptr) return nullptr;
    Py_INCREF(&g_call_type);
    if (PyModule_AddObject(m, "Call", reinterpret_cast<PyObject *>(&g_call_type)) < 0) {
        Py_DECREF(&g_call_type);
        Py_DECREF(m);
        return nullptr;
    }
    return m;
}
