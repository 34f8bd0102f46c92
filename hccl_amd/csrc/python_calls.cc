// CPython module _hccl_calls: calls of the C entry points without ctypes' conversions.
//
// A collective among n virtual ranks is n calls, and a small one is over before Python has made them.  8 ranks x 1001 fp32
// take 10.4 us through ctypes (a foreign-function call of seven converted arguments each time), 6.3 through Call from a method
// written in Python and 5.2 through Method; an AlltoAll among 32 ranks 40.9, 22.2 and 9.5 (of which not making its tables of
// equal counts in every call is about half).
//
// Call(address, kinds, Array): one character of kinds per argument.  "i": an int (wraps like ctypes' integers); "p": an
// address, an int, None or a ctypes array; "l": a list or tuple of up to 64 ints or Nones (an array of addresses).  Given
// anything else it returns NotImplemented and the caller goes through ctypes, which converts or refuses it.  The GIL is
// released during the call, as ctypes does.  Every argument of the entry points is of INTEGER class (pointers, 32- and
// 64-bit integers), which the x86-64 System V calling convention passes in one 8-byte register or stack slot each whatever
// its width.
//
// Method(call, function, order): a Python method of a class of communicators in native code.  Called as
// object.name(rank, ...) it passes object.comms[rank] and the arguments that `order` names to `call`; whatever it cannot pass
// (keywords, another number of arguments, a rank that is no index, arguments of other types) goes to `function`, the same
// method written in Python.  order: one byte per argument of the entry point, the place of the method's argument (the object is
// place 0, the rank 1), plus 64 where it has to be a ctypes array; 255: the communicator.
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

constexpr unsigned char kTheComm = 255;
constexpr unsigned char kTable = 64;

struct Method {
    PyObject_HEAD
    Call *call;
    PyObject *function;
    PyObject *comms;   // the attribute's name
    Py_ssize_t nargs;  // of the method
    unsigned char order[kMaxArgs];
    PyObject *weakrefs;
    vectorcallfunc vectorcall;
};

PyObject *call_method(PyObject *self, PyObject *const *args, size_t nargsf, PyObject *kwnames)
{
    const Method *m = reinterpret_cast<const Method *>(self);
    const bool plain = PyVectorcall_NARGS(nargsf) == m->nargs && (kwnames == nullptr || PyTuple_GET_SIZE(kwnames) == 0);
    if (plain && PyLong_CheckExact(args[1])) {
        PyObject *comms = PyObject_GetAttr(args[0], m->comms);
        if (comms == nullptr) PyErr_Clear();   // the function reports it
        const Py_ssize_t rank = PyLong_AsSsize_t(args[1]);
        if (rank == -1 && PyErr_Occurred()) PyErr_Clear();
        if (comms != nullptr && PyList_CheckExact(comms) && rank >= 0 && rank < PyList_GET_SIZE(comms)) {
            // (held: asking an argument for its class may run code that empties the list)
            PyObject *comm = PyList_GET_ITEM(comms, rank);
            Py_INCREF(comm);
            PyObject *a[kMaxArgs];
            bool fits = true;
            for (Py_ssize_t k = 0; fits && k < m->call->nargs; ++k) {
                if (m->order[k] == kTheComm) {
                    a[k] = comm;
                    continue;
                }
                a[k] = args[m->order[k] & (kTable - 1)];
                if (m->order[k] >= kTable) fits = PyObject_IsInstance(a[k], m->call->array_type) == 1;
            }
            PyObject *result = nullptr;
            if (fits) {
                result = call(reinterpret_cast<PyObject *>(m->call), a, static_cast<size_t>(m->call->nargs), nullptr);
            } else if (PyErr_Occurred()) {
                PyErr_Clear();
            }
            Py_DECREF(comm);
            Py_DECREF(comms);
            if (fits && result != Py_NotImplemented) return result;
            Py_XDECREF(result);
        } else {
            Py_XDECREF(comms);
        }
    }
    return PyObject_Vectorcall(m->function, args, nargsf, kwnames);
}

PyObject *make_method(PyTypeObject *type, PyObject *args, PyObject *)
{
    PyObject *call_object = nullptr;
    PyObject *function = nullptr;
    const char *order = nullptr;
    Py_ssize_t n = 0;
    Py_ssize_t nargs = 0;
    if (!PyArg_ParseTuple(args, "O!Oy#n", &g_call_type, &call_object, &function, &order, &n, &nargs)) return nullptr;
    bool known = n == reinterpret_cast<Call *>(call_object)->nargs && nargs >= 2;
    for (Py_ssize_t k = 0; known && k < n; ++k) {
        const unsigned char at = static_cast<unsigned char>(order[k]);
        known = at == kTheComm || (at < 2 * kTable && (at & (kTable - 1)) < nargs);
    }
    if (!known) {
        PyErr_SetString(PyExc_ValueError, "one place of the method's arguments per argument of the call expected");
        return nullptr;
    }
    Method *m = reinterpret_cast<Method *>(type->tp_alloc(type, 0));
    if (m == nullptr) return nullptr;
    m->comms = PyUnicode_InternFromString("comms");
    if (m->comms == nullptr) {
        Py_DECREF(m);
        return nullptr;
    }
    Py_INCREF(call_object);
    Py_INCREF(function);
    m->call = reinterpret_cast<Call *>(call_object);
    m->function = function;
    m->nargs = nargs;
    for (Py_ssize_t k = 0; k < n; ++k) m->order[k] = static_cast<unsigned char>(order[k]);
    m->vectorcall = call_method;
    return reinterpret_cast<PyObject *>(m);
}

void drop_method(PyObject *self)
{
    Method *m = reinterpret_cast<Method *>(self);
    if (m->weakrefs != nullptr) PyObject_ClearWeakRefs(self);
    Py_XDECREF(reinterpret_cast<PyObject *>(m->call));
    Py_XDECREF(m->function);
    Py_XDECREF(m->comms);
    Py_TYPE(self)->tp_free(self);
}

PyObject *bind_method(PyObject *self, PyObject *object, PyObject *)
{
    if (object == nullptr || object == Py_None) {
        Py_INCREF(self);
        return self;
    }
    return PyMethod_New(self, object);
}

// What a program asks of a method is what the function says: its name, module, documentation, code and class, and attributes of
// the program's own.
PyObject *method_attribute(PyObject *self, PyObject *name)
{
    PyObject *found = PyObject_GenericGetAttr(self, name);
    if (found != nullptr || !PyErr_ExceptionMatches(PyExc_AttributeError)) return found;
    PyErr_Clear();
    return PyObject_GetAttr(reinterpret_cast<Method *>(self)->function, name);
}

int set_method_attribute(PyObject *self, PyObject *name, PyObject *value)
{
    return PyObject_SetAttr(reinterpret_cast<Method *>(self)->function, name, value);
}

PyObject *repr_method(PyObject *self) { return PyObject_Repr(reinterpret_cast<Method *>(self)->function); }

// (these two the type of any object has, so the lookup above would end there)
PyObject *of_the_function(PyObject *self, void *name)
{
    return PyObject_GetAttrString(reinterpret_cast<Method *>(self)->function, static_cast<const char *>(name));
}
char g_doc[] = "__doc__";
char g_class[] = "__class__";
PyGetSetDef g_method_getset[] = {{g_doc, of_the_function, nullptr, nullptr, g_doc},
                                 {g_class, of_the_function, nullptr, nullptr, g_class},
                                 {nullptr, nullptr, nullptr, nullptr, nullptr}};

// pickled and copied by name, as a function is
PyObject *reduce_method(PyObject *self, PyObject *)
{
    return PyObject_GetAttrString(reinterpret_cast<Method *>(self)->function, "__qualname__");
}
PyMethodDef g_method_methods[] = {{"__reduce__", reduce_method, METH_NOARGS, nullptr}, {nullptr, nullptr, 0, nullptr}};

PyMemberDef g_method_members[] = {{"__wrapped__", T_OBJECT, offsetof(Method, function), READONLY, nullptr},
                                  {nullptr, 0, 0, 0, nullptr}};

PyTypeObject g_method_type = {PyVarObject_HEAD_INIT(nullptr, 0)};

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
    g_method_type.tp_name = "_hccl_calls.Method";
    g_method_type.tp_basicsize = sizeof(Method);
    // (a method descriptor: an interpreter that calls object.name(...) passes the object without making a bound method)
    g_method_type.tp_flags = Py_TPFLAGS_DEFAULT | Py_TPFLAGS_HAVE_VECTORCALL | Py_TPFLAGS_METHOD_DESCRIPTOR;
    g_method_type.tp_vectorcall_offset = offsetof(Method, vectorcall);
    g_method_type.tp_call = PyVectorcall_Call;
    g_method_type.tp_new = make_method;
    g_method_type.tp_dealloc = drop_method;
    g_method_type.tp_descr_get = bind_method;
    g_method_type.tp_members = g_method_members;
    g_method_type.tp_getset = g_method_getset;
    g_method_type.tp_methods = g_method_methods;
    g_method_type.tp_getattro = method_attribute;
    g_method_type.tp_setattro = set_method_attribute;
    g_method_type.tp_repr = repr_method;
    g_method_type.tp_weaklistoffset = offsetof(Method, weakrefs);
    if (PyType_Ready(&g_method_type) < 0) return nullptr;
    PyObject *m = PyModule_Create(&g_module);
    if (m == nullptr) return nullptr;
    Py_INCREF(&g_call_type);
    if (PyModule_AddObject(m, "Call", reinterpret_cast<PyObject *>(&g_call_type)) < 0) {
        Py_DECREF(&g_call_type);
        Py_DECREF(m);
        return nullptr;
    }
    Py_INCREF(&g_method_type);
    if (PyModule_AddObject(m, "Method", reinterpret_cast<PyObject *>(&g_method_type)) < 0) {
        Py_DECREF(&g_method_type);
        Py_DECREF(m);
        return nullptr;
    }
    return m;
}
