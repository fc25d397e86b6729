// The part of the scripting mirror that a program goes through for every node of an expression: the Array handle with its arithmetic
// operators and inspection, the factories of elementwise operators, reductions and products, and evaluation (dali/array/array.h,
// dali/array/op.h). The rest of the mirror calls the same entry points of include/dali_front.h through ctypes, which costs 0.3 us a call
// and 0.8 to 2 us a node where this takes 0.1 to 0.3 (an expression of eight operators: 11.3 us to build, now 2.9; with its evaluation 16.8, now 8.3).
//
// Calls on operands give up the interpreter lock, as ctypes does: building a node may evaluate what it stands on, and observers of that may be
// Python functions of another thread. So does the release of the last handle to a buffer, or to a node that may hold the last reference to one: it
// waits for transfers that still use the memory. Inspection, literals and the release of operands that a node keeps alive hold it (giving
// it up costs 0.04 us).
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <vector>

#include "../../include/dali_front.h"

namespace {

struct ArrayObject {
    PyObject_HEAD
    dali_array_t handle;
};

PyTypeObject* g_array = nullptr;  // the Python class built on Handle below
PyObject* g_error = nullptr;      // DaliError
PyObject* g_as_array = nullptr;   // what becomes of operands that are neither arrays nor Python numbers

extern PyTypeObject HandleType;

// the call of a native function without the interpreter lock
template <typename F>
auto unlocked(F&& call) {
    PyThreadState* state = PyEval_SaveThread();
    auto r = call();
    PyEval_RestoreThread(state);
    return r;
}

void release(dali_array_t handle) {
    if (dali_fe_is_last_handle(handle)) {
        unlocked([&] {
            dali_fe_release(handle);
            return 0;
        });
    } else {
        dali_fe_release(handle);
    }
}

PyObject* fail(const char* what) {
    PyErr_Format(g_error, "%s failed: %s", what, dali_fe_last_error());
    return nullptr;
}

PyObject* wrap(dali_array_t handle, const char* what) {
    if (!handle) return fail(what);
    PyObject* o = g_array->tp_alloc(g_array, 0);
    if (!o) {
        release(handle);
        return nullptr;
    }
    ((ArrayObject*)o)->handle = handle;
    return o;
}

// An operand: an array, a number (which becomes a literal for the duration of the call), or whatever as_array makes of it
struct Operand {
    dali_array_t handle = nullptr, literal = nullptr;
    PyObject* kept = nullptr;
    Operand() = default;
    Operand(const Operand&) = delete;
    Operand& operator=(const Operand&) = delete;
    ~Operand() {
        if (literal) dali_fe_release(literal);
        Py_XDECREF(kept);
    }
    bool set(PyObject* o) {
        if (PyObject_TypeCheck(o, &HandleType)) {
            Py_INCREF(o);  // (the call may give up the interpreter lock)
            kept = o;
            handle = ((ArrayObject*)o)->handle;
            return true;
        }
        if (PyLong_Check(o)) {
            const unsigned long bits = PyLong_AsUnsignedLongMask(o);
            if (bits == (unsigned long)-1 && PyErr_Occurred()) return false;
            handle = literal = dali_fe_scalar_int((int)bits);
        } else if (PyFloat_Check(o)) {
            handle = literal = dali_fe_scalar_double(PyFloat_AS_DOUBLE(o));
        } else {
            kept = PyObject_CallOneArg(g_as_array, o);
            if (!kept) return false;
            if (!PyObject_TypeCheck(kept, &HandleType)) {
                PyErr_SetString(PyExc_TypeError, "as_array returned no Array");
                return false;
            }
            handle = ((ArrayObject*)kept)->handle;
            return true;
        }
        if (!handle) fail("scalar");
        return handle != nullptr;
    }
};

bool count_is(Py_ssize_t n, Py_ssize_t want, const char* what) {
    if (n == want) return true;
    PyErr_Format(PyExc_TypeError, "%s takes %zd arguments (got %zd)", what, want, n);
    return false;
}

bool whole_number(PyObject* o, int* v) {
    PyObject* n = PyNumber_Long(o);
    if (!n) return false;
    *v = (int)PyLong_AsUnsignedLongMask(n);
    Py_DECREF(n);
    return !PyErr_Occurred();
}

// one axis, or several
bool whole_numbers(PyObject* o, std::vector<int>* out) {
    if (PyLong_Check(o)) {
        out->resize(1);
        return whole_number(o, out->data());
    }
    PyObject* s = PySequence_Tuple(o);  // (converting an entry may run the program's code, which could change a list)
    if (!s) return false;
    const Py_ssize_t n = PyTuple_GET_SIZE(s);
    out->resize(n);
    bool ok = true;
    for (Py_ssize_t i = 0; ok && i < n; ++i) ok = whole_number(PyTuple_GET_ITEM(s, i), &(*out)[i]);
    Py_DECREF(s);
    return ok;
}

// ------------------------------------------------------------------------------------------------ Handle
int handle_init(PyObject* self, PyObject* args, PyObject* kwargs) {
    PyObject* handle = nullptr;
    static const char* names[] = {"handle", nullptr};
    if (!PyArg_ParseTupleAndKeywords(args, kwargs, "O", (char**)names, &handle)) return -1;
    void* h = nullptr;
    if (handle != Py_None) {
        h = PyLong_AsVoidPtr(handle);
        if (!h && PyErr_Occurred()) return -1;
    }
    dali_array_t old = ((ArrayObject*)self)->handle;
    ((ArrayObject*)self)->handle = h;
    if (old && old != h) release(old);
    return 0;
}

void handle_dealloc(PyObject* self) {
    dali_array_t h = ((ArrayObject*)self)->handle;
    if (h) release(h);
    Py_TYPE(self)->tp_free(self);
}

dali_array_t of(PyObject* self) { return ((ArrayObject*)self)->handle; }

PyObject* get_handle(PyObject* self, void*) {
    if (!of(self)) Py_RETURN_NONE;
    return PyLong_FromVoidPtr(of(self));
}

// (the handle is exchanged, not released: whoever assigns None has taken it over)
int set_handle(PyObject* self, PyObject* value, void*) {
    void* h = nullptr;
    if (value && value != Py_None) {
        h = PyLong_AsVoidPtr(value);
        if (!h && PyErr_Occurred()) return -1;
    }
    ((ArrayObject*)self)->handle = h;
    return 0;
}

PyObject* extents(PyObject* self, int (*read)(dali_array_t, int*), const char* what) {
    const int nd = dali_fe_ndim(of(self));
    if (nd < 0) return fail(what);
    std::vector<int> v(nd + 1);
    if (read(of(self), v.data()) != 0) return fail(what);
    PyObject* t = PyTuple_New(nd);
    for (int i = 0; t && i < nd; ++i) {
        PyObject* n = PyLong_FromLong(v[i]);
        if (!n) {
            Py_DECREF(t);
            return nullptr;
        }
        PyTuple_SET_ITEM(t, i, n);
    }
    return t;
}

PyObject* get_shape(PyObject* self, void*) { return extents(self, dali_fe_shape, "shape"); }
PyObject* get_strides(PyObject* self, void*) { return extents(self, dali_fe_strides, "strides"); }
PyObject* get_ndim(PyObject* self, void*) { return PyLong_FromLong(dali_fe_ndim(of(self))); }
PyObject* get_dtype(PyObject* self, void*) { return PyLong_FromLong(dali_fe_dtype(of(self))); }
PyObject* get_offset(PyObject* self, void*) { return PyLong_FromLong(dali_fe_offset(of(self))); }

PyObject* handle_eval(PyObject* self, PyObject*) {
    Py_INCREF(self);
    if (unlocked([&] { return dali_fe_eval(of(self)); }) != 0) {
        Py_DECREF(self);
        return fail("eval");
    }
    return self;
}

PyObject* handle_device_ptr(PyObject* self, PyObject*) {
    void* p = unlocked([&] { return dali_fe_device_ptr(of(self)); });
    return p ? PyLong_FromVoidPtr(p) : fail("device_ptr");
}

PyObject* combine(const char* name, PyObject* a, PyObject* b) {
    Operand l, r;
    if (!l.set(a) || !r.set(b)) return nullptr;
    return wrap(unlocked([&] { return dali_fe_binary(name, l.handle, r.handle); }), name);
}

PyObject* nb_add(PyObject* a, PyObject* b) { return combine("add", a, b); }
PyObject* nb_subtract(PyObject* a, PyObject* b) { return combine("subtract", a, b); }
PyObject* nb_multiply(PyObject* a, PyObject* b) { return combine("eltmul", a, b); }
PyObject* nb_divide(PyObject* a, PyObject* b) { return combine("eltdiv", a, b); }
PyObject* nb_negative(PyObject* a) {
    Operand l, r;
    l.handle = l.literal = dali_fe_scalar_int(-1);
    if (!l.handle) return fail("scalar");
    return r.set(a) ? wrap(unlocked([&] { return dali_fe_binary("eltmul", l.handle, r.handle); }), "eltmul") : nullptr;
}

PyGetSetDef handle_getset[] = {{"_h", get_handle, set_handle, "the native handle", nullptr},
                               {"shape", get_shape, nullptr, nullptr, nullptr},
                               {"strides", get_strides, nullptr, nullptr, nullptr},
                               {"ndim", get_ndim, nullptr, nullptr, nullptr},
                               {"dtype", get_dtype, nullptr, nullptr, nullptr},
                               {"offset", get_offset, nullptr, nullptr, nullptr},
                               {nullptr, nullptr, nullptr, nullptr, nullptr}};
PyMethodDef handle_methods[] = {{"eval", handle_eval, METH_NOARGS, nullptr}, {"device_ptr", handle_device_ptr, METH_NOARGS, nullptr}, {nullptr, nullptr, 0, nullptr}};
PyNumberMethods handle_number = {};
PyTypeObject HandleType = {PyVarObject_HEAD_INIT(nullptr, 0)};

// ------------------------------------------------------------------------------------------------ functions
// (those that take a name take it first, those with an axis list as last but one)
PyObject* f_register(PyObject*, PyObject* const* args, Py_ssize_t n) {
    if (!count_is(n, 3, "register")) return nullptr;
    if (!PyType_Check(args[0]) || !PyType_IsSubtype((PyTypeObject*)args[0], &HandleType)) {
        PyErr_SetString(PyExc_TypeError, "register needs a class built on Handle");
        return nullptr;
    }
    for (int i = 0; i < 3; ++i) Py_INCREF(args[i]);
    Py_XDECREF((PyObject*)g_array);
    Py_XDECREF(g_error);
    Py_XDECREF(g_as_array);
    g_array = (PyTypeObject*)args[0];
    g_error = args[1];
    g_as_array = args[2];
    Py_RETURN_NONE;
}

PyObject* f_unary(PyObject*, PyObject* const* args, Py_ssize_t n) {
    Operand a;
    if (!count_is(n, 2, "unary")) return nullptr;
    const char* name = PyUnicode_AsUTF8(args[0]);
    return name && a.set(args[1]) ? wrap(unlocked([&] { return dali_fe_unary(name, a.handle); }), name) : nullptr;
}

PyObject* f_binary(PyObject*, PyObject* const* args, Py_ssize_t n) {
    if (!count_is(n, 3, "binary")) return nullptr;
    const char* name = PyUnicode_AsUTF8(args[0]);
    return name ? combine(name, args[1], args[2]) : nullptr;
}

PyObject* f_all_reduce(PyObject*, PyObject* const* args, Py_ssize_t n) {
    Operand a;
    if (!count_is(n, 2, "all_reduce")) return nullptr;
    const char* name = PyUnicode_AsUTF8(args[0]);
    return name && a.set(args[1]) ? wrap(unlocked([&] { return dali_fe_all_reduce(name, a.handle); }), name) : nullptr;
}

PyObject* f_axis_reduce(PyObject*, PyObject* const* args, Py_ssize_t n) {
    Operand a;
    std::vector<int> axes;
    if (!count_is(n, 4, "axis_reduce")) return nullptr;
    const char* name = PyUnicode_AsUTF8(args[0]);
    if (!name || !a.set(args[1]) || !whole_numbers(args[2], &axes)) return nullptr;
    const int keepdims = PyObject_IsTrue(args[3]);
    return keepdims < 0 ? nullptr : wrap(unlocked([&] { return dali_fe_axis_reduce(name, a.handle, axes.data(), (int)axes.size(), keepdims); }), name);
}

PyObject* f_arg_axis_reduce(PyObject*, PyObject* const* args, Py_ssize_t n) {
    Operand a;
    int axis;
    if (!count_is(n, 4, "arg_axis_reduce")) return nullptr;
    const char *name = PyUnicode_AsUTF8(args[0]), *what = PyUnicode_AsUTF8(args[3]);
    return name && what && a.set(args[1]) && whole_number(args[2], &axis) ? wrap(unlocked([&] { return dali_fe_arg_axis_reduce(name, a.handle, axis); }), what) : nullptr;
}

PyObject* f_softmax(PyObject*, PyObject* const* args, Py_ssize_t n) {
    Operand a;
    int axis;
    return count_is(n, 2, "softmax") && a.set(args[0]) && whole_number(args[1], &axis) ? wrap(unlocked([&] { return dali_fe_softmax(a.handle, axis); }), "softmax") : nullptr;
}

// two operands to one array; building a product or a gather may evaluate operands
PyObject* pair(PyObject* const* args, Py_ssize_t n, dali_array_t (*make)(dali_array_t, dali_array_t), const char* what) {
    Operand a, b;
    if (!count_is(n, 2, what) || !a.set(args[0]) || !b.set(args[1])) return nullptr;
    return wrap(unlocked([&] { return make(a.handle, b.handle); }), what);
}
PyObject* f_dot(PyObject*, PyObject* const* args, Py_ssize_t n) { return pair(args, n, dali_fe_dot, "dot"); }
PyObject* f_gather(PyObject*, PyObject* const* args, Py_ssize_t n) { return pair(args, n, dali_fe_gather, "gather"); }
PyObject* f_gather_from_rows(PyObject*, PyObject* const* args, Py_ssize_t n) { return pair(args, n, dali_fe_gather_from_rows, "gather_from_rows"); }

PyObject* f_transpose(PyObject*, PyObject* const* args, Py_ssize_t n) {
    Operand a;
    std::vector<int> axes;
    if (!count_is(n, 2, "transpose") || !a.set(args[0]) || !whole_numbers(args[1], &axes)) return nullptr;
    return wrap(unlocked([&] { return dali_fe_transpose(a.handle, axes.data(), (int)axes.size()); }), "transpose");
}

PyObject* f_assign(PyObject*, PyObject* const* args, Py_ssize_t n) {
    Operand dest, source;
    int op;
    if (!count_is(n, 3, "assign") || !dest.set(args[0]) || !whole_number(args[1], &op) || !source.set(args[2])) return nullptr;
    if (unlocked([&] { return dali_fe_assign(dest.handle, op, source.handle); }) != 0) return fail("assign");
    Py_RETURN_NONE;
}

PyObject* wrapped(dali_array_t* handles, int n, const char* what) {
    PyObject* t = PyTuple_New(n);
    for (int i = 0; i < n; ++i) {
        PyObject* o = t ? wrap(handles[i], what) : nullptr;
        if (o) {
            PyTuple_SET_ITEM(t, i, o);
            continue;
        }
        for (int j = i + (t ? 1 : 0); j < n; ++j)
            if (handles[j]) release(handles[j]);
        Py_XDECREF(t);
        return nullptr;
    }
    return t;
}

PyObject* f_softmax_cross_entropy(PyObject*, PyObject* const* args, Py_ssize_t n) {
    Operand logits, targets;
    if (!count_is(n, 2, "softmax_cross_entropy") || !logits.set(args[0]) || !targets.set(args[1])) return nullptr;
    dali_array_t r[3] = {};
    const int status = unlocked([&] { return dali_fe_softmax_cross_entropy(logits.handle, targets.handle, &r[0], &r[1], &r[2]); });
    return status != 0 ? fail("softmax_cross_entropy") : wrapped(r, 3, "softmax_cross_entropy");
}

// x, h, c, W, U, b
PyObject* f_lstm_step(PyObject*, PyObject* const* args, Py_ssize_t n) {
    Operand a[6];
    if (!count_is(n, 6, "lstm_step")) return nullptr;
    for (int i = 0; i < 6; ++i)
        if (!a[i].set(args[i])) return nullptr;
    dali_array_t r[2] = {};
    const int status = unlocked([&] { return dali_fe_lstm_step(a[0].handle, a[1].handle, a[2].handle, a[3].handle, a[4].handle, a[5].handle, &r[0], &r[1]); });
    return status != 0 ? fail("lstm_step") : wrapped(r, 2, "lstm_step");
}

#define FUNCTION(name) {#name, (PyCFunction)(void (*)(void))f_##name, METH_FASTCALL, nullptr}
PyMethodDef functions[] = {FUNCTION(register),        FUNCTION(unary),     FUNCTION(binary),  FUNCTION(all_reduce), FUNCTION(axis_reduce),
                           FUNCTION(arg_axis_reduce), FUNCTION(softmax),   FUNCTION(dot),     FUNCTION(gather),     FUNCTION(gather_from_rows),
                           FUNCTION(transpose),       FUNCTION(assign),    FUNCTION(softmax_cross_entropy),         FUNCTION(lstm_step),
                           {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_bind", nullptr, -1, functions, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__bind(void) {
    handle_number.nb_add = nb_add;
    handle_number.nb_subtract = nb_subtract;
    handle_number.nb_multiply = nb_multiply;
    handle_number.nb_true_divide = nb_divide;
    handle_number.nb_negative = nb_negative;
    HandleType.tp_name = "dali_amd._bind.Handle";
    HandleType.tp_basicsize = sizeof(ArrayObject);
    HandleType.tp_flags = Py_TPFLAGS_DEFAULT | Py_TPFLAGS_BASETYPE;
    HandleType.tp_new = PyType_GenericNew;
    HandleType.tp_init = handle_init;
    HandleType.tp_dealloc = handle_dealloc;
    HandleType.tp_getset = handle_getset;
    HandleType.tp_methods = handle_methods;
    HandleType.tp_as_number = &handle_number;
    if (PyType_Ready(&HandleType) < 0) return nullptr;
    PyObject* m = PyModule_Create(&module);
    if (!m) return nullptr;
    Py_INCREF(&HandleType);
    if (PyModule_AddObject(m, "Handle", (PyObject*)&HandleType) < 0) {
        Py_DECREF(&HandleType);
        Py_DECREF(m);
        return nullptr;
    }
    return m;
}
