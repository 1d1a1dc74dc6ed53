// Python calls into libcf_fp8.so without ctypes: one callable per declared function, its arguments converted by templates over
// the header's own prototypes.  A pass over a small layer is bound by its host calls; through ctypes and a Python loop over the
// arguments a GEMM's nineteen took 4.7 us beside a launch of about two, here 0.8.  An FP8 linear layer, four calls and five launches: 512 x 1024 x 1024,
// where the GPU takes over, 23.2 to 25.7 -> 18.8 to 21.2 us in five pairs of runs (two runs of one side differ by 3 to 24 %); smaller passes that the
// host bounds 24.4 -> 20.1 and 13.2 -> 11.4 (within 2 %).
//
// A pointer is None, an int or an object with data_ptr() (a torch tensor).  Whatever is not plainly one of the types a parameter
// takes, and any other number of arguments, goes to the ctypes callable that each of these carries, which converts it or raises.
// The GIL is released around the call, as ctypes does.
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#include <structmember.h>

#include <cstddef>
#include <cstring>
#include <tuple>
#include <type_traits>
#include <utility>

#include "cf_fp8.h"

namespace {

PyObject* g_data_ptr = nullptr;      // the interned method name

struct Callable {
    PyObject_HEAD
    vectorcallfunc vectorcall;
    void* fn;                        // the function in the library this callable was made for
    PyObject* fallback;              // the same call through ctypes
    PyObject* failed;                // called with a non-zero return code; raises
    PyObject* name;
};

// false: not plainly of the parameter's type, or data_ptr() raised (what it raised is then set)
template <class T>
bool convert(PyObject* o, T& out) {
    if constexpr (std::is_pointer_v<T>) {
        if (o == Py_None) {
            out = nullptr;
            return true;
        }
        if (PyLong_CheckExact(o)) {
            out = reinterpret_cast<T>(static_cast<uintptr_t>(PyLong_AsUnsignedLongLongMask(o)));
            return true;
        }
        PyObject* r = PyObject_VectorcallMethod(g_data_ptr, &o, 1 | PY_VECTORCALL_ARGUMENTS_OFFSET, nullptr);
        if (!r) {
            if (PyErr_ExceptionMatches(PyExc_AttributeError)) PyErr_Clear();       // no such method: not a tensor
            return false;
        }
        const bool ok = PyLong_CheckExact(r);
        if (ok) out = reinterpret_cast<T>(static_cast<uintptr_t>(PyLong_AsUnsignedLongLongMask(r)));
        Py_DECREF(r);
        return ok;
    } else if constexpr (std::is_floating_point_v<T>) {
        if (PyFloat_CheckExact(o)) {
            out = static_cast<T>(PyFloat_AS_DOUBLE(o));
            return true;
        }
        return false;
    } else {
        static_assert(std::is_integral_v<T>);
        if (!PyLong_Check(o)) return false;
        out = static_cast<T>(PyLong_AsUnsignedLongLongMask(o));
        return true;
    }
}

template <class F>
struct Thunk;
template <class... A>
struct Thunk<int (*)(A...)> {
    template <std::size_t... I>
    static bool convert_all(PyObject* const* args, std::tuple<A...>& v, std::index_sequence<I...>) {
        return (convert(args[I], std::get<I>(v)) && ...);
    }
    static PyObject* call(PyObject* self, PyObject* const* args, size_t nargsf, PyObject* names) {
        auto* c = reinterpret_cast<Callable*>(self);
        std::tuple<A...> v;
        if (names || PyVectorcall_NARGS(nargsf) != static_cast<Py_ssize_t>(sizeof...(A)) ||
            !convert_all(args, v, std::index_sequence_for<A...>{}))
            return PyErr_Occurred() ? nullptr : PyObject_Vectorcall(c->fallback, args, nargsf, names);
        int rc;
        auto fn = reinterpret_cast<int (*)(A...)>(c->fn);
        Py_BEGIN_ALLOW_THREADS
        rc = std::apply(fn, v);
        Py_END_ALLOW_THREADS
        if (rc == 0) Py_RETURN_NONE;
        PyObject* code = PyLong_FromLong(rc);
        if (!code) return nullptr;
        PyObject* r = PyObject_CallOneArg(c->failed, code);
        Py_DECREF(code);
        return r;
    }
};

struct Entry { const char* name; vectorcallfunc call; };
#define CF_CALL(name) {#name, &Thunk<decltype(&name)>::call},
const Entry kEntries[] = {
#include "call_names.inc"       // CF_CALL(f) for every function of the header that returns int; written by build.py
};
#undef CF_CALL

int traverse(PyObject* self, visitproc visit, void* arg) {
    auto* c = reinterpret_cast<Callable*>(self);
    Py_VISIT(c->fallback);
    Py_VISIT(c->failed);
    Py_VISIT(c->name);
    return 0;
}
int clear(PyObject* self) {
    auto* c = reinterpret_cast<Callable*>(self);
    Py_CLEAR(c->fallback);
    Py_CLEAR(c->failed);
    Py_CLEAR(c->name);
    return 0;
}
void dealloc(PyObject* self) {
    PyObject_GC_UnTrack(self);
    clear(self);
    Py_TYPE(self)->tp_free(self);
}

PyMemberDef kMembers[] = {{"__name__", T_OBJECT_EX, offsetof(Callable, name), READONLY, nullptr}, {nullptr, 0, 0, 0, nullptr}};
PyTypeObject CallableType = {PyVarObject_HEAD_INIT(nullptr, 0)};

// make(name, address, fallback, failed): the callable, or None for a name that is not in the header
PyObject* make(PyObject*, PyObject* args) {
    const char* name;
    unsigned long long address;
    PyObject *fallback, *failed;
    if (!PyArg_ParseTuple(args, "sKOO", &name, &address, &fallback, &failed)) return nullptr;
    for (const Entry& e : kEntries)
        if (std::strcmp(e.name, name) == 0) {
            PyObject* text = PyUnicode_FromString(name);
            if (!text) return nullptr;
            auto* c = PyObject_GC_New(Callable, &CallableType);
            if (!c) {
                Py_DECREF(text);
                return nullptr;
            }
            c->name = text;
            c->vectorcall = e.call;
            c->fn = reinterpret_cast<void*>(static_cast<uintptr_t>(address));
            Py_INCREF(fallback);
            Py_INCREF(failed);
            c->fallback = fallback;
            c->failed = failed;
            PyObject_GC_Track(reinterpret_cast<PyObject*>(c));
            return reinterpret_cast<PyObject*>(c);
        }
    Py_RETURN_NONE;
}

PyMethodDef kMethods[] = {{"make", make, METH_VARARGS, nullptr}, {nullptr, nullptr, 0, nullptr}};
PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_cf_call", nullptr, -1, kMethods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__cf_call() {
    g_data_ptr = PyUnicode_InternFromString("data_ptr");
    if (!g_data_ptr) return nullptr;
    CallableType.tp_name = "_cf_call.Callable";
    CallableType.tp_basicsize = sizeof(Callable);
    CallableType.tp_flags = Py_TPFLAGS_DEFAULT | Py_TPFLAGS_HAVE_GC | Py_TPFLAGS_HAVE_VECTORCALL;
    CallableType.tp_vectorcall_offset = offsetof(Callable, vectorcall);
    CallableType.tp_call = PyVectorcall_Call;
    CallableType.tp_traverse = traverse;
    CallableType.tp_members = kMembers;
    CallableType.tp_clear = clear;
    CallableType.tp_dealloc = dealloc;
    if (PyType_Ready(&CallableType) < 0) return nullptr;
    PyObject* module = PyModule_Create(&kModule);
    // the text these prototypes came from: the binding goes by what it reads, and uses none of them if that is another
    if (module && PyModule_AddStringConstant(module, "header", CF_HEADER_HASH) < 0) Py_CLEAR(module);
    return module;
}
