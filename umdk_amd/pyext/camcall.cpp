// Python caller of the two-phase C ABI (include/camhip.h): one extension function per entry point that converts its
// arguments, sizes the workspace, has it allocated and launches.  Through ctypes the two calls of an operator with some
// thirty arguments cost 8 us of host time, as much as its launches, and the smallest operator calls are bound by the
// host (one token through moe_route and fused_deep_moe: 39 us a pass through ctypes, 34 us through this; the five-operator
// chain at T = 1021: 90 and 75 us).
//
// name(alloc, workspace, workspace_bytes, stream, *args) -> buffer or None
//   args: the GetWorkspaceSize arguments (pointers as int or None, sizes as any integer), without the two outputs;
//   alloc: called with the workspace size when it is not 0, returns a tensor (its data_ptr is used and the tensor is
//          returned); None: the caller's workspace is used;
//   a failed call raises bind's exception with the library's message.
// bind(handle, error): takes the entry points from an open library (a dlopen handle), the one its Python loader has
// loaded; this module links to none, so a diagnostic build loaded in the library's place gets every call.
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#include <dlfcn.h>

#include <tuple>
#include <type_traits>
#include <utility>

#include "camhip.h"

namespace {

PyObject *g_error = nullptr;
decltype(&camhipGetLastErrorMsg) g_last_error = nullptr;
decltype(&camhipReleaseExecutor) g_release = nullptr;

template <typename A> bool convert(PyObject *o, A &out)
{
    if constexpr (std::is_pointer_v<A>) {
        if (o == Py_None) {
            out = nullptr;
            return true;
        }
        if (!PyLong_Check(o)) {
            PyErr_SetString(PyExc_TypeError, "a pointer argument must be an int or None");
            return false;
        }
        out = (A)PyLong_AsVoidPtr(o);
    } else {
        // any integer type, numpy's among them, through __index__ (a float has none: TypeError); taken modulo 2^64
        out = (A)PyLong_AsUnsignedLongLongMask(o);
    }
    return !PyErr_Occurred();
}

PyObject *failed(const char *name, const char *phase, int status)
{
    PyErr_Format(g_error, "%s%s failed (%d): %s", name, phase, status,
                 g_last_error());
    return nullptr;
}

using RunFn = camhipStatus (*)(void *, uint64_t, camhipExecutor *, void *);
constexpr Py_ssize_t FIXED = 4;

template <typename... P, size_t... I>
PyObject *invoke(const char *name, camhipStatus (*get)(P...), RunFn run, PyObject *const *argv, Py_ssize_t n,
                 std::index_sequence<I...>)
{
    if (n != FIXED + (Py_ssize_t)sizeof...(I)) {
        PyErr_Format(PyExc_TypeError, "%s takes %zd arguments (%zd given)", name, (Py_ssize_t)sizeof...(I), n - FIXED);
        return nullptr;
    }
    if (!g_error) {
        PyErr_SetString(PyExc_RuntimeError, "_camcall is not bound to a library");
        return nullptr;
    }
    std::tuple<P...> a{};
    void *ws = nullptr, *stream = nullptr;
    int64_t have = 0;
    if (!convert(argv[1], ws) || !convert(argv[2], have) || !convert(argv[3], stream) ||
        !(convert(argv[FIXED + I], std::get<I>(a)) && ...))
        return nullptr;
    uint64_t need = 0;
    camhipExecutor *ex = nullptr;
    std::get<sizeof...(I)>(a) = &need;
    std::get<sizeof...(I) + 1>(a) = &ex;
    int st = std::apply(get, a);
    if (st != CAMHIP_SUCCESS)
        return failed(name, "GetWorkspaceSize", st);
    PyObject *buf = nullptr;
    if (argv[0] != Py_None && need > 0) {
        PyObject *size = PyLong_FromUnsignedLongLong(need);
        buf = size ? PyObject_CallOneArg(argv[0], size) : nullptr;
        Py_XDECREF(size);
        PyObject *p = buf ? PyObject_CallMethod(buf, "data_ptr", nullptr) : nullptr;
        const bool ok = p && convert(p, ws);
        Py_XDECREF(p);
        if (!ok) {
            Py_XDECREF(buf);
            g_release(ex);
            return nullptr;
        }
        have = (int64_t)need;
    }
    Py_BEGIN_ALLOW_THREADS
    st = run(ws, (uint64_t)have, ex, stream);
    Py_END_ALLOW_THREADS
    if (st != CAMHIP_SUCCESS) {
        Py_XDECREF(buf);
        return failed(name, "", st);
    }
    if (buf)
        return buf;
    Py_RETURN_NONE;
}

template <typename... P>
PyObject *entry(const char *name, camhipStatus (*get)(P...), RunFn run, PyObject *const *argv, Py_ssize_t n)
{
    return invoke(name, get, run, argv, n, std::make_index_sequence<sizeof...(P) - 2>{});
}

#define ENTRIES(X)                                                                                                   \
    X(camhipMoeRoute)                                                                                                \
    X(camhipDispatchLayout)                                                                                          \
    X(camhipNotifyDispatch)                                                                                          \
    X(camhipMoeDispatchNormal)                                                                                       \
    X(camhipMoeCombineNormal)                                                                                        \
    X(camhipGroupedMatmulSwiglu)                                                                                     \
    X(camhipGroupedMatmul)                                                                                           \
    X(camhipFusedDeepMoe)                                                                                            \
    X(camhipMoePrefillDispatch)                                                                                      \
    X(camhipMoePrefillCombine)                                                                                       \
    X(camhipMoeExperts)

#define DEFINE(f)                                                                                                    \
    decltype(&f##GetWorkspaceSize) get_##f = nullptr;                                                                \
    RunFn run_##f = nullptr;                                                                                         \
    PyObject *py_##f(PyObject *, PyObject *const *argv, Py_ssize_t n)                                                \
    {                                                                                                                \
        if (n < FIXED) {                                                                                             \
            PyErr_SetString(PyExc_TypeError, #f ": alloc, workspace, workspace_bytes and stream come first");        \
            return nullptr;                                                                                          \
        }                                                                                                            \
        return entry(#f, get_##f, run_##f, argv, n);                                                                 \
    }
ENTRIES(DEFINE)

template <typename F> bool resolve(void *lib, const char *name, F &out)
{
    out = (F)dlsym(lib, name);
    if (!out)
        PyErr_Format(PyExc_ImportError, "the library has no %s", name);
    return out != nullptr;
}

PyObject *bind(PyObject *, PyObject *args)
{
    PyObject *handle, *type;
    void *lib = nullptr;
    if (!PyArg_ParseTuple(args, "OO", &handle, &type) || !convert(handle, lib))
        return nullptr;
#define RESOLVE(f)                                                                                                   \
    if (!resolve(lib, #f "GetWorkspaceSize", get_##f) || !resolve(lib, #f, run_##f))                                 \
        return nullptr;
    ENTRIES(RESOLVE)
    if (!resolve(lib, "camhipGetLastErrorMsg", g_last_error) || !resolve(lib, "camhipReleaseExecutor", g_release))
        return nullptr;
    Py_INCREF(type);
    Py_XSETREF(g_error, type);
    Py_RETURN_NONE;
}

#define METHOD(f) {#f, (PyCFunction)(void (*)(void))py_##f, METH_FASTCALL, nullptr},
PyMethodDef g_methods[] = {ENTRIES(METHOD){"bind", bind, METH_VARARGS, nullptr}, {nullptr, nullptr, 0, nullptr}};
PyModuleDef g_module = {PyModuleDef_HEAD_INIT, "_camcall", nullptr, -1, g_methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__camcall(void) { return PyModule_Create(&g_module); }
