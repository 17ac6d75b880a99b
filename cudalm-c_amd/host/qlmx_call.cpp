/* qlmx_call.cpp -- Python's way into the calls of libqlmx.so that a program makes per layer and step.
 *
 * Through ctypes a call costs its caller the conversion of every argument in Python and again in ctypes: 5 us for a
 * GEMM, 15 for the optimizer step with its 30 arguments, as long as the kernels themselves where the work is small. Here
 * the argument types come from include/qlmx.h at compile time and a call is converted and made in 0.5 to 2 us. The library is not
 * linked: `bind` makes a Python function from the address that the caller's loaded library has for the name.
 * Pointers: None, an integer, anything with data_ptr() (a torch tensor), or a numpy array. As with ctypes the calls run
 * without the interpreter lock. */
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#include <string.h>
#include <tuple>
#include <type_traits>
#include <utility>
#include "qlmx.h"

static PyObject *s_data_ptr, *s_ctypes, *s_data;

static bool as_address(PyObject *o, unsigned long long &v){
    if(o == Py_None){ v = 0; return true; }
    if(!PyLong_Check(o)){
        PyObject *n = PyObject_CallMethodNoArgs(o, s_data_ptr);
        if(!n){
            if(!PyErr_ExceptionMatches(PyExc_AttributeError)) return false;
            PyErr_Clear();
            PyObject *c = PyObject_GetAttr(o, s_ctypes);
            if(c){ n = PyObject_GetAttr(c, s_data); Py_DECREF(c); }
            else { PyErr_Clear(); n = PyNumber_Index(o); }
            if(!n){ PyErr_Format(PyExc_TypeError, "cannot take a pointer of %R", (PyObject *)Py_TYPE(o)); return false; }
        }
        v = PyLong_AsUnsignedLongLongMask(n);
        Py_DECREF(n);
    } else v = PyLong_AsUnsignedLongLongMask(o);
    return !(v == ~0ULL && PyErr_Occurred());
}
template<class T> static bool convert(PyObject *o, T &v){
    if constexpr(std::is_pointer_v<T>){
        unsigned long long a;
        if(!as_address(o, a)) return false;
        v = (T)(uintptr_t)a;
        return true;
    } else if constexpr(std::is_floating_point_v<T>){
        const double d = PyFloat_AsDouble(o);
        v = (T)d;
        return !(d == -1.0 && PyErr_Occurred());
    } else {
        const unsigned long long a = PyLong_AsUnsignedLongLongMask(o);
        v = (T)a;
        return !(a == ~0ULL && PyErr_Occurred());
    }
}
template<class F> struct Call;
template<class... A> struct Call<int (*)(A...)> {
    template<size_t... I> static PyObject *make(PyObject *address, PyObject *const *args, std::index_sequence<I...>){
        std::tuple<A...> v;
        if(!(convert(args[I], std::get<I>(v)) && ...)) return nullptr;
        int (*f)(A...) = (int (*)(A...))PyLong_AsVoidPtr(address);
        int rc;
        Py_BEGIN_ALLOW_THREADS
        rc = f(std::get<I>(v)...);
        Py_END_ALLOW_THREADS
        return PyLong_FromLong(rc);
    }
    static PyObject *call(PyObject *address, PyObject *const *args, Py_ssize_t n){
        if(n != (Py_ssize_t)sizeof...(A)) return PyErr_Format(PyExc_TypeError, "takes %d arguments, %zd given", (int)sizeof...(A), n);
        return make(address, args, std::index_sequence_for<A...>());
    }
};

#define ENTRY(NAME) {#NAME, (PyCFunction)(void (*)(void))Call<decltype(&NAME)>::call, METH_FASTCALL, nullptr}
static PyMethodDef entries[] = {
    ENTRY(qlmx_encode), ENTRY(qlmx_render), ENTRY(qlmx_servo), ENTRY(qlmx_step), ENTRY(qlmx_step_touched), ENTRY(qlmx_sqsum), ENTRY(qlmx_gnorm),
    ENTRY(qlmx_moe_gemm_nn), ENTRY(qlmx_moe_gemm_tn), ENTRY(qlmx_moe_gemm_nt), ENTRY(qlmx_moe_gemm_tn_pair), ENTRY(qlmx_moe_gemm_nn_swiglu),
    ENTRY(qlmx_moe_gemm_nn_gather), ENTRY(qlmx_moe_gemm_nn_gather_swiglu), ENTRY(qlmx_moe_gemm_nn_scatter), ENTRY(qlmx_moe_gemm_tn_swiglu_bwd),
    ENTRY(qlmx_moe_gemm_tn_pair_scatter), ENTRY(qlmx_pair_begin), ENTRY(qlmx_pair_end),
    ENTRY(qlmx_moe_decode_forward), ENTRY(qlmx_moe_decode_forward_noalloc),
    ENTRY(qlmx_router_topk), ENTRY(qlmx_moe_perm), ENTRY(qlmx_moe_gather), ENTRY(qlmx_moe_scatter_gate), ENTRY(qlmx_moe_scatter_add),
    ENTRY(qlmx_moe_dgate), ENTRY(qlmx_moe_dgate_merged), ENTRY(qlmx_moe_merge_rows), ENTRY(qlmx_moe_combine),
    ENTRY(qlmx_swiglu), ENTRY(qlmx_swiglu_bwd),
};

static PyObject *bind(PyObject *, PyObject *args){
    const char *name; PyObject *address;
    if(!PyArg_ParseTuple(args, "sO!", &name, &PyLong_Type, &address)) return nullptr;
    for(PyMethodDef &e : entries)
        if(strcmp(e.ml_name, name) == 0) return PyCFunction_New(&e, address);
    return PyErr_Format(PyExc_KeyError, "%s", name);
}
static PyObject *names(PyObject *, PyObject *){
    PyObject *t = PyTuple_New((Py_ssize_t)(sizeof entries / sizeof entries[0]));
    for(size_t i = 0; t && i < sizeof entries / sizeof entries[0]; i++) PyTuple_SET_ITEM(t, (Py_ssize_t)i, PyUnicode_FromString(entries[i].ml_name));
    return t;
}
static PyMethodDef methods[] = {
    {"bind", bind, METH_VARARGS, "bind(name, address): the library function of that name at that address as a Python function"},
    {"names", names, METH_NOARGS, "the names that bind knows"},
    {nullptr, nullptr, 0, nullptr}};
static PyModuleDef module = {PyModuleDef_HEAD_INIT, "_qlmx_call", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};
PyMODINIT_FUNC PyInit__qlmx_call(void){
    s_data_ptr = PyUnicode_InternFromString("data_ptr");
    s_ctypes = PyUnicode_InternFromString("ctypes");
    s_data = PyUnicode_InternFromString("data");
    return s_data_ptr && s_ctypes && s_data ? PyModule_Create(&module) : nullptr;
}
