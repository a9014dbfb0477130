// Calls of the C-ABI launchers from Python without ctypes: one vectorcall function per launcher, whose argument
// conversions are generated from the launcher's prototype in include/cpmk.h.  A decode step is some thirty calls of a few
// microseconds each, and the conversions of ctypes with the status check in Python cost 1.5-2 us of every one.
//
// The library itself is loaded by library/base.py (search order, one HIP runtime per process); bind() is given the
// address of a launcher in it.  Conversions are those of ctypes: integers of any size are taken modulo the parameter's width, pointers
// are integers, None or ctypes.c_void_p (anything else that ctypes accepts goes through the callable of
// init(), as ctypes numbers do), and the call runs without the interpreter lock.  A non-zero status raises RuntimeError("HIP Error: ...").
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#include <cstdint>
#include <cstring>
#include <tuple>
#include <type_traits>
#include <utility>
#include "../../include/cpmk.h"

namespace {

const char* (*g_error_string)(int) = nullptr;
// callable: object -> address, for the pointer arguments that are neither int nor None;
// (object, bytes of the integer parameter or 0 for a float one) -> number, for what is no Python number
PyObject* g_value = nullptr;

bool convert(PyObject* o, float& out) {
    const PyNumberMethods* m = Py_TYPE(o)->tp_as_number;
    if (m == nullptr || (m->nb_float == nullptr && m->nb_index == nullptr)) {
        PyObject* f = PyObject_CallFunction(g_value, "Oi", o, 0);
        if (f == nullptr) return false;
        const double d = PyFloat_AsDouble(f);
        Py_DECREF(f);
        if (d == -1.0 && PyErr_Occurred()) return false;
        out = (float)d;
        return true;
    }
    const double d = PyFloat_AsDouble(o);
    if (d == -1.0 && PyErr_Occurred()) return false;
    out = (float)d;
    return true;
}

template <class T>
std::enable_if_t<std::is_integral_v<T>, bool> convert(PyObject* o, T& out) {
    if (!PyLong_Check(o)) {
        PyObject* i = PyIndex_Check(o) ? PyNumber_Index(o) : PyObject_CallFunction(g_value, "Oi", o, (int)sizeof(T));
        if (i == nullptr) return false;
        const bool ok = convert(i, out);
        Py_DECREF(i);
        return ok;
    }
    const unsigned long long v = PyLong_AsUnsignedLongLongMask(o);
    if (v == (unsigned long long)-1 && PyErr_Occurred()) return false;
    out = (T)v;
    return true;
}

template <class T>
bool convert(PyObject* o, T*& out) {
    if (o == Py_None) {
        out = nullptr;
        return true;
    }
    if (!PyLong_Check(o)) {
        PyObject* i = PyObject_CallOneArg(g_value, o);
        if (i == nullptr) return false;
        const bool ok = PyLong_Check(i) || i == Py_None ? convert(i, out) : (PyErr_SetString(PyExc_TypeError, "a device address is an integer"), false);
        Py_DECREF(i);
        return ok;
    }
    const unsigned long long v = PyLong_AsUnsignedLongLongMask(o);
    if (v == (unsigned long long)-1 && PyErr_Occurred()) return false;
    out = reinterpret_cast<T*>((uintptr_t)v);
    return true;
}

template <class Fn>
struct Launcher;

template <class... A>
struct Launcher<int (*)(A...)> {
    template <size_t... I>
    static int apply(void* fn, std::tuple<A...>& a, std::index_sequence<I...>) {
        return reinterpret_cast<int (*)(A...)>(fn)(std::get<I>(a)...);
    }
    template <size_t... I>
    static bool parse(PyObject* const* args, std::tuple<A...>& a, std::index_sequence<I...>) {
        return (... && convert(args[I], std::get<I>(a)));
    }
    static PyObject* call(PyObject* self, PyObject* const* args, Py_ssize_t n) {
        if (n != (Py_ssize_t)sizeof...(A)) {
            PyErr_Format(PyExc_TypeError, "this launcher takes %zd arguments (%zd given)", (Py_ssize_t)sizeof...(A), n);
            return nullptr;
        }
        std::tuple<A...> a;
        if (!parse(args, a, std::index_sequence_for<A...>{})) return nullptr;
        void* fn = PyCapsule_GetPointer(self, nullptr);
        int rc;
        Py_BEGIN_ALLOW_THREADS
        rc = apply(fn, a, std::index_sequence_for<A...>{});
        Py_END_ALLOW_THREADS
        if (rc != 0) {
            PyErr_Format(PyExc_RuntimeError, "HIP Error: %s", g_error_string ? g_error_string(rc) : "unknown");
            return nullptr;
        }
        Py_RETURN_NONE;
    }
};

#define CPMK_ENTRY(name) {#name, (PyCFunction)(void (*)(void))&Launcher<decltype(&name)>::call, METH_FASTCALL, "Launcher of include/cpmk.h."},
PyMethodDef g_launchers[] = {
    CPMK_ENTRY(cpmk_gemm_calc_scale)
    CPMK_ENTRY(cpmk_gemm_calc_scale_transpose)
    CPMK_ENTRY(cpmk_gemm_round)
    CPMK_ENTRY(cpmk_gemm_round_transpose)
    CPMK_ENTRY(cpmk_gemm_scale)
    CPMK_ENTRY(cpmk_gemm_scale_x)
    CPMK_ENTRY(cpmk_gemm_scale_y)
    CPMK_ENTRY(cpmk_gemm_int8)
    CPMK_ENTRY(cpmk_gemm_int8_scale)
    CPMK_ENTRY(cpmk_gemm_quantize)
    CPMK_ENTRY(cpmk_gemm_quantize_pair)
    CPMK_ENTRY(cpmk_gemm_quantize_cols)
    CPMK_ENTRY(cpmk_gemm_fp16)
    CPMK_ENTRY(cpmk_gemm_quantize_cols_ld)
    CPMK_ENTRY(cpmk_gemm_quantize_pair_ld)
    CPMK_ENTRY(cpmk_gemm_backward_round_scale_ld)
    CPMK_ENTRY(cpmk_gemm_int8_scale_one)
    CPMK_ENTRY(cpmk_transpose_i8_ld)
    CPMK_ENTRY(cpmk_gemm_int8_scale_sum)
    CPMK_ENTRY(cpmk_gemm_fp16_sum)
    CPMK_ENTRY(cpmk_gemm_quantize_cols_rows)
    CPMK_ENTRY(cpmk_gemm_backward_quantize_both)
    CPMK_ENTRY(cpmk_gemm_int8_scale_split)
    CPMK_ENTRY(cpmk_gemm_fp16_split)
    CPMK_ENTRY(cpmk_gemm_int8_scale_parts)
    CPMK_ENTRY(cpmk_gemm_fp16_parts)
    CPMK_ENTRY(cpmk_gemm_add_parts)
    CPMK_ENTRY(cpmk_gemv_fp16)
    CPMK_ENTRY(cpmk_gemv_fp16_transpose)
    CPMK_ENTRY(cpmk_gemv_broadcast_mat_fp16)
    CPMK_ENTRY(cpmk_embedding_forward)
    CPMK_ENTRY(cpmk_embedding_step)
    CPMK_ENTRY(cpmk_copy_data_to_kv)
    CPMK_ENTRY(cpmk_gemv_calc_scale)
    CPMK_ENTRY(cpmk_gemv_round)
    CPMK_ENTRY(cpmk_gemv_broadcast_mat_int8)
    CPMK_ENTRY(cpmk_layernorm_forward)
    CPMK_ENTRY(cpmk_layernorm_forward_noalloc)
    CPMK_ENTRY(cpmk_layernorm_step)
    CPMK_ENTRY(cpmk_layernorm_affine_forward)
    CPMK_ENTRY(cpmk_layernorm_affine_forward_stats)
    CPMK_ENTRY(cpmk_layernorm_affine_backward)
    CPMK_ENTRY(cpmk_softmax_forward)
    CPMK_ENTRY(cpmk_softmax_step_inplace)
    CPMK_ENTRY(cpmk_gelu_forward)
    CPMK_ENTRY(cpmk_position_embedding_init)
    CPMK_ENTRY(cpmk_position_embedding_forward)
    CPMK_ENTRY(cpmk_position_embedding_step)
    CPMK_ENTRY(cpmk_arith_ln_mul_add)
    CPMK_ENTRY(cpmk_arith_ln_mul)
    CPMK_ENTRY(cpmk_arith_element_add)
    CPMK_ENTRY(cpmk_mask)
    CPMK_ENTRY(cpmk_arith_global_scale)
    CPMK_ENTRY(cpmk_arith_element_mul)
    CPMK_ENTRY(cpmk_arith_batch_add_forward)
    CPMK_ENTRY(cpmk_arith_batch_add_backward)
    CPMK_ENTRY(cpmk_arith_ln_add)
    CPMK_ENTRY(cpmk_arith_ln_div)
    CPMK_ENTRY(cpmk_arith_ln_sub_div)
    CPMK_ENTRY(cpmk_arith_ln_mul_backward)
    CPMK_ENTRY(cpmk_arith_ln_add_backward)
    CPMK_ENTRY(cpmk_arith_batch_mul_add)
    CPMK_ENTRY(cpmk_arith_batch_mul)
    CPMK_ENTRY(cpmk_gelu_backward)
    CPMK_ENTRY(cpmk_softmax_backward)
    CPMK_ENTRY(cpmk_layernorm_forward_v)
    CPMK_ENTRY(cpmk_layernorm_forward_mv)
    CPMK_ENTRY(cpmk_layernorm_backward_v)
    CPMK_ENTRY(cpmk_layernorm_backward_mv)
    CPMK_ENTRY(cpmk_gemm_backward_round_scale)
    CPMK_ENTRY(cpmk_gemm_backward_scale_round)
    CPMK_ENTRY(cpmk_position_embedding_backward)
    CPMK_ENTRY(cpmk_embedding_backward_stage1)
    CPMK_ENTRY(cpmk_embedding_backward_stage2)
    CPMK_ENTRY(cpmk_embedding_order_ids)
    CPMK_ENTRY(cpmk_embedding_backward_rows)
    CPMK_ENTRY(cpmk_embedding_backward_prepare)
    CPMK_ENTRY(cpmk_transpose)
    CPMK_ENTRY(cpmk_transpose_i8)
    CPMK_ENTRY(cpmk_array_add)
    CPMK_ENTRY(cpmk_adjustify_logits)
    CPMK_ENTRY(cpmk_copy_extend_buffer)
    CPMK_ENTRY(cpmk_has_nan_inf)
    CPMK_ENTRY(cpmk_copy_pos_hidden)
    CPMK_ENTRY(cpmk_async_status)
    CPMK_ENTRY(cpmk_selftest_exchange_timeout)
};

// init(address of cpmk_error_string, callable object[, size] -> address or number)
PyObject* init(PyObject*, PyObject* args) {
    unsigned long long err;
    PyObject* value;
    if (!PyArg_ParseTuple(args, "KO", &err, &value)) return nullptr;
    g_error_string = reinterpret_cast<const char* (*)(int)>((uintptr_t)err);
    Py_INCREF(value);
    Py_XDECREF(g_value);
    g_value = value;
    Py_RETURN_NONE;
}

// bind(name, address) -> a callable for the launcher at that address
PyObject* bind(PyObject*, PyObject* args) {
    const char* name;
    unsigned long long address;
    if (!PyArg_ParseTuple(args, "sK", &name, &address)) return nullptr;
    for (PyMethodDef& d : g_launchers)
        if (std::strcmp(d.ml_name, name) == 0) {
            PyObject* self = PyCapsule_New(reinterpret_cast<void*>((uintptr_t)address), nullptr, nullptr);
            if (self == nullptr) return nullptr;
            PyObject* f = PyCFunction_NewEx(&d, self, nullptr);
            Py_DECREF(self);
            return f;
        }
    PyErr_Format(PyExc_KeyError, "no launcher named %s", name);
    return nullptr;
}

PyObject* names(PyObject*, PyObject*) {
    PyObject* l = PyList_New(0);
    if (l == nullptr) return nullptr;
    for (PyMethodDef& d : g_launchers) {
        PyObject* s = PyUnicode_FromString(d.ml_name);
        if (s == nullptr || PyList_Append(l, s) != 0) {
            Py_XDECREF(s);
            Py_DECREF(l);
            return nullptr;
        }
        Py_DECREF(s);
    }
    return l;
}

PyMethodDef g_methods[] = {
    {"init", init, METH_VARARGS, "init(address of cpmk_error_string, callable object[, size] -> address or number)"},
    {"bind", bind, METH_VARARGS, "bind(name, address) -> callable"},
    {"names", names, METH_NOARGS, "names of the launchers"},
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef g_module = {PyModuleDef_HEAD_INIT, "_cpmk_call", "Launcher calls of libcpmk_hip.so.", -1, g_methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__cpmk_call() { return PyModule_Create(&g_module); }
