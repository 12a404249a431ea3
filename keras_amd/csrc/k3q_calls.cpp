// Python module _k3q_calls: the entry points of include/k3q.h as built-in functions of integers, floats and None.
//
// A layer call at decode sizes is 9 to 12 us of Python around 5 to 9 us of kernel, and 3 us of that went into ctypes, which
// boxes every pointer and converts a dozen arguments through descriptors (16 rows of 4096 x 4096 int8: 3.1 us a call, 0.4
// here).  The conversions here are chosen from the declared types at compile time.  Entry points that take pointers to
// structures stay with ctypes, as does every use of the library outside the package's own hot calls.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <limits.h>
#include <stdint.h>

#include <tuple>
#include <utility>

#include "../../include/k3q.h"

namespace {

bool convert(PyObject* o, int64_t* v) {
    const long long r = PyLong_AsLongLong(o);
    if (r == -1 && PyErr_Occurred()) return false;
    *v = r;
    return true;
}
bool convert(PyObject* o, int* v) {
    const long r = PyLong_AsLong(o);
    if (r == -1 && PyErr_Occurred()) return false;
    if (r > INT_MAX || r < INT_MIN) {
        PyErr_SetString(PyExc_OverflowError, "argument does not fit an int");
        return false;
    }
    *v = (int)r;
    return true;
}
bool convert(PyObject* o, float* v) {
    const double r = PyFloat_AsDouble(o);
    if (r == -1.0 && PyErr_Occurred()) return false;
    *v = (float)r;
    return true;
}
template <class T>
bool convert(PyObject* o, T** v) {  // an address, or None
    if (o == Py_None) {
        *v = nullptr;
        return true;
    }
    void* r = PyLong_AsVoidPtr(o);
    if (!r && PyErr_Occurred()) return false;
    *v = (T*)r;
    return true;
}

template <auto kFn>
struct Entry;
template <class R, class... A, R (*kFn)(A...)>
struct Entry<kFn> {
    template <size_t... kI>
    static PyObject* run(PyObject* const* args, std::index_sequence<kI...>) {
        std::tuple<A...> v;
        if (!(convert(args[kI], &std::get<kI>(v)) && ...)) return nullptr;
        R r;
        Py_BEGIN_ALLOW_THREADS;
        r = kFn(std::get<kI>(v)...);
        Py_END_ALLOW_THREADS;
        return PyLong_FromLongLong((long long)r);
    }
    static PyObject* call(PyObject*, PyObject* const* args, Py_ssize_t n) {
        if (n != (Py_ssize_t)sizeof...(A)) {
            PyErr_Format(PyExc_TypeError, "expected %zd arguments, got %zd", (Py_ssize_t)sizeof...(A), n);
            return nullptr;
        }
        return run(args, std::index_sequence_for<A...>{});
    }
};

#define K3Q_ENTRY(name) {#name, (PyCFunction)(void (*)(void))Entry<&name>::call, METH_FASTCALL, nullptr}

PyMethodDef methods[] = {
    K3Q_ENTRY(k3q_version),
    K3Q_ENTRY(k3q_absmax_quantize),
    K3Q_ENTRY(k3q_weight_absmax_quantize),
    K3Q_ENTRY(k3q_weight_quantize_grouped),
    K3Q_ENTRY(k3q_weight_quantize_grouped_int4),
    K3Q_ENTRY(k3q_pack_int4),
    K3Q_ENTRY(k3q_unpack_int4),
    K3Q_ENTRY(k3q_gemm_i8_workspace_bytes),
    K3Q_ENTRY(k3q_gemm_i8_split_bytes),
    K3Q_ENTRY(k3q_prepack_kernel_i8),
    K3Q_ENTRY(k3q_gemm_i8),
    K3Q_ENTRY(k3q_gemm_i8_addend),
    K3Q_ENTRY(k3q_gemm_w8_workspace_bytes),
    K3Q_ENTRY(k3q_gemm_w8),
    K3Q_ENTRY(k3q_gemm_wbf16_workspace_bytes),
    K3Q_ENTRY(k3q_gemm_wbf16),
    K3Q_ENTRY(k3q_gemv_w4_workspace_bytes),
    K3Q_ENTRY(k3q_gemv_w4),
    K3Q_ENTRY(k3q_gemv_w4_counters_bytes),
    K3Q_ENTRY(k3q_gemv_w4_fused),
    K3Q_ENTRY(k3q_gemv_w4_addend),
    K3Q_ENTRY(k3q_gemv_w4_static_max_bytes),
    K3Q_ENTRY(k3q_gemv_w4_static),
    K3Q_ENTRY(k3q_w4s_shadow_bytes),
    K3Q_ENTRY(k3q_w4s_params_bytes),
    K3Q_ENTRY(k3q_w4s_pack),
    K3Q_ENTRY(k3q_w4s_pack_params),
    K3Q_ENTRY(k3q_gemv_w4s_supported),
    K3Q_ENTRY(k3q_gemv_w4s),
    K3Q_ENTRY(k3q_w4s_rows_params_bytes),
    K3Q_ENTRY(k3q_w4s_rows_pack_params),
    K3Q_ENTRY(k3q_gemv_w4s_rows_launches),
    K3Q_ENTRY(k3q_gemv_w4s_rows),
    K3Q_ENTRY(k3q_gemv_w4s_rows_plain_launches),
    K3Q_ENTRY(k3q_gemv_w4s_rows_plain),
    K3Q_ENTRY(k3q_w4_kmajor_pack),
    K3Q_ENTRY(k3q_gemm_w4_rows_workspace_bytes),
    K3Q_ENTRY(k3q_gemm_w4_rows),
    K3Q_ENTRY(k3q_gemm_w4_kmajor_workspace_bytes),
    K3Q_ENTRY(k3q_gemm_w4_kmajor),
    K3Q_ENTRY(k3q_gemm_w4_strip),
    K3Q_ENTRY(k3q_gemv_w4_nk),
    K3Q_ENTRY(k3q_embedding_lookup),
    K3Q_ENTRY(k3q_w8s_shadow_bytes),
    K3Q_ENTRY(k3q_w8s_pack),
    K3Q_ENTRY(k3q_dense_i8_w8s_supported),
    K3Q_ENTRY(k3q_dense_i8_w8s),
    K3Q_ENTRY(k3q_gemm_i8_w8s_supported),
    K3Q_ENTRY(k3q_gemm_i8_w8s),
    K3Q_ENTRY(k3q_dense_i8_workspace_bytes),
    K3Q_ENTRY(k3q_dense_i8),
    K3Q_ENTRY(k3q_decode_attention),
    K3Q_ENTRY(k3q_rope_cache),
    K3Q_ENTRY(k3q_prompt_attention),
    K3Q_ENTRY(k3q_rmsnorm),
    K3Q_ENTRY(k3q_silu_mul),
    {nullptr, nullptr, 0, nullptr},
};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_k3q_calls", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__k3q_calls(void) {
    PyObject* m = PyModule_Create(&module);
    if (m && PyModule_AddStringConstant(m, "header_digest", K3Q_HEADER_DIGEST) < 0) {
        Py_DECREF(m);
        return nullptr;
    }
    return m;
}
