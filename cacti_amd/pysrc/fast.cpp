// Operator entry points of the C ABI as CPython functions.  A ctypes call converts every argument through a Python-level
// type object, 1 us for 7 arguments and 2 us for 14, which on a small operator is as much as the launch; here an argument
// costs some 10 ns.  Pointers are integers or None; every function returns the entry point's status.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <stdint.h>

#include <tuple>
#include <type_traits>
#include <utility>

#include "../../include/cacti_gpu_hip_ffi.h"

namespace {

template <class T>
bool convert(PyObject *o, T *out)
{
    if constexpr (std::is_pointer_v<T>) {
        *out = o == Py_None ? nullptr : (T)PyLong_AsVoidPtr(o);
        return *out || o == Py_None || !PyErr_Occurred();
    } else if constexpr (std::is_floating_point_v<T>) {
        *out = (T)PyFloat_AsDouble(o);
        return !PyErr_Occurred();
    } else {
        const long long v = PyLong_AsLongLong(o);
        if (v == -1 && PyErr_Occurred()) return false;
        *out = (T)v;
        if ((long long)*out != v) {
            PyErr_SetString(PyExc_OverflowError, "argument does not fit the C type");
            return false;
        }
        return true;
    }
}

// f with the arguments of a function of type R (*)(A...)
template <class F, class R, class... A, size_t... I>
PyObject *apply(const F &f, R (*)(A...), PyObject *const *args, Py_ssize_t n, std::index_sequence<I...>)
{
    if (n != (Py_ssize_t)sizeof...(A)) {
        PyErr_Format(PyExc_TypeError, "%d arguments expected, %d given", (int)sizeof...(A), (int)n);
        return nullptr;
    }
    std::tuple<A...> v;
    if (!(convert(args[I], &std::get<I>(v)) && ...)) return nullptr;
    R r;
    Py_BEGIN_ALLOW_THREADS
    r = f(std::get<I>(v)...);
    Py_END_ALLOW_THREADS
    if constexpr (std::is_signed_v<R>) return PyLong_FromLongLong((long long)r);
    else return PyLong_FromUnsignedLongLong((unsigned long long)r);
}

template <class R, class... A>
PyObject *apply(R (*fn)(A...), PyObject *const *args, Py_ssize_t n)
{
    return apply(fn, fn, args, n, std::index_sequence_for<A...>{});
}

// cacti_hip_gemm_f16_ws without ws_need: 0 done, > 0 the bytes of workspace it wants, < 0 failed with status -r - 1000000
PyObject *gemm_f16_ws(PyObject *, PyObject *const *args, Py_ssize_t n)
{
    typedef int64_t (*Type)(int, int, int64_t, int64_t, int64_t, float, const void *, int64_t, const void *, int64_t, float, void *,
                            int64_t, void *, size_t, void *);
    auto f = [](int ta, int tb, int64_t M, int64_t N, int64_t K, float alpha, const void *A, int64_t lda, const void *B, int64_t ldb,
                float beta, void *C, int64_t ldc, void *ws, size_t ws_bytes, void *stream) -> int64_t {
        size_t need = 0;
        const int rc = cacti_hip_gemm_f16_ws(ta, tb, M, N, K, alpha, A, lda, B, ldb, beta, C, ldc, ws, ws_bytes, &need, stream);
        return rc ? -1000000 - (int64_t)rc : need > ws_bytes ? (int64_t)need : 0;
    };
    return apply(f, Type(nullptr), args, n, std::make_index_sequence<16>{});
}

// cacti_hip_read_i32 (device pointer, stream): (status, value)
PyObject *read_i32(PyObject *, PyObject *const *args, Py_ssize_t n)
{
    const void *p = nullptr;
    void *st = nullptr;
    if (n != 2 || !convert(args[0], &p) || !convert(args[1], &st)) {
        if (!PyErr_Occurred()) PyErr_SetString(PyExc_TypeError, "2 arguments expected");
        return nullptr;
    }
    int32_t v = 0;
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = cacti_hip_read_i32(p, &v, st);
    Py_END_ALLOW_THREADS
    return Py_BuildValue("(ii)", rc, (int)v);
}

#define FN(name)                                                                                      \
    {#name, (PyCFunction)(void (*)(void))(+[](PyObject *, PyObject *const *args, Py_ssize_t n) {       \
         return apply(&cacti_hip_##name, args, n);                                                    \
     }),                                                                                              \
     METH_FASTCALL, nullptr}

PyMethodDef methods[] = {
    {"gemm_f16_ws", (PyCFunction)(void (*)(void))gemm_f16_ws, METH_FASTCALL, nullptr},
    FN(gemm_f16_strided_batched_tri),
    FN(accumulate_1d_f32),
    FN(accumulate_1d_f16),
    FN(accumulate_1d_u16),
    FN(rms_norm_fwd),
    FN(add_rms_norm_fwd),
    FN(rms_norm_bwd_workspace),
    FN(rms_norm_bwd),
    FN(rope_tables),
    FN(rope_fwd),
    FN(rope_bwd),
    FN(silu_gate_fwd),
    FN(silu_gate_bwd),
    FN(causal_softmax_fwd),
    FN(causal_softmax_bwd),
    FN(attention_stats_bytes),
    FN(attention_fwd),
    FN(attention_bwd_workspace),
    FN(attention_bwd),
    FN(softmax_ce_fwd),
    FN(softmax_ce_bwd),
    FN(embed_fwd),
    FN(embed_bwd),
    FN(add_f16),
    FN(nan_count_f16),
    FN(abs_log2_hist8_f16),
    FN(digests_scratch_bytes),
    FN(online_average_scale_f16_f32),
    FN(online_average_square_scale_f16_f32),
    FN(online_adamw_update_f32),
    FN(cast_f32_f16),
    FN(cast_f16_f32),
    FN(raw_cast_bf16_f16),
    FN(raw_cast_bf16_f32),
    FN(raw_cast_f32_bf16),
    FN(raw_cast_f16_bf16),
    FN(adamw32_scratch_bytes),
    {"read_i32", (PyCFunction)(void (*)(void))read_i32, METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr},
};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_fast", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__fast(void) { return PyModule_Create(&module); }
