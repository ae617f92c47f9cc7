// The operators of ops.py as CPython functions.  A small operator is host work: of the 6 to 7 us that a call took in Python
// over the C ABI some 2 were the launch (which the device needs as well, 2.3 us from one small kernel to the next); the
// rest went into allocating the results (torch.empty: 1.5 us each from Python, a third of it here), a Python call for
// every property of a tensor that is looked at, and the conversion of arguments.  us per call from Python, before ->
// here: gemm 6.3 -> 4.0, rms_norm 4.8 -> 3.7, its adjoint (two kernels) 10.6 -> 8.0, silu_gate 4.8 -> 3.7.
//
// Tensors come as torch hands them over; what an operator wants of them is checked as before (AssertionError), a status of
// the C ABI that is not 0 is raised by ffi.check.  The other entry points (FN) take pointers as integers or None and
// return the status.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/ATen.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <stdint.h>

#include <tuple>
#include <type_traits>
#include <utility>
#include <vector>

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

// ---------------------------------------------------------------- operators on tensors
PyObject *g_check = nullptr;                   // ffi.check

struct PyFailed {};                            // a Python exception is set
[[noreturn]] void fail(PyObject *type, const char *what)
{
    PyErr_SetString(type, what);
    throw PyFailed();
}
void require(bool ok, const char *what)
{
    if (!ok) fail(PyExc_AssertionError, what);
}

const at::Tensor &tensor(PyObject *o)
{
    if (!THPVariable_Check(o)) fail(PyExc_TypeError, "a tensor expected");
    return THPVariable_Unpack(o);
}
const at::Tensor &checked(const at::Tensor &t, at::ScalarType dtype)
{
    if (!(t.is_cuda() && t.is_contiguous() && t.scalar_type() == dtype)) {
        PyErr_Format(PyExc_AssertionError, "contiguous %s tensor on the GPU expected, got %s on %s%s", c10::toString(dtype),
                     c10::toString(t.scalar_type()), t.device().str().c_str(), t.is_contiguous() ? "" : ", strided");
        throw PyFailed();
    }
    return t;
}
const at::Tensor &f16(PyObject *o) { return checked(tensor(o), at::kHalf); }
const at::Tensor &f32(PyObject *o) { return checked(tensor(o), at::kFloat); }

at::Tensor empty(at::IntArrayRef sizes, const at::Tensor &like, at::ScalarType dtype)
{
    return at::empty(sizes, at::TensorOptions().dtype(dtype).device(like.device()));
}
at::Tensor new_like(const at::Tensor &t) { return empty(t.sizes(), t, t.scalar_type()); }

void *stream() { return c10::hip::getCurrentHIPStream().stream(); }

template <class T>
T number(PyObject *o)
{
    T v;
    if (!convert(o, &v)) throw PyFailed();
    return v;
}
int truth(PyObject *o)
{
    const int v = PyObject_IsTrue(o);
    if (v < 0) throw PyFailed();
    return v;
}

// the call itself runs without the interpreter lock (taken again also where it throws: a tensor without storage does); a
// status that is not 0 becomes the exception ffi.check raises
struct Unlocked {
    PyThreadState *st = PyEval_SaveThread();
    ~Unlocked() { PyEval_RestoreThread(st); }
};
template <class F>
auto unlocked(F f)
{
    const Unlocked u;
    return f();
}
void raise_status(int rc)
{
    PyObject *r = PyObject_CallFunction(g_check, "i", rc);
    Py_XDECREF(r);
    if (r) PyErr_SetString(PyExc_RuntimeError, "status of an entry point");
    throw PyFailed();
}
template <class F>
void run(F f)
{
    const int rc = unlocked(f);
    if (rc) raise_status(rc);
}

PyObject *wrap(at::Tensor t)
{
    PyObject *o = THPVariable_Wrap(std::move(t));
    if (!o) throw PyFailed();
    return o;
}
// a result tensor: the argument it accumulates into (the same object is returned) or a new one
struct Result {
    at::Tensor t;
    PyObject *arg;
    int acc() const { return arg != nullptr; }
    void *ptr() const { return t.data_ptr(); }
    PyObject *take() const
    {
        if (!arg) return wrap(t);
        Py_INCREF(arg);
        return arg;
    }
};
Result result(PyObject *acc, const at::Tensor &like)
{
    if (acc == Py_None) return {new_like(like), nullptr};
    return {f16(acc), acc};
}
PyObject *take2(const Result &a, const Result &b)
{
    PyObject *x = a.take(), *y = b.take(), *r = PyTuple_New(2);
    PyTuple_SET_ITEM(r, 0, x);
    PyTuple_SET_ITEM(r, 1, y);
    return r;
}

// The tensors of a list or tuple, held: another thread may change the list while a call runs without the interpreter lock.
struct Tensors {
    std::vector<at::Tensor> t;
    explicit Tensors(PyObject *o)
    {
        PyObject *seq = PySequence_Fast(o, "a sequence of tensors expected");
        if (!seq) throw PyFailed();
        const Py_ssize_t n = PySequence_Fast_GET_SIZE(seq);
        t.reserve(n);
        for (Py_ssize_t i = 0; i < n; i++) {
            PyObject *e = PySequence_Fast_GET_ITEM(seq, i);
            if (!THPVariable_Check(e)) {
                Py_DECREF(seq);
                fail(PyExc_TypeError, "a tensor expected");
            }
            t.push_back(THPVariable_Unpack(e));
        }
        Py_DECREF(seq);
    }
    size_t size() const { return t.size(); }
    const at::Tensor &operator[](size_t i) const { return t[i]; }
    std::vector<void *> pointers() const
    {
        std::vector<void *> p(t.size());
        for (size_t i = 0; i < t.size(); i++) p[i] = t[i].data_ptr();
        return p;
    }
};

void gemm_into(int ta, int tb, int64_t M, int64_t N, int64_t K, float alpha, const at::Tensor &a, const at::Tensor &b, float beta,
               const at::Tensor &out)
{
    void *st = stream();
    size_t need = 0;
    auto call = [&](void *ws, size_t bytes) {
        return cacti_hip_gemm_f16_ws(ta, tb, M, N, K, alpha, a.data_ptr(), a.stride(0), b.data_ptr(), b.stride(0), beta, out.data_ptr(),
                                     out.stride(0), ws, bytes, &need, st);
    };
    run([&] { return call(nullptr, 0); });
    if (need > 0) {                              // not launched: the product wants a workspace
        const at::Tensor ws = empty({(int64_t)need}, a, at::kByte);
        const size_t bytes = need;
        run([&] { return call(ws.data_ptr(), bytes); });
    }
}

struct Shape {
    int64_t M, N, K;
};
Shape product_shape(const at::Tensor &a, const at::Tensor &b, int ta, int tb)
{
    require(a.dim() == 2 && b.dim() == 2 && a.stride(1) == 1 && b.stride(1) == 1, "gemm: matrices with contiguous rows expected");
    const Shape s = {a.size(ta ? 1 : 0), b.size(tb ? 0 : 1), a.size(ta ? 0 : 1)};
    require(s.K == b.size(tb ? 1 : 0), "gemm: inner dimensions differ");
    return s;
}

// (a, b, ta, tb, alpha, beta, out)
PyObject *gemm(PyObject *const *v)
{
    const at::Tensor &a = tensor(v[0]), &b = tensor(v[1]);
    const int ta = truth(v[2]), tb = truth(v[3]);
    const float alpha = number<float>(v[4]), beta = number<float>(v[5]);
    const Shape s = product_shape(a, b, ta, tb);
    if (v[6] == Py_None) {
        require(beta == 0.f, "gemm: beta without out");
        at::Tensor out = empty({s.M, s.N}, a, at::kHalf);
        gemm_into(ta, tb, s.M, s.N, s.K, alpha, a, b, beta, out);
        return wrap(std::move(out));
    }
    const at::Tensor &out = tensor(v[6]);
    require(out.dim() == 2 && out.size(0) == s.M && out.size(1) == s.N && out.stride(1) == 1, "gemm: shape of out");
    gemm_into(ta, tb, s.M, s.N, s.K, alpha, a, b, beta, out);
    Py_INCREF(v[6]);
    return v[6];
}

// (As, Bs, outs, ta, tb, alpha, beta)
PyObject *gemm_batched(PyObject *const *v)
{
    const Tensors as(v[0]), bs(v[1]), outs(v[2]);
    const int ta = truth(v[3]), tb = truth(v[4]);
    const float alpha = number<float>(v[5]), beta = number<float>(v[6]);
    const size_t n = as.size();
    require(n > 0 && bs.size() == n && outs.size() == n, "gemm_batched: lists of one length expected");
    const at::Tensor &a = as[0], &b = bs[0], &o = outs[0];
    const Shape s = product_shape(a, b, ta, tb);
    const std::vector<void *> pa = as.pointers(), pb = bs.pointers(), po = outs.pointers();
    bool aligned = true;
    for (int64_t x : {a.size(1), b.size(1), s.N, a.stride(0), b.stride(0), o.stride(0)}) aligned = aligned && x % 8 == 0;
    for (const std::vector<void *> *v : {&pa, &pb, &po})
        for (void *p : *v) aligned = aligned && reinterpret_cast<uintptr_t>(p) % 16 == 0;
    if (!aligned) {
        // operands whose rows are not all 16-byte aligned run one after another; each may want a workspace
        for (size_t z = 0; z < n; z++) gemm_into(ta, tb, s.M, s.N, s.K, alpha, as[z], bs[z], beta, outs[z]);
        Py_RETURN_NONE;
    }
    void *st = stream();
    run([&] {
        return cacti_hip_gemm_f16_batched(ta, tb, (int64_t)n, s.M, s.N, s.K, alpha, pa.data(), a.stride(0), pb.data(), b.stride(0), beta,
                                          po.data(), o.stride(0), st);
    });
    Py_RETURN_NONE;
}

// (q, k, v, alpha)
PyObject *attention_fwd(PyObject *const *v)
{
    const at::Tensor &q = f16(v[0]), &k = f16(v[1]), &w = f16(v[2]);
    const float alpha = number<float>(v[3]);
    require(q.dim() == 3, "attention: [S, H, Dh] expected");
    const int64_t S = q.size(0), H = q.size(1), Dh = q.size(2);
    const Result o = {new_like(q), nullptr};
    const Result stats = {empty({(int64_t)(cacti_hip_attention_stats_bytes(S, H) / 4)}, q, at::kFloat), nullptr};
    void *st = stream();
    run([&] { return cacti_hip_attention_fwd(S, H, Dh, alpha, q.data_ptr(), k.data_ptr(), w.data_ptr(), H * Dh, o.ptr(), stats.ptr(), st); });
    return take2(o, stats);
}

// (q, k, v, dO, stats, alpha, acc, o)
PyObject *attention_bwd(PyObject *const *v)
{
    const at::Tensor &q = f16(v[0]), &k = f16(v[1]), &w = f16(v[2]), &dO = f16(v[3]), &stats = tensor(v[4]);
    const float alpha = number<float>(v[5]);
    const void *o = v[7] == Py_None ? nullptr : f16(v[7]).data_ptr();
    require(q.dim() == 3, "attention: [S, H, Dh] expected");
    const int64_t S = q.size(0), H = q.size(1), Dh = q.size(2);
    const bool into = v[6] != Py_None;
    auto given = [&]() {
        const Tensors acc(v[6]);
        require(acc.size() == 3, "attention_bwd: acc = (dq, dk, dv)");
        return acc.t;
    };
    const std::vector<at::Tensor> d = into ? given() : std::vector<at::Tensor>{new_like(q), new_like(q), new_like(q)};
    const size_t bytes = cacti_hip_attention_bwd_workspace_used(S, H, Dh, H * Dh);
    const at::Tensor ws = empty({(int64_t)bytes}, q, at::kByte);
    void *st = stream();
    run([&] {
        return cacti_hip_attention_bwd(S, H, Dh, alpha, q.data_ptr(), k.data_ptr(), w.data_ptr(), o, dO.data_ptr(), H * Dh, stats.data_ptr(),
                                       d[0].data_ptr(), into, d[1].data_ptr(), into, d[2].data_ptr(), into, ws.data_ptr(), bytes, st);
    });
    PyObject *r = PyTuple_New(3);
    if (!r) throw PyFailed();
    for (int i = 0; i < 3; i++) PyTuple_SET_ITEM(r, i, THPVariable_Wrap(d[i]));     // (a tensor that was given: its own object)
    return r;
}

// (x, w, eps)
PyObject *rms_norm_fwd(PyObject *const *v)
{
    const at::Tensor &x = f16(v[0]), &w = f16(v[1]);
    const float eps = number<float>(v[2]);
    require(x.dim() == 2, "rms_norm: [N, D] expected");
    at::Tensor y = new_like(x);
    void *st = stream();
    run([&] { return cacti_hip_rms_norm_fwd(x.size(0), x.size(1), x.data_ptr(), w.data_ptr(), eps, y.data_ptr(), st); });
    return wrap(std::move(y));
}

// (a, b, w, eps)
PyObject *add_rms_norm_fwd(PyObject *const *v)
{
    const at::Tensor &a = f16(v[0]), &b = f16(v[1]), &w = f16(v[2]);
    const float eps = number<float>(v[3]);
    require(a.dim() == 2, "add_rms_norm: [N, D] expected");
    const Result s = {new_like(a), nullptr}, y = {new_like(a), nullptr};
    void *st = stream();
    run([&] {
        return cacti_hip_add_rms_norm_fwd(a.size(0), a.size(1), a.data_ptr(), b.data_ptr(), w.data_ptr(), eps, s.ptr(), y.ptr(), st);
    });
    return take2(s, y);
}

// (x, w, eps, dy, dx_acc, dw_acc)
PyObject *rms_norm_bwd(PyObject *const *v)
{
    const at::Tensor &x = f16(v[0]), &w = f16(v[1]), &dy = f16(v[3]);
    const float eps = number<float>(v[2]);
    require(x.dim() == 2, "rms_norm: [N, D] expected");
    const Result dx = result(v[4], x), dw = result(v[5], w);
    const size_t bytes = cacti_hip_rms_norm_bwd_workspace(x.size(0), x.size(1));
    const at::Tensor ws = empty({(int64_t)bytes}, x, at::kByte);
    void *st = stream();
    run([&] {
        return cacti_hip_rms_norm_bwd(x.size(0), x.size(1), x.data_ptr(), w.data_ptr(), eps, dy.data_ptr(), dx.ptr(), dx.acc(), dw.ptr(),
                                      dw.acc(), ws.data_ptr(), bytes, st);
    });
    return take2(dx, dw);
}

// (x, cos, sin)
PyObject *rope_fwd(PyObject *const *v)
{
    const at::Tensor &x = f16(v[0]), &c = f16(v[1]), &s = f16(v[2]);
    require(x.dim() == 3, "rope: [S, H, Dh] expected");
    at::Tensor y = new_like(x);
    void *st = stream();
    run([&] {
        return cacti_hip_rope_fwd(x.size(0), x.size(1), x.size(2), x.data_ptr(), c.data_ptr(), s.data_ptr(), y.data_ptr(), st);
    });
    return wrap(std::move(y));
}

// (dy, cos, sin, dx_acc)
PyObject *rope_bwd(PyObject *const *v)
{
    const at::Tensor &dy = f16(v[0]), &c = f16(v[1]), &s = f16(v[2]);
    require(dy.dim() == 3, "rope: [S, H, Dh] expected");
    const Result dx = result(v[3], dy);
    void *st = stream();
    run([&] {
        return cacti_hip_rope_bwd(dy.size(0), dy.size(1), dy.size(2), dy.data_ptr(), c.data_ptr(), s.data_ptr(), dx.ptr(), dx.acc(), st);
    });
    return dx.take();
}

// (g, u)
PyObject *silu_gate_fwd(PyObject *const *v)
{
    const at::Tensor &g = f16(v[0]), &u = f16(v[1]);
    at::Tensor h = new_like(g);
    void *st = stream();
    run([&] { return cacti_hip_silu_gate_fwd(g.numel(), g.data_ptr(), u.data_ptr(), h.data_ptr(), st); });
    return wrap(std::move(h));
}

// (g, u, dh, dg_acc, du_acc)
PyObject *silu_gate_bwd(PyObject *const *v)
{
    const at::Tensor &g = f16(v[0]), &u = f16(v[1]), &dh = f16(v[2]);
    const Result dg = result(v[3], g), du = result(v[4], u);
    void *st = stream();
    run([&] {
        return cacti_hip_silu_gate_bwd(g.numel(), g.data_ptr(), u.data_ptr(), dh.data_ptr(), dg.ptr(), dg.acc(), du.ptr(), du.acc(), st);
    });
    return take2(dg, du);
}

// (a, b, out)
PyObject *add_f16(PyObject *const *v)
{
    const at::Tensor &a = tensor(v[0]), &b = tensor(v[1]);
    // (element for element in memory order: the result has a's strides, whatever they are)
    const Result out = v[2] == Py_None ? Result{at::empty_like(a), nullptr} : Result{tensor(v[2]), v[2]};
    void *st = stream();
    run([&] { return cacti_hip_add_f16(a.numel(), a.data_ptr(), b.data_ptr(), out.ptr(), st); });
    return out.take();
}

// (logit, tok, scale, acc)
PyObject *softmax_ce_bwd(PyObject *const *v)
{
    const at::Tensor &logit = f16(v[0]), &tok = tensor(v[1]), &scale = f32(v[2]);
    require(logit.dim() == 2, "softmax_ce: [N, V] expected");
    const Result d = result(v[3], logit);
    void *st = stream();
    run([&] {
        return cacti_hip_softmax_ce_bwd(logit.size(0), logit.size(1), logit.data_ptr(), tok.data_ptr(), scale.data_ptr(), d.ptr(), d.acc(), st);
    });
    return d.take();
}

// (xs)
PyObject *digests(PyObject *const *v)
{
    const Tensors xs(v[0]);
    std::vector<int64_t> ns(xs.size());
    for (size_t i = 0; i < xs.size(); i++) ns[i] = checked(xs[i], at::kHalf).numel();
    require(xs.size() > 0, "digests: no tensors");
    const at::Tensor out = empty({(int64_t)xs.size(), 257}, xs[0], at::kLong);
    const std::vector<void *> p = xs.pointers();
    void *st = stream();
    run([&] { return cacti_hip_digests_f16_batch((int)p.size(), p.data(), ns.data(), out.data_ptr(), nullptr, st); });
    return take2({out.narrow(1, 0, 256), nullptr}, {out.select(1, 256), nullptr});
}

// (grads, avgs, avg2s, masters, params, scalars)
PyObject *adamw32_step(PyObject *const *v)
{
    const Tensors g(v[0]), a(v[1]), b(v[2]), w(v[3]), p(v[4]);
    const size_t n = g.size();
    require(a.size() == n && b.size() == n && w.size() == n && p.size() == n, "adamw32_step: lists of one length expected");
    float sc[7];
    PyObject *seq = PySequence_Fast(v[5], "adamw32_step: seven scalars expected");
    if (!seq) throw PyFailed();
    bool ok = PySequence_Fast_GET_SIZE(seq) == 7;
    for (int i = 0; ok && i < 7; i++) ok = convert(PySequence_Fast_GET_ITEM(seq, i), &sc[i]);
    Py_DECREF(seq);
    if (PyErr_Occurred()) throw PyFailed();
    require(ok, "adamw32_step: seven scalars expected");
    std::vector<int64_t> ns(n);
    for (size_t i = 0; i < n; i++) {
        ns[i] = checked(g[i], at::kHalf).numel();
        require(checked(a[i], at::kFloat).numel() == ns[i] && checked(b[i], at::kFloat).numel() == ns[i] &&
                    checked(w[i], at::kFloat).numel() == ns[i] && checked(p[i], at::kHalf).numel() == ns[i],
                "adamw32_step: tensors of one size expected");
    }
    if (n == 0) Py_RETURN_NONE;
    const std::vector<void *> pg = g.pointers(), pa = a.pointers(), pb = b.pointers(), pw = w.pointers(), pp = p.pointers();
    void *st = stream();
    run([&] {
        return cacti_hip_adamw32_step_f16_batch((int)n, pg.data(), pa.data(), pb.data(), pw.data(), pp.data(), ns.data(), sc, nullptr, st);
    });
    Py_RETURN_NONE;
}

// (iter_nr, grad_scale, lr, wd, a1, a2, eps)
PyObject *adamw32_scalars(PyObject *const *v)
{
    float out[7];
    const int iter_nr = number<int>(v[0]);
    float in[6];
    for (int i = 0; i < 6; i++) in[i] = number<float>(v[1 + i]);
    const int rc = cacti_adamw32_scalars(iter_nr, in[0], in[1], in[2], in[3], in[4], in[5], out);
    if (rc) raise_status(rc);
    PyObject *r = PyList_New(7);
    for (int i = 0; i < 7; i++) PyList_SET_ITEM(r, i, PyFloat_FromDouble(out[i]));
    return r;
}

// an operator of N arguments as a CPython function
template <PyObject *(*F)(PyObject *const *), int N>
PyObject *entry(PyObject *, PyObject *const *args, Py_ssize_t n)
{
    HANDLE_TH_ERRORS
    if (n != N) {
        PyErr_Format(PyExc_TypeError, "%d arguments expected, %d given", N, (int)n);
        return nullptr;
    }
    try {
        return F(args);
    } catch (const PyFailed &) {
        return nullptr;
    }
    END_HANDLE_TH_ERRORS
}

PyObject *set_check(PyObject *, PyObject *f)
{
    Py_INCREF(f);
    Py_XSETREF(g_check, f);
    Py_RETURN_NONE;
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

#define OP(name, n) {#name, (PyCFunction)(void (*)(void))(&entry<name, n>), METH_FASTCALL, nullptr}

PyMethodDef methods[] = {
    {"set_check", set_check, METH_O, nullptr},
    OP(gemm, 7),
    OP(gemm_batched, 7),
    OP(attention_fwd, 4),
    OP(attention_bwd, 8),
    OP(rms_norm_fwd, 3),
    OP(add_rms_norm_fwd, 4),
    OP(rms_norm_bwd, 6),
    OP(rope_fwd, 3),
    OP(rope_bwd, 4),
    OP(silu_gate_fwd, 2),
    OP(silu_gate_bwd, 5),
    OP(add_f16, 3),
    OP(softmax_ce_bwd, 4),
    OP(digests, 1),
    OP(adamw32_step, 6),
    OP(adamw32_scalars, 7),
    FN(gemm_f16_strided_batched_tri),
    FN(accumulate_1d_f32),
    FN(accumulate_1d_f16),
    FN(accumulate_1d_u16),
    FN(rope_tables),
    FN(causal_softmax_fwd),
    FN(causal_softmax_bwd),
    FN(softmax_ce_fwd),
    FN(embed_fwd),
    FN(embed_bwd),
    FN(nan_count_f16),
    FN(abs_log2_hist8_f16),
    FN(online_average_scale_f16_f32),
    FN(online_average_square_scale_f16_f32),
    FN(online_adamw_update_f32),
    FN(cast_f32_f16),
    FN(cast_f16_f32),
    FN(raw_cast_bf16_f16),
    FN(raw_cast_bf16_f32),
    FN(raw_cast_f32_bf16),
    FN(raw_cast_f16_bf16),
    {"read_i32", (PyCFunction)(void (*)(void))read_i32, METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr},
};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_fast", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__fast(void) { return PyModule_Create(&module); }
