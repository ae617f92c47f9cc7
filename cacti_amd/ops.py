"""Operator-level Python mirror of the thunks on cacti's LLaMA backward path.

Each function is one `ThunkImpl::apply` (or `accumulate` when an `*_acc` tensor is
given) in the reference's terms (src/thunk/mod.rs:347-351), executed by the HIP kernels
behind the C ABI.  torch is used only to own device memory and name the stream; every
computation goes through libcacti_gpu_hip_ffi.so and fails if it is not built.
"""
import torch

from . import ffi

F16 = torch.float16
F32 = torch.float32

# A small operator is host work (8 us of it in Python against some 3 us on the device), so the operators of the model's path
# are CPython functions that take the tensors themselves (ffi.fast, pysrc/fast.cpp); the others reach the C ABI through it
# with pointers and a stream that is read without building a torch.cuda.Stream (2.7 us).
_raw_stream = getattr(torch._C, "_cuda_getCurrentRawStream", None)
_current_device = getattr(torch._C, "_cuda_getDevice", None)


def _stream():
    return _raw_stream(_current_device()) if _raw_stream else torch.cuda.current_stream().cuda_stream


class _Calls:
    """The library's entry points without their prefix, raising on a status that is not 0."""

    def __getattr__(self, name):
        f = getattr(ffi.fast(), name)

        def call(*args):
            rc = f(*args)
            if rc:
                ffi.check(rc)

        setattr(self, name, call)
        return call


class _Operators:
    """The operators of pysrc/fast.cpp."""

    def __getattr__(self, name):
        f = getattr(ffi.fast(), name)
        setattr(self, name, f)
        return f


_do = _Calls()
_op = _Operators()


def _p(t):
    return None if t is None else t.data_ptr()


def _chk(t, dtype=F16):
    assert t.is_cuda and t.is_contiguous() and t.dtype is dtype, (t.dtype, t.device, t.shape)
    return t


def selftest_wave_reduce():
    out = torch.zeros(4, dtype=torch.float32, device="cuda")
    ffi.call("cacti_hip_selftest_wave_reduce", out.data_ptr(), _stream())
    return out.cpu().tolist()


# ---------------------------------------------------------------- GEMM
def gemm(a, b, ta=False, tb=False, alpha=1.0, beta=0.0, out=None):
    """out = f16(alpha op(a) op(b) + beta out); a, b 2-d row-major f16 (rows may be strided)."""
    return _op.gemm(a, b, ta, tb, alpha, beta, out)


def gemm_batched(As, Bs, ta=False, tb=False, alpha=1.0, beta=0.0, outs=None):
    """Pointer-array batch: outs[z] = f16(alpha op(As[z]) op(Bs[z]) + beta outs[z]), one shape."""
    if outs is None:
        assert beta == 0.0
        shape = (As[0].shape[1 if ta else 0], Bs[0].shape[0 if tb else 1])
        outs = [torch.empty(shape, dtype=F16, device=As[0].device) for _ in As]
    _op.gemm_batched(As, Bs, outs, ta, tb, alpha, beta)
    return outs


def gemm_strided_batched(ta, tb, nblk, M, N, K, alpha, a, lda, sa, b, ldb, sb, beta, c, ldc, sc,
                         tri=0):
    """tri: 0 dense; 1 only tril(C) wanted (rest unwritten); 2 A = tril; 3 A^T with A = tril."""
    _do.gemm_f16_strided_batched_tri(int(ta), int(tb), nblk, M, N, K, alpha,
             a.data_ptr(), lda, sa, b.data_ptr(), ldb, sb, beta, c.data_ptr(), ldc, sc, int(tri),
             _stream())
    return c


def block_matmul_qk(q, k, alpha, causal=False):
    """S16[i,h,j] = f16(alpha q[i,h,:] . k[j,h,:]) on [S,H,Dh] tensors (src/librarium/llama.rs:501).
    causal: only the tiles touching j <= i are computed; the rest of S16 is left unwritten."""
    S, H, Dh = q.shape
    s16 = torch.empty((S, H, S), dtype=F16, device=q.device)
    return gemm_strided_batched(False, True, H, S, S, Dh, alpha, q, H * Dh, Dh, k, H * Dh, Dh, 0.0,
                                s16, H * S, S, tri=1 if causal else 0)


def block_matmul_pv(p16, v, causal=False):
    """O[i,h,:] = f16(sum_j p16[i,h,j] v[j,h,:]) (src/librarium/llama.rs:506).
    causal: p16 is lower triangular (as the causal softmax writes it)."""
    S, H, _ = p16.shape
    Dh = v.shape[2]
    o = torch.empty((S, H, Dh), dtype=F16, device=v.device)
    return gemm_strided_batched(False, False, H, S, Dh, S, 1.0, p16, H * S, S, v, H * Dh, Dh, 0.0, o,
                                H * Dh, Dh, tri=2 if causal else 0)


def attention_fwd(q, k, v, alpha):
    """Fused causal attention on [S,H,Dh] tensors: returns (o, stats); stats feeds attention_bwd."""
    return _op.attention_fwd(q, k, v, alpha)


def attention_bwd(q, k, v, dO, stats, alpha, acc=None, o=None):
    """Adjoint of attention_fwd: returns (dq, dk, dv); acc = (dq, dk, dv) to accumulate into; o = the forward
    output (lets blocks of queries with spread probabilities skip the pass that forms the row sums)."""
    return _op.attention_bwd(q, k, v, dO, stats, alpha, acc, o)


# ---------------------------------------------------------------- fused thunks
def rms_norm_fwd(x, w, eps):
    return _op.rms_norm_fwd(x, w, eps)


def add_rms_norm_fwd(a, b, w, eps):
    """(f16(a + b), rms_norm of it): the residual add and the norm that follows, one launch."""
    return _op.add_rms_norm_fwd(a, b, w, eps)


def rms_norm_bwd(x, w, eps, dy, dx_acc=None, dw_acc=None):
    """Returns (dx, dw).  dx_acc / dw_acc: tensors to accumulate into (updated in place)."""
    return _op.rms_norm_bwd(x, w, eps, dy, dx_acc, dw_acc)


def rope_tables(S, Dh, device="cuda"):
    cos = torch.empty((S, Dh), dtype=F16, device=device)
    sin = torch.empty((S, Dh), dtype=F16, device=device)
    _do.rope_tables(S, Dh, cos.data_ptr(), sin.data_ptr(), _stream())
    return cos, sin


def rope_fwd(x, cos, sin):
    return _op.rope_fwd(x, cos, sin)


def rope_bwd(dy, cos, sin, dx_acc=None):
    return _op.rope_bwd(dy, cos, sin, dx_acc)


def silu_gate_fwd(g, u):
    return _op.silu_gate_fwd(g, u)


def silu_gate_bwd(g, u, dh, dg_acc=None, du_acc=None):
    return _op.silu_gate_bwd(g, u, dh, dg_acc, du_acc)


def causal_softmax_fwd(s16):
    _chk(s16)
    S, H, S2 = s16.shape
    assert S == S2
    # the kernel writes j <= i and zeros only up to the next multiple of 256 columns:
    # start from zeros so that dense consumers may read the whole row
    p = torch.zeros_like(s16)
    _do.causal_softmax_fwd(S, H, s16.data_ptr(), p.data_ptr(), _stream())
    return p


def causal_softmax_bwd(s16, dp16):
    _chk(s16), _chk(dp16)
    S, H, _ = s16.shape
    ds = torch.zeros_like(s16)
    _do.causal_softmax_bwd(S, H, s16.data_ptr(), dp16.data_ptr(), ds.data_ptr(),
             _stream())
    return ds


def _raise_index(status, what):
    rc, v = ffi.fast().read_i32(status.data_ptr(), _stream())
    if rc:
        ffi.check(rc)
    if v:
        raise IndexError("%s: id out of range at row %d" % (what, v - 1))


def softmax_ce_fwd(logit, tok, want_prob=True):
    """Returns (prob f32 or None, loss f32 [N], amax u16-as-int16 bits [N])."""
    _chk(logit)
    N, V = logit.shape
    prob = torch.empty((N, V), dtype=torch.float32, device=logit.device) if want_prob else None
    loss = torch.empty((N,), dtype=torch.float32, device=logit.device)
    amax = torch.empty((N,), dtype=torch.int16, device=logit.device)
    status = torch.zeros(1, dtype=torch.int32, device=logit.device)
    _do.softmax_ce_fwd(N, V, logit.data_ptr(), tok.data_ptr(), _p(prob),
             loss.data_ptr(), amax.data_ptr(), status.data_ptr(), _stream())
    _raise_index(status, "softmax_ce_fwd")
    return prob, loss, amax


def softmax_ce_bwd(logit, tok, scale, acc=None):
    return _op.softmax_ce_bwd(logit, tok, scale, acc)


def embed_fwd(W, tok):
    _chk(W)
    V, D = W.shape
    S = tok.numel()
    y = torch.empty((S, D), dtype=F16, device=W.device)
    status = torch.zeros(1, dtype=torch.int32, device=W.device)
    _do.embed_fwd(V, D, W.data_ptr(), S, tok.data_ptr(), y.data_ptr(),
             status.data_ptr(), _stream())
    _raise_index(status, "embed_fwd")
    return y


def embed_bwd(V, tok, dy, acc=None):
    _chk(dy)
    S, D = dy.shape
    dW = torch.empty((V, D), dtype=F16, device=dy.device) if acc is None else _chk(acc)
    _do.embed_bwd(V, D, S, tok.data_ptr(), dy.data_ptr(), dW.data_ptr(),
             int(acc is not None), _stream())
    return dW


def add_f16(a, b, out=None):
    return _op.add_f16(a, b, out)


def accumulate_1d(dst, src):
    name = {torch.float32: "f32", torch.float16: "f16", torch.int16: "u16"}[dst.dtype]
    getattr(_do, "accumulate_1d_" + name)(dst.data_ptr(), src.data_ptr(), dst.numel(),
             _stream())
    return dst


# ---------------------------------------------------------------- numerical-health digests
def nan_count(x):
    """Number of NaNs of an f16 tensor as a 0-d int64 device tensor (src/thunk/op.rs:273-349)."""
    _chk(x)
    out = torch.empty((), dtype=torch.int64, device=x.device)
    _do.nan_count_f16(x.numel(), x.data_ptr(), out.data_ptr(), _stream())
    return out


def abs_log2_hist8(x):
    """int64[256] histogram of the floor(log2 |x|) classes of an f16 tensor (src/thunk/op.rs:351-441)."""
    _chk(x)
    out = torch.empty(256, dtype=torch.int64, device=x.device)
    _do.abs_log2_hist8_f16(x.numel(), x.data_ptr(), out.data_ptr(), _stream())
    return out


def digests(xs):
    """Both digests of a list of f16 tensors, up to 64 in a launch: (hist int64[n,256], nan int64[n])
    (the per-cycle loop of examples/open_llama_3b_train.rs:409-424)."""
    if len(xs) == 0:
        out = torch.empty((0, 257), dtype=torch.int64, device="cuda")
        return out[:, :256], out[:, 256]
    return _op.digests(xs)


# ---------------------------------------------------------------- optimiser thunks (AdamW32)
def _f(x):
    return _chk(x, torch.float32)


def online_average_scale_(u, v, src_scale, rate):
    """v += rate * (src_scale * f32(u) - v) in place (src/thunk/op.rs:3884-3939)."""
    _chk(u), _f(v)
    assert u.numel() == v.numel()
    _do.online_average_scale_f16_f32(u.numel(), u.data_ptr(), v.data_ptr(), src_scale, rate,
             _stream())
    return v


def online_average_square_scale_(u, v, src_scale, rate):
    """v += rate * ((src_scale * f32(u))^2 - v) in place (src/thunk/op.rs:3941-4002)."""
    _chk(u), _f(v)
    assert u.numel() == v.numel()
    _do.online_average_square_scale_f16_f32(u.numel(), u.data_ptr(), v.data_ptr(), src_scale,
             rate, _stream())
    return v


def online_adamw_update_(g1, g2, w, signed_lr, lr_unbias, lamda, eps):
    """w += signed_lr * (lr_unbias * (g1 / (sqrt(g2) + eps)) + lamda * w) in place
    (src/thunk/op.rs:4004-4062)."""
    _f(g1), _f(g2), _f(w)
    assert g1.numel() == g2.numel() == w.numel()
    _do.online_adamw_update_f32(w.numel(), g1.data_ptr(), g2.data_ptr(), w.data_ptr(),
             signed_lr, lr_unbias, lamda, eps, _stream())
    return w


def cast_f32_f16(x):
    _f(x)
    y = torch.empty(x.shape, dtype=torch.float16, device=x.device)
    _do.cast_f32_f16(x.numel(), x.data_ptr(), y.data_ptr(), _stream())
    return y


def cast_f16_f32(x):
    _chk(x)
    y = torch.empty(x.shape, dtype=torch.float32, device=x.device)
    _do.cast_f16_f32(x.numel(), x.data_ptr(), y.data_ptr(), _stream())
    return y


def adamw32_scalars(iter_nr, grad_scale, lr, wd, a1, a2, eps):
    """The seven f32 scalars of one AdamW32 step (host arithmetic of src/librarium/adamw.rs:45-60 and
    src/op.rs:984-1023) as a list; raises for iter_nr <= 0."""
    return _op.adamw32_scalars(int(iter_nr), grad_scale or 0.0, lr, wd, a1, a2, eps)


def adamw32_step_(grads, avgs, avg2s, masters, params, scalars):
    """One AdamW32 step of a list of tensors, up to 64 in a launch, in place (avgs, avg2s, masters updated,
    params overwritten with f16(master))."""
    _op.adamw32_step(grads, avgs, avg2s, masters, params, scalars)


# ---------------------------------------------------------------- bf16 raw casts (src/thunk/op.rs:665-803)
def _raw_cast(name, x, in_dtype, out_dtype):
    _chk(x, in_dtype)
    y = torch.empty(x.shape, dtype=out_dtype, device=x.device)
    getattr(_do, name)(x.numel(), x.data_ptr(), y.data_ptr(), _stream())
    return y


def raw_cast_bf16_f16(u):
    """bf16 bit patterns (int16 tensor) -> f16."""
    return _raw_cast("raw_cast_bf16_f16", u, torch.int16, torch.float16)


def raw_cast_bf16_f32(u):
    return _raw_cast("raw_cast_bf16_f32", u, torch.int16, torch.float32)


def raw_cast_f32_bf16(x):
    """f32 -> bf16 bit patterns (int16 tensor), truncating."""
    return _raw_cast("raw_cast_f32_bf16", x, torch.float32, torch.int16)


def raw_cast_f16_bf16(x):
    return _raw_cast("raw_cast_f16_bf16", x, torch.float16, torch.int16)
