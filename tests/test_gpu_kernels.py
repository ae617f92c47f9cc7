"""Parity of every HIP kernel against the CPU oracle on the same seeded inputs (MI355X).

All calls go through the C ABI (cacti_amd.ops is a thin layer over it).  Tolerances:
tests/util.py (rel-L2 <= 1e-3, max element relative error <= 2e-2); gather / argmax /
index results bit-exact.  Elementwise kernels reproduce the oracle's rounding points, so
most of them are in fact compared bit for bit (`exact_frac`).
"""
import numpy as np
import pytest
import torch

from tests.util import assert_parity, rng, randn16

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    assert torch.cuda.is_available(), "these tests need the MI355X"
    from cacti_amd import ops as o
    return o


def dev(a):
    if a.dtype == np.uint16:
        a = a.view(np.int16)
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def host(t):
    a = t.detach().cpu().numpy()
    return a


def exact_frac(a, b):
    return float(np.mean(a.view(np.uint16) == b.view(np.uint16)))


def assert_bits(a, b, name=""):
    """Bit-for-bit equality of two f16 arrays, with a short message instead of an array dump."""
    eq = a.view(np.uint16) == b.view(np.uint16)
    assert eq.all(), "%s: %d of %d elements differ" % (name, int((~eq).sum()), eq.size)


def say(*a):
    print(*a, flush=True)


# ---------------------------------------------------------------- wave reduce
def test_wave_reduce_selftest(ops):
    s, rs, m, cnt = ops.selftest_wave_reduce()
    assert s == rs and cnt == 64.0, (s, rs, m, cnt)


# ---------------------------------------------------------------- RMSNorm
@pytest.mark.parametrize("N,D", [(2048, 3200), (128, 256), (37, 4096), (5, 8), (16, 8192)])
def test_rms_norm_fwd(ops, oracle, N, D):
    say("rms_norm_fwd", N, D)
    r = rng(100 + D)
    x, w = randn16(r, (N, D)), randn16(r, (D,))
    want, _, _ = oracle.rmsnorm_fwd(x, w, 1e-6)
    got = host(ops.rms_norm_fwd(dev(x), dev(w), 1e-6))
    assert_parity(got, want, "rms_norm_fwd")
    assert exact_frac(got, want) > 0.999


@pytest.mark.parametrize("N,D", [(2048, 3200), (37, 4096), (5, 8)])
def test_add_rms_norm_fwd_equals_the_two_thunks(ops, oracle, N, D):
    """One launch for x = a + b and rms_norm(x): bit for bit the add thunk followed by the norm."""
    say("add_rms_norm_fwd", N, D)
    r = rng(120 + N)
    a, b, w = randn16(r, (N, D)), randn16(r, (N, D)), (randn16(r, (D,), 0.1) + np.float16(1))
    s, y = ops.add_rms_norm_fwd(dev(a), dev(b), dev(w), 1e-6)
    want_s = oracle.accumulate_f16(a, b)
    assert_bits(host(s), want_s, "sum")
    assert_bits(host(y), host(ops.rms_norm_fwd(dev(want_s), dev(w), 1e-6)), "norm vs unfused kernel")
    assert_parity(host(y), oracle.rmsnorm_fwd(want_s, w, 1e-6)[0], "norm vs oracle")


# (beyond 4096 a row is more than 8 chunks of 512 and its dx is read late; blocks of 8 rows with rows missing)
@pytest.mark.parametrize("N,D", [(2048, 3200), (128, 256), (37, 4096), (5, 8), (16, 8192), (19, 4104), (300, 4608), (9, 6000), (41, 6152)])
@pytest.mark.parametrize("acc", [False, True])
def test_rms_norm_bwd(ops, oracle, N, D, acc):
    say("rms_norm_bwd", N, D, acc)
    r = rng(200 + D + acc)
    x, w, dy = randn16(r, (N, D)), randn16(r, (D,)), randn16(r, (N, D))
    dx0 = randn16(r, (N, D)) if acc else None
    dw0 = randn16(r, (D,)) if acc else None
    wdx, wdw = oracle.rmsnorm_bwd(x, w, 1e-6, dy, dx0, dw0)
    gdx, gdw = ops.rms_norm_bwd(dev(x), dev(w), 1e-6, dev(dy), dev(dx0) if acc else None,
                                dev(dw0) if acc else None)
    assert_parity(host(gdx), wdx, "dx")
    assert_parity(host(gdw), wdw, "dw")
    assert exact_frac(host(gdx), wdx) > 0.99


# ---------------------------------------------------------------- RoPE
def test_rope_tables(ops, oracle):
    for S, Dh in [(2048, 100), (128, 64)]:
        c, s = ops.rope_tables(S, Dh)
        wc, ws = oracle.rope_tables(S, Dh)
        # device cos/sin/pow differ from libm in the last ulp of f32: allow one f16 ulp
        assert np.max(np.abs(host(c).astype(np.float32) - wc.astype(np.float32))) <= 2 ** -10
        assert np.max(np.abs(host(s).astype(np.float32) - ws.astype(np.float32))) <= 2 ** -10
        assert exact_frac(host(c), wc) > 0.99 and exact_frac(host(s), ws) > 0.99


@pytest.mark.parametrize("S,H,Dh", [(2048, 32, 100), (128, 4, 64), (7, 2, 12), (33, 32, 100)])
def test_rope_fwd_bwd(ops, oracle, S, H, Dh):
    say("rope", S, H, Dh)
    r = rng(300 + S)
    x, dy, dx0 = randn16(r, (S, H, Dh)), randn16(r, (S, H, Dh)), randn16(r, (S, H, Dh))
    cos, sin = oracle.rope_tables(S, Dh)
    dc, ds = dev(cos), dev(sin)
    assert_bits(host(ops.rope_fwd(dev(x), dc, ds)), oracle.rope_fwd(x, cos, sin), "fwd")
    assert_bits(host(ops.rope_bwd(dev(dy), dc, ds)), oracle.rope_bwd(dy, cos, sin), "bwd")
    assert_bits(host(ops.rope_bwd(dev(dy), dc, ds, dev(dx0))), oracle.rope_bwd(dy, cos, sin, dx0),
                "bwd+")


def test_rope_bwd_in_place(ops, oracle):
    r = rng(310)
    S, H, Dh = 64, 32, 100
    dy = randn16(r, (S, H, Dh))
    cos, sin = oracle.rope_tables(S, Dh)
    t, dc, ds = dev(dy), dev(cos), dev(sin)
    from cacti_amd import ffi
    ffi.call("cacti_hip_rope_bwd", S, H, Dh, t.data_ptr(), dc.data_ptr(), ds.data_ptr(),
             t.data_ptr(), 0, torch.cuda.current_stream().cuda_stream)
    assert_bits(host(t), oracle.rope_bwd(dy, cos, sin), "in place")


# ---------------------------------------------------------------- SiLU gate
@pytest.mark.parametrize("shape", [(2048, 8640), (128, 688), (1, 8)])
def test_silu_gate(ops, oracle, shape):
    say("silu_gate", shape)
    r = rng(400 + shape[1])
    g, u, dh = randn16(r, shape, 2.0), randn16(r, shape), randn16(r, shape)
    _, wh = oracle.silu_gate_fwd(g, u)
    gh = host(ops.silu_gate_fwd(dev(g), dev(u)))
    assert_parity(gh, wh, "h")
    assert exact_frac(gh, wh) > 0.999
    wdg, wdu = oracle.silu_gate_bwd(g, u, dh)
    gdg, gdu = ops.silu_gate_bwd(dev(g), dev(u), dev(dh))
    assert_parity(host(gdg), wdg, "dg"), assert_parity(host(gdu), wdu, "du")
    assert exact_frac(host(gdg), wdg) > 0.999 and exact_frac(host(gdu), wdu) > 0.999
    dg0, du0 = randn16(r, shape), randn16(r, shape)
    wdg, wdu = oracle.silu_gate_bwd(g, u, dh, dg0, du0)
    gdg, gdu = ops.silu_gate_bwd(dev(g), dev(u), dev(dh), dev(dg0), dev(du0))
    assert_parity(host(gdg), wdg, "dg+"), assert_parity(host(gdu), wdu, "du+")


# ---------------------------------------------------------------- causal softmax
@pytest.mark.parametrize("S,H", [(128, 4), (512, 3), (8, 1), (2048, 2), (640, 2)])
def test_causal_softmax(ops, oracle, S, H):
    say("causal_softmax", S, H)
    r = rng(500 + S)
    s16, dp = randn16(r, (S, H, S), 2.0), randn16(r, (S, H, S), 3.0)
    # the kernels read j <= i only (entries above the diagonal may hold anything) and write
    # j <= i plus zeros up to the next multiple of 256 columns; the rest stays untouched
    i, j = np.arange(S)[:, None, None], np.arange(S)[None, None, :]
    upper = np.broadcast_to(j > i, s16.shape)
    written = np.broadcast_to(j < np.minimum(S, (i + 256) // 256 * 256), s16.shape)
    junk = s16.copy(); junk[upper] = np.float16(np.nan)
    wp = oracle.causal_softmax_fwd(s16)
    out = torch.full((S, H, S), 7.0, dtype=torch.float16, device="cuda")
    from cacti_amd import ffi
    dj = dev(junk)
    ffi.call("cacti_hip_causal_softmax_fwd", S, H, dj.data_ptr(), out.data_ptr(),
             torch.cuda.current_stream().cuda_stream)
    gp = host(out)
    assert np.all(gp[~written] == 7.0) and np.all(gp[written & upper] == 0)
    assert_parity(np.where(written, gp, 0), wp, "p16")
    wds = oracle.causal_softmax_bwd(s16, dp)
    djp = dp.copy(); djp[upper] = np.float16(np.nan)
    ddp = dev(djp)
    out = torch.full((S, H, S), 7.0, dtype=torch.float16, device="cuda")
    ffi.call("cacti_hip_causal_softmax_bwd", S, H, dj.data_ptr(), ddp.data_ptr(), out.data_ptr(),
             torch.cuda.current_stream().cuda_stream)
    gds = host(out)
    assert np.all(gds[~written] == 7.0) and np.all(gds[written & upper] == 0)
    assert_parity(np.where(written, gds, 0), wds, "ds16")


# ---------------------------------------------------------------- softmax cross-entropy
@pytest.mark.parametrize("N,V", [(64, 32000), (128, 1024), (3, 8), (5, 40000)])
def test_softmax_ce(ops, oracle, N, V):
    say("softmax_ce", N, V)
    r = rng(600 + V)
    logit = randn16(r, (N, V), 2.0)
    tok = r.integers(0, V, N).astype(np.uint16)
    scale = r.random(N).astype(np.float32)
    scale[0] = 0.0
    wprob, wloss, wamax = oracle.softmax_ce_fwd(logit, tok)
    gprob, gloss, gamax = ops.softmax_ce_fwd(dev(logit), dev(tok))
    assert_parity(host(gprob), wprob, "prob", l2=1e-5, mx=1e-4)
    assert_parity(host(gloss), wloss, "loss", l2=1e-5, mx=1e-4)
    assert (host(gamax).view(np.uint16) == wamax).all()                # index work: bit-exact
    wd = oracle.softmax_ce_bwd(logit, tok, scale)
    gd = host(ops.softmax_ce_bwd(dev(logit), dev(tok), dev(scale)))
    assert_parity(gd, wd, "dlogit")
    assert gd.size < 10000 or exact_frac(gd, wd) > 0.995
    assert np.all(gd[0] == 0)
    d0 = randn16(r, (N, V), 0.01)
    ga = host(ops.softmax_ce_bwd(dev(logit), dev(tok), dev(scale), dev(d0)))
    assert_parity(ga, oracle.accumulate_f16(d0, wd), "dlogit+")


# the label and the maximum are one lane's business each: in a row's first and last element, on both sides of a lane's eight, of
# the block's 8192 and of the row's last, partly filled round; the maximum twice, the later one in another lane, wave and round;
# a row of one value, of -infinity but for one
@pytest.mark.gpu
@pytest.mark.parametrize("V", [8, 64, 1000, 8192, 8200, 16384, 24576, 32000])
def test_softmax_ce_places_of_label_and_maximum(ops, oracle, V):
    say("softmax_ce places", V)
    places = sorted({p for p in (0, 7, 8, 511, 512, 8191, 8192, 8199, V - 8, V - 1) if 0 <= p < V})
    N = 2 * len(places) + 2
    r = rng(660 + V)
    logit, tok = randn16(r, (N, V)), np.zeros(N, np.uint16)
    for i, p in enumerate(places):
        tok[i], tok[len(places) + i] = p, places[-1 - i]
        logit[i, p] = logit[len(places) + i, p] = logit[len(places) + i, V - 1] = 9.0
    logit[-2], logit[-1], logit[-1, V // 2] = 1.5, -np.inf, 0.25
    tok[-2:] = V - 1, V // 2
    wprob, wloss, wamax = oracle.softmax_ce_fwd(logit, tok)
    gprob, gloss, gamax = ops.softmax_ce_fwd(dev(logit), dev(tok))
    assert (host(gamax).view(np.uint16) == wamax).all() and wamax[-2] == 0
    assert_parity(host(gprob), wprob, "prob", l2=1e-5, mx=1e-4)
    assert_parity(host(gloss), wloss, "loss", l2=1e-5, mx=1e-4)
    scale = np.linspace(0.5, 2, N).astype(np.float32)
    assert_parity(host(ops.softmax_ce_bwd(dev(logit), dev(tok), dev(scale))), oracle.softmax_ce_bwd(logit, tok, scale), "dlogit")


def test_softmax_ce_argmax_ties_and_bad_token(ops, oracle):
    logit = np.zeros((2, 64), np.float16)
    logit[0, [9, 40]] = 2.0
    logit[1, 63] = 1.0
    tok = np.array([1, 2], np.uint16)
    _, _, amax = ops.softmax_ce_fwd(dev(logit), dev(tok), want_prob=False)
    assert host(amax).view(np.uint16).tolist() == [9, 63]
    with pytest.raises(IndexError):
        ops.softmax_ce_fwd(dev(logit), dev(np.array([1, 64], np.uint16)))


# ---------------------------------------------------------------- embedding
@pytest.mark.parametrize("V,D,S", [(32000, 3200, 2048), (1024, 256, 128), (16, 8, 50)])
def test_embedding(ops, oracle, V, D, S):
    say("embedding", V, D, S)
    r = rng(700 + V)
    W = randn16(r, (V, D), 0.02)
    tok = r.integers(0, V, S).astype(np.uint16)
    tok[S // 2] = tok[0]                                   # force a repeated id
    got = host(ops.embed_fwd(dev(W), dev(tok)))
    assert_bits(got, oracle.embed_fwd(W, tok), "gather")
    dy = randn16(r, (S, D))
    want = oracle.embed_bwd(V, tok, dy)
    got = host(ops.embed_bwd(V, dev(tok), dev(dy)))
    assert_parity(got, want, "dW")
    assert exact_frac(got, want) > 0.9999
    never = np.setdiff1d(np.arange(V), tok)
    assert np.all(got[never] == 0)
    bad = tok.copy()
    bad[1] = V
    with pytest.raises(IndexError):
        ops.embed_fwd(dev(W), dev(bad))


# ---------------------------------------------------------------- accumulate / add
def test_accumulate_and_add(ops, oracle):
    r = rng(800)
    a, b = randn16(r, (100003,)), randn16(r, (100003,))
    got = host(ops.add_f16(dev(a), dev(b)))
    assert_bits(got, oracle.accumulate_f16(a, b), "add")
    t, tb = dev(a), dev(b)
    ops.accumulate_1d(t, tb)
    assert_bits(host(t), oracle.accumulate_f16(a, b), "accumulate")
    f, g = r.standard_normal(1000).astype(np.float32), r.standard_normal(1000).astype(np.float32)
    t, tg = dev(f), dev(g)
    ops.accumulate_1d(t, tg)
    assert (host(t) == f + g).all()
    u, v = r.integers(0, 30000, 1000).astype(np.uint16), r.integers(0, 30000, 1000).astype(np.uint16)
    t, tv = dev(u), dev(v)
    ops.accumulate_1d(t, tv)
    assert (host(t).view(np.uint16) == (u + v).astype(np.uint16)).all()


def test_add_of_transposed_operands(ops):
    # element for element in memory order: the result has the operands' strides
    a, b = (torch.randn(33, 50, device="cuda").half().t() for _ in range(2))
    got = ops.add_f16(a, b)
    assert got.stride() == a.stride()
    assert torch.equal(got, a + b)


def test_operators_run_on_the_current_stream(ops):
    """A chain of operators, with a product that wants a workspace, captured on another stream and replayed on new inputs."""
    x, y = (torch.empty(64, 250, dtype=torch.float16, device="cuda") for _ in range(2))
    W = torch.randn(35, 250, device="cuda").half()
    chain = lambda: ops.gemm(ops.silu_gate_fwd(ops.add_f16(x, y), y), W, tb=True)
    eager = []
    inputs = [[torch.randn_like(x) for _ in range(2)] for _ in range(3)]
    for u, v in inputs:
        x.copy_(u), y.copy_(v)
        eager.append(chain())
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = chain()
    for (u, v), want in zip(inputs, eager):
        x.copy_(u), y.copy_(v)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)


def test_operators_refuse_tensors_without_memory(ops):
    # a batched tensor has no pointer; the error leaves the operators usable
    x = torch.randn(3, 16, device="cuda").half()
    with pytest.raises(RuntimeError):
        torch.func.vmap(lambda a: ops.add_f16(a, a))(x)
    assert torch.equal(ops.add_f16(x, x), x + x)


# ---------------------------------------------------------------- GEMM
GEMM_SHAPES = [
    (128, 128, 32), (256, 384, 192), (100, 72, 40), (128, 688, 256), (128, 256, 688),
    (61, 35, 27),            # nothing aligned: scalar path
    (64, 100, 64), (64, 64, 100),   # head_dim 100: 8-byte path
    (200, 264, 128), (300, 648, 100), (132, 140, 12),   # short K: several column tiles, ragged edges
]


@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
@pytest.mark.parametrize("M,N,K", GEMM_SHAPES)
def test_gemm_small(ops, oracle, ta, tb, M, N, K):
    say("gemm", ta, tb, M, N, K)
    r = rng(900 + M + 3 * N + 7 * K + 2 * ta + tb)
    A = randn16(r, (K, M) if ta else (M, K))
    B = randn16(r, (N, K) if tb else (K, N))
    C0 = randn16(r, (M, N))
    for alpha, beta in [(1.0, 0.0), (0.1, 1.0)]:
        want = oracle.matmul(ta, tb, A, B, alpha, beta, C0)
        c = dev(C0)
        got = host(ops.gemm(dev(A), dev(B), bool(ta), bool(tb), alpha, beta, c))
        assert_parity(got, want, "gemm")
        assert exact_frac(got, want) > 0.98


# shapes that reach the direct-to-LDS kernels (outputs of at least 1024 x 1024, 16-byte aligned,
# K % 64 == 0) with ragged last tiles in both directions, the 256 x 256 and 256 x 192 wgrad tiles,
# and the forward product whose last columns go to a second launch of small tiles
DIRECT_SHAPES = [
    (0, 1, 1096, 1032, 192), (0, 0, 1096, 1032, 192), (1, 0, 1096, 1032, 128), (1, 1, 1032, 1096, 64),
    (1, 0, 2056, 2304, 64),      # 256 x 256 tiles
    (1, 0, 3200, 3200, 64),      # 256 x 192 tiles
    (0, 1, 1024, 8640, 64),      # 64 full-round column tiles + 448 columns on 64 x 64 tiles
    # the same with 5 .. 13 k tiles: the small tiles load five k tiles ahead (shorter than the
    # pipeline, exactly as long, every length of the peeled tail)
    (0, 1, 1024, 8640, 320), (0, 0, 1024, 8640, 384), (0, 1, 1024, 8640, 448), (0, 0, 1024, 8640, 512),
    (0, 1, 1024, 8640, 576), (0, 0, 1024, 8640, 640), (0, 1, 1024, 8640, 704), (0, 0, 1024, 8640, 832),
    (0, 1, 2048, 24584, 64),     # forward product with at least 768 tiles of 256 x 256
]


@pytest.mark.parametrize("ta,tb,M,N,K", DIRECT_SHAPES)
def test_gemm_direct_load_kernels(ops, oracle, ta, tb, M, N, K):
    say("gemm direct", ta, tb, M, N, K)
    r = rng(970 + M + N + K + 2 * ta + tb)
    A = randn16(r, (K, M) if ta else (M, K))
    B = randn16(r, (N, K) if tb else (K, N), 0.1)
    C0 = randn16(r, (M, N))
    for alpha, beta in [(1.0, 0.0), (0.5, 1.0)]:
        want = oracle.matmul(ta, tb, A, B, alpha, beta, C0)
        got = host(ops.gemm(dev(A), dev(B), bool(ta), bool(tb), alpha, beta, dev(C0)))
        assert_parity(got, want, "gemm direct")
        assert exact_frac(got, want) > 0.98


# every tile shape of the direct kernels with a K that ends inside a k tile (also shorter than one), sums in parts of K
# (few tiles, long K; the last part shorter than the others), and operands and results of any alignment
ANY_SHAPES = [
    (0, 1, 72, 200, 1000), (0, 0, 72, 200, 1000), (1, 0, 72, 200, 1001), (1, 1, 72, 200, 136), (1, 0, 256, 264, 8), (0, 0, 136, 72, 24),
    (1, 0, 1032, 1096, 611), (0, 1, 776, 1104, 520), (1, 0, 2056, 2304, 129), (1, 0, 3200, 3200, 37), (0, 0, 1100, 4104, 72),
    (0, 1, 37, 512, 4096), (0, 0, 64, 64, 8200), (1, 0, 136, 64, 3001), (0, 1, 5, 1003, 3000), (1, 0, 40, 72, 2600),
    (0, 1, 61, 35, 127), (0, 0, 129, 257, 193), (1, 0, 130, 258, 65), (1, 1, 7, 9, 130), (0, 0, 300, 1004, 772), (0, 1, 1, 3, 333),
    (0, 0, 33, 31, 4001), (1, 0, 1025, 1027, 67),
]


@pytest.mark.parametrize("ta,tb,M,N,K", ANY_SHAPES)
def test_gemm_tails_parts_and_odd_sizes(ops, oracle, ta, tb, M, N, K):
    say("gemm any", ta, tb, M, N, K)
    r = rng(990 + M + N + K + 2 * ta + tb)
    A = randn16(r, (K, M) if ta else (M, K))
    B = randn16(r, (N, K) if tb else (K, N), 0.1)
    C0 = randn16(r, (M, N))
    for alpha, beta in [(1.0, 0.0), (0.5, 1.0)]:
        want = oracle.matmul(ta, tb, A, B, alpha, beta, C0)
        c = torch.full((M * N + 16,), 7.0, dtype=torch.float16, device="cuda")      # what lies behind C stays
        c[:M * N] = dev(C0).view(-1)
        got = host(ops.gemm(dev(A), dev(B), bool(ta), bool(tb), alpha, beta, c[:M * N].view(M, N)))
        assert_parity(got, want, "gemm any")
        assert exact_frac(got, want) > 0.97
        assert (c[M * N:] == 7.0).all()


# one to four rows against a weight matrix (decoding): the streaming kernel, including a row count
# of columns that is not a multiple of its 4 rows per workgroup, a short K, and a padded weight matrix
SKINNY_SHAPES = [(1, 3200, 3200, 0), (2, 8640, 3200, 0), (3, 3200, 8640, 8), (4, 1000, 136, 0), (1, 32000, 3200, 0),
                 (4, 24, 136, 16)]


@pytest.mark.parametrize("M,N,K,pad", SKINNY_SHAPES)
def test_gemm_few_rows_streams_the_weights(ops, oracle, M, N, K, pad):
    say("gemm skinny", M, N, K, pad)
    r = rng(400 + M + N + K)
    A = randn16(r, (M, K))
    Bp = randn16(r, (N, K + pad), 0.05)
    B = Bp[:, :K]
    for alpha in (1.0, 0.125):
        want = oracle.matmul(0, 1, A, np.ascontiguousarray(B), alpha, 0.0, None)
        got = host(ops.gemm(dev(A), dev(Bp)[:, :K], False, True, alpha, 0.0))
        assert_parity(got, want, "gemm skinny")
        assert exact_frac(got, want) > 0.98


# each way a row of K is cut over the lanes, at both edges (one row: 1 to 5 pieces per lane, then passes of four; two to four
# rows: passes of two or four).  400 columns and more: fp32 sums of 10^4 terms in another order differ by some 1e-6 of a
# typical result, which moves one f16 rounding (5e-4 apart) in 250; of 40 columns a single pair is 5 %.
@pytest.mark.parametrize("M,N,K", [(1, 400, 8), (1, 400, 512), (1, 472, 520), (1, 500, 1032), (1, 466, 2048), (1, 464, 2056),
                                   (1, 464, 4104), (1, 430, 6144), (1, 464, 6152), (1, 464, 8200), (1, 440, 10240), (1, 440, 10248),
                                   (1, 424, 16392), (2, 464, 4096), (2, 464, 4104), (3, 440, 8200), (4, 466, 10248)])
def test_gemm_few_rows_over_their_ranges(ops, oracle, M, N, K):
    test_gemm_few_rows_streams_the_weights(ops, oracle, M, N, K, 0)


@pytest.mark.parametrize("ta,tb,n,M,N,K,off", [(0, 1, 3, 1032, 1096, 192, 0), (1, 0, 2, 1096, 1032, 128, 0), (0, 0, 5, 1024, 1024, 192, 0),
                                             (0, 1, 3, 1032, 1096, 192, 4), (0, 1, 2, 64, 72, 40, 0)])
def test_gemm_pointer_array_batch(ops, oracle, ta, tb, n, M, N, K, off):
    """Products of one shape on separate arrays: one launch for up to four of them (direct-load
    tiles, ragged edges), one after another when an operand is not 16-byte aligned (off) or the
    shape is small; every block against the oracle, with and without accumulation."""
    say("gemm batched", ta, tb, n, M, N, K, off)
    r = rng(300 + n + M + K + off)
    As = [randn16(r, (K, M) if ta else (M, K)) for _ in range(n)]
    Bs = [randn16(r, (N, K) if tb else (K, N), 0.1) for _ in range(n)]
    C0 = [randn16(r, (M, N)) for _ in range(n)]
    shared_a = dev(As[0])

    def place(x):                        # device copy starting `off` elements past an aligned address
        buf = torch.empty(x.size + 8, dtype=torch.float16, device="cuda")
        v = buf[off:off + x.size].view(x.shape)
        v.copy_(dev(x))
        return v
    for alpha, beta in [(1.0, 0.0), (0.5, 1.0)]:
        dA = [shared_a if z == 0 else place(As[z]) for z in range(n)]
        dB = [place(Bs[z]) for z in range(n)]
        dC = [dev(C0[z]) for z in range(n)]
        ops.gemm_batched(dA, dB, bool(ta), bool(tb), alpha, beta, dC)
        for z in range(n):
            want = oracle.matmul(ta, tb, As[z], Bs[z], alpha, beta, C0[z])
            assert_parity(host(dC[z]), want, "gemm batched %d" % z)
            single = host(ops.gemm(dA[z], dB[z], bool(ta), bool(tb), alpha, beta, dev(C0[z])))
            assert np.array_equal(host(dC[z]).view(np.uint16), single.view(np.uint16)), z


# a K that ends inside a k tile, as the weight gradients of a ragged sequence have it (any K where both operands are strided
# in it); the smallest K the shared launch takes; outputs below and above the line of the small ones
@pytest.mark.parametrize("ta,tb,n,M,N,K", [(1, 0, 3, 1032, 1096, 611), (1, 0, 2, 2056, 1032, 129), (0, 1, 3, 1032, 1096, 200),
                                           (0, 0, 4, 520, 1024, 136), (1, 0, 3, 688, 256, 203), (1, 1, 2, 1032, 520, 264),
                                           (0, 1, 5, 203, 1376, 520)])
def test_gemm_pointer_array_batch_with_a_k_tail(ops, oracle, ta, tb, n, M, N, K):
    test_gemm_pointer_array_batch(ops, oracle, ta, tb, n, M, N, K, 0)


@pytest.mark.parametrize("n,M,N,K", [(3, 1, 1096, 264), (2, 4, 1096, 264), (4, 5, 1096, 264)])
def test_gemm_pointer_array_batch_of_few_rows(ops, oracle, n, M, N, K):
    """One to four rows take the streaming kernel in a batch as they do alone: the bits of the single products.  (K = 264:
    ops.gemm lends a workspace, with which an accumulating product of few rows and a longer K is summed in parts.)"""
    test_gemm_pointer_array_batch(ops, oracle, 0, 1, n, M, N, K, 0)


@pytest.mark.parametrize("ta,tb,M,N,K", [(0, 1, 64, 264, 520), (0, 0, 64, 264, 520), (1, 0, 72, 264, 64), (1, 0, 72, 264, 61), (0, 1, 63, 100, 40)])
@pytest.mark.parametrize("ws", [False, True])
def test_gemm_rows_gigabytes_apart(ops, oracle, ta, tb, M, N, K, ws):
    """Rows of A 2^26 elements apart (a column slice of a very wide matrix): beyond a 32-bit offset inside one tile.  Through
    the entry point without a workspace, and with one."""
    from cacti_amd import ffi
    say("gemm far rows", ta, tb, M, N, K, ws)
    r = rng(320 + M + K + ta + 2 * tb)
    A, B = randn16(r, (K, M) if ta else (M, K)), randn16(r, (N, K) if tb else (K, N), 0.1)
    ld = (1 << 26) + 8
    wide = torch.empty((A.shape[0] - 1) * ld + A.shape[1], dtype=torch.float16, device="cuda")
    dA = wide.as_strided(A.shape, (ld, 1))
    dA.copy_(dev(A))
    dB, want = dev(B), oracle.matmul(ta, tb, A, B)
    if ws:
        got = ops.gemm(dA, dB, bool(ta), bool(tb))
    else:
        got = torch.empty((M, N), dtype=torch.float16, device="cuda")
        ffi.call("cacti_hip_gemm_f16", ta, tb, M, N, K, 1.0, dA.data_ptr(), ld, dB.data_ptr(), dB.stride(0), 0.0, got.data_ptr(), N,
                 torch.cuda.current_stream().cuda_stream)
    assert_parity(host(got), want, "far rows")
    del wide, dA
    torch.cuda.empty_cache()


@pytest.mark.parametrize("ta,tb", [(0, 1), (1, 0), (0, 0)])
@pytest.mark.parametrize("off", [1, 4])
def test_gemm_operands_that_start_between_16_byte_boundaries(ops, oracle, ta, tb, off):
    """Rows that are multiples of 8 elements, every array `off` elements past a boundary (slices of larger tensors): a batch
    takes the way of its single products, an aligned copy and the direct kernels, bit for bit; C is written where it
    is, with nothing beside it touched."""
    say("gemm odd bases", ta, tb, off)
    n, M, N, K = 2, 520, 616, 264
    r = rng(310 + 2 * ta + tb + off)
    As = [randn16(r, (K, M) if ta else (M, K)) for _ in range(n)]
    Bs = [randn16(r, (N, K) if tb else (K, N), 0.1) for _ in range(n)]
    C0 = randn16(r, (M, N))

    def place(x):
        buf = torch.full((x.size + 16,), 7.0, dtype=torch.float16, device="cuda")
        buf[off:off + x.size] = dev(x).view(-1)
        return buf, buf[off:off + x.size].view(x.shape)
    dA, dB = [place(x)[1] for x in As], [place(x)[1] for x in Bs]
    assert dA[0].data_ptr() % 16 == 2 * off
    for alpha, beta in [(1.0, 0.0), (0.5, 1.0)]:
        dC = [place(C0) for _ in range(n)]
        ops.gemm_batched(dA, dB, bool(ta), bool(tb), alpha, beta, [c for _, c in dC])
        for z in range(n):
            want = oracle.matmul(ta, tb, As[z], Bs[z], alpha, beta, C0)
            assert_parity(host(dC[z][1]), want, "odd base %d" % z)
            assert exact_frac(host(dC[z][1]), want) > 0.97
            one = place(C0)[1]
            ops.gemm(dA[z], dB[z], bool(ta), bool(tb), alpha, beta, one)
            assert_bits(host(dC[z][1]), host(one), "batch and single product")
            assert (dC[z][0][:off] == 7.0).all() and (dC[z][0][off + M * N:] == 7.0).all()


@pytest.mark.parametrize("tb,n,M,N,K", [(1, 16, 264, 520, 200), (0, 16, 264, 520, 200), (1, 33, 512, 512, 192), (0, 70, 128, 256, 136)])
def test_gemm_batch_of_many_small_outputs(ops, tb, n, M, N, K):
    """More 64 x 64 tiles than run at once, against fp32 torch (the bar of the random shapes above: f16 rounding of the result)."""
    say("gemm batch of small outputs", tb, n, M, N, K)
    torch.manual_seed(n + M)
    A = torch.randn(n, M, K, device="cuda").half()
    B = (torch.randn((n, N, K) if tb else (n, K, N), device="cuda") * 0.1).half()
    for beta in (0.0, 1.0):
        C0 = torch.randn(n, M, N, device="cuda").half()
        got = C0.clone()
        ops.gemm_strided_batched(False, bool(tb), n, M, N, K, 1.0, A, K, M * K, B, K if tb else N, N * K, beta, got, N, M * N)
        for z in range(n):
            ref = A[z].float() @ (B[z].float().T if tb else B[z].float()) + beta * C0[z].float()
            err = ((got[z].float() - ref).norm() / ref.norm()).item()
            mx = ((got[z].float() - ref).abs().max() / ref.abs().max()).item()
            assert err < 6e-4 and mx < 4e-3, (z, beta, err, mx)


@pytest.mark.parametrize("case", ["fwd", "dgrad", "wgrad"])
def test_gemm_projection_shapes(ops, oracle, case):
    """The three GEMMs of one projection at a reduced token count (oracle finishes in seconds)."""
    say("gemm projection", case)
    r = rng(950)
    T, Din, Dout = 256, 3200, 8640
    x, W, dy = randn16(r, (T, Din)), randn16(r, (Dout, Din), 0.02), randn16(r, (T, Dout))
    if case == "fwd":
        got, want = ops.gemm(dev(x), dev(W), False, True), oracle.matmul(0, 1, x, W)
    elif case == "dgrad":
        got, want = ops.gemm(dev(dy), dev(W), False, False), oracle.matmul(0, 0, dy, W)
    else:
        got, want = ops.gemm(dev(dy), dev(x), True, False), oracle.matmul(1, 0, dy, x)
    assert_parity(host(got), want, case)


def test_gemm_linearity_full_size(ops):
    """At full size (no oracle): (A1 + A2) B == A1 B + A2 B up to rounding, against fp32 torch."""
    say("gemm full size")
    torch.manual_seed(0)
    M, N, K = 2048, 3200, 3200
    A = torch.randn(M, K, device="cuda").half()
    B = (torch.randn(N, K, device="cuda") * 0.02).half()
    got = ops.gemm(A, B, False, True)
    ref = (A.float() @ B.float().T)
    err = (got.float() - ref).norm() / ref.norm()
    assert err < 5e-4, err
    got = ops.gemm(A, got, True, False)          # [K,M]^T... (K x N) wgrad-shaped product
    ref = (A.float().T @ ref.half().float())
    assert (got.float() - ref).norm() / ref.norm() < 5e-4


@pytest.mark.parametrize("seed", [0, 1, 2])
def test_gemm_random_shapes_through_the_tile_choice(ops, seed):
    """Seeded random shapes, transpositions and alpha / beta through the automatic choice of kernel and
    tile (direct-load and register tiles, the two-launch column split, the short-K and few-row kernels,
    the element-wise fallback for unaligned operands) against fp32 torch: rel-L2 <= 6e-4 and largest
    error <= 4e-3 of the largest value (f16 rounding of the result is 4.9e-4 relative)."""
    import random
    rnd = random.Random(seed)
    torch.manual_seed(seed)
    for it in range(24):
        ta, tb = rnd.random() < 0.5, rnd.random() < 0.5
        step = rnd.choice([8, 8, 8, 4, 1])                     # alignment class of the leading dimensions
        M = rnd.randrange(1024, 4300, step)
        N = rnd.randrange(1024, 9000, step)
        K = rnd.choice([rnd.randrange(64, 1100, 64), rnd.randrange(8, 600, step), 100])
        if rnd.random() < 0.2:
            N = rnd.choice([3200, 8640, 8192 + 8, 8448])
        if rnd.random() < 0.2:
            M = rnd.choice([2048, 3200, 2056, 1, 3, 4])
        alpha, beta = rnd.choice([1.0, 0.5]), rnd.choice([0.0, 1.0])
        say("gemm random", seed, it, ta, tb, M, N, K, alpha, beta)
        A = torch.randn((K, M) if ta else (M, K), device="cuda").half()
        B = (torch.randn((N, K) if tb else (K, N), device="cuda") * 0.1).half()
        C0 = torch.randn(M, N, device="cuda").half()
        got = ops.gemm(A, B, ta, tb, alpha, beta, C0.clone()).float()
        ref = alpha * ((A.float().T if ta else A.float()) @ (B.float().T if tb else B.float())) + beta * C0.float()
        err = ((got - ref).norm() / ref.norm()).item()
        mx = ((got - ref).abs().max() / ref.abs().max()).item()
        assert err < 6e-4 and mx < 4e-3, (ta, tb, M, N, K, alpha, beta, err, mx)


# sums of products in one launch: small outputs (M32) and others, edges of tiles and one past them, as many k tiles as buffers
# (256) and one more, remainders of all tiles; behind the line what is not for one launch: K below 256 or no multiple of 64, five
# products, rows that are not 16-byte aligned
@pytest.mark.gpu
@pytest.mark.parametrize("n,M,N,K,gap,beta", [
    (2, 1, 8, 256, 0, 0), (3, 64, 64, 256, 0, 0), (4, 65, 72, 320, 8, 0), (2, 33, 264, 384, 0, 0), (3, 512, 512, 256, 0, 0),
    (3, 513, 520, 256, 0, 0), (2, 611, 1032, 1024, 8, 0), (3, 777, 2048, 448, 0, 0), (2, 2049, 1608, 256, 0, 0), (4, 1000, 3200, 512, 0, 0),
    (2, 2048, 8640, 320, 0, 0), (2, 4000, 4104, 256, 0, 0),
    (1, 96, 128, 512, 0, 0), (2, 96, 128, 192, 0, 0), (3, 96, 128, 328, 0, 0), (5, 96, 640, 256, 0, 0), (2, 300, 1028, 256, 0, 0), (3, 512, 520, 256, 0, 1)])
def test_gemm_chain_has_the_bits_of_products_one_by_one(ops, n, M, N, K, gap, beta):
    import ctypes as C
    import torch
    from cacti_amd import ffi
    say("gemm chain", n, M, N, K, gap, beta)
    g = torch.Generator(device="cuda").manual_seed(n + M + N + K)
    st = torch.cuda.current_stream().cuda_stream
    rows = lambda r, c: torch.randn(r, c + gap, device="cuda", generator=g).half()
    A, B, c0 = [rows(M, K) for _ in range(n)], [rows(K, N) for _ in range(n)], rows(M, N)
    got, want = c0.clone(), c0.clone()
    for z in range(n):
        ffi.call("cacti_hip_gemm_f16", 0, 0, M, N, K, 1.0, A[z].data_ptr(), K + gap, B[z].data_ptr(), N + gap, 1.0 if z else float(beta),
                 want.data_ptr(), N + gap, st)
    pa, pb = ((C.c_void_p * n)(*[t.data_ptr() for t in x]) for x in (A, B))
    ffi.call("cacti_hip_gemm_f16_chain", n, M, N, K, C.cast(pa, C.c_void_p), K + gap, C.cast(pb, C.c_void_p), N + gap, float(beta),
             got.data_ptr(), N + gap, st)
    assert_bits(host(got), host(want), "chain")
    ref = sum(a[:, :K].float() @ b[:, :N].float() for a, b in zip(A, B)) + beta * c0[:, :N].float()
    # n roundings of partial sums of the size of the result at most: n half ulps, 2^-12 of a value in the mean
    assert ((got[:, :N].float() - ref).norm() / ref.norm()).item() < n * 3e-4


# all gradients of products that share an input in one launch: small outputs (M32) and the four tiles of others; either one's sums the
# longer; one k tile, a tail of either sum; behind the line what is for separate launches: one small output of two, what fills the device, a chain with a tail,
# five products, rows that are not 16-byte aligned
@pytest.mark.gpu
@pytest.mark.parametrize("beta_x,beta_w", [(0, 0), (1, 1)])
@pytest.mark.parametrize("n,S,N,K,one", [
    (1, 1, 8, 8, 1), (1, 64, 64, 64, 1), (1, 33, 136, 72, 1), (3, 128, 256, 256, 1), (2, 200, 320, 264, 1), (1, 611, 1024, 1024, 1),
    (1, 513, 1032, 1048, 1), (3, 611, 1024, 1024, 1), (2, 611, 2816, 1024, 1), (1, 611, 1024, 2816, 1), (1, 777, 2048, 2048, 1),
    (4, 600, 576, 1032, 1), (1, 1300, 768, 2304, 1), (1, 2000, 1024, 1024, 1),
    (2, 128, 688, 256, 0), (1, 128, 4096, 256, 0), (1, 1600, 2048, 6000, 0), (2, 600, 1000, 1024, 0), (5, 96, 256, 256, 0), (1, 300, 1028, 512, 0)])
def test_gemm_grads_have_the_bits_of_products_one_by_one(ops, n, S, N, K, one, beta_x, beta_w):
    import ctypes as C
    import torch
    from cacti_amd import ffi
    say("gemm grads", n, S, N, K, beta_x, beta_w)
    assert ffi.lib().cacti_hip_gemm_f16_grads_one_launch(n, S, N, K) == one
    g = torch.Generator(device="cuda").manual_seed(n + S + N + K)
    st = torch.cuda.current_stream().cuda_stream
    new = lambda *s: torch.randn(*s, device="cuda", generator=g).half()
    dy, W, x = [new(S, N) for _ in range(n)], [new(N, K) for _ in range(n)], new(S, K)
    dx, dW = new(S, K), [new(N, K) for _ in range(n)]
    want_x, want_w = dx.clone(), [t.clone() for t in dW]
    for z in range(n):
        ffi.call("cacti_hip_gemm_f16", 1, 0, N, K, S, 1.0, dy[z].data_ptr(), N, x.data_ptr(), K, float(beta_w), want_w[z].data_ptr(), K, st)
        ffi.call("cacti_hip_gemm_f16", 0, 0, S, K, N, 1.0, dy[z].data_ptr(), N, W[z].data_ptr(), K, 1.0 if z else float(beta_x),
                 want_x.data_ptr(), K, st)
    pd, pw, pg = ((C.c_void_p * n)(*[t.data_ptr() for t in a]) for a in (dy, W, dW))
    ffi.call("cacti_hip_gemm_f16_grads", n, S, N, K, C.cast(pd, C.c_void_p), C.cast(pw, C.c_void_p), x.data_ptr(), float(beta_x), dx.data_ptr(),
             float(beta_w), C.cast(pg, C.c_void_p), st)
    assert_bits(host(dx), host(want_x), "dx")
    for z in range(n):
        assert_bits(host(dW[z]), host(want_w[z]), "dW %d" % z)


@pytest.mark.parametrize("n,S,N,K", [(1, 611, 1024, 1024), (3, 128, 256, 256), (2, 611, 2816, 1024), (2, 600, 1000, 1024)])
def test_gemm_grads_with_dx_in_place_of_x(ops, n, S, N, K):
    """The weight gradients are those of x, whether or not the sizes would have one launch of all (the last ones have not)."""
    import ctypes as C
    from cacti_amd import ffi
    say("gemm grads in place", n, S, N, K)
    g = torch.Generator(device="cuda").manual_seed(n + S + N + K)
    st = torch.cuda.current_stream().cuda_stream
    new = lambda *s: torch.randn(*s, device="cuda", generator=g).half()
    dy, W, x = [new(S, N) for _ in range(n)], [new(N, K) for _ in range(n)], new(S, K)
    table = lambda ts: C.cast((C.c_void_p * n)(*[t.data_ptr() for t in ts]), C.c_void_p)
    got = []
    for dx in (torch.empty_like(x), x):                  # (the second call overwrites x)
        dW = [torch.empty(N, K, device="cuda", dtype=torch.float16) for _ in range(n)]
        ffi.call("cacti_hip_gemm_f16_grads", n, S, N, K, table(dy), table(W), x.data_ptr(), 0.0, dx.data_ptr(), 0.0, table(dW), st)
        got.append([host(t) for t in [dx] + dW])
    for i, (a, b) in enumerate(zip(*got)):
        assert_bits(b, a, "dx" if i == 0 else "dW %d" % (i - 1))


def test_gemm_colmajor_entry(ops, oracle):
    """The cuBLAS-shaped entry: row-major callers pass operands swapped (thunk/op.rs:4469-4491)."""
    import ctypes as C
    from cacti_amd import ffi
    r = rng(960)
    M, N, K = 96, 80, 64
    x, W = randn16(r, (M, K)), randn16(r, (N, K))
    want = oracle.matmul(0, 1, x, W)             # row-major y = x W^T
    y = torch.empty((M, N), dtype=torch.float16, device="cuda")
    one, zero = C.c_float(1.0), C.c_float(0.0)
    # column-major: y^T (N x M) = W (as col-major K x N, transposed) * x (col-major K x M)
    dW, dx = dev(W), dev(x)
    ffi.call("cacti_hip_gemm_colmajor_f16", 1, 0, N, M, K, C.byref(one), dW.data_ptr(), K,
             dx.data_ptr(), K, C.byref(zero), y.data_ptr(), N,
             torch.cuda.current_stream().cuda_stream)
    assert_parity(host(y), want, "colmajor")


# ---------------------------------------------------------------- attention block
@pytest.mark.parametrize("ta", [0, 1])
def test_head_slab_products_accumulate_in_place(ops, oracle, ta):
    """C[:, h, :] += op(A_h) B[:, h, :] on [S, H, 100] slabs (every other head starts 8 bytes off a
    16-byte boundary): each head's 100 columns get exactly its own product, nothing else moves."""
    say("head slabs accumulate", ta)
    S, H, Dh = 256, 4, 100
    r = rng(1100 + ta)
    a = randn16(r, (S, H, S), 0.1)
    b, c0 = randn16(r, (S, H, Dh)), randn16(r, (S, H, Dh))
    want = np.empty_like(c0)
    for h in range(H):
        want[:, h, :] = oracle.matmul(ta, 0, np.ascontiguousarray(a[:, h, :]),
                                      np.ascontiguousarray(b[:, h, :]), 0.5, 1.0,
                                      np.ascontiguousarray(c0[:, h, :]))
    c = dev(c0)
    ops.gemm_strided_batched(bool(ta), False, H, S, Dh, S, 0.5, dev(a), H * S, S, dev(b), H * Dh, Dh,
                             1.0, c, H * Dh, Dh)
    assert_parity(host(c), want, "slab accumulate")


@pytest.mark.parametrize("S,H,Dh", [(128, 4, 64), (256, 3, 100), (1024, 2, 100), (512, 4, 100), (384, 6, 100)])
@pytest.mark.parametrize("tri", [False, True])
def test_attention_block_via_thunks(ops, oracle, S, H, Dh, tri):
    """Q K^T -> causal softmax -> P V and the adjoint, composed as the reference stages them;
    tri: the products skip the half that the causal mask discards."""
    say("attention", S, H, Dh, tri)
    r = rng(1000 + S)
    alpha = float(np.float32(1.0) / np.sqrt(np.float32(Dh)))
    q, k, v, dO = (randn16(r, (S, H, Dh)) for _ in range(4))
    ws16, wp16, wo = oracle.attention_fwd(q, k, v, alpha)
    dq_, dk_, dv_ = oracle.attention_bwd(q, k, v, dO, alpha)
    Q, K_, V_, DO = dev(q), dev(k), dev(v), dev(dO)
    low = np.broadcast_to(np.arange(S)[:, None, None] >= np.arange(S)[None, None, :], ws16.shape)
    s16 = ops.block_matmul_qk(Q, K_, alpha, causal=tri)
    assert_parity(np.where(low, host(s16), 0), np.where(low, ws16, 0), "s16")
    p16 = ops.causal_softmax_fwd(s16)
    assert_parity(np.where(low, host(p16), 0), wp16, "p16")
    o = ops.block_matmul_pv(p16, V_, causal=tri)
    assert_parity(host(o), wo, "o")
    ld, lds = H * Dh, H * S
    dv = torch.empty_like(V_); dp = torch.empty_like(s16)
    dq = torch.empty_like(Q); dk = torch.empty_like(Q)
    t1, t2, t3 = (1, 2, 3) if tri else (0, 0, 0)
    ops.gemm_strided_batched(True, False, H, S, Dh, S, 1.0, p16, lds, S, DO, ld, Dh, 0.0, dv, ld, Dh, t3)
    ops.gemm_strided_batched(False, True, H, S, S, Dh, 1.0, DO, ld, Dh, V_, ld, Dh, 0.0, dp, lds, S, t1)
    ds = ops.causal_softmax_bwd(s16, dp)
    ops.gemm_strided_batched(True, False, H, S, Dh, S, alpha, ds, lds, S, Q, ld, Dh, 0.0, dk, ld, Dh, t3)
    ops.gemm_strided_batched(False, False, H, S, Dh, S, alpha, ds, lds, S, K_, ld, Dh, 0.0, dq, ld, Dh, t2)
    assert_parity(host(dv), dv_, "dv")
    assert_parity(host(dq), dq_, "dq")
    assert_parity(host(dk), dk_, "dk")


@pytest.mark.parametrize("S,H,Dh", [(128, 4, 64), (256, 3, 100), (200, 2, 100), (72, 2, 128), (1024, 2, 100),
                                    (384, 6, 100), (8, 1, 4), (192, 4, 60), (130, 2, 124), (448, 2, 100)])
def test_fused_attention(ops, oracle, S, H, Dh):
    """The fused forward and adjoint kernels against the oracle's chain of separate thunks: O, the row
    statistics they keep (maximum and sum of exp of the f16 scores), dQ, dK, dV; ragged sequence lengths
    (rows and keys beyond S are masked) and head dims 4 .. 128; accumulation into existing gradients.
    Both ways of loading tiles are covered: straight into LDS (even head counts with Dh % 8 = 4: every other
    head addressed 4 elements before its start, windows of 8, 13 and 16 chunks; Dh % 8 = 0) and through
    registers (3 heads of 100, 1 head of 4).  On 256 compute units the direct ones are the kernels' of 32 rows per workgroup; the
    tile kernels beyond those with tiles straight into LDS: TILE_SHAPES."""
    say("fused attention", S, H, Dh)
    r = rng(1200 + S + Dh)
    alpha = float(np.float32(1.0) / np.sqrt(np.float32(Dh)))
    q, k, v, dO = (randn16(r, (S, H, Dh)) for _ in range(4))
    ws16, wp16, wo = oracle.attention_fwd(q, k, v, alpha)
    dq_, dk_, dv_ = oracle.attention_bwd(q, k, v, dO, alpha)
    Q, K_, V_, DO = dev(q), dev(k), dev(v), dev(dO)
    o, stats = ops.attention_fwd(Q, K_, V_, alpha)
    assert_parity(host(o), wo, "o")
    st = host(stats).reshape(2, H, S)
    low = np.arange(S)[:, None, None] >= np.arange(S)[None, None, :]
    sm = np.where(low, ws16.astype(np.float32), -np.inf)                      # [S, H, S]
    want_m = sm.max(2).T
    want_l = np.exp(sm.astype(np.float64) - sm.max(2, keepdims=True)).sum(2).T
    # up to the few scores whose f16 rounding falls the other way with another fp32 summation order
    assert np.abs(st[0] - want_m).max() <= 2e-3 * max(1.0, np.abs(want_m).max()), "row maxima of the f16 scores"
    assert np.mean(st[0] == want_m) > 0.95
    assert np.abs(st[1] / want_l - 1).max() < 2e-3
    dq, dk, dv = ops.attention_bwd(Q, K_, V_, DO, stats, alpha)
    for name, got, want in (("dv", dv, dv_), ("dq", dq, dq_), ("dk", dk, dk_)):
        assert_parity(host(got), want, name)
    # with the forward output handed over, blocks of queries with spread probabilities take their row sums from
    # dO . O instead of a pass over the keys: the same bar; dV does not depend on the row sums at all
    dq_o, dk_o, dv_o = ops.attention_bwd(Q, K_, V_, DO, stats, alpha, o=o)
    for name, got, want in (("dv", dv_o, dv_), ("dq", dq_o, dq_), ("dk", dk_o, dk_)):
        e2, em = assert_parity(host(got), want, name + " (row sums from dO . O)")
        say("  %s with o: rel_l2 %.2e max_rel %.2e" % (name, e2, em))
    assert_bits(host(dv_o), host(dv), "dv with and without o")
    if S <= 128:                                    # a single block of queries holds row 0: always the pass
        assert_bits(host(dq_o), host(dq), "dq: the first block of queries keeps the pass over the keys")
    # accumulate mode: the product is added to what the tensors hold, one rounding
    base = [randn16(r, (S, H, Dh)) for _ in range(3)]
    acc = tuple(dev(b) for b in base)
    ops.attention_bwd(Q, K_, V_, DO, stats, alpha, acc=acc)
    for name, got, b, plain in zip(("dq", "dk", "dv"), acc, base, (dq, dk, dv)):
        want = b.astype(np.float32) + host(plain).astype(np.float32)
        assert_parity(host(got), want, name + " accumulated", l2=6e-4, mx=2e-3)
    # a second call gives the same bits (no atomics, no order dependence)
    dq2, dk2, dv2 = ops.attention_bwd(Q, K_, V_, DO, stats, alpha)
    for a, b in ((dq, dq2), (dk, dk2), (dv, dv2)):
        assert_bits(host(a), host(b), "repeat")


# Edges of the kernels of 32 rows per workgroup (attention_short.hip): of their blocks of 32 (a single position, one short of, on
# and one past it), of what 4 and 8 waves split (128, 256), of the forms by length (1024, 2048) and by workgroups on 256 CUs (256,
# 512; 768 and 1024 forward), and of the adjoint's other half (2048, 2 of 128: dK, dV in parts; 2080, 4 of 64: no forward; the
# last ones: forward only, neither, and neither with 128 rows of dQ a workgroup, heads to 64); windows, rows longer than the heads, accumulation
SHORT_SHAPES = [(1, 1, 8, 0), (31, 2, 100, 0), (32, 1, 64, 24), (33, 4, 60, 0), (127, 1, 128, 0), (129, 3, 64, 0), (255, 2, 68, 8),
                (257, 1, 32, 0), (512, 16, 100, 0), (513, 16, 64, 0), (1023, 2, 12, 0), (1024, 8, 64, 0), (1025, 2, 128, 0), (2047, 8, 64, 0),
                (2048, 2, 128, 8), (2080, 4, 64, 0), (97, 192, 12, 0), (128, 256, 72, 0), (128, 257, 72, 0), (700, 48, 64, 0)]
# Just past those limits, tiles straight into LDS in the tile kernels (attention.hip), each of its forms for heads to 64, in windows
# and beyond 112, whole tiles and a ragged last one: 64 rows forward and dQ, 64 keys; 128 rows, 128 keys (to 64: 64 keys, then
# 128); up to 1024 positions 128 rows forward (exact: 64); 128 rows, 128 keys up to 128 positions.  Then parts of the queries
# (default arithmetic) beside the dQ kernel of 32 rows, whole ones and a ragged last one.  Then more than one workgroup of 32 rows per
# CU: the tile dQ kernel (default arithmetic) beside dK / dV of 32 keys, and the tile kernels for both
TILE_SHAPES = [(1100, 20, 64, 8), (1057, 16, 100, 0), (1531, 16, 128, 0), (1090, 40, 64, 0), (1025, 64, 64, 0), (1090, 32, 100, 0),
               (1100, 32, 128, 8), (1000, 26, 64, 0), (128, 264, 128, 0),
               (4001, 1, 64, 0), (4096, 1, 64, 24), (1531, 4, 100, 0), (2001, 2, 100, 8), (1471, 4, 128, 8), (2048, 4, 128, 0),
               (450, 24, 64, 0), (385, 28, 100, 8), (699, 18, 128, 0), (300, 36, 64, 0), (500, 32, 100, 0), (420, 34, 128, 8)]


@pytest.mark.gpu
@pytest.mark.parametrize("exact", [False, True])
@pytest.mark.parametrize("S,H,Dh,gap", SHORT_SHAPES + TILE_SHAPES)
def test_attention_of_short_sequences_against_the_register_path(ops, S, H, Dh, gap, exact):
    """Tensors on 16-byte boundaries against the same ones 8 bytes off (tiles through registers, 128 rows): relative L2 to the
    chain in 64 bits of O, dQ, dK, dV no larger, but for the output's own rounding falling otherwise here and there (two sums of
    the same terms in another order: a few of 2^-11 steps, 2e-5 of the norm, measured 1e-6); gap: columns between rows."""
    import torch
    from cacti_amd import ffi
    say("attention of short sequences", S, H, Dh, gap, exact)
    ld, alpha, st = H * Dh + gap, Dh ** -0.5, torch.cuda.current_stream().cuda_stream
    g = torch.Generator(device="cuda").manual_seed(S + H + Dh)
    def tensor(off, like=None):
        x = torch.full((S * ld + 8,), 7.0, dtype=torch.float16, device="cuda")[off:off + S * ld].view(S, ld)
        x[:, :H * Dh] = torch.randn(S, H * Dh, device="cuda", generator=g).half() if like is None else like[:, :H * Dh]
        return x
    q, k, v, dO, base = (tensor(0) for _ in range(5))
    ffi.call("cacti_hip_attention_set_exact", int(exact))
    try:
        size = ffi.lib().cacti_hip_attention_bwd_workspace_best(S, H, Dh)
        got = []
        for off in (0, 4):
            Q, K, V, DO, o = (tensor(off, like) for like in (q, k, v, dO, base))
            stats, ws = torch.empty(2 * S * H, device="cuda"), torch.empty(size, dtype=torch.uint8, device="cuda")
            ffi.call("cacti_hip_attention_fwd", S, H, Dh, alpha, Q.data_ptr(), K.data_ptr(), V.data_ptr(), ld, o.data_ptr(), stats.data_ptr(), st)
            out = [o]
            for with_o, acc in ((1, 0), (0, 0), (1, 1)):
                d = [tensor(off, base) for _ in range(3)]
                ffi.call("cacti_hip_attention_bwd", S, H, Dh, alpha, Q.data_ptr(), K.data_ptr(), V.data_ptr(), o.data_ptr() if with_o else None,
                         DO.data_ptr(), ld, stats.data_ptr(), d[0].data_ptr(), acc, d[1].data_ptr(), acc, d[2].data_ptr(), acc, ws.data_ptr(),
                         size, st)
                out += d
            assert all(bool((x[:, H * Dh:] == 7.0).all()) for x in out), "columns between rows"
            got.append([x[:, :H * Dh].double() for x in out] + [stats.double()])
    finally:
        ffi.call("cacti_hip_attention_set_exact", 0)
    sums = [0.0] * 4, [[0.0] * 10, [0.0] * 10]
    for h in range(H):                              # the chain in 64 bits, a head at a time
        hq, hk, hv, hd, hb = (t[:, h * Dh:(h + 1) * Dh].double() for t in (q, k, v, dO, base))
        low = torch.ones(S, S, dtype=torch.bool, device="cuda").tril()
        p = torch.softmax((alpha * hq @ hk.T.contiguous()).masked_fill(~low, float("-inf")), 1)
        dp = hd @ hv.T.contiguous()
        ds = p * (dp - (p * dp).sum(1, keepdim=True))
        d = [alpha * ds @ hk, alpha * ds.T.contiguous() @ hq, p.T.contiguous() @ hd]
        want = [p @ hv] + d + d + [x + hb for x in d]
        for i, w in enumerate([p @ hv] + d): sums[0][i] += float(w.square().sum())
        for side in (0, 1):
            for i, w in enumerate(want):
                sums[1][side][i] += float((got[side][i][:, h * Dh:(h + 1) * Dh] - w).square().sum())
    for i in range(10):
        norm = max(sums[0][(0, 1, 2, 3)[0 if i == 0 else (i - 1) % 3 + 1]], 1e-30 * S * H * Dh)
        new, old = (sums[1][side][i] ** 0.5 / norm ** 0.5 for side in (0, 1))
        say("  result %d: rel_l2 %.3e, through registers %.3e" % (i, new, old))
        assert new <= old + 2e-5, (i, new, old)
    # the statistics: maxima and sums of the rounded scores, of which a few round otherwise in the other order of summation
    m, l = (torch.stack([got[side][10].view(2, H, S)[j] for side in (0, 1)]) for j in (0, 1))
    assert float((m[0] - m[1]).abs().max()) <= 2e-3 * max(1.0, float(m.abs().max())) and float((l[0] / l[1] - 1).abs().max()) < 2e-3


# One position, a ragged last block, 8 and 4 waves, a wave whose blocks hold no finite score of a row, windows, the form beyond 1024
# positions; both adjoints of 32 rows, heads to 64 and beyond
NOT_FINITE_SHAPES = [(1, 1, 64), (33, 2, 128), (61, 2, 64), (300, 4, 100), (700, 16, 64), (777, 4, 128), (1500, 4, 64)]


def _attention_masks(q, k, v, dO, alpha, off, exact):
    """Which elements of O, dQ, dK, dV are NaN and which infinite, with the tensors `off` elements past a 16-byte boundary (0: tiles
    straight into LDS, 4: through registers)."""
    import torch
    from cacti_amd import ffi
    S, H, Dh = q.shape
    def at(x):
        t = torch.empty(x.numel() + 8, dtype=torch.float16, device="cuda")[off:off + x.numel()].view(x.shape)
        return t.copy_(x)
    Q, K, V, G, o, dq, dk, dv = (at(x) for x in (q, k, v, dO, q, q, q, q))
    st, size = torch.cuda.current_stream().cuda_stream, ffi.lib().cacti_hip_attention_bwd_workspace(S, H)
    stats, ws = torch.empty(2 * S * H, device="cuda"), torch.empty(size, dtype=torch.uint8, device="cuda")
    ffi.call("cacti_hip_attention_set_exact", int(exact))
    try:
        ffi.call("cacti_hip_attention_fwd", S, H, Dh, alpha, Q.data_ptr(), K.data_ptr(), V.data_ptr(), H * Dh, o.data_ptr(), stats.data_ptr(), st)
        ffi.call("cacti_hip_attention_bwd", S, H, Dh, alpha, Q.data_ptr(), K.data_ptr(), V.data_ptr(), o.data_ptr(), G.data_ptr(), H * Dh,
                 stats.data_ptr(), dq.data_ptr(), 0, dk.data_ptr(), 0, dv.data_ptr(), 0, ws.data_ptr(), size, st)
    finally:
        ffi.call("cacti_hip_attention_set_exact", 0)
    return {n: (host(torch.isnan(x)), host(torch.isinf(x))) for n, x in (("o", o), ("dq", dq), ("dk", dk), ("dv", dv))}


def _same_masks(q, k, v, dO, alpha, exact):
    direct, registers = (_attention_masks(q, k, v, dO, alpha, off, exact) for off in (0, 4))
    for n in direct:
        assert (direct[n][0] == registers[n][0]).all(), n + ": NaN"
        assert (direct[n][1] == registers[n][1]).all(), n + ": infinity"
    return direct


@pytest.mark.gpu
@pytest.mark.parametrize("exact", [False, True])
@pytest.mark.parametrize("S,H,Dh", NOT_FINITE_SHAPES)
def test_attention_rows_whose_every_score_overflows(ops, S, H, Dh, exact):
    """Every live score of a row rounds to -infinity: the row has no softmax (its sum is 0), so its output is NaN, and what
    the adjoint makes of it is NaN where the register path has it."""
    import torch
    say("attention, rows of -infinity", S, H, Dh, exact)
    g = torch.Generator(device="cuda").manual_seed(S + H + Dh)
    q, v, dO = (torch.randn(S, H, Dh, device="cuda", generator=g).half() for _ in range(3))
    k = torch.full((S, H, Dh), -300.0, device="cuda", dtype=torch.float16)
    rows = sorted({0, S // 2, S - 1})
    q[rows] = 300.0
    masks = _same_masks(q, k, v, dO, Dh ** -0.5, exact)
    nan = masks["o"][0]
    assert nan[rows].all() and nan.sum() == len(rows) * H * Dh


@pytest.mark.gpu
@pytest.mark.parametrize("S,H,Dh,keys", [(33, 2, 128, 1), (65, 3, 64, 1), (161, 2, 64, 1), (225, 1, 128, 1), (128, 4, 64, 32)])
def test_attention_of_nan_scores_that_are_all_a_wave_has_of_a_row(ops, S, H, Dh, keys):
    """The last keys of a head are NaN, in a block of 32 keys that is one wave's only one: the rows that see no other key of the
    block have no softmax, and every gradient they reach is NaN, as in the chain of separate products (default arithmetic; in the
    other heads nothing is)."""
    import torch
    say("attention, NaN scores", S, H, Dh, keys)
    g = torch.Generator(device="cuda").manual_seed(S + H + Dh)
    q, k, v, dO = (torch.randn(S, H, Dh, device="cuda", generator=g).half() for _ in range(4))
    k[S - keys:, 0] = float("nan")
    masks = _attention_masks(q, k, v, dO, Dh ** -0.5, 0, False)
    for n, (nan, inf) in masks.items():
        first = S - keys if n in ("o", "dq") else 0
        assert nan[first:, 0].all() and nan.sum() == (S - first) * Dh and not inf.any(), n


@pytest.mark.gpu
@pytest.mark.parametrize("exact", [False, True])
@pytest.mark.parametrize("S,H,Dh", NOT_FINITE_SHAPES)
def test_attention_infinity_in_the_last_row(ops, S, H, Dh, exact):
    """The last position's values (then its output gradient) hold an infinity, in a block of 32 that the tensor may not fill:
    the last output row (every dV row) is infinite there and not NaN, nothing beyond the tensor being multiplied with it."""
    import torch
    say("attention, infinity in the last row", S, H, Dh, exact)
    g = torch.Generator(device="cuda").manual_seed(S + H + Dh)
    q, k, v, dO = (torch.randn(S, H, Dh, device="cuda", generator=g).half() for _ in range(4))
    q *= 0.25                                     # (no probability of the last row below what f16 holds)
    x = v.clone()
    x[-1, :, 4:8] = float("inf")
    masks = _same_masks(q, k, x, dO, Dh ** -0.5, exact)
    assert masks["o"][1][-1, :, 4:8].all() and not masks["o"][0][-1].any()
    x = dO.clone()
    x[-1, :, 4:8] = float("inf")
    masks = _same_masks(q, k, v, x, Dh ** -0.5, exact)
    assert masks["dv"][1][:, :, 4:8].all() and not masks["dv"][0].any()


# Rows one short of, on and one past the edges of 64 and 128 query rows at few heads, which on 256 CUs are the kernels' of 32 rows;
# at many small heads the tile kernels with 128 rows (64 for dQ at 480 workgroups of 64 rows, and forward in the exact
# arithmetic; 528, 640: 128 for both), with tiles straight into LDS, in windows (heads of 12, 100) and, exact, in the other
# arithmetic, all against the restatement of the chain
@pytest.mark.gpu
@pytest.mark.parametrize("exact", [False, True])
@pytest.mark.parametrize("S,H,Dh", [(63, 2, 64), (64, 1, 128), (65, 2, 100), (127, 2, 128), (129, 4, 64), (191, 2, 100), (193, 1, 128),
                                    (130, 160, 8), (130, 176, 8), (257, 128, 12), (321, 86, 16)])
def test_fused_attention_by_query_rows(ops, oracle, S, H, Dh, exact):
    from cacti_amd import ffi
    ffi.call("cacti_hip_attention_set_exact", int(exact))
    try:
        test_fused_attention(ops, oracle, S, H, Dh)
    finally:
        ffi.call("cacti_hip_attention_set_exact", 0)


@pytest.mark.gpu
@pytest.mark.parametrize("gain,exact", [(8.0, False), (24.0, True), (2.0, True)])
def test_fused_attention_with_large_scores(ops, oracle, gain, exact):
    """Scores of large magnitude (row maxima in the hundreds for gain 8, 1500 .. 2600 for 24): by default
    the fused kernels fold the row maximum and the logarithm of the row sum into one fp32 exponent offset,
    whose rounding error is common to a row and grows with |m|; the probabilities are nearly one-hot here,
    the case in which the adjoint's dP - sigma cancels exactly in the reference.  The default forms hold
    the literal bar at gain 8; at gain 24 they do not (dQ 7e-3) and cacti_hip_attention_set_exact(1)
    selects the exactly rounded forms, which do -- they are also run once on ordinary scores."""
    from cacti_amd import ffi
    ffi.call("cacti_hip_attention_set_exact", int(exact))
    try:
        _large_scores_case(ops, oracle, gain)
    finally:
        ffi.call("cacti_hip_attention_set_exact", 0)


def _large_scores_case(ops, oracle, gain):
    S, H, Dh = 384, 3, 100
    say("fused attention, large scores, gain", gain)
    r = rng(1300 + int(gain))
    alpha = float(np.float32(1.0) / np.sqrt(np.float32(Dh)))
    q, k = (randn16(r, (S, H, Dh), gain) for _ in range(2))
    v, dO = (randn16(r, (S, H, Dh)) for _ in range(2))
    ws16, _, wo = oracle.attention_fwd(q, k, v, alpha)
    low = np.arange(S)[:, None, None] >= np.arange(S)[None, None, :]
    m = np.where(low, ws16.astype(np.float32), -np.inf).max(2)
    say("  row maxima of the scores: median %.0f, largest %.0f" % (np.median(np.abs(m)), np.abs(m).max()))
    assert np.abs(m).max() > 9 * gain and np.all(np.isfinite(ws16.astype(np.float32)))
    dq_, dk_, dv_ = oracle.attention_bwd(q, k, v, dO, alpha)
    Q, K_, V_, DO = dev(q), dev(k), dev(v), dev(dO)
    o, stats = ops.attention_fwd(Q, K_, V_, alpha)
    e2, em = assert_parity(host(o), wo, "o")
    say("  o  rel_l2 %.2e max_rel %.2e" % (e2, em))
    # the forward output is handed over: rows this concentrated must all fall back to the pass over the keys
    dq, dk, dv = ops.attention_bwd(Q, K_, V_, DO, stats, alpha, o=o)
    for name, got, want in (("dv", dv, dv_), ("dq", dq, dq_), ("dk", dk, dk_)):
        e2, em = assert_parity(host(got), want, name)
        say("  %s rel_l2 %.2e max_rel %.2e" % (name, e2, em))


@pytest.mark.gpu
@pytest.mark.parametrize("S,H,Dh", [(64, 4, 64), (2048, 32, 100), (37, 4, 20), (16, 4, 6)])
def test_rope_on_two_tensors_in_one_launch(S, H, Dh):
    """cacti_hip_rope_{fwd,bwd}_pair: bit for bit what two single launches give, accumulation included
    (Dh = 6 takes the staged kernel, one launch per tensor behind the same entry point)."""
    import torch
    from cacti_amd import ffi, ops
    g = torch.Generator(device="cuda").manual_seed(S + Dh)
    x0, x1, a0, a1 = (torch.randn(S, H, Dh, device="cuda", generator=g).half() for _ in range(4))
    cos, sin = ops.rope_tables(S, Dh)
    st = torch.cuda.current_stream().cuda_stream
    y0, y1 = torch.empty_like(x0), torch.empty_like(x1)
    ffi.call("cacti_hip_rope_fwd_pair", S, H, Dh, x0.data_ptr(), x1.data_ptr(), cos.data_ptr(), sin.data_ptr(),
             y0.data_ptr(), y1.data_ptr(), st)
    assert torch.equal(y0, ops.rope_fwd(x0, cos, sin)) and torch.equal(y1, ops.rope_fwd(x1, cos, sin))
    d0, d1 = a0.clone(), torch.empty_like(x1)
    ffi.call("cacti_hip_rope_bwd_pair", S, H, Dh, x0.data_ptr(), x1.data_ptr(), cos.data_ptr(), sin.data_ptr(),
             d0.data_ptr(), 1, d1.data_ptr(), 0, st)
    w0 = a0.clone()
    ffi.call("cacti_hip_rope_bwd", S, H, Dh, x0.data_ptr(), cos.data_ptr(), sin.data_ptr(), w0.data_ptr(), 1, st)
    assert torch.equal(d0, w0) and torch.equal(d1, ops.rope_bwd(x1, cos, sin))


# dK / dV in parts of the queries (the workspace of ops) against one walk over all of them (the least workspace): parts that
# begin on the diagonal or past it, of whole tiles and of a ragged last one alone, and accumulation; heads up to 64 (two
# output tiles) and beyond, in windows too.  The first six have room for parts (577: the fewest tiles that have), and a walk that
# is the better form with either workspace: the same kernel twice
PART_SHAPES = [(577, 2, 128, True), (1000, 2, 128, False), (1025, 8, 100, False), (641, 4, 36, True), (705, 4, 64, False),
               (1500, 10, 64, True),
               (1531, 4, 100, True), (2001, 2, 100, False), (1471, 4, 128, False), (2048, 4, 128, True), (4001, 1, 64, True),
               (4096, 1, 64, False)]


@pytest.mark.parametrize("S,H,Dh,acc", PART_SHAPES)
def test_attention_bwd_in_parts(ops, S, H, Dh, acc):
    from cacti_amd import ffi
    from tests.util import rel_l2
    least, best = ffi.lib().cacti_hip_attention_bwd_workspace(S, H), ffi.lib().cacti_hip_attention_bwd_workspace_best(S, H, Dh)
    say("attention_bwd in parts", S, H, Dh, acc, least, best)
    assert best > least
    g = torch.Generator(device="cuda")
    g.manual_seed(S + H + Dh)
    q, k, v, dO, d0 = (torch.randn(S, H, Dh, generator=g, device="cuda").half() for _ in range(5))
    alpha = Dh ** -0.5
    o, stats = ops.attention_fwd(q, k, v, alpha)
    got = ops.attention_bwd(q, k, v, dO, stats, alpha, acc=tuple(d0.clone() for _ in range(3)) if acc else None, o=o)
    want = [d0.clone() for _ in range(3)]
    ws = torch.empty(least, dtype=torch.uint8, device="cuda")
    ffi.call("cacti_hip_attention_bwd", S, H, Dh, alpha, q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(), dO.data_ptr(), H * Dh,
             stats.data_ptr(), want[0].data_ptr(), int(acc), want[1].data_ptr(), int(acc), want[2].data_ptr(), int(acc),
             ws.data_ptr(), least, torch.cuda.current_stream().cuda_stream)
    assert_bits(host(got[0]), host(want[0]), "dq")
    for a, b in zip(got[1:], want[1:]):
        # fp32 sums of the same terms in another order, rounded once: a last place (2^-11 of it) here and there
        assert rel_l2(host(a), host(b)) < 2e-4 and exact_frac(host(a), host(b)) > 0.95


# (the last three: the default arithmetic has parts there; the others: room for some)
@pytest.mark.parametrize("S,H,Dh", [(577, 2, 128), (1000, 4, 100), (705, 4, 64), (1531, 4, 100), (1471, 4, 128), (4001, 1, 64)])
def test_attention_bwd_exact_has_no_parts(ops, S, H, Dh):
    """The exact arithmetic asks for no scratch for parts and takes the same kernels whatever the workspace: the same bits
    with the least one and with one that the default arithmetic can have parts in."""
    from cacti_amd import ffi
    best = ffi.lib().cacti_hip_attention_bwd_workspace_best(S, H, Dh)
    least = ffi.lib().cacti_hip_attention_bwd_workspace(S, H)
    assert best > least
    say("attention_bwd, exact", S, H, Dh)
    g = torch.Generator(device="cuda")
    g.manual_seed(S + H + Dh)
    q, k, v, dO = (torch.randn(S, H, Dh, generator=g, device="cuda").half() for _ in range(4))
    alpha, st = Dh ** -0.5, torch.cuda.current_stream().cuda_stream
    ffi.call("cacti_hip_attention_set_exact", 1)
    try:
        o, stats = ops.attention_fwd(q, k, v, alpha)
        assert ffi.lib().cacti_hip_attention_bwd_workspace_best(S, H, Dh) == least
        got = []
        for size in (least, best):
            ws = torch.empty(size, dtype=torch.uint8, device="cuda")
            d = [torch.empty_like(q) for _ in range(3)]
            ffi.call("cacti_hip_attention_bwd", S, H, Dh, alpha, q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(), dO.data_ptr(),
                     H * Dh, stats.data_ptr(), d[0].data_ptr(), 0, d[1].data_ptr(), 0, d[2].data_ptr(), 0, ws.data_ptr(), size, st)
            got.append([host(t) for t in d])
    finally:
        ffi.call("cacti_hip_attention_set_exact", 0)
    for name, a, b in zip(("dq", "dk", "dv"), *got):
        assert_bits(a, b, name)


def test_attention_bwd_scratch_of_rows_without_parts(ops):
    """1000 positions of 3 heads of 100: rows of 300 elements, which no kernel with parts takes; the operator allocates its
    results and the least workspace (each rounded up by the allocator), not 19 MB of fp32 planes."""
    S, H, Dh = 1000, 3, 100
    q, k, v, dO = (torch.randn(S, H, Dh, device="cuda").half() for _ in range(4))
    o, stats = ops.attention_fwd(q, k, v, 0.1)
    torch.cuda.synchronize()
    before = torch.cuda.memory_allocated()
    torch.cuda.reset_peak_memory_stats()
    ops.attention_bwd(q, k, v, dO, stats, 0.1, o=o)
    taken, room = torch.cuda.max_memory_allocated() - before, 3 * q.nbytes + 8 * S * H + 4 * 512
    assert taken <= room


# with parts, then with a walk over all queries although a device of so few workgroups had room for parts, rows without direct tiles
# (heads off the 16-byte grid, a window beyond the row's end), and shapes without parts
@pytest.mark.parametrize("S,H,Dh,ld,parts", [(1531, 4, 100, 400, 5), (1471, 4, 128, 520, 5), (4001, 1, 64, 64, 8),
                                             (1000, 4, 100, 400, 0), (577, 2, 128, 256, 0), (2048, 8, 128, 1024, 0),
                                             (1531, 3, 100, 300, 0), (1531, 3, 100, 304, 6), (1531, 4, 100, 404, 0), (2048, 32, 100, 3200, 0), (128, 4, 64, 256, 0)])
def test_attention_bwd_scratch_is_what_its_kernels_use(ops, S, H, Dh, ld, parts):
    """What the operator allocates and a context's pool lends beside the results: the statistics, and the fp32 planes of the parts
    where the kernel with parts is the one that runs (256 compute units); the exact arithmetic has none."""
    from cacti_amd import ffi
    L = ffi.lib()
    least = L.cacti_hip_attention_bwd_workspace(S, H)
    want = -(-least // 16) * 16 + parts * 2 * H * S * Dh * 4 if parts else least
    assert L.cacti_hip_attention_bwd_workspace_used(S, H, Dh, ld) == want <= L.cacti_hip_attention_bwd_workspace_best(S, H, Dh)
    ffi.call("cacti_hip_attention_set_exact", 1)
    try:
        assert L.cacti_hip_attention_bwd_workspace_used(S, H, Dh, ld) == least
    finally:
        ffi.call("cacti_hip_attention_set_exact", 0)
    if ld != H * Dh:
        return
    q, k, v, dO = (torch.randn(S, H, Dh, device="cuda").half() for _ in range(4))
    o, stats = ops.attention_fwd(q, k, v, 0.1)
    torch.cuda.synchronize()
    before = torch.cuda.memory_allocated()
    torch.cuda.reset_peak_memory_stats()
    ops.attention_bwd(q, k, v, dO, stats, 0.1, o=o)
    # (the allocator leaves up to 1 MiB of a block with the tensor in it)
    assert torch.cuda.max_memory_allocated() - before <= 3 * q.nbytes + want + (4 << 20)


@pytest.mark.parametrize("S,H,Dh", [(577, 2, 128), (576, 2, 128), (611, 16, 64), (777, 16, 128), (449, 3, 100), (1000, 2, 128),
                                    (1025, 8, 100), (2048, 32, 100), (128, 4, 64)])
def test_attention_bwd_parts_fill_this_device(S, H, Dh):
    """As many parts as this device has compute units for, whatever their number, and at most 8, where a part is at least 8
    tiles shorter than the whole walk; no scratch for parts anywhere else."""
    from cacti_amd import ffi
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    tiles, split = -(-S // 64), min(cus // (-(-S // 128) * H), 8)
    least = ffi.lib().cacti_hip_attention_bwd_workspace(S, H)
    want = least
    if split >= 2:
        per = max(2, -(-tiles // split))
        if tiles - per >= 8:
            want = -(-least // 16) * 16 + -(-tiles // per) * 2 * H * S * Dh * 4
    assert ffi.lib().cacti_hip_attention_bwd_workspace_best(S, H, Dh) == want
