"""End-to-end: the tiny LLaMA cycle staged on the spine (reset / stage / vadd_vjp / compile /
resume / resume_put) against the CPU oracle, every parameter gradient (MI355X)."""
import numpy as np
import pytest

from tests.llama_ref import make_inputs
from tests.util import assert_parity, rel_l2, max_rel

pytestmark = pytest.mark.gpu

TINY = dict(S=128, D=256, H=4, Dh=64, F=688, V=1024, L=2, eps=1e-6)


def _model(cfg, pool_bytes=1 << 30, pagelocked=True):
    from cacti_amd.runtime import Ctx, Llama
    ctx = Ctx(0, pool_bytes, pagelocked)
    m = Llama(ctx, cfg.S, cfg.D, cfg.H, cfg.Dh, cfg.F, cfg.V, cfg.L, cfg.eps)
    return ctx, m


def _compare(oracle, cfg, m, ref, env, tag):
    """Every gradient tensor of the device against the oracle's default run, held to the summation-order
    envelope (tests/envelope.py): no further from the oracle than the oracle's own runs with other valid
    fp32 summation orders are from each other, ratio <= 1.0 per tensor."""
    from tests.envelope import assert_inside_envelope
    grads = m.grads()
    assert len(grads) == 3 + 9 * cfg.L
    return assert_inside_envelope(grads, oracle.split_params(cfg, ref["grad"]), env, tag)


@pytest.mark.parametrize("attention", ["fused", "thunks"])
def test_tiny_llama_step_all_gradients(oracle, attention):
    """Healthy-range variant: norm weights ~N(1, 0.02), grad_scale 1024 (the example's); the attention
    block staged as the fused thunk and as the reference's chain of separate thunks."""
    cfg, flat, tok, lm_tok, scale = make_inputs(TINY, seed=0, norm_mean=1.0, grad_scale=1024.0)
    ref = oracle.llama_step(cfg, flat, tok, lm_tok, scale)
    ctx, m = _model(cfg)
    m.set_attention(attention)
    m.put_params_flat(flat)
    out = m.step_explicit(tok, lm_tok, scale, want_prob=True)
    assert_parity(out["loss"], ref["loss"], "loss", l2=1e-4, mx=1e-3)
    assert_parity(out["logit"], ref["logit"], "logit")
    assert np.mean(out["amax"] == ref["amax"]) > 0.99       # ties in f16 logits may differ
    assert abs(out["prob"].sum(1) - 1).max() < 1e-4
    from tests.envelope import order_envelope
    _, env = order_envelope(oracle, cfg, flat, tok, lm_tok, scale)
    _compare(oracle, cfg, m, ref, env, "healthy")
    # and against exact arithmetic (fp64 autograd): no further from the truth than the oracle is
    from tests.llama_ref import torch_step
    _, g64, _ = torch_step(cfg, oracle.split_params(cfg, flat), tok, lm_tok, scale)
    want = oracle.split_params(cfg, ref["grad"])
    for name, g in m.grads().items():
        assert rel_l2(g, g64[name]) <= 1.15 * rel_l2(want[name], g64[name]) + 1e-4, name
    names = ctx.log_names()
    assert names.count("yield_set") == 3 and "unlive" in names and "rms_norm_bwd" in names
    assert ("attention_bwd" in names) == (attention == "fused")
    assert ("causal_softmax_bwd" in names) == (attention == "thunks")
    # a second cycle on the same context (reset GCs the first one's cells) gives the same result
    g1 = m.grads()
    loss2 = m.step(tok, lm_tok, scale)
    assert np.array_equal(loss2, out["loss"])
    for name, g in m.grads().items():
        assert np.array_equal(g.view(np.uint16), g1[name].view(np.uint16)), name
    m.close(); ctx.close()


def test_grouped_products_are_the_separate_thunks_bit_for_bit():
    """Small shapes (outputs of at most 2^18 elements): the grouped stagings of the projections and
    of their weight gradients (modes 1 and 2) give the loss and all gradients of the separate matmul thunks
    (mode 0), bit for bit."""
    cfg, flat, tok, lm_tok, scale = make_inputs(TINY, seed=3, norm_mean=1.0, grad_scale=1024.0)
    got = {}
    for groups in (0, 1, 2):
        ctx, m = _model(cfg)
        m.set_product_groups(groups)
        m.put_params_flat(flat)
        got[groups] = (m.step(tok, lm_tok, scale), m.grads())
        m.close(); ctx.close()
    for groups in (1, 2):
        assert np.array_equal(got[groups][0], got[0][0])
        for n, g in got[groups][1].items():
            assert np.array_equal(g.view(np.uint16), got[0][1][n].view(np.uint16)), (groups, n)


# a sequence of odd length and products of more than 2^18 outputs: the weight gradients sum over 203 positions (a k tile of 64
# ends inside them), and the forward products of the FFN and the head, and all weight gradients but the norms', are past the
# line up to which the tiny model's products keep the instruction of the register path
RAGGED = dict(S=203, D=544, H=8, Dh=68, F=1376, V=2048, L=1, eps=1e-6)


def test_ragged_llama_step_all_gradients(oracle):
    from tests.envelope import order_envelope
    cfg, flat, tok, lm_tok, scale = make_inputs(RAGGED, seed=12, norm_mean=1.0, grad_scale=1024.0)
    ref = oracle.llama_step(cfg, flat, tok, lm_tok, scale)
    ctx, m = _model(cfg)
    m.put_params_flat(flat)
    assert_parity(m.step(tok, lm_tok, scale), ref["loss"], "loss", l2=1e-4, mx=1e-3)
    _, env = order_envelope(oracle, cfg, flat, tok, lm_tok, scale)
    _compare(oracle, cfg, m, ref, env, "ragged")
    m.close(); ctx.close()


def test_grouped_products_of_a_ragged_sequence_are_the_separate_thunks_bit_for_bit():
    cfg, flat, tok, lm_tok, scale = make_inputs(RAGGED, seed=13, norm_mean=1.0, grad_scale=1024.0)
    got = {}
    for groups in (0, 1, 2):
        ctx, m = _model(cfg)
        m.set_product_groups(groups)
        m.put_params_flat(flat)
        got[groups] = (m.step(tok, lm_tok, scale), m.grads())
        m.close(); ctx.close()
    for groups in (1, 2):
        assert np.array_equal(got[groups][0], got[0][0])
        for n, g in got[groups][1].items():
            assert np.array_equal(g.view(np.uint16), got[0][1][n].view(np.uint16)), (groups, n)


@pytest.mark.parametrize("L,thunks", [(7, 1), (8, 2)])
def test_norm_gradients_summed_together(oracle, L, thunks):
    """The sums of the norms' weight gradients wait for one another, up to 16 (7 layers have 15 norms, 8 have 17): each no further
    from the oracle than its own other summation orders are, and twice itself, bit for bit, once a second cycle of the same batch
    has added to it."""
    from tests.envelope import order_envelope
    cfg, flat, tok, lm_tok, scale = make_inputs(dict(S=41, D=64, H=2, Dh=32, F=176, V=256, L=L, eps=1e-6), seed=L, norm_mean=1.0,
                                                grad_scale=64.0)
    ref = oracle.llama_step(cfg, flat, tok, lm_tok, scale)
    ctx, m = _model(cfg)
    m.put_params_flat(flat)
    m.step(tok, lm_tok, scale)
    assert ctx.log_names().count("rms_norm_dw") == thunks
    _, env = order_envelope(oracle, cfg, flat, tok, lm_tok, scale)
    once, want = m.grads(), oracle.split_params(cfg, ref["grad"])
    for name in [n for n in once if n.endswith("norm")]:
        assert rel_l2(once[name], want[name]) <= env[name][0], name
    m.step(tok, lm_tok, scale, accumulate=True)
    for name, g in m.grads().items():
        if name.endswith("norm"):
            assert np.array_equal(g, once[name] + once[name]), name
    m.close(); ctx.close()


def test_sums_of_another_number_of_norms_are_timed_apart():
    """17 norms are a launch of 16 and one of 1: a label each, whose bytes are those of its launches (G partial rows of D values, f32,
    read and D written, f16, by each sum; read as well where they are added to)."""
    cfg, flat, tok, lm_tok, scale = make_inputs(dict(S=41, D=64, H=2, Dh=32, F=176, V=256, L=8, eps=1e-6), seed=8, norm_mean=1.0)
    ctx, m = _model(cfg)
    m.put_params_flat(flat)
    ctx.set_timing(2)
    m.step(tok, lm_tok, scale)
    m.step(tok, lm_tok, scale, accumulate=True)
    ctx.sync()
    rep = {k: v for k, v in ctx.timing_report().items() if k.startswith("rms_norm_dw")}
    G = 6                                                   # eight rows to a workgroup of the adjoint
    assert {k: (n, ctx.operand_bytes[k]) for k, (n, _) in rep.items()} == {
        "rms_norm_dw[%dx64]x16" % G: (1, 16 * (G * 256 + 128)), "rms_norm_dw[%dx64]x1" % G: (1, G * 256 + 128),
        "rms_norm_dw[%dx64,accffff]x16" % G: (1, 16 * (G * 256 + 256)), "rms_norm_dw[%dx64,acc1]x1" % G: (1, G * 256 + 256)}
    ctx.set_timing(0)
    m.close(); ctx.close()


@pytest.mark.parametrize("S,V,D,F", [(64, 8192, 64, 648), (37, 4104, 64, 648), (40, 8192, 256, 3080)])
def test_products_in_parts_of_k(oracle, S, V, D, F):
    """The head's input gradient, and the last time the FFN's last product, as sums of parts (one to four tiles of 64 x 64, K of 3080 to
    8192, a k tile that ends inside K): every gradient no further from the oracle than its own other summation orders are, the same bits from
    every staging of the products and in a pool that spills (the two V x D weights, their gradients and nothing else fit)."""
    from tests.envelope import order_envelope
    cfg, flat, tok, lm_tok, scale = make_inputs(dict(S=S, D=D, H=D // 32, Dh=32, F=F, V=V, L=1, eps=1e-6), seed=S, norm_mean=1.0,
                                                grad_scale=64.0)
    ref = oracle.llama_step(cfg, flat, tok, lm_tok, scale)
    _, env = order_envelope(oracle, cfg, flat, tok, lm_tok, scale)
    want, first = oracle.split_params(cfg, ref["grad"]), None
    for groups, pool in ((2, 1 << 30), (1, 1 << 30), (0, 1 << 30), (2, 8 * D * V)):
        ctx, m = _model(cfg, pool_bytes=pool)
        m.set_product_groups(groups)
        m.put_params_flat(flat)
        ctx.set_timing(2)
        assert_parity(m.step(tok, lm_tok, scale), ref["loss"], "loss", l2=1e-4, mx=1e-3)
        ctx.sync()
        labels = list(ctx.timing_report())
        for name, K in (("NN", V), ("NT", F))[:1 if F == 648 else 2]:           # their labels say so
            assert any(l.startswith("matmul[%s,1x%dx%dx%d,parts" % (name, S, D, K)) for l in labels), labels
        got = m.grads()
        if pool < 1 << 30:
            assert ctx.stats()["n_evict"] > 0
        m.close(); ctx.close()
        first = first or got
        for name, g in got.items():
            assert rel_l2(g, want[name]) <= env[name][0], name
            assert np.array_equal(g.view(np.uint16), first[name].view(np.uint16)), (groups, pool, name)


def test_tiny_llama_literal_config(oracle):
    """The reference's small training configuration as written: every weight ~N(0, 0.02), loss scale 1/(S-1).
    The q/k/gate/up/down gradients (1e-8 .. 1e-11) underflow f16 in the reference's own
    arithmetic, so those tensors are compared in absolute terms (f16 subnormal quanta)."""
    cfg, flat, tok, lm_tok, scale = make_inputs(TINY, seed=0)
    ref = oracle.llama_step(cfg, flat, tok, lm_tok, scale)
    ctx, m = _model(cfg)
    m.put_params_flat(flat)
    loss = m.step(tok, lm_tok, scale)
    assert_parity(loss, ref["loss"], "loss", l2=1e-4, mx=1e-3)
    want = oracle.split_params(cfg, ref["grad"])
    for name, g in m.grads().items():
        w = want[name].astype(np.float64)
        rms = np.sqrt(np.mean(w * w))
        if rms > 2.0 ** -14:                                  # normal f16 range
            assert_parity(g, want[name], name)
        else:
            # within a few f16 subnormal quanta (2^-24) everywhere
            assert np.max(np.abs(g.astype(np.float64) - w)) <= 8 * 2.0 ** -24, name
    m.close(); ctx.close()


def test_bad_token_is_an_error(oracle):
    from cacti_amd.ffi import CactiError
    cfg, flat, tok, lm_tok, scale = make_inputs(dict(TINY, S=16, L=1), seed=1)
    ctx, m = _model(cfg)
    m.put_params_flat(flat)
    bad = lm_tok.copy(); bad[3] = cfg.V
    with pytest.raises(CactiError) as e:
        m.step(tok, bad, scale)
    assert e.value.code == -3
    m.step(tok, lm_tok, scale)                                # the context stays usable
    m.close(); ctx.close()


@pytest.mark.parametrize("pagelocked", [True, False])
def test_capped_pool_spills_and_matches(oracle, pagelocked):
    """Pool capped below the step's footprint: live cells spill to host memory and are
    re-uploaded; results are bit-identical to the uncapped run."""
    cfg, flat, tok, lm_tok, scale = make_inputs(TINY, seed=2, norm_mean=1.0, grad_scale=1024.0)
    ctx, m = _model(cfg)
    m.put_params_flat(flat)
    loss_a = m.step(tok, lm_tok, scale)
    ga = m.grads()
    peak = ctx.stats()["pool_peak"]
    m.close(); ctx.close()
    cap = int(peak * 0.45)
    ctx, m = _model(cfg, pool_bytes=cap, pagelocked=pagelocked)
    m.put_params_flat(flat)
    loss_b = m.step(tok, lm_tok, scale)
    st = ctx.stats()
    print("peak %d cap %d evictions %d d2h %d h2d %d" % (peak, st["pool_cap"], st["n_evict"],
                                                       st["bytes_d2h"], st["bytes_h2d"]), flush=True)
    assert st["n_evict"] > 0 and st["bytes_d2h"] > 0 and st["pool_peak"] <= st["pool_cap"]
    assert np.array_equal(loss_a, loss_b)
    for name, g in m.grads().items():
        assert np.array_equal(g.view(np.uint16), ga[name].view(np.uint16)), name
    m.close(); ctx.close()


def test_grouped_products_run_one_by_one_in_a_pool_too_small_for_the_group():
    """The three projections of a layer and their weight gradients are one thunk each by default; a pool with room for
    one weight matrix of 2 MiB at a time, but not for three, runs them one after another, with the same bits."""
    wide = dict(S=136, D=1024, H=8, Dh=128, F=1024, V=1024, L=1, eps=1e-6)
    cfg, flat, tok, lm_tok, scale = make_inputs(wide, seed=8, norm_mean=1.0, grad_scale=1024.0)
    got = []
    for pool in (1 << 30, 5 << 20):
        ctx, m = _model(cfg, pool_bytes=pool)
        m.put_params_flat(flat)
        got.append((m.step(tok, lm_tok, scale), m.grads()))
        m.close(); ctx.close()
    assert np.array_equal(got[0][0], got[1][0])
    for n, g in got[1][1].items():
        assert np.array_equal(g.view(np.uint16), got[0][1][n].view(np.uint16)), n


def test_timing_labels_of_gradients_in_one_launch():
    """The first micro-batch writes the weights' gradients and the second adds to them: timing entries of their own, with the operand
    bytes of each; the benchmark takes them for the products they are."""
    import bench
    S, D, F = 128, 256, 256
    cfg, flat, tok, lm_tok, scale = make_inputs(dict(S=S, D=D, H=4, Dh=64, F=F, V=512, L=1, eps=1e-6), seed=3, norm_mean=1.0, grad_scale=1024.0)
    ctx, m = _model(cfg, pool_bytes=1 << 30)
    m.put_params_flat(flat)
    ctx.set_timing(2)
    m.step(tok, lm_tok, scale)
    m.step(tok, lm_tok, scale, accumulate=True)
    rep = ctx.timing_report()
    first, more = "matmul_grads[%dx%dx%d]x3" % (S, D, D), "matmul_grads[%dx%dx%d,acce]x3" % (S, D, D)
    assert rep[first][0] == 1 and rep[more][0] == 1, sorted(rep)
    # dy, W and x are read, dx and dW written, the latter read first as well
    least = 2 * (3 * S * D + 3 * D * D + S * D + S * D + 3 * D * D)
    assert ctx.operand_bytes[first] == least and ctx.operand_bytes[more] == least + 2 * 3 * D * D
    assert bench.gemm_flops(first) == bench.gemm_flops(more) == 3 * 2 * 2.0 * S * D * D and bench.kernel_symbol(first) is bench.kernel_symbol(more) is None
    m.close(); ctx.close()


# (1024 positions have room for parts only; a walk over all queries is the better form, so that the smaller pool has what it wants)
@pytest.mark.parametrize("S,cap,parts", [(1024, 24 << 20, False), (1531, 24400000, True)])
def test_attention_scratch_gives_way_to_a_capped_pool(oracle, S, cap, parts):
    """A pool with room for the least scratch of the attention adjoint, but not for what it is fastest with (24.5 MB of fp32
    partial sums at 1531 positions, 4 heads of 100): the cycle runs, with the results of the larger pool up to the
    order of those sums (fp32, rounded once: rel-L2 below one f16 rounding, 2^-11, through the layer below)."""
    from cacti_amd import ffi
    big = dict(S=S, D=400, H=4, Dh=100, F=416, V=512, L=1, eps=1e-6)
    cfg, flat, tok, lm_tok, scale = make_inputs(big, seed=5, norm_mean=1.0, grad_scale=1024.0)
    assert ffi.lib().cacti_hip_attention_bwd_workspace_best(S, 4, 100) > cap > 2 * ffi.lib().cacti_hip_attention_bwd_workspace(S, 4)
    assert (ffi.lib().cacti_hip_attention_bwd_workspace_used(S, 4, 100, 400) > cap) == parts
    got = []
    for pool in (1 << 30, cap):
        ctx, m = _model(cfg, pool_bytes=pool)
        m.put_params_flat(flat)
        got.append((m.step(tok, lm_tok, scale), m.grads()))
        m.close(); ctx.close()
    assert np.array_equal(got[0][0], got[1][0])
    for n, g in got[1][1].items():
        assert rel_l2(g, got[0][1][n]) < 5e-4, n


def test_attention_scratch_of_a_walk_over_all_queries_is_the_least():
    """1000 positions of 4 heads of 100 have no parts of the queries although there is room for some: the pool of a cycle in the
    default arithmetic is no larger than in the exact one, which never has parts (25.6 MB of fp32 sums)."""
    from cacti_amd import ffi
    cfg, flat, tok, lm_tok, scale = make_inputs(dict(S=1000, D=400, H=4, Dh=100, F=416, V=512, L=1, eps=1e-6), seed=5, norm_mean=1.0,
                                                grad_scale=1024.0)
    peaks = []
    for exact in (1, 0):
        ffi.call("cacti_hip_attention_set_exact", exact)
        try:
            ctx, m = _model(cfg, pool_bytes=1 << 30)
            m.put_params_flat(flat)
            m.step(tok, lm_tok, scale)
            peaks.append(ctx.stats()["pool_peak"])
            m.close(); ctx.close()
        finally:
            ffi.call("cacti_hip_attention_set_exact", 0)
    assert peaks[1] == peaks[0]


@pytest.mark.parametrize("capped", [False, True])
def test_digests_of_parameters_and_gradients(oracle, capped):
    """abs_log2_hist8 and nan_count of every parameter and gradient after a cycle, as the
    reference's example takes them (examples/open_llama_3b_train.rs:409-424): bit-exact against
    the oracle's digests of the same tensors; also with cells spilled to the host in between."""
    cfg, flat, tok, lm_tok, scale = make_inputs(TINY, seed=4, norm_mean=1.0, grad_scale=1024.0)
    ctx, m = _model(cfg)
    m.put_params_flat(flat)
    m.step(tok, lm_tok, scale)
    if capped:
        peak = ctx.stats()["pool_peak"]
        m.close(); ctx.close()
        ctx, m = _model(cfg, pool_bytes=int(peak * 0.45))
        m.put_params_flat(flat)
        m.step(tok, lm_tok, scale)
    grads = m.grads()
    gh, gn = m.digests(of_grads=True)
    ph, pn = m.digests(of_grads=False)
    want_p = oracle.split_params(cfg, flat)
    for i, (name, shape) in enumerate(m.params):
        assert np.array_equal(gh[i], oracle.abs_log2_hist8(grads[name])), name
        assert gn[i] == oracle.nan_count(grads[name]) == 0, name
        assert np.array_equal(ph[i], oracle.abs_log2_hist8(want_p[name])), name
        assert pn[i] == 0 and ph[i].sum() == int(np.prod(shape)), name
    m.close(); ctx.close()


@pytest.mark.parametrize("capped", [False, True])
def test_adamw_steps_between_cycles(oracle, capped):
    """The example's minibatch loop (examples/open_llama_3b_train.rs:230-268): master = cast(param),
    zeroed averages, then cycle -> AdamW32 step -> cycle -> step.  Averages, master weights and the
    f16 parameters are bit-exact against the oracle's thunks applied to the gradients the device
    produced; the embedding stays as it was when skipped; the second cycle runs on the updated
    parameters (its loss differs).  Also with a pool so small that the optimiser state spills."""
    opt = dict(grad_scale=1024.0, lr=2.0e-3, wd=0.1, a1=0.1, a2=0.05, eps=1.0e-5)
    cfg, flat, tok, lm_tok, scale = make_inputs(TINY, seed=6, norm_mean=1.0, grad_scale=1024.0)
    ctx, m = _model(cfg)
    m.put_params_flat(flat)
    m.step(tok, lm_tok, scale)
    if capped:
        peak = ctx.stats()["pool_peak"]
        m.close(); ctx.close()
        ctx, m = _model(cfg, pool_bytes=int(peak))          # the cycle fits, the f32 optimiser state does not
        m.put_params_flat(flat)
    want_p = oracle.split_params(cfg, flat)
    names = [n for n, _ in m.params]
    master = {n: want_p[n].astype(np.float32) for n in names}
    avg = {n: np.zeros(want_p[n].shape, np.float32) for n in names}
    avg2 = {n: np.zeros(want_p[n].shape, np.float32) for n in names}
    m.adamw_init()
    losses = []
    for it in (1, 2):
        losses.append(m.step(tok, lm_tok, scale))
        grads = m.grads()
        m.adamw_step(it, skip_embed=(it == 1), **opt)
        sc = oracle.adamw32_scalars(it, **opt)
        for i, n in enumerate(names):
            if it == 1 and n == "embed":
                p16 = want_p[n]
            else:
                avg[n], avg2[n], master[n], p16 = oracle.adamw32_step(grads[n], avg[n], avg2[n], master[n], sc)
                want_p[n] = p16
            assert np.array_equal(m.adamw_state(i, "grad_avg").view(np.uint32), avg[n].view(np.uint32)), (it, n)
            assert np.array_equal(m.adamw_state(i, "grad2_avg").view(np.uint32), avg2[n].view(np.uint32)), (it, n)
            assert np.array_equal(m.adamw_state(i, "master").view(np.uint32), master[n].view(np.uint32)), (it, n)
            assert np.array_equal(m.param(i).view(np.uint16), p16.view(np.uint16)), (it, n)
    assert not np.array_equal(losses[0], losses[1])
    if capped:
        assert ctx.stats()["n_evict"] > 0
    from cacti_amd.ffi import CactiError
    with pytest.raises(CactiError) as e:
        m.adamw_step(0, **opt)
    assert e.value.code == -1
    m.close(); ctx.close()


def test_training_cycles_follow_the_oracle(oracle):
    """The example's loop end to end (examples/open_llama_3b_train.rs:223-531 with one cycle per
    minibatch): cycle -> AdamW32 step on every parameter but the embedding -> cycle ...; four cycles on
    the device against four cycles of the oracle (its own gradients, its own optimiser): per-cycle
    losses agree, the loss of the repeated batch goes down, and the parameters stay together."""
    opt = dict(grad_scale=1024.0, lr=1.0e-3, wd=0.1, a1=0.1, a2=0.05, eps=1.0e-5)
    cfg, flat, tok, lm_tok, scale = make_inputs(TINY, seed=9, norm_mean=1.0, grad_scale=1024.0)
    ctx, m = _model(cfg)
    m.put_params_flat(flat)
    m.adamw_init()
    names = [n for n, _ in m.params]
    o_p = {n: v.copy() for n, v in oracle.split_params(cfg, flat).items()}
    o_master = {n: o_p[n].astype(np.float32) for n in names}
    o_avg = {n: np.zeros(o_p[n].shape, np.float32) for n in names}
    o_avg2 = {n: np.zeros(o_p[n].shape, np.float32) for n in names}
    live = scale > 0
    g_losses, o_losses = [], []
    for it in range(1, 5):
        g_loss = m.step(tok, lm_tok, scale)
        m.adamw_step(it, skip_embed=True, **opt)
        oflat = np.concatenate([o_p[n].reshape(-1) for n in names])
        ref = oracle.llama_step(cfg, oflat, tok, lm_tok, scale)
        og = oracle.split_params(cfg, ref["grad"])
        sc = oracle.adamw32_scalars(it, **opt)
        for n in names[1:]:
            o_avg[n], o_avg2[n], o_master[n], o_p[n] = oracle.adamw32_step(og[n], o_avg[n], o_avg2[n], o_master[n], sc)
        g_losses.append(float(g_loss[live].mean()))
        o_losses.append(float(ref["loss"][live].mean()))
        assert abs(g_losses[-1] - o_losses[-1]) < 2e-3 * abs(o_losses[-1]), (it, g_losses, o_losses)
    assert g_losses[-1] < g_losses[0] - 0.05 and o_losses[-1] < o_losses[0] - 0.05, (g_losses, o_losses)
    for i, n in enumerate(names):
        got, want = m.param(i), o_p[n]
        if n == "embed":
            assert np.array_equal(got.view(np.uint16), want.view(np.uint16))
            continue
        # the step of one cycle is ~lr per element: two runs whose gradients differ in the last
        # bits stay within a small fraction of the total movement
        moved = np.abs(want.astype(np.float32) - oracle.split_params(cfg, flat)[n].astype(np.float32)).max()
        diff = np.abs(got.astype(np.float32) - want.astype(np.float32)).max()
        assert moved > 1e-3 and diff <= 0.35 * moved, (n, moved, diff)
    m.close(); ctx.close()


def test_adamw_step_before_init_is_a_state_error(oracle):
    from cacti_amd.ffi import CactiError
    cfg, flat, tok, lm_tok, scale = make_inputs(TINY, seed=6)
    ctx, m = _model(cfg)
    with pytest.raises(CactiError) as e:
        m.adamw_step(1)
    assert e.value.code == -5
    m.close(); ctx.close()


def test_pool_too_small_is_a_clean_error(oracle):
    from cacti_amd.ffi import CactiError
    cfg, flat, tok, lm_tok, scale = make_inputs(TINY, seed=3)
    ctx, m = _model(cfg, pool_bytes=1 << 19)                  # the head's weight alone fills it
    m.put_params_flat(flat)
    with pytest.raises(CactiError) as e:
        m.step(tok, lm_tok, scale)
    assert e.value.code == -4
    assert "pinned by the running thunk" in str(e.value) and "largest free" in str(e.value)
    # the usage table by class of cell (the reference dumps it before it panics, src/pctx/nvgpu.rs:2424-2440)
    rep = ctx.usage_report()
    print(rep)
    lines = rep.splitlines()
    assert lines[0].startswith("pool: cap=%d " % (1 << 19))
    assert [l.split()[0] for l in lines[1:6]] == ["parameters", "gradients", "optimiser", "tables,", "cycle"]
    n_par = int(lines[1].split("cells=")[1].split()[0])
    assert n_par == 3 + 9 * cfg.L and int(lines[2].split("cells=")[1].split()[0]) == n_par
    m.close(); ctx.close()


def test_full_size_step_properties():
    """The reference's 3B configuration at full shapes (S=2048, D=3200, H=32 x 100, F=8640, V=32000) with
    4 of the 26 layers (the oracle would need a minute per layer): properties that hold at any
    size.  (a) the loss is -log softmax(logit)[target] of the logits the step returns, recomputed
    in fp64; (b) a second cycle is bit-identical; (c) doubling the loss scale (a power of two)
    doubles the gradients: every product and sum on the adjoint path is homogeneous in the
    scale, so elements differ only where a value on the way was an f16 subnormal; (d) embedding rows
    of ids that do not occur get a zero gradient, rows that occur a non-zero one."""
    import bench
    from cacti_amd.runtime import Ctx, Llama
    cfg = dict(bench.LLAMA_3B, L=4)
    ctx = Ctx(0, 24 << 30, True)
    m = Llama(ctx, **cfg)
    bench.synth_params(m)
    tok, lm_tok, scale = bench.synth_inputs(cfg, grad_scale=8192.0)
    out = m.step_explicit(tok, lm_tok, scale)
    lg = out["logit"].astype(np.float64)
    lse = np.log(np.exp(lg - lg.max(1, keepdims=True)).sum(1)) + lg.max(1)
    want_loss = lse - lg[np.arange(cfg["S"]), lm_tok]
    assert np.all(np.isfinite(out["loss"]))
    assert np.abs(out["loss"] - want_loss).max() < 2e-3 * max(1.0, np.abs(want_loss).max())
    assert np.mean(out["amax"] == lg.argmax(1)) > 0.999

    idx = {name: i for i, (name, _) in enumerate(m.params)}
    probe = ["embed", "l0.q", "l0.pre_norm", "l1.down", "l3.gate", "l3.v", "head_norm", "lm_head"]
    g1 = {n: m.grad(idx[n]) for n in probe}
    m.step(tok, lm_tok, scale, want_loss=False)
    for n in probe:
        assert np.array_equal(m.grad(idx[n]).view(np.uint16), g1[n].view(np.uint16)), n

    present = np.zeros(cfg["V"], bool)
    present[tok] = True
    rows = np.abs(g1["embed"].astype(np.float32)).max(1)
    assert np.all(rows[~present] == 0) and np.mean(rows[present] > 0) > 0.99

    m.step(tok, lm_tok, 2.0 * scale, want_loss=False)
    tiny = 2.0 ** -14
    for n in probe:
        a, b = g1[n].astype(np.float32), m.grad(idx[n]).astype(np.float32)
        ok = (np.abs(a) >= tiny) & (np.abs(b) < 65504)
        assert ok.mean() > 0.03, (n, ok.mean())      # embed: only rows of ids that occur
        same = float(np.mean(b[ok] == 2.0 * a[ok]))
        err = rel_l2(b, 2.0 * a)
        print("scale x2: %-12s %.4f of the normal elements doubled exactly, rel_l2 %.2e" % (n, same, err),
              flush=True)
        assert err < 5e-3, (n, same, err)
    m.close(); ctx.close()


@pytest.mark.gpu
def test_cached_gradients_accumulate_micro_batches(oracle):
    """Two micro-batches with the gradients cached in between (g.cache(),
    examples/open_llama_3b_train.rs:334-345) against the oracle doing the same; caching before any cycle
    has written the gradients is an error; a plain cycle afterwards overwrites again."""
    from cacti_amd.ffi import CactiError
    cfg, flat, tok, lm_tok, scale = make_inputs(TINY, seed=0, norm_mean=1.0, grad_scale=1024.0)
    _, _, tok2, lm_tok2, _ = make_inputs(TINY, seed=17, norm_mean=1.0, grad_scale=1024.0)
    ctx, m = _model(cfg)
    m.put_params_flat(flat)
    with pytest.raises(CactiError) as e:
        m.step(tok, lm_tok, scale, accumulate=True)
    assert e.value.code == -5
    m.step(tok, lm_tok, scale)
    first = m.grads()
    loss2 = m.step(tok2, lm_tok2, scale, accumulate=True)
    a = oracle.llama_step(cfg, flat, tok, lm_tok, scale)
    ab = oracle.llama_step(cfg, flat, tok2, lm_tok2, scale, grad_cached=a["grad"])
    assert_parity(loss2, ab["loss"], "loss", l2=1e-4, mx=1e-3)
    from tests.envelope import assert_inside_envelope, order_envelope
    want = oracle.split_params(cfg, ab["grad"])
    got = m.grads()
    # the same rule as for one cycle: inside the envelope of the oracle's own summation orders, here of the
    # second cycle accumulating onto the oracle's first-cycle gradients
    _, env2 = order_envelope(oracle, cfg, flat, tok2, lm_tok2, scale, grad_cached=a["grad"])
    _, env1 = order_envelope(oracle, cfg, flat, tok, lm_tok, scale)
    env = {t: (env1[t][0] + env2[t][0], env1[t][1] + env2[t][1]) for t in env2}   # two free-running cycles
    assert_inside_envelope(got, want, env, "accumulated")
    for name, g in got.items():
        assert not np.array_equal(g, first[name]), name
    # from the device's own first gradients the accumulation adds exactly one micro-batch: got - first ~ b
    b = oracle.split_params(cfg, oracle.llama_step(cfg, flat, tok2, lm_tok2, scale)["grad"])
    for name, g in got.items():
        d = g.astype(np.float32) - first[name].astype(np.float32)
        assert rel_l2(d, b[name]) < 5e-3, name
    m.step(tok2, lm_tok2, scale)
    _, envb = order_envelope(oracle, cfg, flat, tok2, lm_tok2, scale)
    assert_inside_envelope(m.grads(), b, envb, "overwritten")
    m.close(); ctx.close()


@pytest.mark.gpu
def test_copy_forwarding_changes_no_bit(tmp_path):
    """The compile pass that turns the adjoint copies of a residual add into storage moves must not change
    any result: one cycle in a child process with the pass, one with CACTI_NO_COPY_FORWARD=1 (the switch is
    read once per process), gradients and loss compared byte for byte."""
    import os
    import subprocess
    import sys
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    code = (
        "import sys, numpy as np\n"
        "sys.path.insert(0, %r)\n"
        "from tests.llama_ref import make_inputs\n"
        "from tests.test_gpu_llama import TINY, _model\n"
        "cfg, flat, tok, lm_tok, scale = make_inputs(TINY, seed=4, norm_mean=1.0, grad_scale=1024.0)\n"
        "ctx, m = _model(cfg)\n"
        "m.put_params_flat(flat)\n"
        "loss = m.step(tok, lm_tok, scale)\n"
        "g = m.grads()\n"
        "np.savez(sys.argv[1], loss=loss, **{k: v.view(np.uint16) for k, v in g.items()})\n"
        "print(ctx.stats())\n" % root)
    outs = []
    for tag, extra in (("fwd", {}), ("plain", {"CACTI_NO_COPY_FORWARD": "1"})):
        path = str(tmp_path / (tag + ".npz"))
        env = dict(os.environ, **extra)
        r = subprocess.run([sys.executable, "-c", code, path], env=env, capture_output=True, text=True, timeout=110)
        assert r.returncode == 0, r.stderr[-2000:]
        outs.append(np.load(path))
    a, b = outs
    assert sorted(a.files) == sorted(b.files) and len(a.files) == 3 + 9 * TINY["L"] + 1
    for k in a.files:
        assert a[k].tobytes() == b[k].tobytes(), k


@pytest.mark.gpu
def test_capped_pool_spills_at_full_shapes():
    """The host-spill path at the OpenLLaMA-3B shapes (4 of the 26 layers): with the pool capped at 0.45 of
    the uncapped peak -- below what parameters and gradients alone take -- live cells are downloaded on the
    copy stream, victims chosen by their next use in the compiled log, and uploaded again ahead of their
    use; loss and every probed gradient are bit-identical to the uncapped run, over two cycles."""
    import bench
    from cacti_amd.runtime import Ctx, Llama
    cfg = dict(bench.LLAMA_3B, L=4)
    tok, lm_tok, scale = bench.synth_inputs(cfg, grad_scale=8192.0)
    probe = ["embed", "l0.q", "l0.pre_norm", "l1.down", "l2.up", "l3.gate", "l3.v", "head_norm", "lm_head"]

    def run(pool_bytes):
        ctx = Ctx(0, pool_bytes, True)
        m = Llama(ctx, **cfg)
        bench.synth_params(m)
        idx = {name: i for i, (name, _) in enumerate(m.params)}
        out = []
        for _ in range(2):
            loss = m.step(tok, lm_tok, scale)
            out.append((loss, {n: m.grad(idx[n]) for n in probe}))
        st = ctx.stats()
        m.close(); ctx.close()
        return out, st

    ref, st0 = run(24 << 30)
    assert st0["n_evict"] == 0
    cap = int(st0["pool_peak"] * 0.45)
    got, st = run(cap)
    print("peak %.2f GB, cap %.2f GB: %d evictions, %.2f GB down, %.2f GB up over two cycles"
          % (st0["pool_peak"] / 1e9, cap / 1e9, st["n_evict"], st["bytes_d2h"] / 1e9, st["bytes_h2d"] / 1e9), flush=True)
    assert st["n_evict"] > 0 and st["bytes_d2h"] > 0 and st["pool_peak"] <= st["pool_cap"]
    for cyc in range(2):
        assert np.array_equal(ref[cyc][0], got[cyc][0]), "loss, cycle %d" % cyc
        for n in probe:
            assert np.array_equal(ref[cyc][1][n].view(np.uint16), got[cyc][1][n].view(np.uint16)), (cyc, n)


def test_full_depth_step_on_a_16_gib_pool():
    """The whole 26-layer OpenLLaMA-3B-shaped step on a pool capped at 16 GiB (the reference's card,
    examples/open_llama_3b_train.rs): two cycles; the loss and twelve probed gradients (first and last
    layers, every kind of tensor, embedding and LM head) are bit-identical to the uncapped run's, and the
    capped run really spilled."""
    import bench
    from cacti_amd.runtime import Ctx, Llama
    cfg = dict(bench.LLAMA_3B)
    assert cfg["L"] == 26
    tok, lm_tok, scale = bench.synth_inputs(cfg)

    def run(pool_bytes):
        print("26 layers on a pool of %.0f GiB" % (pool_bytes / 2 ** 30), flush=True)
        ctx = Ctx(0, pool_bytes, True)
        m = Llama(ctx, **cfg)
        bench.synth_params(m)
        out = []
        for _ in range(2):
            loss = m.step(tok, lm_tok, scale)
            out.append((loss, bench.probe_grads(m, cfg)))
        st = ctx.stats()
        m.close(); ctx.close()
        return out, st

    got, st = run(bench.CAPPED_POOL_BYTES)
    ref, st0 = run(40 << 30)
    print("uncapped peak %.2f GB; at 16 GiB: %d evictions, %.2f GB down, %.2f GB up over two cycles"
          % (st0["pool_peak"] / 1e9, st["n_evict"], st["bytes_d2h"] / 1e9, st["bytes_h2d"] / 1e9), flush=True)
    assert st0["n_evict"] == 0
    assert st["n_evict"] > 0 and st["bytes_d2h"] > 0 and st["bytes_h2d"] > 0 and st["pool_peak"] <= st["pool_cap"]
    for cyc in range(2):
        assert np.all(np.isfinite(ref[cyc][0]))
        assert np.array_equal(ref[cyc][0], got[cyc][0]), "loss, cycle %d" % cyc
        assert len(ref[cyc][1]) >= 12
        for n, g in ref[cyc][1].items():
            assert np.array_equal(g.view(np.uint16), got[cyc][1][n].view(np.uint16)), (cyc, n)


# An FFN width that is no multiple of 8: the down projection and its input gradient, which a cycle lends a workspace, take operands
# and results of any alignment; a K of 22 and of 79 k tiles, the latter in parts
@pytest.mark.parametrize("S,D,H,F,V", [(256, 512, 8, 1367, 1024), (200, 256, 4, 1373, 512), (40, 256, 4, 5003, 512)])
def test_ffn_width_of_any_alignment(oracle, S, D, H, F, V):
    """Loss and every gradient of a cycle, and of a second one that adds to it, inside the oracle's envelope; the bits of the
    separate thunks in every staging of the products."""
    from tests.envelope import assert_inside_envelope, order_envelope
    c = dict(S=S, D=D, H=H, Dh=D // H, F=F, V=V, L=1, eps=1e-6)
    cfg, flat, tok, lm_tok, scale = make_inputs(c, seed=F, norm_mean=1.0, grad_scale=256.0)
    _, _, tok2, lm_tok2, _ = make_inputs(c, seed=F + 1, norm_mean=1.0, grad_scale=256.0)
    print("ffn width", F, flush=True)
    one = oracle.llama_step(cfg, flat, tok, lm_tok, scale)
    two = oracle.llama_step(cfg, flat, tok2, lm_tok2, scale, grad_cached=one["grad"])
    _, env1 = order_envelope(oracle, cfg, flat, tok, lm_tok, scale)
    _, env2 = order_envelope(oracle, cfg, flat, tok2, lm_tok2, scale, grad_cached=one["grad"])
    env12 = {t: (env1[t][0] + env2[t][0], env1[t][1] + env2[t][1]) for t in env2}   # two free-running cycles
    first = None
    for groups in (0, 1, 2):
        ctx, m = _model(cfg)
        m.set_product_groups(groups)
        m.put_params_flat(flat)
        loss = m.step(tok, lm_tok, scale)
        assert_parity(loss, one["loss"], "loss", l2=1e-4, mx=1e-3)
        got = m.grads()
        m.step(tok2, lm_tok2, scale, accumulate=True)
        both = m.grads()
        m.close(); ctx.close()
        if first is None:
            first = (got, both)
            assert_inside_envelope(got, oracle.split_params(cfg, one["grad"]), env1, "ffn of %d" % F)
            assert_inside_envelope(both, oracle.split_params(cfg, two["grad"]), env12, "ffn of %d, twice" % F)
        for name, g in got.items():
            assert np.array_equal(g.view(np.uint16), first[0][name].view(np.uint16)), (groups, name)
            assert np.array_equal(both[name].view(np.uint16), first[1][name].view(np.uint16)), (groups, name)


# Sequences that the forward kernel of whole tiles takes (more than 1024 positions and 512 workgroups of 32 of them), heads of one and
# of two 64-column halves
@pytest.mark.parametrize("S,H,Dh", [(1100, 16, 64), (1060, 16, 72)])
def test_two_layers_of_a_long_sequence(oracle, S, H, Dh):
    """What one layer's attention rounds goes through the next layer's: loss and gradients of two layers inside the oracle's envelope."""
    from tests.envelope import assert_loss_inside_envelope, order_envelope
    D = H * Dh
    cfg, flat, tok, lm_tok, scale = make_inputs(dict(S=S, D=D, H=H, Dh=Dh, F=512, V=1024, L=2, eps=1e-6), seed=3, norm_mean=1.0,
                                                grad_scale=1024.0)
    print("two layers", S, H, Dh, flush=True)
    ref = oracle.llama_step(cfg, flat, tok, lm_tok, scale)
    _, env = order_envelope(oracle, cfg, flat, tok, lm_tok, scale, count=8)
    print("envelope measured", flush=True)
    ctx, m = _model(cfg, pool_bytes=4 << 30)
    m.put_params_flat(flat)
    assert_loss_inside_envelope(m.step(tok, lm_tok, scale), ref["loss"], env, "two layers")
    _compare(oracle, cfg, m, ref, env, "two layers")
    m.close(); ctx.close()
