"""What a user of this framework has it do, as cases that can be timed and compared.

Eight kinds of work, each through the package's public entry points:

  train      one minibatch of training: forward, loss and full gradient of a LLaMA-shaped model (runtime.Llama.step),
             as one or more micro-batches whose gradients add up, with or without the AdamW step on the device
  generate   one request: a prompt in one call, then one position per call, each fed the previous arg max
             (runtime.LlamaCached)
  layer      forward and backward of one decoder layer written with the operators (cacti_amd.ops), for a program that
             keeps its tensors in torch
  head       LM head product, softmax cross-entropy and their gradients, with the operators
  attention  fused causal attention, forward and backward
  linear     the three products of a linear layer of any size (forward, input gradient, weight gradient)
  pointwise  RMSNorm, rotary embedding and SiLU gate, forward and backward
  optimizer  one AdamW step and the numerical-health digests over a list of tensors

All tensors are f16 with fp32 accumulation, the only element type of the path; optimiser state is f32.
"""
import math

import numpy as np
import torch

from cacti_amd import ops
from cacti_amd.runtime import Ctx, Llama, LlamaCached

EPS = 1e-6


def listed():
    return [
        # the smallest model of the tests; its program runs the optimiser itself and reads every gradient back
        dict(name="train_tiny", kind="train", S=128, D=256, H=4, F=688, V=1024, L=2, micro=1, update=False, read_all=True),
        # a small model on texts of odd length, two micro-batches to a minibatch, AdamW on the device
        dict(name="train_small_ragged", kind="train", S=611, D=1024, H=16, F=2816, V=8192, L=4, micro=2, update=True,
             read_all=False),
        # the benchmark's widths and sequence length (4 of its 26 layers: the layers repeat)
        dict(name="train_3b_width", kind="train", S=2048, D=3200, H=32, F=8640, V=32000, L=4, micro=1, update=False,
             read_all=False),
        # the smallest request: every kernel is short, launches and host work count
        dict(name="generate_tiny", kind="generate", D=256, H=4, F=688, V=1024, L=2, prompt=13, new=32, cap=128, stream=True),
        # a chat turn: a short prompt, logits and tokens handed out as they come
        dict(name="generate_chat", kind="generate", D=3200, H=32, F=8640, V=32000, L=3, prompt=37, new=32, cap=512,
             stream=True),
        # a long document as the prompt, a short answer: prefill counts, decoding runs over a long cache; a generic width
        # with heads of 128
        dict(name="generate_document", kind="generate", D=2048, H=16, F=5504, V=32000, L=4, prompt=1531, new=16, cap=2048,
             stream=False),
        # one layer of that width, ragged sequence
        dict(name="layer_ragged", kind="layer", S=777, D=2048, H=16, F=5504),
        # LM head and loss of the benchmark's configuration
        dict(name="head_3b", kind="head", N=2048, D=3200, V=32000),
        # attention of the benchmark's configuration: one layer, 32 heads of 100
        dict(name="attention_3b", kind="attention", S=2048, H=32, Dh=100),
        # a linear layer with sizes that are multiples of nothing
        dict(name="linear_odd", kind="linear", M=509, N=1003, K=770, count=1),
        # the memory-bound kernels at the benchmark's shapes
        dict(name="pointwise_3b", kind="pointwise", S=2048, H=32, Dh=100, F=8640),
        # optimiser and digests over tensors from a norm weight to a large matrix
        dict(name="optimizer", kind="optimizer", tensors=12, largest=27648000),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


# (width, heads): heads of 64, 100 and 128, from the tiny configuration's width to the benchmark's
_WIDTHS = [(256, 4), (512, 8), (768, 12), (800, 8), (1024, 16), (1600, 16), (2048, 16), (2048, 32), (3200, 32)]


def _ffn(rng, D):
    return int(D * rng.uniform(2.6, 3.6)) // 8 * 8


def draw(rng):
    most = _weight(next(c for c in listed() if c["name"] == "train_3b_width"))
    while True:
        c = _draw(rng)
        if _weight(c) <= most:
            return c


def _weight(case):
    w = work(case)
    return max(w["bytes"], w["flops"] / 50)


def _draw(rng):
    kind = rng.choice(["train", "train", "generate", "generate", "layer", "head", "attention", "linear", "pointwise", "optimizer"])
    D, H = rng.choice(_WIDTHS)
    if kind == "train":
        return dict(kind=kind, S=_log(rng, 33, 2048), D=D, H=H, F=_ffn(rng, D), V=_log(rng, 1000, 32000) // 8 * 8,
                    L=rng.randint(1, 4), micro=rng.choice([1, 1, 2]), update=rng.random() < 0.5, read_all=D <= 256)
    if kind == "generate":
        prompt, new = _log(rng, 2, 1900), rng.randint(8, 48)
        return dict(kind=kind, D=D, H=H, F=_ffn(rng, D), V=_log(rng, 1000, 32000) // 8 * 8, L=rng.randint(1, 3),
                    prompt=prompt, new=new, cap=(prompt + new + 7) // 8 * 8, stream=rng.random() < 0.5)
    if kind == "layer":
        return dict(kind=kind, S=_log(rng, 33, 2048), D=D, H=H, F=_ffn(rng, D))
    if kind == "head":
        return dict(kind=kind, N=_log(rng, 33, 2048), D=D, V=_log(rng, 1000, 50000) // 8 * 8)
    if kind == "attention":
        return dict(kind=kind, S=_log(rng, 33, 2048), H=rng.randint(1, 32), Dh=rng.choice([64, 100, 128]))
    if kind == "linear":
        return dict(kind=kind, M=_log(rng, 5, 4000), N=_log(rng, 50, 5000), K=_log(rng, 50, 5000), count=rng.choice([1, 1, 1, 3]))
    if kind == "pointwise":
        return dict(kind=kind, S=_log(rng, 1, 4096), H=H, Dh=D // H, F=_ffn(rng, D))
    return dict(kind=kind, tensors=rng.randint(1, 14), largest=_log(rng, 1000, 60000000))


# ---------------------------------------------------------------- inputs
def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _randn(g, *shape, std=1.0, mean=0.0):
    x = torch.randn(shape, generator=g, device="cuda", dtype=torch.float16)
    return x.mul_(std).add_(mean) if mean else x.mul_(std)


def _host(x):
    """The tensor as a numpy array in page-locked memory (the copy of gigabytes of weights is quick that way)."""
    h = torch.empty(x.shape, dtype=x.dtype, pin_memory=True)
    h.copy_(x)
    return h.numpy()


class _Model:
    """A model with its context, closed in order when the state goes."""

    def __init__(self, case, S, pool_bytes):
        self.ctx = Ctx(0, pool_bytes, True)
        self.m = Llama(self.ctx, S=S, D=case["D"], H=case["H"], Dh=case["D"] // case["H"], F=case["F"], V=case["V"],
                       L=case["L"], eps=EPS)
        self.cached = None

    def __del__(self):
        if self.cached is not None:
            self.cached.close()
        self.m.close()
        self.ctx.close()


def _num_params(case):
    D, F = case["D"], case["F"]
    return case["L"] * (4 * D * D + 3 * D * F + 2 * D) + 2 * case["V"] * D + D


def _pool_bytes(case, S):
    state = _num_params(case) * (16 if case.get("update") else 4)
    acts = S * case["L"] * (24 * case["D"] + 10 * case["F"]) * 2 + S * case["V"] * 16 + S * S * case["H"] * 4
    return int(1.1 * (state + acts)) + (256 << 20)


def _prepare_train(case, seed):
    g = _gen(seed)
    st = _Model(case, case["S"], _pool_bytes(case, case["S"]))
    # matrices ~N(0, 0.02), norm weights ~N(1, 0.02), ids uniform, labels the ids shifted by one, gradient scale 1024
    for i, (name, shape) in enumerate(st.m.params):
        st.m.put_param(i, _host(_randn(g, *shape, std=0.02, mean=1.0 if name.endswith("norm") else 0.0)))
    if case["update"]:
        st.m.adamw_init()
    S = case["S"]
    st.batches = []
    for _ in range(case["micro"]):
        tok = torch.randint(0, case["V"], (S,), generator=g, device="cuda").cpu().numpy().astype(np.uint16)
        scale = np.full(S, 1024.0 / (S - 1) / case["micro"], np.float32)
        scale[0] = 0.0
        st.batches.append((tok, np.roll(tok, -1), scale))
    names = [n for n, _ in st.m.params]
    # what the program reads back: everything, or what it watches (the norms and the first layer's query projection,
    # whose gradients are the last of the backward pass)
    st.watched = list(range(len(names))) if case["read_all"] else \
        [i for i, n in enumerate(names) if n.endswith("norm") or n == "l0.q"]
    st.updated = names.index("l0.q") if case["update"] else None
    st.iter_nr = 0
    return st


def _run_train(case, st):
    m, losses = st.m, []
    for k, (tok, lm_tok, scale) in enumerate(st.batches):
        losses.append(m.step(tok, lm_tok, scale, accumulate=k > 0))
    out = dict(loss=losses, grads=[m.grad(i) for i in st.watched])
    if case["update"]:
        st.iter_nr += 1
        m.adamw_step(st.iter_nr, grad_scale=1024.0, lr=2e-5)
        out["param"] = m.param(st.updated)
    return out


def _prepare_generate(case, seed):
    g = _gen(seed)
    D, V = case["D"], case["V"]
    st = _Model(case, case["cap"], _pool_bytes(case, case["cap"]))
    # A model that is sure of its next token, as a trained one mostly is: the head of token next(t) points where the
    # embedding of t does.  The layers are random.
    embed = _randn(g, V, D)
    head = torch.empty_like(embed)
    head[torch.randperm(V, generator=g, device="cuda")] = embed * 0.02
    for i, (name, shape) in enumerate(st.m.params):
        w = embed if name == "embed" else head if name == "lm_head" else \
            _randn(g, *shape, std=0.02, mean=1.0 if name.endswith("norm") else 0.0)
        st.m.put_param(i, _host(w))
    st.cached = LlamaCached(st.m, case["cap"])
    st.prompt = torch.randint(0, V, (case["prompt"],), generator=g, device="cuda").cpu().numpy().astype(np.uint16)
    return st


def _run_generate(case, st):
    c, T, logits = st.cached, case["prompt"], []
    c.reset_state()
    c.set_tokens(st.prompt)
    c.apply(0, T)
    for pos in range(T, T + case["new"] - 1):
        if case["stream"]:                       # every position's logits are looked at as they come
            logits.append(c.outputs()["logit"])
        c.apply(pos, pos + 1)
    last = c.outputs()
    return dict(logits=logits + [last["logit"]], tok=last["tok"], tokens=c.tokens())


def _prepare_layer(case, seed):
    g = _gen(seed)
    S, D, F, H = case["S"], case["D"], case["F"], case["H"]
    st = dict(x=_randn(g, S, D), dy=_randn(g, S, D, std=0.1), n1=_randn(g, D, std=0.02, mean=1.0),
              n2=_randn(g, D, std=0.02, mean=1.0))
    for n, shape in dict(q=(D, D), k=(D, D), v=(D, D), o=(D, D), gate=(F, D), up=(F, D), down=(D, F)).items():
        st[n] = _randn(g, *shape, std=0.02)
    st["cos"], st["sin"] = ops.rope_tables(S, D // H)
    return st


def _run_layer(case, s):
    S, D, H = case["S"], case["D"], case["H"]
    Dh = D // H
    alpha = 1.0 / math.sqrt(Dh)
    heads = lambda t: t.view(S, H, Dh)
    flat = lambda t: t.view(S, D)
    h1 = ops.rms_norm_fwd(s["x"], s["n1"], EPS)
    q, k = (ops.rope_fwd(heads(ops.gemm(h1, s[n], tb=True)), s["cos"], s["sin"]) for n in "qk")
    v = heads(ops.gemm(h1, s["v"], tb=True))
    o, stats = ops.attention_fwd(q, k, v, alpha)
    x1, h2 = ops.add_rms_norm_fwd(s["x"], ops.gemm(flat(o), s["o"], tb=True), s["n2"], EPS)
    gate, up = ops.gemm(h2, s["gate"], tb=True), ops.gemm(h2, s["up"], tb=True)
    h = ops.silu_gate_fwd(gate, up)
    y = ops.add_f16(x1, ops.gemm(h, s["down"], tb=True))

    d = {}
    d["down"] = ops.gemm(s["dy"], h, ta=True)
    dgate, dup = ops.silu_gate_bwd(gate, up, ops.gemm(s["dy"], s["down"]))
    d["gate"], d["up"] = ops.gemm(dgate, h2, ta=True), ops.gemm(dup, h2, ta=True)
    dh2 = ops.gemm(dgate, s["gate"])
    ops.gemm(dup, s["up"], beta=1.0, out=dh2)
    dx1, d["n2"] = ops.rms_norm_bwd(x1, s["n2"], EPS, dh2)
    ops.add_f16(dx1, s["dy"], out=dx1)
    d["o"] = ops.gemm(dx1, flat(o), ta=True)
    dq, dk, dv = ops.attention_bwd(q, k, v, heads(ops.gemm(dx1, s["o"])), stats, alpha, o=o)
    dq, dk = flat(ops.rope_bwd(dq, s["cos"], s["sin"])), flat(ops.rope_bwd(dk, s["cos"], s["sin"]))
    dv = flat(dv)
    for n, t in (("q", dq), ("k", dk), ("v", dv)):
        d[n] = ops.gemm(t, h1, ta=True)
    dh1 = ops.gemm(dq, s["q"])
    ops.gemm(dk, s["k"], beta=1.0, out=dh1)
    ops.gemm(dv, s["v"], beta=1.0, out=dh1)
    dx, d["n1"] = ops.rms_norm_bwd(s["x"], s["n1"], EPS, dh1, dx_acc=dx1)
    return dict(y=y, dx=dx, **{"d" + n: t for n, t in d.items()})


def _prepare_head(case, seed):
    g = _gen(seed)
    N, D, V = case["N"], case["D"], case["V"]
    W = _randn(g, V, D, std=0.02)
    tok = torch.randint(0, V, (N,), generator=g, device="cuda")
    # hidden states that lean towards their target, as those of a model in training do: the loss is small, the arg max clear
    x = _randn(g, N, D) + W[tok] * (12.0 / (0.02 * 0.02 * D))
    return dict(x=x, W=W, tok=tok.to(torch.int32).to(torch.int16), scale=torch.full((N,), 1024.0 / N, device="cuda"))


def _run_head(case, s):
    logit = ops.gemm(s["x"], s["W"], tb=True)
    _, loss, amax = ops.softmax_ce_fwd(logit, s["tok"], want_prob=False)
    dlogit = ops.softmax_ce_bwd(logit, s["tok"], s["scale"])
    return dict(loss=loss, amax=amax, dx=ops.gemm(dlogit, s["W"]), dW=ops.gemm(dlogit, s["x"], ta=True))


def _prepare_attention(case, seed):
    g = _gen(seed)
    return dict(qkv=[_randn(g, case["S"], case["H"], case["Dh"]) for _ in range(3)],
                dO=_randn(g, case["S"], case["H"], case["Dh"]))


def _run_attention(case, s):
    alpha = 1.0 / math.sqrt(case["Dh"])
    o, stats = ops.attention_fwd(*s["qkv"], alpha)
    return o, ops.attention_bwd(*s["qkv"], s["dO"], stats, alpha, o=o)


def _prepare_linear(case, seed):
    g = _gen(seed)
    M, N, K, n = case["M"], case["N"], case["K"], case["count"]
    return dict(x=[_randn(g, M, K) for _ in range(n)], W=[_randn(g, N, K, std=0.02) for _ in range(n)],
                dy=[_randn(g, M, N, std=0.1) for _ in range(n)])


def _run_linear(case, s):
    if case["count"] == 1:
        x, W, dy = s["x"][0], s["W"][0], s["dy"][0]
        return ops.gemm(x, W, tb=True), ops.gemm(dy, W), ops.gemm(dy, x, ta=True)
    return ops.gemm_batched(s["x"], s["W"], tb=True), ops.gemm_batched(s["dy"], s["W"]), ops.gemm_batched(s["dy"], s["x"], ta=True)


def _prepare_pointwise(case, seed):
    g = _gen(seed)
    S, H, Dh, F = case["S"], case["H"], case["Dh"], case["F"]
    cos, sin = ops.rope_tables(S, Dh)
    return dict(x=_randn(g, S, H * Dh), w=_randn(g, H * Dh), dy=_randn(g, S, H * Dh), gate=_randn(g, S, F), up=_randn(g, S, F),
                dh=_randn(g, S, F), cos=cos, sin=sin)


def _run_pointwise(case, s):
    heads = lambda t: t.view(case["S"], case["H"], case["Dh"])
    return (ops.rms_norm_fwd(s["x"], s["w"], EPS), ops.rope_fwd(heads(s["x"]), s["cos"], s["sin"]),
            ops.silu_gate_fwd(s["gate"], s["up"]), ops.silu_gate_bwd(s["gate"], s["up"], s["dh"]),
            ops.rope_bwd(heads(s["dy"]), s["cos"], s["sin"]), ops.rms_norm_bwd(s["x"], s["w"], EPS, s["dy"]))


def _sizes(case):
    # from the largest down to a sixteenth and a norm weight's size, ragged
    return [max(1, (case["largest"] >> (i % 5)) - 3 * i) if i % 3 != 2 else 3200 + i for i in range(case["tensors"])]


def _prepare_optimizer(case, seed):
    g = _gen(seed)
    st = dict(grads=[], avgs=[], avg2s=[], masters=[], params=[], iter_nr=0)
    for n in _sizes(case):
        st["grads"].append(_randn(g, n, std=0.01))
        w = torch.randn(n, generator=g, device="cuda") * 0.02
        st["masters"].append(w)
        st["params"].append(w.half())
        st["avgs"].append(torch.randn(n, generator=g, device="cuda") * 1e-6)
        st["avg2s"].append(torch.rand(n, generator=g, device="cuda") * 1e-10)
    return st


def _run_optimizer(case, s):
    s["iter_nr"] += 1
    scalars = ops.adamw32_scalars(s["iter_nr"], 1024.0, 1e-4, 0.01, 0.1, 1e-3, 1e-8)
    state = s["avgs"], s["avg2s"], s["masters"], s["params"]
    ops.adamw32_step_(s["grads"], *state, scalars)
    return state + tuple(ops.digests(s["grads"])) + tuple(ops.digests(s["params"]))


_PREPARE = dict(train=_prepare_train, generate=_prepare_generate, layer=_prepare_layer, head=_prepare_head,
                attention=_prepare_attention, linear=_prepare_linear, pointwise=_prepare_pointwise, optimizer=_prepare_optimizer)
_RUN = dict(train=_run_train, generate=_run_generate, layer=_run_layer, head=_run_head, attention=_run_attention,
            linear=_run_linear, pointwise=_run_pointwise, optimizer=_run_optimizer)


def prepare(case, seed):
    return case, _PREPARE[case["kind"]](case, seed)


def run(state):
    case, st = state
    return _RUN[case["kind"]](case, st)


# ---------------------------------------------------------------- what cannot be done without
def work(case):
    """Bytes: inputs read once, outputs written once (f16 unless said).  Flops: the products, attention by its causal half."""
    kind = case["kind"]
    if kind == "train":
        S, D, L, n = case["S"], case["D"], case["L"], _num_params(case)
        dense = n - case["V"] * D                                         # the embedding is gathered, not multiplied
        flops = case["micro"] * (6 * S * dense + L * 6 * S * S * D)
        # per minibatch: parameters read, gradients written; AdamW reads 14 and writes 14 bytes per parameter
        return dict(bytes=n * 4 + case["micro"] * S * 8 + (28 * n if case["update"] else 0), flops=flops)
    if kind == "generate":
        D, L, V, T, new = case["D"], case["L"], case["V"], case["prompt"], case["new"]
        dense = _num_params(case) - V * D
        kv = lambda rows: L * rows * D * 4                                # both caches, f16
        passes = [T + i for i in range(1, new)]
        # every call reads the weights once and the cache rows so far; the prompt's logits are all formed
        return dict(bytes=2 * dense * new + (T + new - 1) * V * 2 + kv(T) + sum(kv(p) for p in passes),
                    flops=2 * dense * (T + new - 1) + L * 2 * T * T * D + sum(L * 4 * p * D for p in passes))
    if kind == "layer":
        S, D, F = case["S"], case["D"], case["F"]
        n = 4 * D * D + 3 * D * F + 2 * D
        return dict(bytes=2 * (2 * n + 4 * S * D), flops=6 * S * n + 6 * S * S * D)
    if kind == "head":
        N, D, V = case["N"], case["D"], case["V"]
        return dict(bytes=2 * (2 * V * D + 2 * N * D) + 12 * N, flops=6 * N * D * V)
    if kind == "attention":
        S, HD = case["S"], case["H"] * case["Dh"]
        return dict(bytes=2 * 8 * S * HD, flops=6 * S * S * HD)
    if kind == "linear":
        M, N, K, n = case["M"], case["N"], case["K"], case["count"]
        return dict(bytes=n * 2 * 2 * (M * K + N * K + M * N), flops=n * 6 * M * N * K)
    if kind == "pointwise":
        S, D, F = case["S"], case["H"] * case["Dh"], case["F"]
        return dict(bytes=2 * (S * D * (2 + 2 + 2 + 3) + S * F * (3 + 5)), flops=0)
    total = sum(_sizes(case))
    return dict(bytes=28 * total, flops=0)                                # the digests see the same gradients and parameters


def tolerance(case):
    """f16 results of fp32 sums in another order: a last-place flip here and there in one product, and what a chain of
    rounded products makes of such flips (two runs of one layer that differ in summation order alone are 1e-3 apart)."""
    return dict(train={"rel": 5e-3, "max": 0.15}, generate={"rel": 5e-3, "max": 0.1}, layer={"rel": 3e-3, "max": 0.1},
                head={"rel": 2e-3, "max": 0.05}, attention={"rel": 1e-3, "max": 0.03}, linear={"rel": 1e-3, "max": 5e-3},
                pointwise={"rel": 1e-3, "max": 1e-2}, optimizer={"rel": 1e-6, "max": 1e-3})[case["kind"]]
