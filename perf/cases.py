"""What a user of this framework has it compute, as measurable cases.

A case is one pass through the public entry points:

* "linear": one quantized linear, `linear(gpu, x, w, y)`: GPTQ int4 (group
  size 64 / 128 / 256, with or without zero points and act-order) or INT8,
  f32 or f16 x, from one decode token to a prompt of thousands;
* "layer": every linear of one decoder layer (self-attention or DeltaNet),
  called eagerly: `decode` (f32, 1-32 tokens) or `prefill` (f16);
* "step": one token step of a decoder (several layers of both kinds, then an
  int4 lm_head) captured once as a graph and replayed, the model's own ops
  between the linears standing in as plain adds and multiplies (hooks);
* "head": the bf16 lm_head, `bf16_matvec`.

Weights go through the uploads of the loader (`GptqWeight.upload`,
`Int8Weight.upload`: the tiled layout). Activations are normal with a few
large channels, as hidden states of such models are.
"""
import math

import numpy as np
import torch

import shady_thinker_amd as sta

DEV = "cuda:0"
OUTLIER = 16.0  # size of the large activation channels (one in 256)


def listed():
    return [
        # the smallest call: one token through a small linear (a launch's latency)
        dict(name="linear_1", kind="linear", fmt="gptq", m=1, k=2048, n=2048, gs=128, zeros=False, act=False, x="f32"),
        # token by token without a graph: a 7B layer's linears called one after the other
        dict(name="layer_decode_1", kind="layer", mode="decode", attn="self", m=1, hidden=4096, attn_dim=4096, qkv=12288,
             inter=11008, gs=128, zeros=False, act=False),
        # chat, one user: a captured token step (hybrid model, large vocabulary)
        dict(name="step_1", kind="step", m=1, layers=4, hidden=2560, attn_dim=4096, qkv=10240, dn_dim=2048, dn_qkv=6144,
             inter=9728, vocab=151936, gs=128, zeros=False),
        # a few users, or drafted tokens checked together: an act-order checkpoint with zero points
        dict(name="layer_decode_6", kind="layer", mode="decode", attn="self", m=6, hidden=4096, attn_dim=4096, qkv=6144,
             inter=14336, gs=64, zeros=True, act=True),
        # batched serving: a captured token step of 16 users
        dict(name="step_16", kind="step", m=16, layers=4, hidden=2560, attn_dim=4096, qkv=10240, dn_dim=2048, dn_qkv=6144,
             inter=9728, vocab=151936, gs=128, zeros=False),
        # the largest decode batch, a checkpoint with zero points, ragged
        dict(name="step_31", kind="step", m=31, layers=4, hidden=2560, attn_dim=4096, qkv=10240, dn_dim=2048, dn_qkv=6144,
             inter=9728, vocab=151936, gs=128, zeros=True),
        # INT8 serving of 8 users
        dict(name="int8_8", kind="linear", fmt="int8", m=8, k=5120, n=13824, x="f16"),
        # the lm_head of a model that keeps it in bf16
        dict(name="head_1", kind="head", m=1, k=2560, n=151936, x="f32"),
        # a short prompt, ragged (most chat turns)
        dict(name="layer_prefill_77", kind="layer", mode="prefill", attn="self", m=77, hidden=2560, attn_dim=4096, qkv=10240,
             inter=9728, gs=128, zeros=True, act=False),
        # a prompt of ordinary length through a layer
        dict(name="layer_prefill_512", kind="layer", mode="prefill", attn="delta", m=512, hidden=2560, attn_dim=2048,
             qkv=8192, inter=9728, gs=128, zeros=False, act=False),
        # a long prompt through one wide linear of an act-order checkpoint
        dict(name="linear_2048", kind="linear", fmt="gptq", m=2048, k=4096, n=14336, gs=128, zeros=False, act=True, x="f16",
             y="f16"),
        # an INT8 prompt of odd length
        dict(name="int8_333", kind="linear", fmt="int8", m=333, k=5120, n=13824, x="f16", y="f32"),
    ]


def _log(rng, lo, hi, step):
    """A multiple of `step` in [lo, hi], spread over the logarithm."""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return max(lo, min(hi, int(round(v / step)) * step))


def draw(rng):
    kind = rng.choice(["linear", "linear", "linear", "linear", "int8", "int8", "layer", "layer", "layer", "step", "head"])
    gs = rng.choice([128, 128, 128, 64, 256])
    if kind == "head":
        return dict(kind="head", m=rng.randint(1, 8), k=_log(rng, 1024, 4096, 8), n=_log(rng, 8192, 152064, 8),
                    x=rng.choice(["f32", "f16"]))
    if kind == "int8":
        m = rng.choice([rng.randint(1, 32), _log(rng, 33, 1024, 1)])
        return dict(kind="linear", fmt="int8", m=m, k=_log(rng, 1024, 8192, 128), n=_log(rng, 512, 14336, 4), x="f16",
                    y="f32" if m <= 32 else rng.choice(["f32", "f16"]))
    if kind == "linear":
        m = rng.choice([rng.randint(1, 4), rng.randint(5, 32), _log(rng, 33, 2048, 1)])
        k, n = _log(rng, 1024, 11264, 256), _log(rng, 512, 14336, 8)
        return dict(kind="linear", fmt="gptq", m=m, k=k, n=n, gs=gs, zeros=rng.random() < 0.4, act=rng.random() < 0.4,
                    x="f16" if m > 32 else rng.choice(["f32", "f32", "f16"]),
                    y="f32" if m <= 32 else rng.choice(["f32", "f16"]))
    hidden, inter = _log(rng, 1024, 4096, 256), _log(rng, 2816, 14336, 256)
    heads = rng.choice([8, 16, 24, 32])
    if kind == "layer":
        attn = rng.choice(["self", "delta"])
        mode = rng.choice(["decode", "prefill"])
        dim = 128 * heads
        qkv = dim * 2 + rng.choice([512, 1024, 2048]) if attn == "self" else 3 * dim + 1024
        return dict(kind="layer", mode=mode, attn=attn,
                    m=rng.choice([1, rng.randint(2, 32)]) if mode == "decode" else _log(rng, 33, 1024, 1),
                    hidden=hidden, attn_dim=dim, qkv=qkv, inter=inter, gs=gs, zeros=rng.random() < 0.4,
                    act=rng.random() < 0.3)
    dim = 128 * heads
    return dict(kind="step", m=rng.randint(1, 32), layers=rng.randint(2, 4), hidden=min(hidden, 2560), attn_dim=dim,
                qkv=2 * dim + 1024, dn_dim=1024, dn_qkv=3072, inter=min(inter, 9728), vocab=_log(rng, 16000, 128000, 16),
                gs=gs, zeros=rng.random() < 0.4)


# ------------------------------------------------------------------ inputs
def _gen(seed, idx):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed * 4096 + idx)
    return g


def _x(seed, idx, m, k, dtype=torch.float32, small=1.0):
    """Activations: N(0, 1), one channel in 256 OUTLIER times as large."""
    g = _gen(seed, idx)
    x = torch.randn(m, k, device=DEV, generator=g)
    big = torch.randint(0, k, (max(1, k // 256),), device=DEV, generator=g)
    x[:, big] *= OUTLIER
    return (x * small).to(dtype).contiguous()


def _raw_gptq(seed, idx, k, n, gs, zeros, act):
    """A checkpoint's tensors of one GPTQ linear: uniform nibbles (0 made 8,
    so that weights have no mean, as trained ones have none), scales that
    keep outputs near the inputs' size, zero points around 8, an act-order
    g_idx of whole groups."""
    g = _gen(seed, idx)
    qw = torch.randint(0, 2**32, (k // 8, n), device=DEV, generator=g, dtype=torch.int64)
    some = qw | (qw >> 1) | (qw >> 2) | (qw >> 3)
    qw |= (~some & 0x11111111) << 3
    qw = torch.where(qw >= 2**31, qw - 2**32, qw).to(torch.int32)
    s = (torch.rand(k // gs, n, device=DEV, generator=g) + 0.5) * (0.2 / math.sqrt(k))
    qz = gi = None
    if zeros:
        z = torch.randint(6, 11, (k // gs, n // 8, 8), device=DEV, generator=g, dtype=torch.int64)
        sh = 4 * torch.arange(8, device=DEV)
        w = (z << sh).sum(-1)
        qz = torch.where(w >= 2**31, w - 2**32, w).to(torch.int32)
    if act:
        p = torch.randperm(k, device=DEV, generator=g)
        gi = torch.empty(k, dtype=torch.int32, device=DEV)
        gi[p] = (torch.arange(k, device=DEV) // gs).to(torch.int32)
    return qw, s.half(), qz, gi


def _upload(gpu, raw, gs):
    qw, s, qz, gi = (None if t is None else t.cpu().numpy() for t in raw)
    return sta.GptqWeight.upload(gpu, qw, s, gs, qzeros=qz, g_idx=gi)


def _raw_int8(seed, idx, k, n):
    g = _gen(seed, idx)
    w = torch.randint(-127, 128, (n, k), device=DEV, generator=g, dtype=torch.int16).to(torch.int8)
    s = (torch.rand(n, device=DEV, generator=g) + 0.5) / (73.0 * math.sqrt(k))
    return w, s


def _raw_head(seed, idx, k, n):
    return (torch.randn(n, k, device=DEV, generator=_gen(seed, idx)) / math.sqrt(k)).to(torch.bfloat16)


def _dt(c, key, other="f32"):
    return torch.float16 if c.get(key, other) == "f16" else torch.float32


def _layer_shapes(c, attn):
    """(name, K, N) of a layer's linears, as the loader finds them."""
    h = c["hidden"]
    if attn == "self":
        a, qkv = c["attn_dim"], c["qkv"]
        kv = (qkv - (2 * a if qkv > 2 * a and qkv != 3 * a else a)) // 2
        s = [("q", h, qkv - 2 * kv), ("k", h, kv), ("v", h, kv), ("o", a, h)]
    else:
        a, qkv = (c["dn_dim"], c["dn_qkv"] + c["dn_dim"]) if c["kind"] == "step" else (c["attn_dim"], c["qkv"])
        s = [("in_qkv", h, qkv - a), ("in_z", h, a), ("out", a, h)]
    return s + [("gate", h, c["inter"]), ("up", h, c["inter"]), ("down", c["inter"], h)]


def _layer_raw(c, seed, base, attn):
    """A layer's raw tensors. One g_idx for linears on the same input (they
    are quantized on the same activations): the fused calls need it."""
    raw, shared = {}, {}
    for j, (name, k, n) in enumerate(_layer_shapes(c, attn)):
        qw, s, qz, gi = _raw_gptq(seed, base + j, k, n, c["gs"], c["zeros"], c.get("act", False))
        key = {"q": "x", "k": "x", "v": "x", "in_qkv": "x", "in_z": "x", "gate": "xm", "up": "xm"}.get(name, name)
        gi = shared.setdefault(key, gi)
        raw[name] = (qw, s, qz, gi)
    return raw


def _kinds(c):
    """A hybrid decoder: DeltaNet layers, every second one self-attention."""
    return ["delta" if i % 2 == 0 else "self" for i in range(c["layers"])]


def _build_layer(gpu, c, raw, attn):
    ws = [_upload(gpu, raw[name], c["gs"]) for name, _, _ in _layer_shapes(c, attn)]
    return (sta.DecoderLinears if attn == "self" else sta.DeltaNetLinears)(*ws)


class _Model:
    """The model's own ops between a step's linears: the residual adds, and a
    part of the input projection, damped, in place of the attention core (no
    norms: the damping keeps the hidden state in range)."""

    def __init__(self, embedding, dims):
        self.embedding, self.dims = embedding, dims

    def pre_attention(self, i, b):
        if i == 0:
            b.x.copy_(self.embedding)
        else:
            torch.add(b.xm, b.down, alpha=0.25, out=b.x)

    def attention(self, i, b):
        torch.mul(b.qkv[:, : self.dims[i]], 0.25, out=b.attn)

    def post_attention(self, i, b):
        torch.add(b.x, b.o, out=b.xm)

    def final(self, b):
        torch.add(b.xm, b.down, alpha=0.25, out=b.x)


def prepare(case, seed):
    c = case
    gpu = sta.GpuContext(0)
    st = dict(case=c, gpu=gpu)
    if c["kind"] == "linear":
        st["x"] = _x(seed, 1, c["m"], c["k"], _dt(c, "x"))
        st["y"] = torch.empty(c["m"], c["n"], dtype=_dt(c, "y"), device=DEV)
        if c["fmt"] == "int8":
            w, s = _raw_int8(seed, 2, c["k"], c["n"])
            st["w"] = sta.Int8Weight.upload(gpu, w.cpu().numpy(), s.cpu().numpy())
        else:
            st["w"] = _upload(gpu, _raw_gptq(seed, 2, c["k"], c["n"], c["gs"], c["zeros"], c["act"]), c["gs"])
    elif c["kind"] == "head":
        st["x"] = _x(seed, 1, c["m"], c["k"], _dt(c, "x"))
        st["w"] = _raw_head(seed, 2, c["k"], c["n"])
        st["y"] = torch.empty(c["m"], c["n"], device=DEV)
    elif c["kind"] == "layer":
        L = st["layer"] = _build_layer(gpu, c, _layer_raw(c, seed, 8, c["attn"]), c["attn"])
        m, dt = c["m"], torch.float32 if c["mode"] == "decode" else torch.float16
        st["x"] = _x(seed, 1, m, c["hidden"], dt, 0.5)
        st["attn"] = _x(seed, 2, m, c["attn_dim"], dt, 0.5)
        st["xm"] = _x(seed, 3, m, c["hidden"], dt, 0.5)
        e = lambda n: torch.empty(m, n, dtype=dt, device=DEV)
        mid = [e(c["inter"])] if c["mode"] == "decode" else [e(c["inter"]), e(c["inter"])]
        st["out"] = [e(L.qkv.N), e(c["hidden"]), *mid, e(c["hidden"])]
    else:
        kinds = _kinds(c)
        layers = [_build_layer(gpu, c, _layer_raw(c, seed, 8 + 16 * i, a), a) for i, a in enumerate(kinds)]
        lm = _upload(gpu, _raw_gptq(seed, 4, c["hidden"], c["vocab"], c["gs"], c["zeros"], False), c["gs"])
        stack = sta.DecoderStack(layers, lm)
        b = stack.buffers(gpu, c["m"])
        hooks = _Model(_x(seed, 1, c["m"], c["hidden"], small=0.5), [L.attn_dim for L in layers])
        st.update(stack=stack, hooks=hooks, buffers=b, graph=stack.capture(gpu, b, hooks))
    return st


def run(state):
    c, gpu = state["case"], state["gpu"]
    if c["kind"] == "linear":
        sta.linear(gpu, state["x"], state["w"], state["y"])
        return state["y"]
    if c["kind"] == "head":
        sta.bf16_matvec(gpu, state["x"], state["w"], state["y"], c["k"], c["n"])
        return state["y"]
    if c["kind"] == "layer":
        L = state["layer"]
        (L.decode if c["mode"] == "decode" else L.prefill)(gpu, state["x"], state["attn"], *state["out"], xm=state["xm"])
        return state["out"]
    state["graph"].replay()
    b = state["buffers"]
    return dict(logits=b.logits, x=b.x, h=b.h, qkv=b.qkv)


def _gptq_bytes(k, n, gs, zeros, act):
    return k * n / 2 + 2 * (k // gs) * n + (k // gs * n / 2 if zeros else 0) + (4 * k if act else 0)


def work(case):
    c, m = case, case["m"]
    if c["kind"] == "head":
        return dict(bytes=2 * c["k"] * c["n"] + m * (c["k"] * (2 if c["x"] == "f16" else 4) + 4 * c["n"]),
                    flops=2 * m * c["k"] * c["n"])
    if c["kind"] == "linear":
        io = m * (c["k"] * (2 if c["x"] == "f16" else 4) + c["n"] * (2 if c.get("y") == "f16" else 4))
        w = c["k"] * c["n"] + 4 * c["n"] if c["fmt"] == "int8" else _gptq_bytes(c["k"], c["n"], c["gs"], c["zeros"], c["act"])
        return dict(bytes=w + io, flops=2 * m * c["k"] * c["n"])
    by = fl = 0
    kinds = _kinds(c) if c["kind"] == "step" else [c["attn"]]
    size = 2 if c.get("mode") == "prefill" else 4
    for a in kinds:
        for name, k, n in _layer_shapes(c, a):
            by += _gptq_bytes(k, n, c["gs"], c["zeros"], c.get("act", False))
            fl += 2 * m * k * n
        q = sum(n for name, k, n in _layer_shapes(c, a) if name in ("q", "k", "v", "in_qkv", "in_z"))
        ad = next(k for name, k, n in _layer_shapes(c, a) if name in ("o", "out"))
        by += m * size * (4 * c["hidden"] + ad + q + c["inter"])
    if c["kind"] == "step":
        by += _gptq_bytes(c["hidden"], c["vocab"], c["gs"], c["zeros"], False) + 4 * m * (c["hidden"] + c["vocab"])
        fl += 2 * m * c["hidden"] * c["vocab"]
    return dict(bytes=by, flops=fl)


def tolerance(case):
    c = case
    if c["kind"] == "layer" and c["mode"] == "prefill":  # f16 inputs, weights, outputs and products
        return {"rel": 2e-3}
    if c["kind"] == "linear" and c["m"] > 32:
        # GPTQ weights are rounded to f16; int8 products are exact
        if c["fmt"] == "int8":
            return {"rel": 1e-3} if c["y"] == "f16" else {"rel": 2e-6}
        return {"rel": 1e-3}
    if c["kind"] == "head":  # f32 sums
        return {"rel": 2e-6}
    # f32 sums of exact products of x held in 22 bits of its group's range (a step: the same, a few layers deep)
    return {"rel": 5e-6}


# ------------------------------------------------------------ 64-bit values
def _w64(raw, gs):
    """The dequantized weight [K, N] in float64: (q - z) * s of each row's group."""
    qw, s, qz, gi = raw
    k, n = qw.shape[0] * 8, qw.shape[1]
    q = torch.stack([(qw >> (4 * j)) & 15 for j in range(8)], dim=1).reshape(k, n)
    row = torch.arange(k, device=DEV) // gs if gi is None else gi.long()
    w = q.double()
    if qz is None:
        w -= 8.0
    else:
        z = torch.stack([(qz >> (4 * j)) & 15 for j in range(8)], dim=2).reshape(k // gs, n)
        w -= z.double()[row]
    return w.mul_(s.double()[row])


def _mm64(x, raw, gs):
    return x @ _w64(raw, gs)


def _silu64(v):
    return v / (1.0 + torch.exp(-v))


def _layer64(c, raw, attn, x, core, xm=None):
    """(qkv, o, gate, up, h, down, xm): one layer in float64; xm a function of o when callable."""
    gs = c["gs"]
    if attn == "self":
        qkv = torch.cat([_mm64(x, raw[n], gs) for n in ("q", "k", "v")], dim=1)
        a = core(qkv) if callable(core) else core
        o = _mm64(a, raw["o"], gs)
    else:
        q, z = _mm64(x, raw["in_qkv"], gs), _mm64(x, raw["in_z"], gs)
        qkv = torch.cat([q, z], dim=1)
        a = core(qkv) if callable(core) else core
        o = _mm64(_silu64(z) * a, raw["out"], gs)
    xm = xm(o) if callable(xm) else xm
    g, u = _mm64(xm, raw["gate"], gs), _mm64(xm, raw["up"], gs)
    h = _silu64(g) * u
    return qkv, o, g, u, h, _mm64(h, raw["down"], gs), xm


def exact(case, seed):
    c = case
    if c["kind"] == "linear":
        x = _x(seed, 1, c["m"], c["k"], _dt(c, "x")).double()
        if c["fmt"] == "int8":
            w, s = _raw_int8(seed, 2, c["k"], c["n"])
            return (x @ w.double().t()) * s.double()
        return _mm64(x, _raw_gptq(seed, 2, c["k"], c["n"], c["gs"], c["zeros"], c["act"]), c["gs"])
    if c["kind"] == "head":
        return _x(seed, 1, c["m"], c["k"], _dt(c, "x")).double() @ _raw_head(seed, 2, c["k"], c["n"]).double().t()
    if c["kind"] == "layer":
        dt = torch.float32 if c["mode"] == "decode" else torch.float16
        x, a, xm = (_x(seed, i, c["m"], c[key], dt, 0.5).double()
                    for i, key in ((1, "hidden"), (2, "attn_dim"), (3, "hidden")))
        qkv, o, g, u, h, down, _ = _layer64(c, _layer_raw(c, seed, 8, c["attn"]), c["attn"], x, a, xm)
        return [qkv, o, h, down] if c["mode"] == "decode" else [qkv, o, g, u, down]
    x = _x(seed, 1, c["m"], c["hidden"], small=0.5).double()
    for i, attn in enumerate(_kinds(c)):
        a = c["attn_dim"] if attn == "self" else c["dn_dim"]
        raw = _layer_raw(c, seed, 8 + 16 * i, attn)
        core = lambda qkv, a=a: 0.25 * qkv[:, :a]
        qkv, o, g, u, h, down, xm = _layer64(c, raw, attn, x, core, lambda o, x=x: x + o)
        x = xm + 0.25 * down
    return dict(logits=_mm64(x, _raw_gptq(seed, 4, c["hidden"], c["vocab"], c["gs"], c["zeros"], False), c["gs"]), x=x, h=h,
                qkv=qkv)
