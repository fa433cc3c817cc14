"""Timed cases: what a decoder built on this library has it do, through llaisys_amd.Ops.

The shapes are the ones this repository's benchmark and tests use: a Qwen2-1.5B decoder layer
(hidden 1536, 12 q / 2 kv heads of 128, intermediate 8960, vocabulary 151936) and Llama-style 8B
sizes (4096, 32 / 8 heads, 14336), with random weights N(0, 0.02) and activations N(0, 1).
Inputs are made on the GPU with torch and handed over as library tensors; torch views of the
library's output tensors are what run() returns.

Kinds of case, each with a share of `draw`:
  layer   one decoder layer: norm, q / k / v, RoPE, KV append, attention, o, norm, MLP
  mlp     residual add + rms_norm, gate / up, swiglu, down (prefill and few-row steps)
  attn    causal attention of `seq` queries over `past + seq` cached tokens
  ops     the bandwidth-bound layer ops of a prefill (embedding, norms, RoPE, swiglu)
  head    final norm, lm_head projection, greedy and sampled token of each row
  int8    weight quantization and its read-back, KV-cache append and its read-back
"""
import math

import torch

import llaisys_amd as L

HIDDEN, HEADS, KV_HEADS, DIM, INTER, VOCAB = 1536, 12, 2, 128, 8960, 151936
EPS, THETA = 1e-6, 1e6
TORCH = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}
LIB = {"f32": L.DataType.F32, "bf16": L.DataType.BF16, "f16": L.DataType.F16, "i8": L.DataType.I8,
       "i64": L.DataType.I64}
BYTES = {"f32": 4, "bf16": 2, "f16": 2, "i8": 1, "i64": 8}
GPU = "cuda"


def listed():
    return [
        # one generated token, INT8 weights and KV cache: the smallest call and the most frequent
        {"name": "layer decode 1 int8", "kind": "layer", "tokens": 1, "past": 4096, "dtype": "bf16", "weights": "int8",
         "kv": "int8"},
        # a few tokens checked at once (speculative decoding), 16-bit weights, an odd context
        {"name": "layer verify 5 bf16", "kind": "layer", "tokens": 5, "past": 1531, "dtype": "bf16", "weights": "dense",
         "kv": "int8"},
        # a short prompt in f32, the element type a checkpoint is loaded in by default
        {"name": "layer prompt 128 f32", "kind": "layer", "tokens": 128, "past": 0, "dtype": "f32", "weights": "dense",
         "kv": "plain"},
        # a short prompt's MLP: tens of rows, the weights' bytes still count
        {"name": "mlp 37 bf16", "kind": "mlp", "rows": 37, "hidden": HIDDEN, "inter": INTER, "dtype": "bf16",
         "weights": "dense"},
        # the MLP of a long prompt, 16-bit and INT8 weights: the bulk of a prefill's arithmetic
        {"name": "mlp 2048 bf16", "kind": "mlp", "rows": 2048, "hidden": HIDDEN, "inter": INTER, "dtype": "bf16",
         "weights": "dense"},
        {"name": "mlp 2048 int8", "kind": "mlp", "rows": 2048, "hidden": HIDDEN, "inter": INTER, "dtype": "bf16",
         "weights": "int8"},
        # a long prompt's attention in one pass
        {"name": "attn prefill 2048 bf16", "kind": "attn", "seq": 2048, "past": 0, "heads": HEADS, "kv_heads": KV_HEADS,
         "dim": DIM, "dtype": "bf16", "kv": "plain"},
        # one chunk of a long prompt over the INT8 cache of the chunks before it, 16-bit floats
        # with the wider mantissa
        {"name": "attn chunk 300 f16", "kind": "attn", "seq": 300, "past": 1200, "heads": HEADS, "kv_heads": KV_HEADS,
         "dim": DIM, "dtype": "f16", "kv": "int8"},
        # one token over a long INT8 cache
        {"name": "attn decode 32768 int8", "kind": "attn", "seq": 1, "past": 32767, "heads": HEADS,
         "kv_heads": KV_HEADS, "dim": DIM, "dtype": "bf16", "kv": "int8"},
        # the bandwidth-bound ops of a long prompt: the benchmark's own shape
        {"name": "ops 8192 bf16", "kind": "ops", "tokens": 8192, "hidden": HIDDEN, "heads": HEADS, "kv_heads": KV_HEADS,
         "inter": INTER, "dtype": "bf16"},
        # the end of a decode step: the largest weight there is, then the token
        {"name": "head 1 bf16", "kind": "head", "rows": 1, "dtype": "bf16", "weights": "dense", "top_k": 50},
        # weights converted at load, a 32768-token cache written and read back
        {"name": "int8 8960x1536 kv 32768", "kind": "int8", "out": INTER, "in": HIDDEN, "tokens": 32768,
         "kv_heads": KV_HEADS, "dim": DIM, "dtype": "bf16"},
    ]


def _log(rng, lo, hi):
    """A whole number spread over the logarithm of [lo, hi]."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["layer", "layer", "mlp", "mlp", "attn", "attn", "attn", "ops", "head", "int8"])
    dt = rng.choice(["bf16", "bf16", "bf16", "f16", "f32"])
    if kind == "layer":
        if dt == "f32":
            return {"kind": kind, "tokens": _log(rng, 1, 128), "past": 0, "dtype": dt, "weights": "dense", "kv": "plain"}
        if rng.random() < 0.3:
            return {"kind": kind, "tokens": _log(rng, 1, 1024), "past": 0, "dtype": dt,
                    "weights": rng.choice(["int8", "dense"]), "kv": "plain"}
        tokens, past = (600, 8192) if dt == "bf16" else (128, 2048)
        return {"kind": kind, "tokens": _log(rng, 1, tokens), "past": _log(rng, 16, past), "dtype": dt,
                "weights": rng.choice(["int8", "dense"]), "kv": "int8"}
    if kind == "mlp":
        hidden, inter = rng.choice([(1536, 8960), (1536, 8960), (4096, 14336), (1024, 2816)])
        most = 2048 * 1536 * 8960 // (hidden * inter)
        return {"kind": kind, "rows": _log(rng, 2, min(2048, most) if dt != "f32" else min(128, max(2, most // 16))),
                "hidden": hidden, "inter": inter, "dtype": dt,
                "weights": rng.choice(["int8", "dense"]) if dt != "f32" else "dense"}
    if kind == "attn":
        heads, kv_heads = rng.choice([(12, 2), (12, 2), (32, 8), (16, 16)])
        dim = rng.choice([128, 128, 64])
        kv = rng.choice(["plain", "int8"])
        if rng.random() < 0.4:  # decode
            return {"kind": kind, "seq": _log(rng, 1, 8), "past": _log(rng, 64, 32767 if heads == 12 else 8191),
                    "heads": heads, "kv_heads": kv_heads, "dim": dim, "dtype": dt, "kv": kv}
        seq = _log(rng, 16, 2048 if dt == "bf16" and dim == 128 else 400)
        past = rng.choice([0, _log(rng, 16, 4096 if dt == "bf16" and dim == 128 else 1200)])
        if heads > 12:
            seq, past = max(16, seq // 3), past // 3
        return {"kind": kind, "seq": seq, "past": past, "heads": heads, "kv_heads": kv_heads, "dim": dim, "dtype": dt,
                "kv": kv}
    if kind == "ops":
        hidden, heads, kv_heads, inter = rng.choice([(1536, 12, 2, 8960), (4096, 32, 8, 14336)])
        most = 8192 * 1536 // hidden // (2 if dt == "f32" else 1)
        return {"kind": kind, "tokens": _log(rng, 1, most), "hidden": hidden, "heads": heads, "kv_heads": kv_heads,
                "inter": inter, "dtype": dt}
    if kind == "head":
        return {"kind": kind, "rows": _log(rng, 1, 16), "dtype": dt if dt != "f32" else "bf16",
                "weights": rng.choice(["int8", "dense"]), "top_k": rng.choice([1, 50, 1024])}
    out, inn = rng.choice([(8960, 1536), (1536, 8960), (2048, 1536), (4096, 4096)])
    return {"kind": kind, "out": out, "in": inn, "tokens": _log(rng, 1, 32768), "kv_heads": rng.choice([2, 8]),
            "dim": DIM, "dtype": dt}


# ---- library tensors and their torch views --------------------------------------------------


class _Memory:
    """A library tensor's device memory as torch's array protocol wants it."""

    def __init__(self, tensor, shape, dt):
        kind = {"f32": "<f4", "bf16": "<i2", "f16": "<f2", "i8": "|i1", "i64": "<i8"}[dt]
        self.tensor = tensor
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": kind, "data": (tensor.data_ptr(), False),
                                         "version": 2, "strides": None}


class Buf:
    """A library tensor `t` on the GPU and the torch view `v` of the same memory."""

    def __init__(self, shape, dt, values=None):
        self.t = L.Tensor(shape, LIB[dt], L.DeviceType.AMD, 0)
        self.v = torch.as_tensor(_Memory(self.t, shape, dt), device=GPU)
        if dt == "bf16":
            self.v = self.v.view(torch.bfloat16)
        if values is not None:
            self.v.copy_(values)


class Inputs:
    """Seeded torch tensors on the GPU, the same for prepare() and exact()."""

    def __init__(self, case, seed):
        self.gen = torch.Generator(device=GPU)
        self.gen.manual_seed(int(seed))
        self.dt = case["dtype"]

    def normal(self, *shape, scale=1.0, mean=0.0, dt=None):
        x = torch.randn(*shape, generator=self.gen, device=GPU)
        return x.mul_(scale).add_(mean).to(TORCH[dt or self.dt])

    def kv(self, *shape):
        """k / v rows with 1% outliers, scaled up 20 times."""
        x = torch.randn(*shape, generator=self.gen, device=GPU)
        x = torch.where(torch.rand(*shape, generator=self.gen, device=GPU) < 0.01, 20 * x, x)
        return x.to(TORCH[self.dt])

    def ids(self, n, top):
        return torch.randint(0, top, (n,), generator=self.gen, device=GPU)


def _inputs(case, seed):
    """Every input of the case by name, as torch tensors in the case's element type."""
    g, kind = Inputs(case, seed), case["kind"]
    if kind == "layer":
        t, past = case["tokens"], case["past"]
        d = {"x": g.normal(t, HIDDEN), "res": g.normal(t, HIDDEN),
             "n1": g.normal(HIDDEN, scale=0.1, mean=1.0), "n2": g.normal(HIDDEN, scale=0.1, mean=1.0),
             "pos": torch.arange(past, past + t, device=GPU)}
        for name, rows, cols in (("q", HEADS * DIM, HIDDEN), ("k", KV_HEADS * DIM, HIDDEN), ("v", KV_HEADS * DIM, HIDDEN),
                                 ("o", HIDDEN, HEADS * DIM), ("gate_up", 2 * INTER, HIDDEN), ("down", HIDDEN, INTER)):
            d["w_" + name] = g.normal(rows, cols, scale=0.02)
        for name, rows in (("q", HEADS * DIM), ("k", KV_HEADS * DIM), ("v", KV_HEADS * DIM)):
            d["b_" + name] = g.normal(rows, scale=0.1)
        if past:
            d["past_k"], d["past_v"] = g.kv(past, KV_HEADS, DIM), g.kv(past, KV_HEADS, DIM)
        return d
    if kind == "mlp":
        m, h, i = case["rows"], case["hidden"], case["inter"]
        return {"x": g.normal(m, h), "res": g.normal(m, h), "n": g.normal(h, scale=0.1, mean=1.0),
                "w_gate_up": g.normal(2 * i, h, scale=0.02), "w_down": g.normal(h, i, scale=0.02)}
    if kind == "attn":
        total = case["past"] + case["seq"]
        return {"q": g.normal(case["seq"], case["heads"], case["dim"]), "k": g.kv(total, case["kv_heads"], case["dim"]),
                "v": g.kv(total, case["kv_heads"], case["dim"])}
    if kind == "ops":
        t, h, d = case["tokens"], case["hidden"], DIM
        vocab = VOCAB if h == HIDDEN else 128256
        return {"ids": g.ids(t, vocab), "table": g.normal(vocab, h, scale=0.02), "x": g.normal(t, h), "res": g.normal(t, h),
                "n": g.normal(h, scale=0.1, mean=1.0), "q": g.normal(t, case["heads"], d),
                "k": g.normal(t, case["kv_heads"], d), "pos": torch.arange(t, device=GPU),
                "gate": g.normal(t, case["inter"]), "up": g.normal(t, case["inter"])}
    if kind == "head":
        m = case["rows"]
        d = {"w": g.normal(VOCAB, HIDDEN, scale=0.02), "n": g.normal(HIDDEN, scale=0.1, mean=1.0),
             "res": g.normal(m, HIDDEN, scale=0.3)}
        # a trained head is sure of some token: the hidden state leans towards one row of the weights
        d["x"] = (d["res"].float() + 60 * d["w"][g.ids(m, VOCAB)].float()).to(TORCH[case["dtype"]])
        return d
    return {"w": g.normal(case["out"], case["in"], scale=0.02), "k": g.kv(case["tokens"], case["kv_heads"], case["dim"]),
            "v": g.kv(case["tokens"], case["kv_heads"], case["dim"])}


def _quantized(values, dt):
    """Codes and scales of a weight or a cache as a program keeps them."""
    src = Buf(values.shape, dt, values)
    q, s = Buf(values.shape, "i8"), Buf(values.shape[:-1], "f32")
    torch.cuda.synchronize()
    L.Ops.quantize_int8(q.t, s.t, src.t)
    torch.cuda.synchronize()
    return q, s


class State:
    pass


def prepare(case, seed):
    s, x, dt, kind = State(), _inputs(case, seed), case["dtype"], case["kind"]
    s.case = case

    def put(*names):
        for n in names:
            v = x[n]
            setattr(s, n, Buf(v.shape, "i64" if v.dtype == torch.int64 else dt, v))

    def new(name, *shape, dt=dt):
        setattr(s, name, Buf(shape, dt))

    def weight(name, values):
        setattr(s, name, _quantized(values, dt) if case["weights"] == "int8" else (Buf(values.shape, dt, values), None))

    if kind == "layer":
        t, total = case["tokens"], case["past"] + case["tokens"]
        put("x", "res", "n1", "n2", "pos")
        if t == 1 and case["kv"] == "int8":  # one row: q / k / v are one projection, sliced
            weight("w_qkv", torch.cat([x["w_q"], x["w_k"], x["w_v"]]))
            b = torch.cat([x["b_q"], x["b_k"], x["b_v"]])
            s.b_qkv = Buf(b.shape, dt, b)
            n = (HEADS + 2 * KV_HEADS) * DIM
            new("qkv", 1, n)
            flat = s.qkv.t.view(n)
            s.q = flat.slice(0, 0, HEADS * DIM).view(1, HEADS, DIM)
            s.k = flat.slice(0, HEADS * DIM, (HEADS + KV_HEADS) * DIM).view(1, KV_HEADS, DIM)
            s.v = flat.slice(0, (HEADS + KV_HEADS) * DIM, n).view(1, KV_HEADS, DIM)
        else:
            put("b_q", "b_k", "b_v")
            new("xn", t, HIDDEN)
            for n, heads in (("q", HEADS), ("k", KV_HEADS), ("v", KV_HEADS)):
                weight("w_" + n, x["w_" + n])
                new("p_" + n, t, heads * DIM)
                setattr(s, n, getattr(s, "p_" + n).t.view(t, heads, DIM))
        weight("w_o", x["w_o"])
        weight("w_gate_up", x["w_gate_up"])
        weight("w_down", x["w_down"])
        new("h1", t, HIDDEN)
        new("q_rot", t, HEADS, DIM)
        new("att", t, HEADS, DIM)
        s.att_flat = s.att.t.view(t, HEADS * DIM)
        new("o", t, HIDDEN)
        new("h2", t, HIDDEN)
        new("act", t, INTER)
        new("out", t, HIDDEN)
        if case["kv"] == "int8":
            for n in ("k", "v"):
                new("c_" + n, total, KV_HEADS, DIM, dt="i8")
                new("s_" + n, total, KV_HEADS, dt="f32")
                getattr(s, "c_" + n).v.zero_()
                getattr(s, "s_" + n).v.zero_()
                if case["past"]:
                    src = Buf(x["past_" + n].shape, dt, x["past_" + n])
                    torch.cuda.synchronize()
                    L.Ops.kv_append_int8(getattr(s, "c_" + n).t, getattr(s, "s_" + n).t, src.t, 0)
                    torch.cuda.synchronize()
        else:
            new("k_rot", t, KV_HEADS, DIM)
    elif kind == "mlp":
        m, h, i = case["rows"], case["hidden"], case["inter"]
        put("x", "res", "n")
        weight("w_gate_up", x["w_gate_up"])
        weight("w_down", x["w_down"])
        new("h", m, h)
        new("act", m, i)
        new("out", m, h)
    elif kind == "attn":
        put("q")
        if case["kv"] == "int8":
            s.k, s.v = _quantized(x["k"], dt), _quantized(x["v"], dt)
        else:
            put("k", "v")
        new("out", case["seq"], case["heads"], case["dim"])
    elif kind == "ops":
        t, h = case["tokens"], case["hidden"]
        put("ids", "table", "x", "res", "n", "q", "k", "pos", "gate", "up")
        new("emb", t, h)
        new("y1", t, h)
        new("y2", t, h)
        new("h", t, h)
        new("q_rot", t, case["heads"], DIM)
        new("k_rot", t, case["kv_heads"], DIM)
        new("act", t, case["inter"])
    elif kind == "head":
        m = case["rows"]
        put("x", "res", "n")
        weight("w", x["w"])
        new("xn", m, HIDDEN)
        new("h", m, HIDDEN)
        new("logits", m, VOCAB)
        new("best", m, dt="i64")
        new("best_val", m)
        new("token", m, dt="i64")
    else:
        put("w", "k", "v")
        shape = (case["out"], case["in"])
        new("q", *shape, dt="i8")
        new("scale", case["out"], dt="f32")
        new("back", *shape)
        kv = (case["tokens"], case["kv_heads"], case["dim"])
        for n in ("k", "v"):
            new("c_" + n, *kv, dt="i8")
            new("s_" + n, *kv[:2], dt="f32")
            new("back_" + n, *kv)
    torch.cuda.synchronize()
    return s


def _linear(out, x, w, bias=None):
    if w[1] is None:
        L.Ops.linear(out, x, w[0].t, bias)
    else:
        L.Ops.linear_w8a16(out, x, w[0].t, w[1].t, bias)


def run(s):
    O, c = L.Ops, s.case
    kind = c["kind"]
    if kind == "layer":
        scale, past = 1.0 / math.sqrt(DIM), c["past"]
        if c["tokens"] == 1 and c["kv"] == "int8":
            w, sc = s.w_qkv
            O.rms_norm_linear(s.qkv.t, s.x.t, s.n1.t, EPS, w.t, sc and sc.t, s.b_qkv.t, residual=s.res.t,
                              residual_out=s.h1.t)
        else:
            O.add_rms_norm(s.xn.t, s.h1.t, s.x.t, s.res.t, s.n1.t, EPS)
            _linear(s.p_q.t, s.xn.t, s.w_q, s.b_q.t)
            _linear(s.p_k.t, s.xn.t, s.w_k, s.b_k.t)
            _linear(s.p_v.t, s.xn.t, s.w_v, s.b_v.t)
        if c["kv"] == "int8":
            O.rope_kv_append_int8(s.q_rot.t, s.q, s.k, s.v, s.pos.t, THETA, s.c_k.t, s.s_k.t, s.c_v.t, s.s_v.t, past)
            O.self_attention_int8kv(s.att.t, s.q_rot.t, s.c_k.t, s.s_k.t, s.c_v.t, s.s_v.t, scale)
        else:
            O.rope_qk(s.q_rot.t, s.q, s.k_rot.t, s.k, s.pos.t, THETA)
            O.self_attention(s.att.t, s.q_rot.t, s.k_rot.t, s.v, scale)
        _linear(s.o.t, s.att_flat, s.w_o)
        w, sc = s.w_gate_up
        O.rms_norm_linear(s.act.t, s.o.t, s.n2.t, EPS, w.t, sc and sc.t, residual=s.h1.t, residual_out=s.h2.t, swiglu=True)
        _linear(s.out.t, s.act.t, s.w_down)
        r = {"hidden": s.h2.v, "out": s.out.v, "att": s.att.v}
        if c["kv"] == "int8":
            r.update(c_k=s.c_k.v, s_k=s.s_k.v, c_v=s.c_v.v, s_v=s.s_v.v)
        return r
    if kind == "mlp":
        w, sc = s.w_gate_up
        O.rms_norm_linear(s.act.t, s.x.t, s.n.t, EPS, w.t, sc and sc.t, residual=s.res.t, residual_out=s.h.t, swiglu=True)
        _linear(s.out.t, s.act.t, s.w_down)
        return {"hidden": s.h.v, "act": s.act.v, "out": s.out.v}
    if kind == "attn":
        scale = 1.0 / math.sqrt(c["dim"])
        if c["kv"] == "int8":
            O.self_attention_int8kv(s.out.t, s.q.t, s.k[0].t, s.k[1].t, s.v[0].t, s.v[1].t, scale)
        else:
            O.self_attention(s.out.t, s.q.t, s.k.t, s.v.t, scale)
        return {"out": s.out.v}
    if kind == "ops":
        O.embedding(s.emb.t, s.ids.t, s.table.t)
        O.rms_norm(s.y1.t, s.emb.t, s.n.t, EPS)
        O.add_rms_norm(s.y2.t, s.h.t, s.x.t, s.res.t, s.n.t, EPS)
        O.rope_qk(s.q_rot.t, s.q.t, s.k_rot.t, s.k.t, s.pos.t, THETA)
        O.swiglu(s.act.t, s.gate.t, s.up.t)
        return {"emb": s.emb.v, "y1": s.y1.v, "y2": s.y2.v, "h": s.h.v, "q": s.q_rot.v, "k": s.k_rot.v, "act": s.act.v}
    if kind == "head":
        O.add_rms_norm(s.xn.t, s.h.t, s.x.t, s.res.t, s.n.t, EPS)
        _linear(s.logits.t, s.xn.t, s.w)
        O.argmax_rows(s.best.t, s.best_val.t, s.logits.t)
        O.random_sample(s.token.t, s.logits.t, 0.8, c["top_k"], 0.8, 7)
        return {"hidden": s.h.v, "logits": s.logits.v, "best": s.best.v, "best_val": s.best_val.v, "token": s.token.v}
    O.quantize_int8(s.q.t, s.scale.t, s.w.t)
    O.dequantize_int8(s.back.t, s.q.t, s.scale.t)
    O.kv_append_int8_pair(s.c_k.t, s.s_k.t, s.c_v.t, s.s_v.t, s.k.t, s.v.t, 0)
    O.dequantize_int8_pair(s.back_k.t, s.c_k.t, s.s_k.t, s.back_v.t, s.c_v.t, s.s_v.t)
    return {"q": s.q.v, "scale": s.scale.v, "back": s.back.v, "c_k": s.c_k.v, "s_k": s.s_k.v, "c_v": s.c_v.v,
            "s_v": s.s_v.v, "back_k": s.back_k.v, "back_v": s.back_v.v}


# ---- what the work comes to ------------------------------------------------------------------


def _visible(seq, past):
    """Pairs of a query and a key that it sees."""
    return seq * past + seq * (seq + 1) // 2


def work(case):
    e, kind = BYTES[case["dtype"]], case["kind"]
    we = 1 if case.get("weights") == "int8" else e
    if kind == "layer":
        t, total = case["tokens"], case["past"] + case["tokens"]
        n = 2 * (HEADS + KV_HEADS) * DIM * HIDDEN + 3 * HIDDEN * INTER
        kv = 2 * total * KV_HEADS * (DIM + 4) if case["kv"] == "int8" else 0
        return {"bytes": n * we + t * HIDDEN * 4 * e + t * HEADS * DIM * e + kv,
                "flops": 2 * t * n + 4 * HEADS * DIM * _visible(t, case["past"])}
    if kind == "mlp":
        m, h, i = case["rows"], case["hidden"], case["inter"]
        return {"bytes": 3 * h * i * we + m * (4 * h + i) * e, "flops": 2 * m * 3 * h * i}
    if kind == "attn":
        total, row = case["past"] + case["seq"], case["kv_heads"] * (case["dim"] + 4 if case["kv"] == "int8" else case["dim"] * e)
        return {"bytes": 2 * total * row + 2 * case["seq"] * case["heads"] * case["dim"] * e,
                "flops": 4 * case["heads"] * case["dim"] * _visible(case["seq"], case["past"])}
    if kind == "ops":
        t, h = case["tokens"], case["hidden"]
        n = 2 * h + 2 * h + 4 * h + 2 * (case["heads"] + case["kv_heads"]) * DIM + 3 * case["inter"]
        return {"bytes": t * (n * e + 16), "flops": t * (12 * h + 8 * case["inter"])}
    if kind == "head":
        m = case["rows"]
        return {"bytes": VOCAB * HIDDEN * we + m * (VOCAB + 3 * HIDDEN) * e, "flops": 2 * m * VOCAB * HIDDEN}
    w, kv = case["out"] * case["in"], 2 * case["tokens"] * case["kv_heads"] * case["dim"]
    return {"bytes": (w + kv) * (2 * e + 1) + 4 * (case["out"] + 2 * case["tokens"] * case["kv_heads"]),
            "flops": 4 * (w + kv)}


def tolerance(case):
    kind, dt = case["kind"], case["dtype"]
    if kind == "int8":
        return "exact"
    if dt == "f32":
        # f32 sums in another order: 2e-6 off the 64-bit result after a whole layer
        return {"rel": 8e-6, "max": 3e-4}
    # results rounded to 16 bits: a sum in another order moves a few of them by one step, and a
    # code of an INT8 cache where a rounded input moved
    rel = {"bf16": 8e-3, "f16": 2e-3}[dt]
    return {"rel": rel, "max": 0.1 if dt == "bf16" else 0.02, "differ": 0.01 if kind == "layer" else 0.0}


# ---- the same results in 64 bits ---------------------------------------------------------------


def _norm(x, w):
    return x * w / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS)


def _read_back(values):
    """A row-quantized tensor's values, in 64 bits."""
    f = values.float()
    scale = f.abs().amax(-1, keepdim=True) / 127
    q = torch.clamp(torch.round(torch.where(scale > 0, f / scale, torch.zeros_like(f))), -127, 127)
    return q.double() * scale.double()


def _rope(x, pos):
    half = x.shape[-1] // 2
    freq = torch.tensor(THETA, dtype=torch.float64, device=GPU) ** (-2.0 * torch.arange(half, device=GPU).double() / (2 * half))
    a = pos.double()[:, None, None] * freq
    x1, x2 = x[..., :half], x[..., half:]
    return torch.cat([x1 * torch.cos(a) - x2 * torch.sin(a), x2 * torch.cos(a) + x1 * torch.sin(a)], -1)


def _attend(q, k, v):
    seq, heads, d = q.shape
    total, group = k.shape[0], heads // k.shape[1]
    out = torch.empty(seq, heads, v.shape[2], dtype=torch.float64, device=GPU)
    at = torch.arange(total - seq, total, device=GPU)[:, None]
    hide = torch.arange(total, device=GPU)[None, :] > at
    for h in range(heads):
        s = q[:, h] @ k[:, h // group].T.contiguous() / math.sqrt(d)
        out[:, h] = torch.softmax(s.masked_fill_(hide, -math.inf), -1) @ v[:, h // group]
    return out


def _swiglu(y):
    gate, up = y.chunk(2, -1)
    return up * gate / (1 + torch.exp(-gate))


def exact(case, seed):
    x, kind = _inputs(case, seed), case["kind"]
    d = {k: (v if v.dtype == torch.int64 else v.double()) for k, v in x.items()}
    w = {k: (_read_back(x[k]) if case.get("weights") == "int8" else d[k]) for k in x if k == "w" or k.startswith("w_")}
    if kind == "layer":
        t, total = case["tokens"], case["past"] + case["tokens"]
        h1 = d["x"] + d["res"]
        n = _norm(h1, d["n1"])
        q = (n @ w["w_q"].T + d["b_q"]).view(t, HEADS, DIM)
        k = (n @ w["w_k"].T + d["b_k"]).view(t, KV_HEADS, DIM)
        v = (n @ w["w_v"].T + d["b_v"]).view(t, KV_HEADS, DIM)
        q, k = _rope(q, d["pos"]), _rope(k, d["pos"])
        if case["kv"] == "int8":
            k, v = _read_back(k), _read_back(v)
            if case["past"]:
                k, v = torch.cat([_read_back(x["past_k"]), k]), torch.cat([_read_back(x["past_v"]), v])
        att = _attend(q, k, v)
        h2 = h1 + att.reshape(t, -1) @ w["w_o"].T
        r = {"hidden": h2, "out": _swiglu(_norm(h2, d["n2"]) @ w["w_gate_up"].T) @ w["w_down"].T, "att": att}
        if case["kv"] == "int8":
            r.update(c_k=None, s_k=None, c_v=None, s_v=None)
        return r
    if kind == "mlp":
        h = d["x"] + d["res"]
        act = _swiglu(_norm(h, d["n"]) @ w["w_gate_up"].T)
        return {"hidden": h, "act": act, "out": act @ w["w_down"].T}
    if kind == "attn":
        if case["kv"] == "int8":
            d["k"], d["v"] = _read_back(x["k"]), _read_back(x["v"])
        return {"out": _attend(d["q"], d["k"], d["v"])}
    if kind == "ops":
        emb, h, gate = d["table"][d["ids"]], d["x"] + d["res"], d["gate"]
        return {"emb": emb, "y1": _norm(emb, d["n"]), "y2": _norm(h, d["n"]), "h": h, "q": _rope(d["q"], d["pos"]),
                "k": _rope(d["k"], d["pos"]), "act": d["up"] * gate / (1 + torch.exp(-gate))}
    if kind == "head":
        h = d["x"] + d["res"]
        logits = _norm(h, d["n"]) @ w["w"].T
        return {"hidden": h, "logits": logits, "best": None, "best_val": logits.amax(-1), "token": None}
    out = {}
    for name, src in (("", "w"), ("_k", "k"), ("_v", "v")):
        out["back" + name] = _read_back(x[src])
        scale = (x[src].float().abs().amax(-1) / 127).double()
        out["s" + name if name else "scale"] = scale
        out["c" + name if name else "q"] = None
    return out
