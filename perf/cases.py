"""The work a program has this library do, as cases that can be timed and compared.

A case is a dict of plain values with a "kind":

* ``linear``, ``linear_backward``: one linear layer's forward, and its dX / dW / db, through ``laya_amd.ops``;
* ``attention``: one attention layer, forward and backward;
* ``mlp``: an encoder layer's MLP half (LayerNorm, Wi, GeGLU, Wo with the skip add) and its backward, with the
  operands' magnitude words kept beside the buffers as ``laya_amd.opmodel`` keeps them;
* ``norm``: a LayerNorm, forward and backward;
* ``decide``: inference of the whole model (``TrainableDecisionModel.decide``: eval forward and read-out);
* ``train``: a whole optimizer step composed from the per-op entry points (``OpLevelModel.train_step``).

Widths are those of ``laya_amd.config``: ModernBERT-base (768, GeGLU 1152, 12 heads) and ModernBERT-large (1024,
GeGLU 2624, 16 heads), head feed-forward 4 x width. Activations are unit normal (what a LayerNorm leaves), weights
N(0, 0.02), gradients small with rows of unequal size.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from laya_amd import ops
from laya_amd.batch import Batch
from laya_amd.config import modernbert_base
from laya_amd.device import Context, DeviceArray
from laya_amd.model import TrainableDecisionModel
from laya_amd.opmodel import OpBatch, OpLevelModel

VOCAB = 50368
# (in, out, bias) of the linears: the encoder's Wqkv, Wo, mlp.Wi, mlp.Wo and the head's in_proj, linear1, linear2.
LINEARS = [(768, 2304, False), (768, 768, False), (1152, 768, False), (768, 2304, True), (768, 3072, True),
           (3072, 768, True), (1024, 3072, False), (1024, 1024, False), (1024, 5248, False), (2624, 1024, False)]


def listed():
    return [
        # One head layer's attention on a batch of 4 x 128 tokens, training mode: the smallest training batch.
        {"name": "attention head 4x128", "kind": "attention", "segments": 4, "longest": 128, "shortest": 128,
         "heads": 12, "half_window": -1, "theta": 0.0, "dropout": 0.1},
        # A sliding-window encoder layer (two of every three) on a batch of 32 x 512 with trailing padding dropped.
        {"name": "attention sliding 32x512", "kind": "attention", "segments": 32, "longest": 512, "shortest": 358,
         "heads": 12, "half_window": 64, "theta": 10000.0, "dropout": 0.0},
        # A global encoder layer on two sequences of the longest context the configuration allows.
        {"name": "attention global 2x8192", "kind": "attention", "segments": 2, "longest": 8192, "shortest": 8192,
         "heads": 12, "half_window": -1, "theta": 160000.0, "dropout": 0.0},
        # ModernBERT-large's QKV projection on a short document.
        {"name": "linear 404x1024x3072", "kind": "linear", "rows": 404, "in": 1024, "out": 3072, "bias": False,
         "precision": "fp32"},
        # The head's feed-forward input projection over the real tokens of a batch of 32 x 512.
        {"name": "linear 13871x768x3072", "kind": "linear", "rows": 13871, "in": 768, "out": 3072, "bias": True,
         "precision": "fp32"},
        # Backward of an encoder layer's QKV projection on 4 x 128 tokens.
        {"name": "linear bwd 512x768x2304", "kind": "linear_backward", "rows": 512, "in": 768, "out": 2304,
         "bias": False, "precision": "fp32"},
        # Backward of an encoder layer's MLP output projection over the real tokens of a batch of 32 x 512.
        {"name": "linear bwd 13871x1152x768", "kind": "linear_backward", "rows": 13871, "in": 1152, "out": 768,
         "bias": False, "precision": "fp32"},
        # The same of the QKV projection at 32 x 1024 tokens with bf16 operands (mixed-precision training).
        {"name": "linear bwd bf16 32768x768", "kind": "linear_backward", "rows": 32768, "in": 768, "out": 2304,
         "bias": False, "precision": "bf16"},
        # An MLP half of ModernBERT-large on a micro-batch of four sequences, forward and backward.
        {"name": "mlp large 1618", "kind": "mlp", "rows": 1618, "hidden": 1024, "inter": 2624},
        # A LayerNorm (with bias, as the head's) over the real tokens of a batch of 32 x 512.
        {"name": "norm 13871x768", "kind": "norm", "rows": 13871, "n": 768},
        # One decision on one document: the whole base model's inference.
        {"name": "decide 1x189", "kind": "decide", "items": 1, "longest": 189, "shortest": 189, "layers": 22},
        # One optimizer step of a shallow model on a micro-batch.
        {"name": "train 8x512", "kind": "train", "items": 8, "longest": 512, "shortest": 358, "layers": 3},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["linear", "linear", "linear_backward", "linear_backward", "attention", "attention", "mlp",
                       "norm", "decide", "train"])
    if kind in ("linear", "linear_backward"):
        fan_in, fan_out, bias = rng.choice(LINEARS)
        return {"kind": kind, "rows": _log(rng, 60, 32768), "in": fan_in, "out": fan_out, "bias": bias,
                "precision": rng.choice(["fp32", "fp32", "fp32", "bf16"])}
    if kind == "attention":
        head = rng.random() < 0.25  # a decision-head layer: no RoPE, no window, dropout
        window = -1 if head or rng.random() < 0.4 else 64
        longest = _log(rng, 17, 8192)
        tokens = _log(rng, 256, 32768 if window > 0 else max(1024, min(32768, (1 << 26) // longest)))
        return {"kind": kind, "segments": max(1, min(64, tokens // longest)), "longest": longest,
                "shortest": max(1, int(longest * rng.uniform(0.3, 1.0))), "heads": rng.choice([12, 12, 16]),
                "half_window": window, "theta": 0.0 if head else 10000.0 if window > 0 else 160000.0,
                "dropout": 0.1 if head else 0.0}
    if kind == "mlp":
        hidden, inter = rng.choice([(768, 1152), (1024, 2624)])
        return {"kind": kind, "rows": _log(rng, 128, 16384), "hidden": hidden, "inter": inter}
    if kind == "norm":
        return {"kind": kind, "rows": _log(rng, 128, 65536), "n": rng.choice([768, 1024])}
    longest = _log(rng, 48, 512)
    items = _log(rng, 1, 8)
    return {"kind": kind, "items": items, "longest": longest, "shortest": max(20, int(longest * rng.uniform(0.5, 1))),
            "layers": rng.randint(3, 22) if kind == "decide" else rng.randint(2, 4)}


# ------------------------------------------------------------------------------------------ inputs

_contexts = {}


def _context(precision="fp32"):
    if precision not in _contexts:
        _contexts[precision] = Context(0)
        _contexts[precision].set_matmul_precision(precision)
    return _contexts[precision]


class _Window:
    """A device array's memory as torch sees it; keeps the array alive."""

    def __init__(self, owner, ptr, shape, kind="<f4"):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": kind, "data": (ptr, False), "version": 2}


def _tensor(a):
    return torch.as_tensor(_Window(a, a.ptr, a.shape, "<i4" if a.dtype == np.int32 else "<f4"), device="cuda")


def _put(ctx, t):
    """A tensor's values in a device array of the library's."""
    a = DeviceArray(ctx, t.shape, np.int32 if t.dtype == torch.int32 else np.float32, zero=False)
    _tensor(a).copy_(t)
    return a


def _new(ctx, *shape):
    return _put(ctx, torch.zeros(shape, device="cuda"))


def _parameter(ctx, name, t):
    return ops.Parameter(ctx, name, t.cpu().numpy())


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed) * 7919 + 11)


def _normal(g, *shape):
    return torch.randn(shape, generator=g, device="cuda")


def _gradient(g, rows, n):
    """Rows of unequal size, as the gradients of a batch's tokens have."""
    return _normal(g, rows, n) * (1e-4 * torch.exp(_normal(g, rows, 1)))


def _lengths(case, count):
    r = np.random.default_rng([count, case["longest"], case["shortest"]])  # the same for every seed
    return r.integers(case["shortest"], case["longest"] + 1, size=count).astype(np.int32)


def _inputs(case, seed):
    g, kind = _generator(seed), case["kind"]
    if kind in ("linear", "linear_backward"):
        m, k, n = case["rows"], case["in"], case["out"]
        d = {"x": _normal(g, m, k), "W": 0.02 * _normal(g, n, k), "b": 0.02 * _normal(g, n) if case["bias"] else None}
        if kind == "linear_backward":
            d["dy"] = _gradient(g, m, n)
        return d
    if kind == "attention":
        lengths = _lengths(case, case["segments"])
        t, d = int(lengths.sum()), 64 * case["heads"]
        return {"lengths": lengths, "qkv": _normal(g, t, 3 * d), "dcontext": _gradient(g, t, d),
                "seed": int(seed) * 31 + 7}
    if kind == "mlp":
        m, d, i = case["rows"], case["hidden"], case["inter"]
        return {"x": _normal(g, m, d), "dout": _gradient(g, m, d), "gamma": 1 + 0.1 * _normal(g, d),
                "Wi": 0.02 * _normal(g, 2 * i, d), "Wo": 0.02 * _normal(g, d, i)}
    if kind == "norm":
        m, n = case["rows"], case["n"]
        return {"x": 0.3 + 2 * _normal(g, m, n), "gamma": 1 + 0.1 * _normal(g, n), "beta": 0.1 * _normal(g, n),
                "dy": _gradient(g, m, n), "dx": _gradient(g, m, n)}
    r = np.random.default_rng([int(seed), 9])
    lengths = _lengths(case, case["items"])
    kinds = [(0, 8), (1, 4), (2, 2)]  # choice, score, noul
    qtypes = np.array([kinds[i % 3][0] for i in range(len(lengths))], np.int32)
    options = np.array([kinds[i % 3][1] for i in range(len(lengths))], np.int32)
    batch = Batch(lengths=lengths, tokens=r.integers(0, VOCAB, int(lengths.sum())).astype(np.int32), n_options=options,
                  markers=np.concatenate([1 + 2 * np.arange(k) for k in options]).astype(np.int32), qtypes=qtypes)
    targets = np.concatenate([np.eye(k, dtype=np.float32)[r.integers(0, k)] for k in options])
    params = {}
    for name, shape in _shapes(case["layers"]).items():
        if name == "temperature" or (len(shape) == 1 and name.endswith("weight")):
            params[name] = torch.ones(shape, device="cuda")
        else:
            params[name] = 0.02 * _normal(g, *shape)
    return {"batch": batch, "targets": targets, "params": params, "seed": int(seed) * 31 + 7}


def _shapes(layers):
    """The checkpoint's tensors, in its order, of a ModernBERT-base decision model with this many layers."""
    d, inter, s = 768, 1152, {}
    s["encoder.embeddings.tok_embeddings.weight"] = (VOCAB, d)
    s["encoder.embeddings.norm.weight"] = (d,)
    for i in range(layers):
        p = f"encoder.layers.{i}."
        if i:
            s[p + "attn_norm.weight"] = (d,)
        s[p + "attn.Wqkv.weight"] = (3 * d, d)
        s[p + "attn.Wo.weight"] = (d, d)
        s[p + "mlp_norm.weight"] = (d,)
        s[p + "mlp.Wi.weight"] = (2 * inter, d)
        s[p + "mlp.Wo.weight"] = (d, inter)
    s["encoder.final_norm.weight"] = (d,)
    for i in range(2):
        p = f"head.layers.{i}."
        for name, out, fan_in in (("self_attn.in_proj_", 3 * d, d), ("self_attn.out_proj.", d, d),
                                  ("linear1.", 4 * d, d), ("linear2.", d, 4 * d)):
            s[p + name + "weight"], s[p + name + "bias"] = (out, fan_in), (out,)
        for name in ("norm1.", "norm2."):
            s[p + name + "weight"], s[p + name + "bias"] = (d,), (d,)
    s["type_emb.weight"] = (3, d)
    for name, shape in (("scorer.0.", (d,)), ("scorer.1.", (d, d)), ("scorer.3.", (1, d)), ("act_head.0.", (256, d + 4)),
                        ("act_head.2.", (2, 256))):
        s[name + "weight"], s[name + "bias"] = shape, (shape[0],)
    s["temperature"] = (3,)
    return s


# ------------------------------------------------------------------------------- prepare and run

def prepare(case, seed):
    state = globals()["_prepare_" + case["kind"]](case, _inputs(case, seed))
    torch.cuda.synchronize()
    return state


def run(state):
    return state["run"](state)


def _prepare_linear(case, v):
    ctx = _context(case["precision"])
    y = _new(ctx, case["rows"], case["out"])
    return {"run": _run_linear, "W": _parameter(ctx, "weight", v["W"]),
            "b": _parameter(ctx, "bias", v["b"]) if case["bias"] else None, "x": _put(ctx, v["x"]),
            "rows": case["rows"], "y": y, "out": [_tensor(y)]}


def _run_linear(s):
    ops.linear(s["W"], s["b"], s["x"], s["rows"], s["y"])
    return s["out"]


def _prepare_linear_backward(case, v):
    ctx = _context(case["precision"])
    s = _prepare_linear(case, v)
    dx = _new(ctx, case["rows"], case["in"])
    out = {"dx": _tensor(dx), "dW": _tensor(s["W"].gradient_buffer())}
    if case["bias"]:
        out["db"] = _tensor(s["b"].gradient_buffer())
    del s["y"]
    ctx.sync()
    return {**s, "run": _run_linear_backward, "dy": _put(ctx, v["dy"]), "dx": dx, "out": out}


def _run_linear_backward(s):  # dW and db accumulate from pass to pass, as over micro-batches
    ops.linear_backward(s["W"], s["b"], s["x"], s["dy"], s["rows"], s["dx"])
    return s["out"]


def _prepare_attention(case, v):
    ctx = _context()
    t, d = v["qkv"].shape[0], 64 * case["heads"]
    rotary = ops.Rotary(ctx, 64, case["theta"], case["longest"]) if case["theta"] else None
    shape = ops.AttentionShape(d, case["heads"], ops.default_scale(64), case["half_window"], rotary, case["dropout"],
                               v["seed"])
    s = {"run": _run_attention, "segments": ops.Segments(ctx, v["lengths"]), "shape": shape,
         "qkv": _put(ctx, v["qkv"]), "dcontext": _put(ctx, v["dcontext"]), "context": _new(ctx, t, d),
         "lse": _new(ctx, t * case["heads"]), "dqkv": _new(ctx, t, 3 * d)}
    s["out"] = {k: _tensor(s[k]) for k in ("context", "lse", "dqkv")}
    return s


def _run_attention(s):
    ops.attention_forward(s["qkv"], s["segments"], s["shape"], s["context"], s["lse"])
    ops.attention_backward(s["qkv"], s["segments"], s["shape"], s["dcontext"], s["dqkv"], s["context"], s["lse"])
    return s["out"]


def _prepare_mlp(case, v):
    ctx = _context()
    m, d, i = case["rows"], case["hidden"], case["inter"]
    s = {"run": _run_mlp, "ctx": ctx, "rows": m, "hidden": d, "inter": i}
    for k in ("gamma", "Wi", "Wo"):
        s[k] = _parameter(ctx, k, v[k])
        s["d" + k] = _tensor(s[k].gradient_buffer())
    s["x"], s["dout"], s["dx"] = _put(ctx, v["x"]), _put(ctx, v["dout"]), _put(ctx, v["dout"])
    for k, shape in (("normed", (m, d)), ("mean", (m,)), ("rstd", (m,)), ("wide", (m, 2 * i)), ("act", (m, i)),
                     ("y", (m, d)), ("dact", (m, i)), ("dwide", (m, 2 * i)), ("dnormed", (m, d))):
        s[k] = _new(ctx, *shape)
    for k in ("normed", "act", "dwide"):
        s[k + " words"] = ops.magnitude_words(ctx)
    s["out"] = {"y": _tensor(s["y"]), "dx": _tensor(s["dx"]), "dgamma": s.pop("dgamma"), "dWi": s.pop("dWi"),
                "dWo": s.pop("dWo")}
    ctx.sync()
    return s


def _run_mlp(s):
    ctx, m, d, i = s["ctx"], s["rows"], s["hidden"], s["inter"]
    ops.layer_norm(s["x"], m, d, s["gamma"], None, 1e-5, s["normed"], s["mean"], s["rstd"], y_words=s["normed words"])
    ops.linear(s["Wi"], None, s["normed"], m, s["wide"], x_words=s["normed words"])
    ops.geglu(ctx, s["wide"], m, i, s["act"], act_words=s["act words"])
    ops.linear(s["Wo"], None, s["act"], m, s["y"], residual=s["x"], x_words=s["act words"])
    ops.linear_backward(s["Wo"], None, s["act"], s["dout"], m, s["dact"], x_words=s["act words"])
    ops.geglu_backward(ctx, s["wide"], s["dact"], m, i, s["dwide"], dwide_words=s["dwide words"])
    ops.linear_backward(s["Wi"], None, s["normed"], s["dwide"], m, s["dnormed"], x_words=s["normed words"],
                        dy_words=s["dwide words"])
    ops.layer_norm_backward(s["x"], m, d, s["gamma"], None, 1e-5, s["dnormed"], s["dx"], s["mean"], s["rstd"])
    return s["out"]


def _prepare_norm(case, v):
    ctx = _context()
    m, n = case["rows"], case["n"]
    s = {"run": _run_norm, "rows": m, "n": n, "gamma": _parameter(ctx, "gamma", v["gamma"]),
         "beta": _parameter(ctx, "beta", v["beta"]), "x": _put(ctx, v["x"]), "dy": _put(ctx, v["dy"]),
         "dx": _put(ctx, v["dx"]), "y": _new(ctx, m, n), "mean": _new(ctx, m), "rstd": _new(ctx, m)}
    s["out"] = {"y": _tensor(s["y"]), "dx": _tensor(s["dx"]), "dgamma": _tensor(s["gamma"].gradient_buffer()),
                "dbeta": _tensor(s["beta"].gradient_buffer())}
    ctx.sync()
    return s


def _run_norm(s):
    ops.layer_norm(s["x"], s["rows"], s["n"], s["gamma"], s["beta"], 1e-5, s["y"], s["mean"], s["rstd"])
    ops.layer_norm_backward(s["x"], s["rows"], s["n"], s["gamma"], s["beta"], 1e-5, s["dy"], s["dx"], s["mean"],
                            s["rstd"])
    return s["out"]


def _prepare_decide(case, v):
    model = TrainableDecisionModel(modernbert_base(case["layers"]), _context())
    model.set_params({k: t.cpu().numpy() for k, t in v["params"].items()})
    return {"run": _run_decide, "model": model, "batch": v["batch"]}


def _run_decide(s):
    return [list(item) for item in s["model"].decide(s["batch"])]


def _prepare_train(case, v):
    ctx = _context()
    model = OpLevelModel(modernbert_base(case["layers"]), {k: t.cpu().numpy() for k, t in v["params"].items()}, ctx)
    batch = OpBatch(ctx, v["batch"], v["targets"], VOCAB)
    ctx.sync()
    logits = model.s.get("logits", (batch.n_markers,))
    return {"run": _run_train, "model": model, "batch": batch, "seed": v["seed"],
            "out": {"logits": torch.as_tensor(_Window(model, logits.ptr, logits.shape), device="cuda"),
                    "weights": _tensor(model.arena["P"]), "moment": _tensor(model.arena["M1"])}}


def _run_train(s):
    s["model"].train_step(s["batch"], seed=s["seed"], loss_scale=float(s["batch"].n_items))
    return s["out"]


# ------------------------------------------------------------------------------ work and tolerance

def _pairs(lengths, half_window):
    """Query-key pairs inside the window, over all segments."""
    total = 0
    for n in (int(x) for x in lengths):
        w = n if half_window < 0 else half_window
        total += sum(min(n - 1, q + w) - max(0, q - w) + 1 for q in range(n)) if w < n else n * n
    return total


def work(case):
    kind = case["kind"]
    if kind in ("linear", "linear_backward"):
        m, k, n = case["rows"], case["in"], case["out"]
        if kind == "linear":
            return {"bytes": 4 * (m * k + n * k + m * n), "flops": 2 * m * k * n}
        return {"bytes": 4 * (2 * m * k + m * n + 3 * n * k), "flops": 4 * m * k * n}
    if kind == "attention":
        mean = (case["longest"] + case["shortest"]) // 2
        t, d = case["segments"] * mean, 64 * case["heads"]
        # forward: qkv in, context out; backward: qkv, context, dcontext in, dqkv out
        return {"bytes": 4 * t * d * 12, "flops": 14 * d * _pairs([mean] * case["segments"], case["half_window"])}
    if kind == "mlp":
        m, d, i = case["rows"], case["hidden"], case["inter"]
        return {"bytes": 4 * (5 * m * d + 4 * 3 * d * i), "flops": 18 * m * d * i}
    if kind == "norm":
        return {"bytes": 4 * case["rows"] * case["n"] * 6, "flops": 20 * case["rows"] * case["n"]}
    mean = (case["longest"] + case["shortest"]) // 2
    t, layers = case["items"] * mean, case["layers"]
    matrices = layers * 768 * (4 * 768 + 3 * 1152) + 2 * 768 * 768 * 12
    pairs = case["items"] * 768 * (sum(_pairs([mean], -1 if i % 3 == 0 else 64) for i in range(layers))
                                   + 2 * mean * mean)
    if kind == "decide":
        return {"bytes": 4 * (matrices + t * 768), "flops": 2 * t * matrices + 4 * pairs}
    parameters = matrices + VOCAB * 768
    return {"bytes": 4 * 7 * parameters, "flops": 6 * t * matrices + 14 * pairs}


def tolerance(case):
    """About four times what each path was measured to differ from its 64-bit result by (3e-7 to 1.4e-6 for sums in
    32 bits). bf16 operands are rounded before the product, alike in every implementation, so only the sums differ."""
    kind = case["kind"]
    if kind == "train":
        # A ReLU input within rounding of zero may fall on its other side, and Adam's first steps take the sign of
        # gradients near zero.
        return {"rel": 2e-4, "max": 0.05}
    return {"rel": {"linear": 2e-6, "linear_backward": 2e-6, "norm": 1e-6, "mlp": 4e-6, "attention": 6e-6,
                    "decide": 4e-6}[kind], "max": 4e-4}


# ------------------------------------------------------------------------------------- in 64 bits

def exact(case, seed):
    with torch.no_grad():
        return globals()["_exact_" + case["kind"]](case, _inputs(case, seed))


def _rounded(t, case):
    return t.to(torch.bfloat16).double() if case["precision"] == "bf16" else t.double()


def _exact_linear(case, v):
    y = _rounded(v["x"], case) @ _rounded(v["W"], case).T
    return [y if v["b"] is None else y + v["b"].double()]


def _exact_linear_backward(case, v):
    dy = _rounded(v["dy"], case)
    out = {"dx": dy @ _rounded(v["W"], case), "dW": dy.T @ _rounded(v["x"], case)}
    if v["b"] is not None:
        out["db"] = v["dy"].double().sum(0)
    return out


def _shift(z, n):
    """Logical right shift of a 64-bit pattern held in int64."""
    return (z >> n) & ((1 << (64 - n)) - 1)


def _signed(v):
    v &= (1 << 64) - 1
    return v - (1 << 64) if v >> 63 else v


def _keep(index, p, seed):
    """Inverted dropout's factors at the counter generator's indices."""
    z = _signed(seed) + (index + 1) * _signed(0x9E3779B97F4A7C15)
    z = (z ^ _shift(z, 30)) * _signed(0xBF58476D1CE4E5B9)
    z = (z ^ _shift(z, 27)) * _signed(0x94D049BB133111EB)
    u = _shift(z ^ _shift(z, 31), 40).float() / float(1 << 24)
    p = float(np.float32(p))
    return torch.where(u < p, 0.0, 1.0 / (1.0 - p)).double()


def _turn(t, theta, back=False):
    if not theta:
        return t
    n, half = t.shape[0], t.shape[1] // 2
    i = torch.arange(half, dtype=torch.float64, device=t.device)
    angle = torch.arange(n, dtype=torch.float64, device=t.device)[:, None] * theta ** (-2.0 * i / (2 * half))
    c, s = torch.cos(angle), torch.sin(angle) * (-1 if back else 1)
    a, b = t[:, :half], t[:, half:]
    return torch.cat([a * c - b * s, b * c + a * s], 1)


def _probabilities(q, k, row, head, half_window, p, seed):
    """Softmax of one head's scaled scores, its base-2 log-sum-exp and the dropout factors (None without)."""
    n = q.shape[0]
    scores = (q @ k.T) * 0.125
    at = torch.arange(n, device=q.device)
    if 0 <= half_window < n:
        scores.masked_fill_((at[:, None] - at[None, :]).abs() > half_window, float("-inf"))
    keep = _keep((head << 42) | ((at[:, None] + row) << 21) | at[None, :], p, seed) if p else None
    return torch.softmax(scores, 1), torch.logsumexp(scores, 1) / math.log(2.0), keep


def _exact_attention(case, v):
    heads, theta = case["heads"], case["theta"]
    d = 64 * heads
    qkv, do = v["qkv"], v["dcontext"]
    context = torch.zeros(qkv.shape[0], d, dtype=torch.float64, device="cuda")
    lse = torch.zeros(qkv.shape[0], heads, dtype=torch.float64, device="cuda")
    dqkv = torch.zeros(qkv.shape, dtype=torch.float64, device="cuda")
    row = 0
    for n in (int(x) for x in v["lengths"]):
        rows = slice(row, row + n)
        for h in range(heads):
            at = [slice(j * d + 64 * h, j * d + 64 * h + 64) for j in range(3)]
            q, k, w = (qkv[rows, a].double() for a in at)
            q, k = _turn(q, theta), _turn(k, theta)
            p, lse[rows, h], keep = _probabilities(q, k, row, h, case["half_window"], case["dropout"], v["seed"])
            g = do[rows, at[0]].double()
            kept = p if keep is None else p * keep
            o = kept @ w
            context[rows, at[0]] = o
            dqkv[rows, at[2]] = kept.T @ g
            dp = g @ w.T
            if keep is not None:
                dp *= keep
            ds = p * (dp - (g * o).sum(1, keepdim=True)) * 0.125
            dqkv[rows, at[0]] = _turn(ds @ k, theta, back=True)
            dqkv[rows, at[1]] = _turn(ds.T @ q, theta, back=True)
        row += n
    return {"context": context, "lse": lse.reshape(-1), "dqkv": dqkv}


def _gelu(x):
    return 0.5 * x * (1 + torch.erf(x / math.sqrt(2.0)))


def _norm_of(x, gamma, beta=None, eps=1e-5):
    return torch.nn.functional.layer_norm(x, (x.shape[-1],), gamma, beta, eps)


def _exact_mlp(case, v):
    i = case["inter"]
    x, gamma, wi, wo = (v[k].double().requires_grad_() for k in ("x", "gamma", "Wi", "Wo"))
    with torch.enable_grad():
        wide = _norm_of(x, gamma) @ wi.T
        y = x + (_gelu(wide[:, :i]) * wide[:, i:]) @ wo.T
    dx, dgamma, dwi, dwo = torch.autograd.grad(y, [x, gamma, wi, wo], v["dout"].double())
    return {"y": y.detach(), "dx": dx, "dgamma": dgamma, "dWi": dwi, "dWo": dwo}


def _exact_norm(case, v):
    x, gamma, beta = (v[k].double().requires_grad_() for k in ("x", "gamma", "beta"))
    with torch.enable_grad():
        y = _norm_of(x, gamma, beta)
    dx, dgamma, dbeta = torch.autograd.grad(y, [x, gamma, beta], v["dy"].double())
    return {"y": y.detach(), "dx": v["dx"].double() + dx, "dgamma": dgamma, "dbeta": dbeta}


def _mix(seed, salt):
    m = (1 << 64) - 1
    z = (seed ^ ((salt * 0xD1B54A32D192ED03 + 0x8CB92BA72F3D8DD7) & m)) & m
    z = ((z ^ (z >> 33)) * 0xFF51AFD7ED558CCD) & m
    return z ^ (z >> 33)


def _attend(qkv, lengths, theta, half_window, p, seed):
    d = qkv.shape[1] // 3
    rows, row = [], 0
    for n in (int(x) for x in lengths):
        out = []
        for h in range(d // 64):
            q, k, w = (qkv[row:row + n, j * d + 64 * h:j * d + 64 * h + 64] for j in range(3))
            pr, _, keep = _probabilities(_turn(q, theta), _turn(k, theta), row, h, half_window, p, seed)
            out.append((pr if keep is None else pr * keep) @ w)
        rows.append(torch.cat(out, 1))
        row += n
    return torch.cat(rows, 0)


def _model(case, v, P, p):
    """The decision model's option logits and the head's output rows, in plain torch."""
    b, seed = v["batch"], v["seed"]
    x = _norm_of(P["encoder.embeddings.tok_embeddings.weight"][torch.from_numpy(b.tokens).long().cuda()],
                 P["encoder.embeddings.norm.weight"])
    for i in range(case["layers"]):
        w = {k: P.get(f"encoder.layers.{i}.{k}.weight") for k in ("attn_norm", "attn.Wqkv", "attn.Wo", "mlp_norm",
                                                                 "mlp.Wi", "mlp.Wo")}
        qkv = (x if i == 0 else _norm_of(x, w["attn_norm"])) @ w["attn.Wqkv"].T
        x = x + _attend(qkv, b.lengths, *((160000.0, -1) if i % 3 == 0 else (10000.0, 64)), 0.0, 0) @ w["attn.Wo"].T
        wide = _norm_of(x, w["mlp_norm"]) @ w["mlp.Wi"].T
        x = x + (_gelu(wide[:, :1152]) * wide[:, 1152:]) @ w["mlp.Wo"].T
    x = _norm_of(x, P["encoder.final_norm.weight"])
    x = x + P["type_emb.weight"][torch.from_numpy(np.repeat(b.qtypes, b.lengths)).long().cuda()]

    def drop(t, layer, site):
        if not p:
            return t
        index = torch.arange(t.numel(), device="cuda").reshape(t.shape)
        return t * _keep(index, p, _mix(seed, layer * 16 + site + 1))

    for i in range(2):
        def lin(name, t):
            return t @ P[f"head.layers.{i}.{name}weight"].T + P[f"head.layers.{i}.{name}bias"]

        def norm(name, t):
            return _norm_of(t, P[f"head.layers.{i}.{name}.weight"], P[f"head.layers.{i}.{name}.bias"])

        att = _attend(lin("self_attn.in_proj_", norm("norm1", x)), b.lengths, 0.0, -1, p, _mix(seed, i * 16 + 1))
        x = x + drop(lin("self_attn.out_proj.", att), i, 1)
        x = x + drop(lin("linear2.", drop(torch.relu(lin("linear1.", norm("norm2", x))), i, 2)), i, 3)
    m = _norm_of(x[torch.from_numpy(b.marker_rows()).long().cuda()], P["scorer.0.weight"], P["scorer.0.bias"])
    m = _gelu(m @ P["scorer.1.weight"].T + P["scorer.1.bias"])
    return (m @ P["scorer.3.weight"].T + P["scorer.3.bias"])[:, 0], x


def _exact_decide(case, v):
    P = {k: t.double() for k, t in v["params"].items()}
    logits, x = _model(case, v, P, 0.0)
    out, at, row = [], 0, 0
    for n, k in zip(v["batch"].lengths, v["batch"].n_options):
        mine = logits[at:at + int(k)]
        pr = torch.softmax(mine, 0)
        top = torch.sort(pr, descending=True)[0]
        entropy = -(pr * torch.log(torch.clamp(pr, min=1e-9))).sum() / math.log(max(2, int(k)))
        extra = torch.stack([top[0], top[0] - top[1], entropy, torch.tensor(max(2, int(k)) / 255.0, device="cuda").double()])
        h = _gelu(P["act_head.0.weight"] @ torch.cat([x[row], extra]) + P["act_head.0.bias"])
        out.append([mine, torch.softmax(P["act_head.2.weight"] @ h + P["act_head.2.bias"], 0)])
        at, row = at + int(k), row + int(n)
    return out


def _exact_train(case, v):
    P = {k: t.double().requires_grad_() for k, t in v["params"].items()}
    b = v["batch"]
    targets = torch.from_numpy(v["targets"]).double().cuda()
    with torch.enable_grad():
        logits, _ = _model(case, v, P, 0.1)
        loss, at = 0.0, 0
        for k in (int(x) for x in b.n_options):  # summed over the items
            loss = loss - (targets[at:at + k] * torch.log_softmax(logits[at:at + k], 0)).sum()
            at += k
    names = list(P)
    grads = torch.autograd.grad(loss, [P[k] for k in names], allow_unused=True)
    grads = [torch.zeros_like(P[k]) if g is None else g for k, g in zip(names, grads)]
    norm = math.sqrt(sum(float(g.square().sum()) for g in grads))
    clip = min(1.0, 1.0 / (norm + 1e-6))
    weights, moment = [], []
    for k, g in zip(names, grads):  # the arenas hold every tensor from a multiple of 64 floats on
        g, w = g.reshape(-1) * clip, P[k].detach().reshape(-1)
        pad = torch.zeros(-g.numel() % 64, dtype=torch.float64, device="cuda")
        if k != "temperature":
            w = w * (1 - 3e-5 * 0.01) - 3e-5 * g / (g.abs() + 1e-8)  # the first step: m and v equal g and g squared
        weights += [w, pad]
        moment += [0.1 * g, pad]
    return {"logits": logits.detach(), "weights": torch.cat(weights), "moment": torch.cat(moment)}
