"""The work that a program using torch_gcu asks of the device, as timed cases.

Each case is one call (or the few calls that belong together) through the
public entry points on tensors of the "gcu" device: torch ops and autograd,
``torch.gcu.efficient`` and the decoder layer of ``torch_gcu.utils``.  The
kinds, and the range each one stands for:

  embed_norm_rope  embedding, RMSNorm, RoPE, the append to the key cache,
                   SiLU-mul and the residual add of a token batch, from one
                   token of a decode step to a prefill of 8192
  linear           F.linear forward in 16 bits: 1 .. 64 rows are a decode
                   step of that many sequences, up to 8192 a prefill
  linear_train     F.linear with bias, forward and backward, bf16 or fp32
  int8_linear      the int8 weight-only linear, decode and prefill rows
  attention        scaled_dot_product_attention over a whole prompt (causal)
                   and of a decode step (one or a few queries on a long cache)
  logits           log_softmax forward and backward over a vocabulary, sum and
                   amax of the same rows, and a mean over rows
  layer_norm       layer_norm forward and backward
  adamw            one step of torch.optim.AdamW(fused=True)
  decoder          the whole decoder layer, returning its hidden states
"""
from __future__ import annotations

import math
import os
import sys

import torch
import torch.nn.functional as F

sys.path.insert(0, os.path.join(os.getcwd(), "torch-gcu_amd"))

import torch_gcu  # noqa: E402,F401  (registers the device)
from torch_gcu.utils import decoder_layer as dl  # noqa: E402

EPS = 1e-6
THETA = 10000.0
DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}


def listed():
    return [
        # a decode step of 8 sequences around its matmuls: the smallest calls, where
        # launches and latency count
        {"name": "embed_norm_rope_decode", "kind": "embed_norm_rope", "tokens": 8, "past": 2048,
         "hidden": 4096, "heads": 32, "head_dim": 128, "ffn": 11008, "vocab": 32000},
        # the up projection of a decode step of 8 sequences
        {"name": "linear_decode", "kind": "linear", "m": 8, "n": 11008, "k": 4096,
         "dtype": "bf16", "bias": False},
        # the down projection of a short prompt of 777 tokens
        {"name": "linear_prefill", "kind": "linear", "m": 777, "n": 4096, "k": 11008,
         "dtype": "bf16", "bias": False},
        # training: an attention projection over 8192 tokens, with its three gradients
        {"name": "linear_train_bf16", "kind": "linear_train", "m": 8192, "n": 4096, "k": 4096,
         "dtype": "bf16"},
        # training in full precision: a model of ordinary width
        {"name": "linear_train_f32", "kind": "linear_train", "m": 2000, "n": 2048, "k": 1024,
         "dtype": "f32"},
        # quantised decode of 24 sequences
        {"name": "int8_decode", "kind": "int8_linear", "m": 24, "n": 11008, "k": 4096,
         "dtype": "bf16", "bias": False},
        # a prompt of 1500 tokens with grouped-query heads
        {"name": "attention_prefill", "kind": "attention", "b": 4, "h": 32, "hk": 8, "sq": 1500,
         "sk": 1500, "d": 128, "dtype": "bf16", "causal": True, "heads_inner": True},
        # one new token of 8 sequences against caches of 4000
        {"name": "attention_decode", "kind": "attention", "b": 8, "h": 32, "hk": 8, "sq": 1,
         "sk": 4000, "d": 128, "dtype": "bf16", "causal": False, "heads_inner": True},
        # the loss head of a training step, and the reductions that logging does
        {"name": "logits", "kind": "logits", "rows": 2048, "vocab": 32000, "dtype": "bf16"},
        # a training layer norm
        {"name": "layer_norm_train", "kind": "layer_norm", "rows": 8192, "hidden": 4096,
         "dtype": "bf16"},
        # an optimizer step over two blocks of a small decoder
        {"name": "adamw", "kind": "adamw", "blocks": 2, "hidden": 1024, "ffn": 2816},
        # a whole layer over four prompts: the largest call
        {"name": "decoder_prefill", "kind": "decoder", "b": 4, "s": 2048, "hidden": 4096,
         "heads": 32, "head_dim": 128, "ffn": 11008, "vocab": 32000},
    ]


def _log(rng, lo, hi):
    """A whole number between lo and hi, spread over its logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))))))


def _width(rng, lo, hi):
    """A layer width: most are multiples of 64, some of 8, a few are odd."""
    w = _log(rng, lo, hi)
    step = rng.choice([64, 64, 64, 64, 8, 1])
    return max(step, w // step * step)


def draw(rng):
    kind = rng.choice(["embed_norm_rope", "linear", "linear", "linear_train", "int8_linear",
                       "attention", "attention", "logits", "layer_norm", "adamw", "decoder"])
    if kind == "embed_norm_rope":
        heads = rng.choice([8, 16, 32])
        return {"kind": kind, "tokens": _log(rng, 1, 8192), "past": _log(rng, 1, 8192),
                "hidden": heads * 128, "heads": heads, "head_dim": 128,
                "ffn": _width(rng, 1024, 11008), "vocab": 32000}
    if kind == "linear":
        return {"kind": kind, "m": _log(rng, 1, 8192), "n": _width(rng, 256, 11008),
                "k": _width(rng, 256, 11008), "dtype": rng.choice(["bf16", "bf16", "f16"]),
                "bias": rng.random() < 0.5}
    if kind == "linear_train":
        dtype = rng.choice(["bf16", "f32"])
        n, k = (_width(rng, 128, 4096 if dtype == "bf16" else 2048) for _ in range(2))
        most = 8192 if dtype == "bf16" else min(4096, 2000 * 2048 * 1024 // (n * k))
        return {"kind": kind, "m": _log(rng, 32, most), "n": n, "k": k, "dtype": dtype}
    if kind == "int8_linear":
        return {"kind": kind, "m": _log(rng, 1, 4096), "n": _width(rng, 1024, 11008),
                "k": _width(rng, 1024, 11008), "dtype": rng.choice(["bf16", "bf16", "f16"]),
                "bias": rng.random() < 0.5}
    if kind == "attention":
        d = rng.choice([64, 128, 128])
        hk = rng.choice([4, 8, 16, 32])
        h = hk * rng.choice([g for g in (1, 1, 2, 4, 8) if hk * g <= 32])
        common = {"kind": kind, "h": h, "hk": hk, "d": d, "dtype": rng.choice(["bf16", "bf16", "f16"]),
                  "heads_inner": rng.random() < 0.5}
        if rng.random() < 0.5:
            s = _log(rng, 16, 4096)
            return {**common, "b": max(1, min(8, rng.randint(1, 8) * 1024 // s)), "sq": s, "sk": s,
                    "causal": rng.random() < 0.8}
        return {**common, "b": _log(rng, 1, 16), "sq": rng.choice([1, 1, 1, 2, 5, 8]),
                "sk": _log(rng, 64, 16384), "causal": False}
    if kind == "logits":
        vocab = rng.choice([32000, 50257, _log(rng, 1000, 128000)])
        return {"kind": kind, "rows": max(1, min(_log(rng, 1, 4096), 100_000_000 // vocab)),
                "vocab": vocab, "dtype": rng.choice(["bf16", "bf16", "f16", "f32"])}
    if kind == "layer_norm":
        return {"kind": kind, "rows": _log(rng, 1, 8192), "hidden": _width(rng, 128, 8192),
                "dtype": rng.choice(["bf16", "f32"])}
    if kind == "adamw":
        hidden = _width(rng, 128, 2048)
        return {"kind": kind, "blocks": rng.randint(1, 2), "hidden": hidden, "ffn": hidden * 8 // 3}
    heads = rng.choice([8, 16, 32])
    s = _log(rng, 1, 2048)
    return {"kind": kind, "b": rng.randint(1, max(1, min(8, 4096 // s))), "s": s,
            "hidden": heads * 128, "heads": heads, "head_dim": 128, "ffn": heads * 344,
            "vocab": 32000}


class _Inputs:
    """Seeded tensors.  They are drawn on the GPU (quick at the sizes here) and
    reach the gcu device through host memory, as a program's inputs do."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda").manual_seed(seed)

    def normal(self, shape, std=1.0, mean=0.0, dtype=torch.bfloat16):
        t = torch.randn(shape, generator=self.g, device="cuda")
        return (t * std + mean).to(dtype)

    def uniform(self, shape, lo, hi, dtype=torch.float32):
        t = torch.rand(shape, generator=self.g, device="cuda")
        return (t * (hi - lo) + lo).to(dtype)

    def whole(self, shape, lo, hi, dtype=torch.int64):
        return torch.randint(lo, hi, shape, generator=self.g, device="cuda", dtype=dtype)


def _adamw_shapes(c):
    h, f = c["hidden"], c["ffn"]
    return ([(h, h)] * 4 + [(f, h)] * 2 + [(h, f), (h,), (h,)]) * c["blocks"]


def _layer_config(c):
    return dl.LayerConfig(vocab=c["vocab"], hidden=c["hidden"], heads=c["heads"],
                          head_dim=c["head_dim"], ffn=c["ffn"], theta=THETA, eps=EPS)


def _tensors(c, seed):
    """The case's inputs as a dict of tensors (lists for adamw) on the GPU."""
    r, kind = _Inputs(seed), c["kind"]
    dt = DTYPES[c.get("dtype", "bf16")]
    if kind == "embed_norm_rope":
        t, h, hd, d = c["tokens"], c["hidden"], c["heads"], c["head_dim"]
        pos = torch.arange(c["past"], c["past"] + t, device="cuda")
        return {"ids": r.whole((t,), 0, c["vocab"]), "table": r.normal((c["vocab"], h), 0.02),
                "w": r.normal((h,), 0.02, 1.0), "q": r.normal((t, hd, d)), "k": r.normal((t, hd, d)),
                "pos": pos, "past": r.normal((c["past"], hd, d)), "gate": r.normal((t, c["ffn"])),
                "up": r.normal((t, c["ffn"])), "res": r.normal((t, h))}
    if kind in ("linear", "linear_train"):
        t = {"x": r.normal((c["m"], c["k"]), dtype=dt), "w": r.normal((c["n"], c["k"]), 0.02, dtype=dt)}
        if kind == "linear_train" or c["bias"]:
            t["bias"] = r.normal((c["n"],), 0.02, dtype=dt)
        if kind == "linear_train":
            t["dy"] = r.normal((c["m"], c["n"]), dtype=dt)
        return t
    if kind == "int8_linear":
        t = {"x": r.normal((c["m"], c["k"]), dtype=dt),
             "w": r.whole((c["n"], c["k"]), -127, 128, torch.int8),
             "scales": r.uniform((c["n"],), 0.001, 0.01)}
        if c["bias"]:
            t["bias"] = r.normal((c["n"],), 0.02, dtype=dt)
        return t
    if kind == "attention":
        shapes = {"q": (c["b"], c["h"], c["sq"]), "k": (c["b"], c["hk"], c["sk"]),
                  "v": (c["b"], c["hk"], c["sk"])}
        if c["heads_inner"]:  # [batch, sequence, heads, d], as the projections write them
            shapes = {n: (b, s, h) for n, (b, h, s) in shapes.items()}
        return {n: r.normal(s + (c["d"],), dtype=dt) for n, s in shapes.items()}
    if kind == "logits":
        n = (c["rows"], c["vocab"])
        return {"x": r.normal(n, 4.0, dtype=dt), "dy": r.normal(n, 1e-3, dtype=dt),
                "m": r.normal((c["rows"] * 2, 4096), dtype=torch.float32)}
    if kind == "layer_norm":
        n = (c["rows"], c["hidden"])
        return {"x": r.normal(n, 2.0, 0.5, dtype=dt), "w": r.normal(n[1:], 0.02, 1.0, dtype=dt),
                "bias": r.normal(n[1:], 0.02, dtype=dt), "dy": r.normal(n, dtype=dt)}
    if kind == "adamw":
        s = _adamw_shapes(c)
        f = torch.float32
        return {"p": [r.normal(x, 0.02, dtype=f) for x in s],
                "g": [r.normal(x, 1e-3, dtype=f) for x in s],
                "m": [r.normal(x, 1e-4, dtype=f) for x in s],
                "v": [r.uniform(x, 1e-7, 1e-6) for x in s]}
    cfg = _layer_config(c)
    h, f = cfg.hidden, cfg.ffn
    w = {"embed": r.normal((cfg.vocab, h), 0.02), "attn_norm": r.normal((h,), 0.02, 1.0),
         "ffn_norm": r.normal((h,), 0.02, 1.0), "w_gate": r.normal((f, h), 0.02),
         "w_up": r.normal((f, h), 0.02), "w_down": r.normal((h, f), 0.02)}
    w.update({n: r.normal((h, h), 0.02) for n in ("wq", "wk", "wv", "wo")})
    return {"ids": r.whole((c["b"], c["s"]), 0, cfg.vocab), **w}


def _heads_first(c, t):
    """q, k, v as [batch, heads, sequence, d]."""
    return {n: t[n].transpose(1, 2) if c["heads_inner"] else t[n] for n in ("q", "k", "v")}


def prepare(case, seed):
    t = _tensors(case, seed)
    s = {n: [x.cpu().to("gcu") for x in v] if isinstance(v, list) else v.cpu().to("gcu")
         for n, v in t.items()}
    kind = case["kind"]
    if kind == "attention":
        s.update(_heads_first(case, s))
    elif kind == "linear_train":
        for n in ("x", "w", "bias"):
            s[n].requires_grad_()
    elif kind == "logits":
        s["leaf"] = s["x"].detach().requires_grad_()
    elif kind == "layer_norm":
        for n in ("x", "w", "bias"):
            s[n].requires_grad_()
    elif kind == "adamw":
        params = [torch.nn.Parameter(p) for p in s["p"]]
        opt = torch.optim.AdamW(params, lr=1e-3, betas=(0.9, 0.95), eps=1e-8, weight_decay=0.1,
                                fused=True)
        for p, g, m, v in zip(params, s["g"], s["m"], s["v"]):
            p.grad = g
            opt.state[p] = {"step": torch.tensor(10.0).to("gcu"), "exp_avg": m, "exp_avg_sq": v}
        s["params"], s["opt"] = params, opt
    elif kind == "decoder":
        ids = s.pop("ids")
        s = {"weights": s, "ids": ids, "cfg": _layer_config(case),
             "pos": dl.positions(case["b"], case["s"], "gcu")}
    s["case"] = case
    return s


def run(state):
    s, c = state, state["case"]
    kind = c["kind"]
    if kind == "embed_norm_rope":
        x = F.embedding(s["ids"], s["table"])
        h = torch.gcu.efficient.rms_norm(x, s["w"], EPS)
        q, k = torch.gcu.efficient.rope(s["q"], s["k"], s["pos"], THETA)
        cache = torch.cat((s["past"], k), 0)
        m = torch.gcu.efficient.silu_mul(s["gate"], s["up"])
        return {"h": h, "q": q, "cache": cache, "m": m, "sum": x + s["res"]}
    if kind == "linear":
        return F.linear(s["x"], s["w"], s.get("bias"))
    if kind == "linear_train":
        y = F.linear(s["x"], s["w"], s["bias"])
        dx, dw, db = torch.autograd.grad(y, (s["x"], s["w"], s["bias"]), s["dy"])
        return {"y": y.detach(), "dx": dx, "dw": dw, "db": db}
    if kind == "int8_linear":
        return torch.gcu.efficient.int8_linear(s["x"], s["w"], s["scales"], s.get("bias"))
    if kind == "attention":
        return F.scaled_dot_product_attention(s["q"], s["k"], s["v"], is_causal=c["causal"],
                                              enable_gqa=c["h"] != c["hk"])
    if kind == "logits":
        y = torch.log_softmax(s["leaf"], -1)
        (dx,) = torch.autograd.grad(y, s["leaf"], s["dy"])
        return {"y": y.detach(), "dx": dx, "sum": s["x"].sum(-1), "max": s["x"].amax(-1),
                "mean": s["m"].mean(0)}
    if kind == "layer_norm":
        y = F.layer_norm(s["x"], (c["hidden"],), s["w"], s["bias"], 1e-5)
        dx, dw, db = torch.autograd.grad(y, (s["x"], s["w"], s["bias"]), s["dy"])
        return {"y": y.detach(), "dx": dx, "dw": dw, "db": db}
    if kind == "adamw":
        s["opt"].step()
        return {"p": [p.detach() for p in s["params"]], "m": s["m"], "v": s["v"]}
    return dl.forward(s["weights"], s["ids"], s["cfg"], s["pos"])


def _size(c):
    return 4 if c.get("dtype") == "f32" else 2


def work(case):
    c, e = case, _size(case)
    kind = c["kind"]
    if kind == "embed_norm_rope":
        t, h, qk = c["tokens"], c["hidden"], c["heads"] * c["head_dim"]
        n = (8 * t + 8 * t  # ids, positions
             + 2 * (t * h + t * h + h)  # rows gathered once, normed rows written, weight
             + 2 * (2 * t * qk + t * qk)  # q, k read, rotated q written
             + 2 * (2 * c["past"] * qk + t * qk)  # the cache read and written with the new keys
             + 2 * 3 * t * c["ffn"] + 2 * 2 * t * h)
        return {"bytes": n, "flops": t * (4 * h + 6 * qk + 6 * c["ffn"] + h)}
    if kind in ("linear", "linear_train", "int8_linear"):
        m, n, k = c["m"], c["n"], c["k"]
        if kind == "int8_linear":
            return {"bytes": n * k + 4 * n + 2 * m * (k + n), "flops": 2 * m * n * k}
        if kind == "linear":
            return {"bytes": e * (m * k + n * k + m * n + (n if c["bias"] else 0)),
                    "flops": 2 * m * n * k}
        return {"bytes": e * (2 * m * k + 2 * n * k + 2 * m * n + 2 * n), "flops": 6 * m * n * k}
    if kind == "attention":
        pairs = c["sq"] * c["sk"]
        if c["causal"]:
            pairs = sum(min(i + 1, c["sk"]) for i in range(c["sq"]))
        n = 2 * c["b"] * c["d"] * (2 * c["h"] * c["sq"] + 2 * c["hk"] * c["sk"])
        return {"bytes": n, "flops": 4 * c["b"] * c["h"] * c["d"] * pairs}
    if kind == "logits":
        n = c["rows"] * c["vocab"]
        return {"bytes": e * (4 * n + 2 * c["rows"]) + 4 * 4096 * (2 * c["rows"] + 1),
                "flops": 12 * n}
    if kind == "layer_norm":
        n = c["rows"] * c["hidden"]
        return {"bytes": e * (4 * n + 4 * c["hidden"]), "flops": 16 * n}
    if kind == "adamw":
        n = sum(math.prod(s) for s in _adamw_shapes(c))
        return {"bytes": 28 * n, "flops": 14 * n}
    cfg = _layer_config(c)
    t, h, f = c["b"] * c["s"], cfg.hidden, cfg.ffn
    return {"bytes": 2 * (4 * h * h + 3 * h * f + 2 * h + 2 * t * h) + 16 * t,
            "flops": dl.flops(cfg, c["b"], c["s"])}


def tolerance(case):
    """Errors measured against 64 bits: 16-bit results 1.6e-3 to 2.3e-3 (one
    rounding, attention two), fp32 matmuls and norms up to 8e-7, AdamW 4e-8, and
    1.1e-2 for a whole layer, whose roundings travel through all its ops."""
    kind = case["kind"]
    if kind == "adamw":
        return {"rel": 5e-7, "max": 1e-5}
    if case.get("dtype") == "f32":
        return {"rel": 5e-6, "max": 1e-4}
    if kind == "decoder":
        return {"rel": 2e-2, "max": 0.2}
    return {"rel": 8e-3, "max": 4e-2}


def _rotated(x, pos):
    d = x.shape[-1]
    inv = THETA ** -(torch.arange(0, d, 2, dtype=torch.float64, device="cuda") / d)
    ang = pos.double()[:, None] * inv
    cos, sin = ang.cos()[:, None], ang.sin()[:, None]
    a, b = x[..., : d // 2], x[..., d // 2:]
    return torch.cat((a * cos - b * sin, b * cos + a * sin), -1)


def _normed(x, w):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * w


def _attended(q, k, v, causal):
    """[heads, sequence, d] attention of one sequence, a head at a time."""
    out, group = torch.empty_like(q), q.shape[0] // k.shape[0]
    keep = torch.ones(q.shape[1], k.shape[1], dtype=torch.bool, device="cuda")
    keep = keep.tril() if causal else None
    for i in range(q.shape[0]):
        s = (q[i] @ k[i // group].t().contiguous()) / math.sqrt(q.shape[-1])
        if causal:
            s.masked_fill_(~keep, -math.inf)
        out[i] = torch.softmax(s, -1) @ v[i // group]
    return out


def exact(case, seed):
    c, kind = case, case["kind"]
    t = _tensors(case, seed)
    if kind == "adamw":
        out = {"p": [], "m": [], "v": []}
        for p, g, m, v in zip(*([x.double() for x in t[n]] for n in ("p", "g", "m", "v"))):
            p, m, v = p * (1 - 1e-3 * 0.1), 0.9 * m + 0.1 * g, 0.95 * v + 0.05 * g * g
            p = p - 1e-3 / (1 - 0.9 ** 11) * m / ((v / (1 - 0.95 ** 11)).sqrt() + 1e-8)
            for n, x in zip("pmv", (p, m, v)):
                out[n].append(x)
        return out
    if kind == "attention":
        x = _heads_first(c, t)
        return torch.stack([_attended(*(x[n][b].double().contiguous() for n in ("q", "k", "v")),
                                      c["causal"]) for b in range(c["b"])])
    if kind == "decoder":
        w = {n: x.double() for n, x in t.items() if n != "ids"}
        hd, d = c["heads"], c["head_dim"]
        outs = []
        for ids in t["ids"]:
            pos = torch.arange(c["s"], device="cuda")
            x = w["embed"][ids]
            h = _normed(x, w["attn_norm"])
            q, k, v = ((h @ w[n].t()).view(-1, hd, d) for n in ("wq", "wk", "wv"))
            q, k = _rotated(q, pos), _rotated(k, pos)
            a = _attended(*(y.transpose(0, 1).contiguous() for y in (q, k, v)), True)
            x = x + a.transpose(0, 1).reshape(-1, hd * d) @ w["wo"].t()
            h = _normed(x, w["ffn_norm"])
            outs.append(x + (F.silu(h @ w["w_gate"].t()) * (h @ w["w_up"].t())) @ w["w_down"].t())
        return torch.cat(outs)
    if kind == "logits":
        y, dy = torch.log_softmax(t["x"].double(), -1), t["dy"].double()
        dx = dy - y.exp() * dy.sum(-1, keepdim=True)
        return {"y": y, "dx": dx, "sum": t["x"].double().sum(-1), "max": t["x"].double().amax(-1),
                "mean": t["m"].double().mean(0)}
    t = {n: x.double() if x.is_floating_point() else x for n, x in t.items()}
    if kind == "embed_norm_rope":
        x = t["table"][t["ids"]]
        return {"h": _normed(x, t["w"]), "q": _rotated(t["q"], t["pos"]),
                "cache": torch.cat((t["past"], _rotated(t["k"], t["pos"]))),
                "m": F.silu(t["gate"]) * t["up"], "sum": x + t["res"]}
    if kind == "layer_norm":
        x, dy = t["x"], t["dy"]
        rstd = torch.rsqrt(x.var(-1, unbiased=False, keepdim=True) + 1e-5)
        xh, g = (x - x.mean(-1, keepdim=True)) * rstd, dy * t["w"]
        dx = rstd * (g - g.mean(-1, keepdim=True) - xh * (g * xh).mean(-1, keepdim=True))
        return {"y": xh * t["w"] + t["bias"], "dx": dx, "dw": (dy * xh).sum(0), "db": dy.sum(0)}
    if kind == "int8_linear":
        y = (t["x"] @ t["w"].double().t()) * t["scales"]
        return y + t["bias"] if c["bias"] else y
    y = t["x"] @ t["w"].t()
    if "bias" in t:
        y = y + t["bias"]
    if kind == "linear":
        return y
    return {"y": y, "dx": t["dy"] @ t["w"], "dw": t["dy"].t() @ t["x"], "db": t["dy"].sum(0)}
