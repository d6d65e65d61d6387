"""The calls whose speed this library is judged by, as a user's program makes them.

``listed()`` names them; ``draw(rng)`` gives more of the same kinds over their whole ranges;
``prepare`` makes on the GPU what a program holds before the call; ``run`` is one pass through
the public entry points; ``exact`` is the same answer in 64 bits from plain torch.

The kinds (``op``):

* ``attention``  -- ``attention`` forward and backward (training) or forward alone (prefill),
  causal or not, GQA, contiguous ``[B, H, T, D]`` or a module's transposed ``[B, T, H, D]``;
* ``rope_attention`` -- ``rope`` on q and k, then causal ``attention``, forward and backward:
  an attention layer between its projections;
* ``decode``     -- ``attention`` with one query row per head against a slice of a KV cache;
* ``linear_ce``  -- ``linear_cross_entropy`` forward and backward, 1% of the targets ignored;
* ``norm``       -- ``residual_rmsnorm`` forward and backward, or forward alone (inference);
* ``swiglu``     -- ``swiglu`` forward and backward, or forward alone;
* ``adamw``      -- ``adamw_step_multi`` over a decoder's float32 parameter list;
* ``gpt``        -- ``HipGPT.train_step``: forward, backward and update of the whole model.
"""

from __future__ import annotations

import math

import torch
import torch.nn.functional as F

import helion_amd as tritium
from helion_amd import gpt

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
ESIZE = {"bf16": 2, "fp16": 2, "fp32": 4}
ADAMW = {"lr": 3e-4, "beta1": 0.9, "beta2": 0.95, "eps": 1e-8, "weight_decay": 0.1}
THETA = 10000.0
NORM_EPS = 1e-6
IGNORE = -100


def listed():
    return [
        # one layer of a long-context training step: the large attention of the benchmark
        {"name": "attention_train_long", "op": "attention", "dtype": "bf16", "batch": 4,
         "heads": 32, "kv_heads": 32, "seq": 4096, "head_dim": 128, "causal": True,
         "module_layout": False, "backward": True},
        # the attention layer of the benchmark's GPT block, RoPE included
        {"name": "rope_attention_train", "op": "rope_attention", "dtype": "bf16", "batch": 16,
         "heads": 12, "seq": 1024, "head_dim": 64},
        # one request's prompt at inference: grouped heads, a ragged length, forward alone
        {"name": "attention_prefill_gqa", "op": "attention", "dtype": "bf16", "batch": 1,
         "heads": 32, "kv_heads": 8, "seq": 1531, "head_dim": 128, "causal": True,
         "module_layout": True, "backward": False},
        # float32 modules (what a model is unless it is cast), a small training batch
        {"name": "attention_train_fp32", "op": "attention", "dtype": "fp32", "batch": 4,
         "heads": 12, "kv_heads": 12, "seq": 1024, "head_dim": 64, "causal": True,
         "module_layout": True, "backward": True},
        # a serving step: a batch of requests against long caches
        {"name": "decode_batch", "op": "decode", "dtype": "bf16", "batch": 8, "heads": 32,
         "kv_heads": 8, "cache": 8192, "head_dim": 128},
        # the smallest call: one request, a short odd-sized cache, where latency counts
        {"name": "decode_single", "op": "decode", "dtype": "fp16", "batch": 1, "heads": 12,
         "kv_heads": 12, "cache": 517, "head_dim": 64},
        # the head of a large-vocabulary model: the largest call
        {"name": "linear_ce_large", "op": "linear_ce", "dtype": "bf16", "tokens": 8192,
         "hidden": 4096, "vocab": 128256},
        # the head of a small model on a ragged batch (packed sequences), odd vocabulary
        {"name": "linear_ce_ragged", "op": "linear_ce", "dtype": "bf16", "tokens": 4091,
         "hidden": 768, "vocab": 50257},
        # the row work of a training step at the benchmark's activations
        {"name": "norm_train", "op": "norm", "dtype": "bf16", "rows": 16384, "hidden": 4096,
         "backward": True},
        {"name": "swiglu_train", "op": "swiglu", "dtype": "bf16", "rows": 16384, "hidden": 11008,
         "backward": True},
        # one optimizer step over GPT-2 small's 148 tensors
        {"name": "adamw_gpt2", "op": "adamw", "layers": 12, "width": 768, "vocab": 50257,
         "positions": 1024},
        # the whole training step of the benchmark's GPT
        {"name": "gpt_train_step", "op": "gpt", "layers": 12, "batch": 16, "seq": 1024,
         "vocab": 50304},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _draw_attention(rng):
    backward = rng.random() < 0.6
    dtype = rng.choice(["bf16", "bf16", "fp16", "fp32"])
    d = rng.choice([64, 128])
    heads = rng.choice([8, 12, 16, 32])
    group = rng.choice([1, 1, 4]) if heads % 4 == 0 else 1
    seq = _log_int(rng, 16, 2048 if dtype == "fp32" else 8192)
    # batches up to the listed cases' number of visible pairs
    most = (1 << 26) if dtype == "fp32" else (1 << 31)
    cap = max(1, min(32, most // (heads * seq * seq), (1 << 17) // seq))
    return {"op": "attention", "dtype": dtype, "batch": _log_int(rng, 1, cap), "heads": heads,
            "kv_heads": heads // group, "seq": seq, "head_dim": d,
            "causal": rng.random() < 0.85, "module_layout": rng.random() < 0.6,
            "backward": backward}


def _draw_rope_attention(rng):
    heads = rng.choice([8, 12, 16, 32])
    seq = _log_int(rng, 64, 4096)
    cap = max(1, min(32, (1 << 29) // (heads * seq * seq)))
    return {"op": "rope_attention", "dtype": rng.choice(["bf16", "fp16"]),
            "batch": _log_int(rng, 1, cap), "heads": heads, "seq": seq,
            "head_dim": rng.choice([64, 128])}


def _draw_decode(rng):
    heads = rng.choice([8, 12, 16, 32])
    group = rng.choice([1, 2, 4, 8]) if heads % 8 == 0 else rng.choice([1, 4])
    cache = _log_int(rng, 16, 16384)
    cap = max(1, min(64, (1 << 20) // (cache * (heads // group))))
    return {"op": "decode", "dtype": rng.choice(["bf16", "fp16"]), "batch": _log_int(rng, 1, cap),
            "heads": heads, "kv_heads": heads // group, "cache": cache,
            "head_dim": rng.choice([64, 128])}


def _draw_linear_ce(rng):
    hidden = rng.choice([512, 768, 1024, 2048, 4096])
    vocab = rng.choice([32000, 50257, 50304, 128256, _log_int(rng, 4000, 128256)])
    dtype = rng.choice(["bf16", "bf16", "fp16", "fp32"])
    most = 1 << (37 if dtype == "fp32" else 41)
    tokens = min(_log_int(rng, 128, 16384), most // (hidden * vocab))
    return {"op": "linear_ce", "dtype": dtype, "tokens": tokens, "hidden": hidden, "vocab": vocab}


def _draw_rows(rng, op, widths):
    hidden = rng.choice(widths + [8 * _log_int(rng, widths[0] // 8, widths[-1] // 8)])
    rows = min(_log_int(rng, 1, 32768), (1 << 27) // hidden)
    return {"op": op, "dtype": rng.choice(["bf16", "bf16", "fp16", "fp32"]), "rows": rows,
            "hidden": hidden, "backward": rng.random() < 0.7}


def draw(rng):
    """One more case of the listed kinds, its sizes over the whole range."""
    op = rng.choice(["attention", "attention", "rope_attention", "decode", "linear_ce", "norm",
                     "swiglu", "adamw", "gpt"])
    if op == "attention":
        return _draw_attention(rng)
    if op == "rope_attention":
        return _draw_rope_attention(rng)
    if op == "decode":
        return _draw_decode(rng)
    if op == "linear_ce":
        return _draw_linear_ce(rng)
    if op == "norm":
        return _draw_rows(rng, "norm", [512, 768, 1000, 1024, 2048, 4096, 5120, 8192])
    if op == "swiglu":
        return _draw_rows(rng, "swiglu", [1024, 2048, 3072, 4096, 11008, 14336])
    if op == "adamw":
        return {"op": "adamw", "layers": rng.randint(1, 16), "width": 64 * rng.randint(2, 16),
                "vocab": _log_int(rng, 4000, 50304), "positions": rng.choice([256, 1024, 2048])}
    seq = _log_int(rng, 64, 1024)
    return {"op": "gpt", "layers": rng.randint(2, 6), "batch": _log_int(rng, 1, 8192 // seq),
            "seq": seq, "vocab": rng.choice([8192, 32000, 50304])}


# ------------------------------------------------------------------ inputs --
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _randn(g, shape, dtype=torch.float32, scale=1.0, mean=0.0):
    t = torch.randn(shape, generator=g, device="cuda", dtype=torch.float32)
    return t.mul_(scale).add_(mean).to(dtype)


def _heads(g, batch, heads, seq, dim, dtype, module_layout):
    """[B, H, T, D], contiguous or as the transposed view of a projection's [B, T, H, D]."""
    if module_layout:
        return _randn(g, (batch, seq, heads, dim), dtype).transpose(1, 2)
    return _randn(g, (batch, heads, seq, dim), dtype)


def _rope_tables(seq, dim):
    half = dim // 2
    inv = 1.0 / (THETA ** (torch.arange(half, device="cuda", dtype=torch.float64) / half))
    angle = torch.outer(torch.arange(seq, device="cuda", dtype=torch.float64), inv)
    return angle.cos().float(), angle.sin().float()


def _adamw_shapes(case):
    """A GPT-2 style decoder's tensors (fused q/k/v, biases, two norms a layer)."""
    d = case["width"]
    shapes = [(case["vocab"], d), (case["positions"], d)]
    for _ in range(case["layers"]):
        shapes += [(d,), (d,), (d, 3 * d), (3 * d,), (d, d), (d,),
                   (d,), (d,), (d, 4 * d), (4 * d,), (4 * d, d), (d,)]
    return shapes + [(d,), (d,)]


def _gpt_config(case):
    cfg = gpt.GPTConfig(vocab_size=case["vocab"], n_layers=case["layers"])
    return cfg, gpt.TrainConfig(batch=case["batch"], seq_len=case["seq"])


def _gpt_inputs(case, seed):
    """Initial float32 weights (N(0, 0.02), ones for norms) and one batch of uniform tokens."""
    cfg, _ = _gpt_config(case)
    g = _gen(seed)
    init = {name: torch.ones(shape, device="cuda") if len(shape) == 1
            else _randn(g, shape, scale=0.02) for name, shape in gpt.param_shapes(cfg)}
    tokens = torch.randint(cfg.vocab_size, (case["batch"], case["seq"] + 1), generator=g,
                           device="cuda")
    return init, tokens[:, :-1].contiguous(), tokens[:, 1:].contiguous()


def prepare(case, seed):
    op, g = case["op"], _gen(seed)
    if op == "gpt":
        cfg, tc = _gpt_config(case)
        init, tokens, targets = _gpt_inputs(case, seed)
        return {"op": op, "tokens": tokens, "targets": targets,
                "model": gpt.HipGPT(cfg, tc, init, torch.device("cuda"))}
    if op == "adamw":
        shapes = _adamw_shapes(case)
        return {"op": op, "step": 0,
                "params": [_randn(g, s, scale=0.02) for s in shapes],
                "grads": [_randn(g, s, scale=1e-2) for s in shapes],
                "m": [torch.zeros(s, device="cuda") for s in shapes],
                "v": [torch.zeros(s, device="cuda") for s in shapes]}
    dtype = DTYPES[case["dtype"]]
    if op in ("attention", "decode"):
        b, h, hkv, d = case["batch"], case["heads"], case["kv_heads"], case["head_dim"]
        if op == "decode":
            # the cache is allocated in steps of 1024 positions and filled up to `cache`
            n = case["cache"]
            room = -(-n // 1024) * 1024
            return {"op": op, "q": _randn(g, (b, h, 1, d), dtype),
                    "k": _randn(g, (b, hkv, room, d), dtype)[:, :, :n],
                    "v": _randn(g, (b, hkv, room, d), dtype)[:, :, :n]}
        t, ml = case["seq"], case["module_layout"]
        q = _heads(g, b, h, t, d, dtype, ml)
        k = _heads(g, b, hkv, t, d, dtype, ml)
        v = _heads(g, b, hkv, t, d, dtype, ml)
        state = {"op": op, "causal": case["causal"], "backward": case["backward"]}
        if case["backward"]:
            for x in (q, k, v):
                x.requires_grad_(True)
            state["do"] = _heads(g, b, h, t, d, dtype, ml)
        return {**state, "q": q, "k": k, "v": v}
    if op == "rope_attention":
        b, h, t, d = case["batch"], case["heads"], case["seq"], case["head_dim"]
        q, k, v = (_randn(g, (b * t, h, d), dtype).requires_grad_(True) for _ in range(3))
        cos, sin = _rope_tables(t, d)
        return {"op": op, "b": b, "q": q, "k": k, "v": v, "cos": cos, "sin": sin,
                "pos": torch.arange(t, device="cuda").repeat(b),
                "do": _randn(g, (b, t, h, d), dtype).transpose(1, 2)}
    if op == "linear_ce":
        n, d, vocab = case["tokens"], case["hidden"], case["vocab"]
        target = torch.randint(vocab, (n,), generator=g, device="cuda")
        drop = torch.rand(n, generator=g, device="cuda") < 0.01
        return {"op": op, "hidden": _randn(g, (n, d), dtype).requires_grad_(True),
                "weight": _randn(g, (vocab, d), dtype, 0.02).requires_grad_(True),
                "target": target.masked_fill(drop, IGNORE)}
    rows, d, back = case["rows"], case["hidden"], case["backward"]
    state = {"op": op, "backward": back,
             "x": _randn(g, (rows, d), dtype).requires_grad_(back),
             "r": _randn(g, (rows, d), dtype).requires_grad_(back)}
    if op == "norm":
        state["w"] = _randn(g, (d,), dtype, 0.02, 1.0).requires_grad_(back)
    if back:
        state["dy"] = _randn(g, (rows, d), dtype)
        state["dr"] = _randn(g, (rows, d), dtype) if op == "norm" else None
    return state


# -------------------------------------------------------------------- pass --
def _rope_attention(s):
    q, k = tritium.rope(s["q"], s["k"], s["cos"], s["sin"], position_ids=s["pos"])
    tokens, h, d = s["q"].shape
    b, t = s["b"], tokens // s["b"]
    o = tritium.attention(*(x.view(b, t, h, d).transpose(1, 2) for x in (q, k, s["v"])))
    return (o, *torch.autograd.grad(o, (s["q"], s["k"], s["v"]), s["do"]))


def run(state):
    s, op = state, state["op"]
    if op == "attention":
        o = tritium.attention(s["q"], s["k"], s["v"], is_causal=s["causal"])
        if not s["backward"]:
            return o
        return (o, *torch.autograd.grad(o, (s["q"], s["k"], s["v"]), s["do"]))
    if op == "rope_attention":
        return _rope_attention(s)
    if op == "decode":
        return tritium.attention(s["q"], s["k"], s["v"], is_causal=False)
    if op == "linear_ce":
        loss = tritium.linear_cross_entropy(s["hidden"], s["weight"], s["target"])
        return (loss, *torch.autograd.grad(loss, (s["hidden"], s["weight"])))
    if op == "norm":
        y, z = tritium.residual_rmsnorm(s["x"], s["r"], s["w"], NORM_EPS)
        if not s["backward"]:
            return y, z
        # the gradient of x and of the residual is one tensor
        dx, _, dw = torch.autograd.grad((y, z), (s["x"], s["r"], s["w"]), (s["dy"], s["dr"]))
        return y, z, dx, dw
    if op == "swiglu":
        y = tritium.swiglu(s["x"], s["r"])
        if not s["backward"]:
            return y
        return (y, *torch.autograd.grad(y, (s["x"], s["r"]), s["dy"]))
    if op == "adamw":
        s["step"] += 1
        tritium.adamw_step_multi(s["params"], s["grads"], s["m"], s["v"], step=s["step"], **ADAMW)
        # the largest matrices of each kind, with their moments
        keep = [0] + list(range(4, len(s["params"]), 6))[:6]
        return [s[k][i] for k in ("params", "m", "v") for i in keep]
    model = s["model"]
    loss = model.train_step(s["tokens"], s["targets"])
    return loss, model.master.flat, model.exp_avg, model.exp_avg_sq


# ------------------------------------------------------------- what it costs --
def _pairs(b, h, tq, tkv, causal):
    """Visible (query, key) pairs over all heads; the mask is top-left aligned."""
    if not causal:
        return b * h * tq * tkv
    return b * h * sum(min(i + 1, tkv) for i in range(tq))


def work(case):
    op = case["op"]
    if op == "gpt":
        cfg, tc = _gpt_config(case)
        tokens, n = tc.batch * tc.seq_len, gpt.n_params(cfg)
        attn = 14 * cfg.head_dim * _pairs(tc.batch, cfg.n_heads, tc.seq_len, tc.seq_len, True)
        # each weight's product forward, its two backward; the update's 7 float32 streams
        return {"bytes": 28.0 * n, "flops": 6.0 * n * tokens + cfg.n_layers * attn}
    if op == "adamw":
        return {"bytes": 28.0 * sum(math.prod(s) for s in _adamw_shapes(case)), "flops": 0}
    e = ESIZE[case["dtype"]]
    if op in ("attention", "rope_attention"):
        b, h, t, d = case["batch"], case["heads"], case["seq"], case["head_dim"]
        hkv, back = case.get("kv_heads", h), case.get("backward", True)
        pairs = _pairs(b, h, t, t, case.get("causal", True))
        qo, kv = b * h * t * d * e, b * hkv * t * d * e
        # forward: q, k, v in, o out; backward: those, o and do in, three gradients out
        return {"bytes": float(2 * qo + 2 * kv + ((4 * qo + 4 * kv) if back else 0)),
                "flops": float((14 if back else 4) * d * pairs)}
    if op == "decode":
        b, h, hkv, d, n = (case[k] for k in ("batch", "heads", "kv_heads", "head_dim", "cache"))
        return {"bytes": float(2 * b * hkv * n * d * e + 2 * b * h * d * e),
                "flops": 4.0 * b * h * n * d}
    if op == "linear_ce":
        n, d, vocab = case["tokens"], case["hidden"], case["vocab"]
        # the logits are a product of the forward; their gradient's two products follow
        return {"bytes": float(3 * (n + vocab) * d * e), "flops": 6.0 * n * vocab * d}
    x = case["rows"] * case["hidden"] * e
    if op == "norm":  # x, r in, y, z out; dy, dz, z in, dx out
        return {"bytes": float(x * (8 if case["backward"] else 4)), "flops": 0}
    return {"bytes": float(x * (8 if case["backward"] else 3)), "flops": 0}


def tolerance(case):
    """About four times the relative error measured against ``exact``: 0.8e-6 to 2.4e-6 for the
    float32 sums of attention and the cross-entropy, 0.002 to 0.004 where results are 16-bit,
    0.015 for the gradients of the whole bf16 model."""
    if case["op"] == "adamw":
        return {"rel": 1e-6, "max": 1e-4}
    if case["op"] == "gpt":
        return {"rel": 0.03, "max": 0.99}
    if case["dtype"] == "fp32":
        return {"rel": 1e-5, "max": 1e-3}
    return {"rel": 1e-2, "max": 0.4}


# -------------------------------------------------------------- 64-bit answer --
def _attention64(q, k, v, do, causal):
    """Softmax attention and its gradients in float64, head by head, 1024 queries at a time."""
    b, h, t, d = q.shape
    group, tkv, scale = h // k.shape[1], k.shape[2], d ** -0.5
    o = torch.zeros(q.shape, device=q.device, dtype=torch.float64)
    dq = torch.zeros_like(o)
    dk = torch.zeros(k.shape, device=q.device, dtype=torch.float64)
    dv = torch.zeros_like(dk)
    col = torch.arange(tkv, device=q.device)
    for i in range(b):
        for j in range(h):
            kk, vv = k[i, j // group].double(), v[i, j // group].double()
            for r in range(0, t, 1024):
                rows = slice(r, min(r + 1024, t))
                qq = q[i, j, rows].double()
                s = qq @ kk.t() * scale
                if causal:
                    row = torch.arange(rows.start, rows.stop, device=q.device)
                    s = s.masked_fill(col[None, :] > row[:, None], float("-inf"))
                p = s.softmax(-1)
                o[i, j, rows] = p @ vv
                if do is None:
                    continue
                dd = do[i, j, rows].double()
                dv[i, j // group] += p.t() @ dd
                ds = p * (dd @ vv.t() - (dd * o[i, j, rows]).sum(-1, keepdim=True)) * scale
                dq[i, j, rows] = ds @ kk
                dk[i, j // group] += ds.t() @ qq
    return o if do is None else (o, dq, dk, dv)


def _rotate64(x, cos, sin):
    a, b = x.double().chunk(2, -1)
    return torch.cat([a * cos - b * sin, b * cos + a * sin], -1)


def _linear_ce64(hidden, weight, target):
    """Loss and gradients in float64, 1024 tokens at a time."""
    h, w = hidden.detach().double(), weight.detach().double()
    valid = target != IGNORE
    count = valid.sum()
    loss = torch.zeros((), device=h.device, dtype=torch.float64)
    dh, dw = torch.zeros_like(h), torch.zeros_like(w)
    for r in range(0, h.shape[0], 1024):
        hr, tr, ok = h[r:r + 1024], target[r:r + 1024].clamp(min=0), valid[r:r + 1024]
        logits = hr @ w.t()
        lse = logits.logsumexp(-1)
        loss += ((lse - logits.gather(1, tr[:, None])[:, 0]) * ok).sum() / count
        g = (logits - lse[:, None]).exp_()
        g.scatter_add_(1, tr[:, None], torch.full_like(lse, -1.0)[:, None])
        g *= (ok / count)[:, None]
        dh[r:r + 1024] = g @ w
        dw.addmm_(g.t(), hr)
    return loss, dh, dw


def _gpt_loss64(cfg, w, tokens, targets):
    b, s = tokens.shape
    nh, hd = cfg.n_heads, cfg.head_dim
    cos, sin = (x.double().view(1, s, 1, hd // 2) for x in _rope_tables(s, hd))

    def norm(x, weight):
        return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + cfg.eps) * weight

    x = w["embed"][tokens]
    for i in range(cfg.n_layers):
        p = "blocks.%d." % i
        n = norm(x, w[p + "attn_norm"])
        q, k, v = ((n @ w[p + name].t()).view(b, s, nh, hd) for name in ("wq", "wk", "wv"))
        q, k, v = (y.transpose(1, 2).contiguous()
                   for y in (_rotate64(q, cos, sin), _rotate64(k, cos, sin), v))
        mask = torch.ones((s, s), device=x.device, dtype=torch.bool).triu(1)
        scores = (q @ k.transpose(2, 3).contiguous() * hd ** -0.5).masked_fill(mask, -math.inf)
        o = (scores.softmax(-1) @ v).transpose(1, 2).reshape(b, s, nh * hd)
        x = x + o @ w[p + "wo"].t()
        n = norm(x, w[p + "ffn_norm"])
        x = x + (F.silu(n @ w[p + "w_gate"].t()) * (n @ w[p + "w_up"].t())) @ w[p + "w_down"].t()
    logits = norm(x, w["final_norm"]).view(-1, cfg.d_model) @ w["embed"].t()
    return F.cross_entropy(logits, targets.reshape(-1))


def _adamw64(p, g, hp):
    """The first step from zero moments."""
    m, v = (1 - hp["beta1"]) * g, (1 - hp["beta2"]) * g * g
    p = p * (1 - hp["lr"] * hp["weight_decay"])
    return p - hp["lr"] * g / (g.abs() + hp["eps"]), m, v


def _gpt64(case, seed):
    cfg, tc = _gpt_config(case)
    init, tokens, targets = _gpt_inputs(case, seed)
    names = [name for name, _ in gpt.param_shapes(cfg)]
    # the forward and backward run on the weights rounded to bf16, as the model's do
    w = {n: init[n].to(torch.bfloat16).double().requires_grad_(True) for n in names}
    loss = _gpt_loss64(cfg, w, tokens, targets)
    grads = torch.autograd.grad(loss, [w[n] for n in names])
    hp = {"lr": tc.lr, "beta1": tc.beta1, "beta2": tc.beta2, "eps": tc.eps,
          "weight_decay": tc.weight_decay}
    new = [_adamw64(init[n].double(), g, hp) for n, g in zip(names, grads)]
    # the update of a weight whose gradient is near zero is a rounding's sign: the moments
    # carry the gradients, and the updated weights are compared between implementations
    return (loss, None, *(torch.cat([x[k].reshape(-1) for x in new]) for k in (1, 2)))


def exact(case, seed):
    op = case["op"]
    if op == "gpt":
        return _gpt64(case, seed)
    s = prepare(case, seed)
    if op == "adamw":
        new = [_adamw64(p.double(), g.double(), ADAMW) for p, g in zip(s["params"], s["grads"])]
        keep = [0] + list(range(4, len(new), 6))[:6]
        return [new[i][k] for k in range(3) for i in keep]
    with torch.no_grad():
        if op in ("attention", "decode"):
            return _attention64(s["q"], s["k"], s["v"], s.get("do"), s.get("causal", False))
        if op == "rope_attention":
            t, h, d = case["seq"], case["heads"], case["head_dim"]
            cos, sin = (x[s["pos"]].double()[:, None] for x in (s["cos"], s["sin"]))
            q, k, v = (x.view(s["b"], t, h, d).transpose(1, 2) for x in
                       (_rotate64(s["q"], cos, sin), _rotate64(s["k"], cos, sin), s["v"]))
            o, dq, dk, dv = _attention64(q, k, v, s["do"], True)
            dq, dk, dv = (x.transpose(1, 2).reshape(-1, h, d) for x in (dq, dk, dv))
            return o, _rotate64(dq, cos, -sin), _rotate64(dk, cos, -sin), dv
        if op == "linear_ce":
            return _linear_ce64(s["hidden"], s["weight"], s["target"])
    x, r = (s[k].detach().double().requires_grad_(case["backward"]) for k in ("x", "r"))
    if op == "norm":
        w = s["w"].detach().double().requires_grad_(case["backward"])
        z = x + r

        def norm(t):
            return t * torch.rsqrt(t.square().mean(-1, keepdim=True) + NORM_EPS) * w

        if not case["backward"]:
            return norm(z), z
        # the gradients are those at the stored sum, which is rounded to the inputs' type
        zs = z.detach().to(s["x"].dtype).double().requires_grad_(True)
        dz, dw = torch.autograd.grad(norm(zs), (zs, w), s["dy"].double())
        return norm(z), z, dz + s["dr"].double(), dw
    y = F.silu(x) * r
    if not case["backward"]:
        return y
    return (y, *torch.autograd.grad(y, (x, r), s["dy"].double()))
