"""The work that a program using this package gives it, as cases that can be timed and checked.

A case is a dict of plain values. ``prepare`` makes what such a program holds before the call (inputs, weights, a
captured graph), ``run`` is one pass through the public operators, ``work`` the bytes and operations that a pass
cannot do without, ``tolerance`` how far two correct implementations may differ, and ``exact`` the same outputs in
float64 from plain torch. Widths are those of the 8B Llama layer that the benchmark and the decode step use (hidden
4096, 32 query and 8 key/value heads of 128, intermediate 14336) or generic ones around them.

A pass over decode weights goes through several layers' weights, as a decode step does, so that they come from HBM.
"""

from __future__ import annotations

import math

import torch

import fused_decode as fd
from fused_decode.rowsq import (linear_fp8_sumsq, linear_sumsq, post_attn_mlp_fp8_sumsq, post_attn_mlp_sumsq,
                                pre_attn_qkv_fp8_sumsq, pre_attn_qkv_sumsq, sumsq_buffer)

EPS = 1e-5
DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16, "fp32": torch.float32}
HEAD = 128


def listed():
    return [
        # One token's residual add and norm: the smallest call of a decode loop, latency and launch.
        {"name": "token_norm", "op": "add_norm", "rows": 1, "n": 4096, "dtype": "fp16", "wdtype": "fp16"},
        # The same over a long prompt (or a batch of them): streaming.
        {"name": "prompt_norm", "op": "add_norm", "rows": 8192, "n": 4096, "dtype": "bf16", "wdtype": "bf16"},
        # The heads of a prompt, views of its QKV buffer: a norm over each query and key head, then RoPE with
        # float32 tables, one position a token.
        {"name": "prompt_heads", "op": "heads", "rows": 2048, "q": 32, "kv": 8, "d": 128, "dtype": "fp16",
         "wdtype": "fp32"},
        # A prompt's SwiGLU on the halves of the gate/up product.
        {"name": "prompt_swiglu", "op": "swiglu", "rows": 2048, "n": 14336, "dtype": "bf16"},
        # The attention output projection with the residual, 13 sequences at a time, eight layers' weights.
        {"name": "out_proj", "op": "linear", "rows": 13, "n": 4096, "k": 4096, "layers": 8, "dtype": "fp16",
         "bias": "none", "weight": "nk"},
        # A projection whose checkpoint keeps it as [in, out], passed as its transposed view, with its bias.
        {"name": "in_out_proj", "op": "linear", "rows": 4, "n": 4096, "k": 4096, "layers": 8, "dtype": "bf16",
         "bias": "fp32", "weight": "kn"},
        # The MLP block of four layers for one token (the headline of the benchmark).
        {"name": "token_mlp", "op": "mlp", "rows": 1, "h": 4096, "i": 14336, "layers": 4, "dtype": "fp16",
         "weights": "same"},
        # The same for eight sequences, in bfloat16.
        {"name": "batch_mlp", "op": "mlp", "rows": 8, "h": 4096, "i": 14336, "layers": 4, "dtype": "bf16",
         "weights": "same"},
        # Four whole layers but for the attention, 16 sequences, captured in a graph as a serving loop does.
        {"name": "step_fp16", "op": "step", "rows": 16, "h": 4096, "i": 14336, "layers": 4, "dtype": "fp16",
         "weights": "same"},
        # The same with E4M3 weights for eight sequences.
        {"name": "step_fp8", "op": "step", "rows": 8, "h": 4096, "i": 14336, "layers": 4, "dtype": "fp16",
         "weights": "fp8"},
        # A prompt through one MLP block, an odd number of tokens.
        {"name": "prompt_mlp", "op": "mlp", "rows": 777, "h": 4096, "i": 14336, "layers": 1, "dtype": "fp16",
         "weights": "same"},
        # More sequences (or a short prompt) than the decode kernels' 16 rows through E4M3 MLP blocks.
        {"name": "batch_mlp_fp8", "op": "mlp", "rows": 120, "h": 4096, "i": 14336, "layers": 2, "dtype": "bf16",
         "weights": "fp8"},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _multiple(v, of):
    return max(of, v // of * of)


def draw(rng):
    op = rng.choice(["add_norm", "heads", "swiglu", "linear", "linear", "mlp", "mlp", "step"])
    dtype = rng.choice(["fp16", "bf16"])
    if op == "add_norm":
        n = _log(rng, 512, 8192)
        n = n | 1 if rng.random() < 0.25 else _multiple(n, 8)
        rows = _log(rng, 1, min(8192, 33_000_000 // n))
        return {"op": op, "rows": rows, "n": n, "dtype": dtype, "wdtype": rng.choice([dtype, "fp32"])}
    if op == "heads":
        kv = rng.choice([1, 2, 4, 8])
        return {"op": op, "rows": _log(rng, 1, 2048), "q": kv * rng.choice([1, 3, 4, 5]), "kv": kv,
                "d": rng.choice([64, 80, 96, 128]), "dtype": dtype, "wdtype": rng.choice([dtype, "fp32"])}
    if op == "swiglu":
        n = _log(rng, 1024, 14336)
        n = n | 1 if rng.random() < 0.25 else _multiple(n, 8)
        return {"op": op, "rows": _log(rng, 1, 2048), "n": n, "dtype": dtype}
    if op == "linear":
        k, n = _multiple(_log(rng, 1024, 14336), 8), _log(rng, 1024, 30000)
        weight = rng.choice(["nk", "nk", "kn"])
        if weight == "kn":
            n = _multiple(n, 8)
        return {"op": op, "rows": rng.randint(1, 16), "n": n, "k": k, "layers": max(1, min(8, 250_000_000 // (n * k))),
                "dtype": dtype, "bias": rng.choice(["none", dtype, "fp32"]), "weight": weight}
    weights = rng.choice(["same", "fp8"])
    h = _multiple(_log(rng, 1024, 6144), 128 if op == "step" else 64)
    i = _multiple(int(h * rng.uniform(2.5, 3.5)), 16)
    few = h > 4096  # no more than the listed cases' weights
    if op == "step":
        return {"op": op, "rows": rng.randint(1, 16), "h": h, "i": i, "layers": 2 if few else rng.randint(2, 4),
                "dtype": dtype, "weights": weights}
    rows = _log(rng, 1, 16) if rng.random() < 0.5 else _log(rng, 17, 300 if weights == "fp8" else 777)
    rows = min(rows, max(16, 777 * 4096 * 14336 // (h * i)))
    layers = 1 if rows > (16 if few else 300) else rng.randint(1, 2) if rows > 16 or few else rng.randint(2, 4)
    return {"op": op, "rows": rows, "h": h, "i": i, "layers": layers, "dtype": dtype, "weights": weights}


# ------------------------------------------------------------------ inputs


def _rnd(g, *shape, dtype, scale=1.0, mean=0.0):
    t = torch.randn(*shape, generator=g, device="cuda", dtype=torch.float32)
    return t.mul_(scale).add_(mean).to(dtype)


def _codes(w):
    """E4M3 codes [N, K] and float32 row scales [N]: max|row| at the largest code."""
    w = w.float()
    amax = w.abs().amax(dim=1)
    scale = torch.where(amax > 0, amax * (1.0 / 448.0), torch.ones_like(amax))
    return (w / scale[:, None]).clamp(-448.0, 448.0).to(torch.float8_e4m3fn), scale


def _angles(first, count, d, dtype):
    """cos/sin [count, 1, d] of positions first, first + 1, ... (theta 500000)."""
    inv = 500000.0 ** (-torch.arange(0, d, 2, dtype=torch.float64, device="cuda") / d)
    ang = torch.arange(first, first + count, dtype=torch.float64, device="cuda")[:, None] * inv[None]
    ang = torch.cat((ang, ang), 1)[:, None, :]
    return ang.cos().to(dtype), ang.sin().to(dtype)


def _step_sizes(case):
    """Query heads, key (and value) heads and QKV columns of a layer of this hidden width."""
    q = case["h"] // HEAD
    kv = max(1, q // 4)
    return q, kv, (q + 2 * kv) * HEAD


def _inputs(case, seed):
    """The tensors of a case, from the seed alone."""
    g = torch.Generator(device="cuda").manual_seed(int(seed))
    dt, m = DTYPES[case["dtype"]], case["rows"]
    op = case["op"]
    if op == "add_norm":
        n = case["n"]
        return {"x": _rnd(g, m, n, dtype=dt), "r": _rnd(g, m, n, dtype=dt),
                "w": _rnd(g, n, dtype=DTYPES[case["wdtype"]], scale=0.1, mean=1.0)}
    if op == "heads":
        q, kv, d = case["q"], case["kv"], case["d"]
        cos, sin = _angles(0, m, d, torch.float32)
        wdt = DTYPES[case["wdtype"]]
        return {"qkv": _rnd(g, m, (q + 2 * kv) * d, dtype=dt), "wq": _rnd(g, d, dtype=wdt, scale=0.1, mean=1.0),
                "wk": _rnd(g, d, dtype=wdt, scale=0.1, mean=1.0), "cos": cos, "sin": sin}
    if op == "swiglu":
        return {"gu": _rnd(g, m, 2 * case["n"], dtype=dt, scale=2.0)}
    if op == "linear":
        n, k = case["n"], case["k"]
        s = {"x": _rnd(g, m, k, dtype=dt), "r": _rnd(g, m, n, dtype=dt), "b": [], "w": []}
        for _ in range(case["layers"]):
            w = _rnd(g, n, k, dtype=dt, scale=k ** -0.5)
            s["w"].append(w.t().contiguous().t() if case["weight"] == "kn" else w)
            s["b"].append(None if case["bias"] == "none" else _rnd(g, n, dtype=DTYPES[case["bias"]]))
        return s
    h, i = case["h"], case["i"]
    keep = _codes if case["weights"] == "fp8" else (lambda w: (w,))
    s = {"x": _rnd(g, m, h, dtype=dt), "layers": []}
    for _ in range(case["layers"]):
        w = {"mlp_norm": _rnd(g, h, dtype=dt, scale=0.1, mean=1.0),
             "gate_up": keep(_rnd(g, 2 * i, h, dtype=dt, scale=h ** -0.5)),
             "down": keep(_rnd(g, h, i, dtype=dt, scale=i ** -0.5))}
        if op == "step":
            w["attn_norm"] = _rnd(g, h, dtype=dt, scale=0.1, mean=1.0)
            w["qkv"] = keep(_rnd(g, _step_sizes(case)[2], h, dtype=dt, scale=h ** -0.5))
            w["o"] = keep(_rnd(g, h, h, dtype=dt, scale=h ** -0.5))
            w["attn"] = _rnd(g, m, h, dtype=dt)  # what the attention of this layer gives
        s["layers"].append(w)
    if op == "step":
        s["cos"], s["sin"] = _angles(1024, m, HEAD, dt)
    return s


# ------------------------------------------------------------------ passes


def _step(case, s):
    """Layers minus attention: QKV with its norm and RoPE, output projection with the residual, MLP. From five rows
    each launch hands its row sums to the next norm."""
    fp8, rope_cols = case["weights"] == "fp8", (_step_sizes(case)[0] + _step_sizes(case)[1]) * HEAD
    x, outs, ss_x = s["x"], [], None
    m, h = x.shape
    handoff = m >= 5
    for w in s["layers"]:
        if ss_x is None:
            qkv_op = fd.pre_attn_qkv_fp8 if fp8 else fd.pre_attn_qkv
            qkv = qkv_op(x, w["attn_norm"], *w["qkv"], s["cos"], s["sin"], EPS, rope_cols=rope_cols)
        else:
            qkv_op = pre_attn_qkv_fp8_sumsq if fp8 else pre_attn_qkv_sumsq
            qkv = qkv_op(x, w["attn_norm"], *w["qkv"], s["cos"], s["sin"], EPS, rope_cols=rope_cols, ss_in=ss_x,
                         out=x.new_empty(m, _step_sizes(case)[2]))
        if handoff:
            hid, ss_h, ss_x = torch.empty_like(x), sumsq_buffer(h, x.device), sumsq_buffer(h, x.device)
            (linear_fp8_sumsq if fp8 else linear_sumsq)(w["attn"], *w["o"], row_add=x, out=hid, ss_out=ss_h)
            mlp = post_attn_mlp_fp8_sumsq if fp8 else post_attn_mlp_sumsq
            x = mlp(hid, w["mlp_norm"], *w["gate_up"], *w["down"], EPS, out=torch.empty_like(x), ss_in=ss_h,
                    ss_out=ss_x)
        else:
            hid = (fd.linear_decode_fp8 if fp8 else fd.linear_decode)(w["attn"], *w["o"], row_add=x)
            mlp = fd.post_attn_mlp_fp8 if fp8 else fd.post_attn_mlp
            x = mlp(hid, w["mlp_norm"], *w["gate_up"], *w["down"], EPS)
        outs += [qkv, hid, x]
    return outs


def prepare(case, seed):
    s = _inputs(case, seed)
    s["case"] = case
    if case["op"] == "step":
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            _step(case, s)
        torch.cuda.current_stream().wait_stream(side)
        torch.cuda.synchronize()
        s["graph"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(s["graph"]):
            s["outs"] = _step(case, s)
    return s


def _heads(case, s):
    q, kv, d = case["q"], case["kv"], case["d"]
    qkv = s["qkv"]
    return (qkv[:, : q * d].unflatten(-1, (q, d)), qkv[:, q * d : (q + kv) * d].unflatten(-1, (kv, d)))


def run(state):
    s, case = state, state["case"]
    op = case["op"]
    if op == "add_norm":
        return fd.add_rms_norm(s["x"], s["r"], s["w"], EPS)
    if op == "heads":
        q, k = _heads(case, s)
        q, k = fd.rms_norm(q, s["wq"], EPS), fd.rms_norm(k, s["wk"], EPS)
        return q, k, fd.rope(q, s["cos"], s["sin"]), fd.rope(k, s["cos"], s["sin"])
    if op == "swiglu":
        gate, up = s["gu"].split(case["n"], dim=-1)
        return fd.swiglu(gate, up)
    if op == "linear":
        return [fd.linear_decode(s["x"], w, b, row_add=s["r"]) for w, b in zip(s["w"], s["b"])]
    if op == "mlp":
        mlp = fd.post_attn_mlp_fp8 if case["weights"] == "fp8" else fd.post_attn_mlp
        x, outs = s["x"], []
        for w in s["layers"]:
            x = mlp(x, w["mlp_norm"], *w["gate_up"], *w["down"], EPS)
            outs.append(x)
        return outs
    s["graph"].replay()
    return s["outs"]


# ------------------------------------------------------------------ what a pass cannot do without


def work(case):
    m, op = case["rows"], case["op"]
    size = {"fp16": 2, "bf16": 2, "fp32": 4, "none": 0}
    if op == "add_norm":
        n = case["n"]
        return {"bytes": 8 * m * n + n * size[case["wdtype"]], "flops": 6 * m * n}
    if op == "heads":
        heads, d = case["q"] + case["kv"], case["d"]
        # the heads read, normed and rotated heads written (both are results); both tables
        return {"bytes": 3 * m * heads * d * 2 + 2 * m * d * 4 + 2 * d * size[case["wdtype"]],
                "flops": 8 * m * heads * d}
    if op == "swiglu":
        return {"bytes": 6 * m * case["n"], "flops": 5 * m * case["n"]}
    if op == "linear":
        n, k = case["n"], case["k"]
        per = 2 * n * k + n * size[case["bias"]] + 2 * m * n
        return {"bytes": 2 * m * (k + n) + case["layers"] * per, "flops": case["layers"] * 2 * m * n * k}
    h, i = case["h"], case["i"]
    cells, rows = 3 * h * i, 2 * i + h
    outs, more = m * h, h
    if op == "step":
        qkv = _step_sizes(case)[2]
        cells, rows = cells + qkv * h + h * h, rows + qkv + h
        outs, more = outs + m * (qkv + h), more + h + m * h  # the norm weight and the attention's output
    weights = cells + 4 * rows if case["weights"] == "fp8" else 2 * cells
    return {"bytes": case["layers"] * (weights + 2 * more + 2 * outs) + 2 * m * h,
            "flops": case["layers"] * 2 * m * cells}


def tolerance(case):
    """About four times the measured distance to ``exact``. One rounding of the result (norm, SwiGLU, a projection):
    2.1e-4 in float16, 1.8e-3 in bfloat16, 2.9e-4 and 2.3e-3 where RoPE reads a rounded norm. Blocks and layers round
    their normed rows, products and residual stream, up to four of them in a row: 7.0e-4 and 5.6e-3."""
    bf16 = case["dtype"] == "bf16"
    if case["op"] in ("mlp", "step"):
        return {"rel": 2e-2 if bf16 else 2.8e-3}
    return {"rel": 1e-2 if bf16 else 1.2e-3}


# ------------------------------------------------------------------ the same in float64


def _norm64(x, w):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * w.double()


def _rope64(x, cos, sin):
    a, b = x.chunk(2, -1)
    return x * cos.double() + torch.cat((-b, a), -1) * sin.double()


def _mul64(x, w):
    """x [M, K] against a weight (w,) or its codes and row scales (codes, scale)."""
    y = x @ w[0].double().t()
    return y * w[1].double() if len(w) == 2 else y


def exact(case, seed):
    s, op = _inputs(case, seed), case["op"]
    if op == "add_norm":
        t = s["x"].double() + s["r"].double()
        return _norm64(t, s["w"]), t
    if op == "heads":
        q, k = (_norm64(t.double(), w) for t, w in zip(_heads(case, s), (s["wq"], s["wk"])))
        return q, k, _rope64(q, s["cos"], s["sin"]), _rope64(k, s["cos"], s["sin"])
    if op == "swiglu":
        gate, up = s["gu"].double().split(case["n"], dim=-1)
        return gate * torch.sigmoid(gate) * up
    if op == "linear":
        x, r = s["x"].double(), s["r"].double()
        return [x @ w.double().t() + (0.0 if b is None else b.double()) + r for w, b in zip(s["w"], s["b"])]
    x, outs = s["x"].double(), []
    for w in s["layers"]:
        if op == "step":
            q, kv, n = _step_sizes(case)
            qkv = _mul64(_norm64(x, w["attn_norm"]), w["qkv"])
            heads = qkv[:, : (q + kv) * HEAD].unflatten(-1, (q + kv, HEAD))
            qkv = torch.cat((_rope64(heads, s["cos"], s["sin"]).flatten(1), qkv[:, (q + kv) * HEAD :]), 1)
            x = x + _mul64(w["attn"].double(), w["o"])
            outs += [qkv, x]
        gate, up = _mul64(_norm64(x, w["mlp_norm"]), w["gate_up"]).split(case["i"], dim=-1)
        x = x + _mul64(gate * torch.sigmoid(gate) * up, w["down"])
        outs.append(x)
    return outs
