"""The work a user of this library has it do on one GPU, as timed cases.

Every case is one call of the public host layer (``diskmule_amd.HipContext``)
as a decode step or a prefill makes it, with weights resident in HBM:

* ``matvec``       one projection of a decode step, 1 to 16 tokens
                   (``matvec_device``), in the GGUF types models hold;
* ``head``         the output head with the greedy argmax
                   (``matvec_argmax_device``), one token;
* ``ffn``          the dense gated FFN of a decode step (``ffn_device``);
* ``moe``          a routed-expert layer of a decode step whose experts are
                   all resident (``moe_layer``);
* ``gemm``         a projection of a prefill of more than 16 tokens
                   (``gemm_device``);
* ``attention``    decode attention over a KV ring, full or sliding
                   (``attention_cached_device``);
* ``safetensor``   a GLM safetensors projection
                   (``matvec_safetensor_device``), one token.

Encoded weights are drawn directly as blocks: uniform codes, the scale bytes
a quantizer leaves (6-bit scales and mins of Q4_K, signed 8-bit scales of
Q6_K up to their full range), super-block scales that give weights of
standard deviation about 0.02.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from diskmule_amd import ExpertCache, ExpertLayerLayout, HipContext
from diskmule_amd.hip import PinnedHostBuffer

GGML = {"F16": 1, "Q5_0": 6, "Q8_0": 8, "Q4_K": 12, "Q6_K": 14}
BLOCK = {"F16": (1, 2), "Q5_0": (32, 22), "Q8_0": (32, 34), "Q4_K": (256, 144), "Q6_K": (256, 210)}
EPSILON = 1e-6
PAD = 512  # bytes kept readable past each matrix, as the library's own buffers are padded
MOST = 2048 * 12288 * 4096  # multiply-adds of the largest prefill product

_context = None


def context() -> HipContext:
    """The program's one context on the GPU."""
    global _context
    if _context is None:
        _context = HipContext(0)
    return _context


# --------------------------------------------------------------------------
# The cases
# --------------------------------------------------------------------------
def listed():
    return [
        # one attention projection of a 4096-wide model, one token: the smallest call
        {"name": "proj_q4k_b1", "op": "matvec", "type": "Q4_K", "rows": 4096, "columns": 4096, "batch": 1},
        # the output head of a 152k vocabulary with the greedy argmax: the largest matrix of a decode step
        {"name": "head_q6k_argmax", "op": "head", "rows": 151936, "columns": 4096},
        # the dense FFN of a 4096/12288 model, one user
        {"name": "ffn_b1", "op": "ffn", "hidden": 4096, "ffn": 12288, "batch": 1},
        # the same FFN with eight sequences decoded together
        {"name": "ffn_b8", "op": "ffn", "hidden": 4096, "ffn": 12288, "batch": 8},
        # a 128-expert top-8 layer, one user
        {"name": "moe_b1", "op": "moe", "hidden": 2048, "width": 768, "experts": 128, "k": 8, "batch": 1},
        # the same layer with sixteen sequences decoded together
        {"name": "moe_b16", "op": "moe", "hidden": 2048, "width": 768, "experts": 128, "k": 8, "batch": 16},
        # the FFN's gate projection over a 512-token prompt
        {"name": "prefill_q4k_512", "op": "gemm", "type": "Q4_K", "m": 512, "n": 12288, "k": 4096},
        # its down projection over a prompt whose length fits no tile
        {"name": "prefill_q6k_333", "op": "gemm", "type": "Q6_K", "m": 333, "n": 4096, "k": 12288},
        # a long prompt: the largest product
        {"name": "prefill_q4k_2048", "op": "gemm", "type": "Q4_K", "m": 2048, "n": 12288, "k": 4096},
        # a full-attention layer deep into a long conversation
        {"name": "attn_full_32k", "op": "attention", "query_heads": 16, "kv_heads": 2, "head_dim": 512,
         "positions": 32768, "window": 0},
        # a sliding-window layer whose ring has wrapped
        {"name": "attn_sliding_1k", "op": "attention", "query_heads": 16, "kv_heads": 8, "head_dim": 256,
         "positions": 3000, "window": 1024},
        # a grouped-INT4 projection of a 6144-wide model
        {"name": "st_int4_b1", "op": "safetensor", "dtype": "I4", "rows": 12288, "columns": 6144},
    ]


def _log(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def _blocks(rng, low, high, step=256):
    return step * max(1, round(_log(rng, low, high) / step))


def draw(rng):
    op = rng.choice(["matvec", "matvec", "head", "ffn", "ffn", "moe", "moe", "gemm", "gemm", "attention",
                     "safetensor"])
    if op == "matvec":
        kind = rng.choice(["Q4_K", "Q4_K", "Q6_K", "Q8_0", "Q5_0", "F16"])
        return {"op": op, "type": kind, "rows": _log(rng, 512, 32768), "columns": _blocks(rng, 1024, 12288),
                "batch": rng.choice([1, 1, 2, 3, 4, 6, 8, 11, 16])}
    if op == "head":
        return {"op": op, "rows": _log(rng, 32000, 151936), "columns": _blocks(rng, 2048, 4096)}
    if op == "ffn":
        return {"op": op, "hidden": _blocks(rng, 1024, 5120), "ffn": _blocks(rng, 2048, 16384),
                "batch": rng.choice([1, 2, 3, 4, 5, 8, 13, 16])}
    if op == "moe":
        return {"op": op, "hidden": _blocks(rng, 1024, 4096), "width": _blocks(rng, 512, 1536),
                "experts": rng.choice([32, 60, 64, 128]), "k": rng.choice([2, 4, 6, 8]),
                "batch": rng.choice([1, 2, 4, 7, 8, 12, 16])}
    if op == "gemm":
        m, k = _log(rng, 17, 2048), _blocks(rng, 1024, 12288)
        n = min(_log(rng, 512, 12288), MOST // (m * k))
        return {"op": op, "type": rng.choice(["Q4_K", "Q4_K", "Q6_K", "Q8_0"]), "m": m, "n": n, "k": k}
    if op == "attention":
        heads = rng.choice([(16, 2, 512), (16, 8, 256), (32, 8, 128)])
        return {"op": op, "query_heads": heads[0], "kv_heads": heads[1], "head_dim": heads[2],
                "positions": _log(rng, 64, 32768), "window": rng.choice([0, 0, 1024])}
    return {"op": op, "dtype": rng.choice(["BF16", "F8_E4M3", "I8", "I4"]), "rows": _log(rng, 512, 16384),
            "columns": _blocks(rng, 1024, 8192, 128)}


# --------------------------------------------------------------------------
# Inputs
# --------------------------------------------------------------------------
def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _bytes(g, *shape):
    return torch.randint(0, 256, shape, generator=g, device="cuda", dtype=torch.uint8)


def _uniform(g, n, low, high):
    return torch.rand(n, generator=g, device="cuda") * (high - low) + low


def _half_bytes(v):
    return v.to(torch.float16).view(torch.uint8).reshape(-1, 2)


def _normal(g, *shape):
    return torch.randn(shape, generator=g, device="cuda")


def _encoded(g, kind, rows, columns):
    """`rows` encoded rows of `columns` values (a flat byte tensor, PAD readable bytes after it)."""
    elements, size = BLOCK[kind]
    n = rows * (columns // elements)
    out = torch.zeros(n * size + PAD, dtype=torch.uint8, device="cuda")
    b = out[: n * size].view(n, size)
    if kind == "F16":
        b.copy_(_half_bytes(_normal(g, n) * 0.02))
        return out
    step = 1 << 21  # blocks drawn at a time
    for lo in range(0, n, step):
        c = b[lo:lo + step]
        c.copy_(_bytes(g, *c.shape))
        m = c.shape[0]
        if kind == "Q4_K":  # 16 six-bit scales and mins in 12 bytes: the packing covers every bit pattern
            d = _uniform(g, m, 0.8, 1.2) * 1.1e-4
            c[:, 0:2] = _half_bytes(d)
            c[:, 2:4] = _half_bytes(d * 7.5)
        elif kind == "Q6_K":
            c[:, 208:210] = _half_bytes(_uniform(g, m, 0.8, 1.2) * 1.4e-5)
        elif kind == "Q8_0":
            c[:, 0:2] = _half_bytes(_uniform(g, m, 0.8, 1.2) * 2.7e-4)
        else:
            c[:, 0:2] = _half_bytes(_uniform(g, m, 0.8, 1.2) * 2.2e-3)
    return out


def _length(kind, rows, columns):
    elements, size = BLOCK[kind]
    return rows * (columns // elements) * size


def _router(g, experts, hidden):
    return (_normal(g, experts, hidden) * 0.02).to(torch.bfloat16)


def _safetensor(g, case):
    """(encoded bytes, scales or None)"""
    rows, columns, dtype = case["rows"], case["columns"], case["dtype"]
    if dtype == "BF16":
        w = (_normal(g, rows * columns) * 0.02).to(torch.bfloat16).view(torch.uint8)
        return torch.cat([w, w.new_zeros(PAD)]), None
    if dtype == "F8_E4M3":
        w = _bytes(g, rows * columns)
        w = torch.where((w & 0x7F) == 0x7F, w & 0x80, w)  # no NaN codes in a checkpoint
        scales = _uniform(g, -(-rows // 128) * -(-columns // 128), 1e-4, 3e-4)
    elif dtype == "I8":
        w = _bytes(g, rows * columns)
        scales = _uniform(g, rows, 1e-4, 4e-4)
    else:
        w = _bytes(g, rows * columns // 2)
        scales = _uniform(g, rows * (columns // 32), 2e-3, 6e-3)
    return torch.cat([w, w.new_zeros(PAD)]), scales


def _inputs(case, seed):
    """Every tensor the case reads, from the seed alone."""
    g, op = _generator(seed), case["op"]
    if op in ("matvec", "head"):
        kind, batch = case.get("type", "Q6_K"), case.get("batch", 1)
        return {"x": _normal(g, batch, case["columns"]), "w": _encoded(g, kind, case["rows"], case["columns"])}
    if op == "ffn":
        hidden, ffn = case["hidden"], case["ffn"]
        return {"x": _normal(g, case["batch"], hidden), "gate": _encoded(g, "Q4_K", ffn, hidden),
                "up": _encoded(g, "Q4_K", ffn, hidden), "down": _encoded(g, "Q6_K", hidden, ffn)}
    if op == "moe":
        experts, hidden, width = case["experts"], case["hidden"], case["width"]
        return {"x": _normal(g, case["batch"], hidden), "router": _router(g, experts, hidden),
                "gate_up": _encoded(g, "Q4_K", experts * 2 * width, hidden),
                "down": _encoded(g, "Q6_K", experts * hidden, width)}
    if op == "gemm":
        # channels of different sizes, as activations have
        a = _normal(g, case["m"], case["k"]) * torch.exp(0.5 * _normal(g, 1, case["k"]))
        return {"a": a.to(torch.bfloat16), "w": _encoded(g, case["type"], case["n"], case["k"])}
    if op == "attention":
        width = case["kv_heads"] * case["head_dim"]
        return {"q": _normal(g, case["query_heads"], case["head_dim"]) * (2.0 / math.sqrt(case["head_dim"])),
                "keys": _normal(g, case["positions"], width), "values": _normal(g, case["positions"], width)}
    w, scales = _safetensor(g, case)
    return {"w": w, "scales": scales, "x": _normal(g, case["columns"])}


def prepare(case, seed):
    ctx, op = context(), case["op"]
    state = {"op": op, "case": dict(case), "ctx": ctx}
    t = _inputs(case, seed)
    if op == "matvec":
        t["y"] = torch.zeros(case["batch"], case["rows"], device="cuda")
    elif op == "head":
        t["y"] = torch.zeros(case["rows"], device="cuda")
        t["index"] = torch.zeros(1, dtype=torch.int32, device="cuda")
    elif op == "ffn":
        t["y"] = torch.zeros(case["batch"], case["hidden"], device="cuda")
        need = ctx.ffn_workspace_bytes(case["batch"], case["hidden"], case["ffn"])
        t["workspace"] = torch.zeros(need, dtype=torch.uint8, device="cuda")
    elif op == "moe":
        t["y"] = torch.zeros(case["batch"], case["hidden"], device="cuda")
        experts, hidden, width = case["experts"], case["hidden"], case["width"]
        gate_up, down = _length("Q4_K", 2 * width, hidden), _length("Q6_K", hidden, width)
        source = PinnedHostBuffer(experts * (gate_up + down))
        host = torch.from_numpy(source.array)
        host[: experts * gate_up].copy_(t.pop("gate_up")[: experts * gate_up])
        host[experts * gate_up:].copy_(t.pop("down")[: experts * down])
        layout = ExpertLayerLayout(experts, 0, gate_up, experts * gate_up, down)
        cache = ExpertCache(ctx, source, [layout], experts)
        for e in range(experts):  # a layer in service has loaded its experts
            cache.release(0, cache.acquire(0, e)[0])
        state["source"], state["cache"] = source, cache
    elif op == "gemm":
        t["c"] = torch.zeros(case["m"], case["n"], device="cuda")
        t["workspace"] = torch.zeros(ctx.gemm_workspace_bytes(case["m"], case["k"]), dtype=torch.uint8, device="cuda")
    elif op == "attention":
        width = case["kv_heads"] * case["head_dim"]
        layer = ctx.new_kv_layer(width, case["positions"], case["window"] or None)
        keys, values = t.pop("keys"), t.pop("values")
        torch.cuda.synchronize()
        k, v = keys.data_ptr(), values.data_ptr()
        for p in range(case["positions"]):
            ctx.append_kv_device(layer, p, k + p * width * 4, width, v + p * width * 4, width)
        ctx.synchronize()
        state["layer"] = layer
        t["out"] = torch.zeros(case["query_heads"], case["head_dim"], device="cuda")
    else:
        t["y"] = torch.zeros(case["rows"], device="cuda")
        state["w_len"] = t["w"].numel() - PAD
    torch.cuda.synchronize()
    state["t"] = t
    state["p"] = {k: v.data_ptr() for k, v in t.items() if v is not None}
    return state


def run(state):
    op, case, ctx, t, p = state["op"], state["case"], state["ctx"], state["t"], state["p"]
    if op == "matvec":
        ctx.matvec_device(GGML[case["type"]], case["rows"], case["columns"], p["w"], case["batch"], p["x"], p["y"])
        return t["y"]
    if op == "head":
        ctx.matvec_argmax_device(GGML["Q6_K"], case["rows"], case["columns"], p["w"], p["x"], p["y"], p["index"])
        return {"logits": t["y"], "index": t["index"]}
    if op == "ffn":
        ctx.ffn_device(case["batch"], case["hidden"], case["ffn"], GGML["Q4_K"], p["gate"], GGML["Q4_K"], p["up"],
                       GGML["Q6_K"], p["down"], EPSILON, p["x"], p["y"], p["workspace"], t["workspace"].numel())
        return t["y"]
    if op == "moe":
        ids, probabilities = ctx.moe_layer(state["cache"], 0, case["batch"], case["hidden"], case["width"],
                                           case["experts"], case["k"], p["router"], GGML["Q4_K"], GGML["Q6_K"],
                                           p["x"], p["y"])
        return {"ids": ids, "probabilities": probabilities, "y": t["y"]}
    if op == "gemm":
        ctx.gemm_device(GGML[case["type"]], case["m"], case["n"], case["k"], p["a"], p["w"], p["c"], p["workspace"],
                        t["workspace"].numel())
        return t["c"]
    if op == "attention":
        n = case["query_heads"] * case["head_dim"]
        ctx.attention_cached_device(p["q"], n, state["layer"], case["query_heads"], case["kv_heads"],
                                    case["head_dim"], p["out"], n)
        return t["out"]
    scales = t["scales"]
    ctx.matvec_safetensor_device("U8" if case["dtype"] in ("I8", "I4") else case["dtype"], case["rows"],
                                 case["columns"], p["w"], state["w_len"], None if scales is None else p["scales"],
                                 0 if scales is None else scales.numel(), p["x"], p["y"])
    return t["y"]


# --------------------------------------------------------------------------
# What a pass cannot do without
# --------------------------------------------------------------------------
def work(case):
    op = case["op"]
    if op in ("matvec", "head"):
        rows, columns, batch = case["rows"], case["columns"], case.get("batch", 1)
        return {"bytes": _length(case.get("type", "Q6_K"), rows, columns) + 4 * batch * (rows + columns),
                "flops": 2.0 * rows * columns * batch}
    if op == "ffn":
        hidden, ffn, batch = case["hidden"], case["ffn"], case["batch"]
        return {"bytes": 2 * _length("Q4_K", ffn, hidden) + _length("Q6_K", hidden, ffn) + 8 * batch * hidden,
                "flops": 6.0 * hidden * ffn * batch}
    if op == "moe":
        hidden, width, experts, batch, k = (case[n] for n in ("hidden", "width", "experts", "batch", "k"))
        distinct = experts * (1.0 - (1.0 - k / experts) ** batch)  # expected over tokens
        expert = _length("Q4_K", 2 * width, hidden) + _length("Q6_K", hidden, width)
        return {"bytes": 2.0 * experts * hidden + distinct * expert + 8.0 * batch * hidden,
                "flops": 2.0 * batch * hidden * (experts + 3.0 * k * width)}
    if op == "gemm":
        m, n, k = case["m"], case["n"], case["k"]
        return {"bytes": 2 * m * k + _length(case["type"], n, k) + 4 * m * n, "flops": 2.0 * m * n * k}
    if op == "attention":
        visible = min(case["positions"], case["window"] or case["positions"])
        width, query = case["kv_heads"] * case["head_dim"], case["query_heads"] * case["head_dim"]
        return {"bytes": 8 * visible * width + 8 * query, "flops": 4.0 * visible * query}
    rows, columns, dtype = case["rows"], case["columns"], case["dtype"]
    scales = {"BF16": 0, "F8_E4M3": -(-rows // 128) * -(-columns // 128), "I8": rows, "I4": rows * (columns // 32)}
    weight = {"BF16": 2, "F8_E4M3": 1, "I8": 1, "I4": 0.5}[dtype] * rows * columns
    return {"bytes": weight + 4 * scales[dtype] + 4 * (rows + columns), "flops": 2.0 * rows * columns}


def tolerance(case):
    """About four times the distance from `exact` that was measured."""
    if case["op"] == "gemm":  # 3.8e-4: weights rounded to fp16, one rounding per factor
        return {"rel": 1.5e-3, "max": 8e-3}
    if case["op"] == "attention":  # 2.4e-6: 32-bit scores of up to 512 terms inside the exponential
        return {"rel": 1e-5, "max": 1e-4}
    # 8e-7: activations of 22 bits and 32-bit sums; expert ids and the argmax are exact
    return {"rel": 4e-6, "max": 5e-5, "differ": 0.0}


# --------------------------------------------------------------------------
# The same in 64 bits
# --------------------------------------------------------------------------
def _half(b):
    return b.contiguous().view(torch.float16).to(torch.float64)


def _decode(kind, b):
    """[n, block bytes] -> [n, block values] in float64."""
    if kind == "F16":
        return _half(b)
    if kind == "Q8_0":
        return _half(b[:, 0:2]) * b[:, 2:34].contiguous().view(torch.int8).to(torch.float64)
    if kind == "Q5_0":
        bits = torch.arange(8, device=b.device, dtype=torch.uint8)
        high = ((b[:, 2:6, None] >> bits) & 1).reshape(-1, 32)
        low = torch.cat([b[:, 6:22] & 15, b[:, 6:22] >> 4], dim=1)
        return _half(b[:, 0:2]) * ((low | (high << 4)).to(torch.float64) - 16.0)
    if kind == "Q4_K":
        s = b[:, 4:16]
        scale = torch.cat([s[:, 0:4] & 63, (s[:, 8:12] & 15) | ((s[:, 0:4] >> 6) << 4)], dim=1).to(torch.float64)
        low = torch.cat([s[:, 4:8] & 63, (s[:, 8:12] >> 4) | ((s[:, 4:8] >> 6) << 4)], dim=1).to(torch.float64)
        q = b[:, 16:144].reshape(-1, 4, 32)
        q = torch.stack([q & 15, q >> 4], dim=2).reshape(-1, 8, 32).to(torch.float64)
        w = (_half(b[:, 0:2]) * scale)[:, :, None] * q - (_half(b[:, 2:4]) * low)[:, :, None]
        return w.reshape(-1, 256)
    low, high = b[:, 0:128].reshape(-1, 2, 2, 32), b[:, 128:192].reshape(-1, 2, 32)
    q = torch.stack([(low[:, :, 0] & 15) | ((high & 3) << 4), (low[:, :, 1] & 15) | (((high >> 2) & 3) << 4),
                     (low[:, :, 0] >> 4) | (((high >> 4) & 3) << 4), (low[:, :, 1] >> 4) | ((high >> 6) << 4)], dim=2)
    scale = b[:, 192:208].contiguous().view(torch.int8).to(torch.float64)
    w = (q.reshape(-1, 16, 16).to(torch.float64) - 32.0) * (_half(b[:, 208:210]) * scale)[:, :, None]
    return w.reshape(-1, 256)


def _rows(kind, w, rows, columns):
    """Decoded rows in pieces of about 2^26 values: (first row, [rows, columns] in float64)."""
    elements, size = BLOCK[kind]
    per = columns // elements
    b = w[: rows * per * size].view(rows, per * size)
    step = max(1, (1 << 26) // columns)
    for lo in range(0, rows, step):
        part = b[lo:lo + step]
        yield lo, _decode(kind, part.reshape(-1, size)).reshape(part.shape[0], columns)


def _product(kind, w, rows, columns, x):
    """x [m, columns] times the matrix's rows: [m, rows]."""
    out = torch.empty(x.shape[0], rows, dtype=torch.float64, device=x.device)
    for lo, part in _rows(kind, w, rows, columns):
        out[:, lo:lo + part.shape[0]] = x @ part.T
    return out


def _silu(v):
    return v / (1.0 + torch.exp(-v))


def exact(case, seed):
    op = case["op"]
    t = _inputs(case, seed)
    x = t["x"].to(torch.float64) if "x" in t else None
    if op == "matvec":
        return _product(case["type"], t["w"], case["rows"], case["columns"], x)
    if op == "head":
        y = _product("Q6_K", t["w"], case["rows"], case["columns"], x)[0]
        return {"logits": y, "index": None}
    if op == "ffn":
        hidden, ffn = case["hidden"], case["ffn"]
        n = x / torch.sqrt((x * x).mean(dim=1, keepdim=True) + EPSILON)
        a = _silu(_product("Q4_K", t["gate"], ffn, hidden, n)) * _product("Q4_K", t["up"], ffn, hidden, n)
        return _product("Q6_K", t["down"], hidden, ffn, a)
    if op == "moe":
        hidden, width, k = case["hidden"], case["width"], case["k"]
        logits = x @ t["router"].to(torch.float64).T
        top, ids = torch.sort(logits, dim=1, descending=True, stable=True)
        p = torch.softmax(top[:, :k], dim=1)
        gate_up, down = _length("Q4_K", 2 * width, hidden), _length("Q6_K", hidden, width)
        y = torch.zeros_like(x)
        for e in torch.unique(ids[:, :k]).tolist():
            token, slot = torch.nonzero(ids[:, :k] == e, as_tuple=True)
            gu = _product("Q4_K", t["gate_up"][e * gate_up:], 2 * width, hidden, x[token])
            a = _silu(gu[:, :width]) * gu[:, width:]
            y[token] += _product("Q6_K", t["down"][e * down:], hidden, width, a) * p[token, slot][:, None]
        return {"ids": None, "probabilities": p, "y": y}
    if op == "gemm":
        return _product(case["type"], t["w"], case["n"], case["k"], t["a"].to(torch.float64))
    if op == "attention":
        q, heads, dim = t["q"].to(torch.float64), case["kv_heads"], case["head_dim"]
        visible = min(case["positions"], case["window"] or case["positions"])
        keys = t["keys"][-visible:].to(torch.float64).view(visible, heads, dim)
        values = t["values"][-visible:].to(torch.float64).view(visible, heads, dim)
        group = case["query_heads"] // heads
        out = torch.empty_like(q)
        for h in range(heads):
            p = torch.softmax(q[h * group:(h + 1) * group] @ keys[:, h].T, dim=1)
            out[h * group:(h + 1) * group] = p @ values[:, h]
        return out
    rows, columns, dtype = case["rows"], case["columns"], case["dtype"]
    w = t["w"][:-PAD]
    if dtype == "BF16":
        m = w.view(torch.bfloat16).to(torch.float64).view(rows, columns)
    elif dtype == "F8_E4M3":
        s = t["scales"].to(torch.float64).view(-(-rows // 128), -(-columns // 128))
        s = s.repeat_interleave(128, 0)[:rows].repeat_interleave(128, 1)[:, :columns]
        m = w.view(torch.float8_e4m3fn).to(torch.float64).view(rows, columns) * s
    elif dtype == "I8":
        m = w.view(torch.int8).to(torch.float64).view(rows, columns) * t["scales"].to(torch.float64)[:, None]
    else:
        q = torch.stack([w & 15, w >> 4], dim=1).view(rows, columns).to(torch.float64) - 8.0
        m = q * t["scales"].to(torch.float64).view(rows, -1).repeat_interleave(32, 1)
    return m @ x
