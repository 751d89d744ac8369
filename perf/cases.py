"""The measured workloads of this library: the calls an inference engine makes of it, per layer.

A case is one call (or the few calls of one step) through the public Python binding:

  linear     y = W x                 one projection (or the LM head)
  residual   y = W x + r             attention output / FFN down projection with its residual
  gate_up    y = silu(Wg x) * Wu x   the SwiGLU pair
  shared     three projections of one quantized activation (Q, K and V: N, N/4 and N/4 rows)
  attention  write the step's K and V rows into the paged cache, then attend over the cache

Weights are quantized rows laid out as GGUF files hold them, made here from normal values; the
activations are normal with a few large channels, as the residual stream has them.
"""
import math

import torch

import densecore_amd as dc

TYPES = {"Q4_0": dc.TYPE_Q4_0, "Q8_0": dc.TYPE_Q8_0, "Q8_0_RS": dc.TYPE_Q8_0_RS, "Q4_K": dc.TYPE_Q4_K,
         "Q5_K": dc.TYPE_Q5_K, "Q6_K": dc.TYPE_Q6_K}
ROW_BYTES = {"Q4_0": (18, 32), "Q8_0": (34, 32), "Q8_0_RS": (34, 32), "Q4_K": (144, 256), "Q5_K": (176, 256),
             "Q6_K": (210, 256)}
CACHE_TYPES = {"F32": dc.TYPE_F32, "F16": dc.TYPE_F16, "Q8_0": dc.TYPE_Q8_0}
CACHE_ROW = {"F32": 4.0, "F16": 2.0, "Q8_0": 34 / 32}  # bytes per value
MAX_FLOPS = 4 * 2048 * 9728 * 2560  # of the largest listed case
LAYERS, LAYER = 2, 1  # layers of a drawn or listed cache, and the one attended


def _linear(name, op, wtype, m, n, k, scratch="kept"):
    return {"name": name, "op": op, "type": wtype, "m": m, "n": n, "k": k, "scratch": scratch}


def _attention(name, cache, tokens, past, heads, kv_heads, head_dim):
    return {"name": name, "op": "attention", "cache": cache, "tokens": tokens, "past": past, "heads": heads,
            "kv_heads": kv_heads, "head_dim": head_dim}


def listed():
    return [
        # one token through a small model's FFN: launch latency, 3 MB of weights
        _linear("decode_small_q8_0", "linear", "Q8_0", 1, 3072, 1024),
        # one token through a 4B model's SwiGLU pair, the largest weights of its layer
        _linear("decode_gate_up_q4_k", "gate_up", "Q4_K", 1, 9728, 2560),
        # one token's logits over a 151,936-entry vocabulary
        _linear("lm_head_q6_k", "linear", "Q6_K", 1, 151936, 2560),
        # a ragged small batch (requests decoded together, or drafted tokens) in the quantize tool's default type
        _linear("batch13_residual_q4_0", "residual", "Q4_0", 13, 4096, 4096),
        # a full decode batch through a 1B model's FFN
        _linear("batch64_q4_k", "linear", "Q4_K", 64, 8192, 2048),
        # a short prompt's Q, K and V from one quantized activation
        _linear("prompt200_qkv_q5_k", "shared", "Q5_K", 200, 4096, 2560),
        # a ragged chunk of a prompt through an FFN down projection and its residual
        _linear("chunk515_down_q6_k", "residual", "Q6_K", 515, 2560, 9728),
        # long prompts: the 1B model's FFN up projection, and the 4B model's SwiGLU pair
        _linear("prompt2048_q8_0", "linear", "Q8_0", 2048, 8192, 2048),
        _linear("prompt2048_gate_up_q4_k", "gate_up", "Q4_K", 2048, 9728, 2560),
        # one token over a full 4096-token context
        _attention("attention_decode_q8_0", "Q8_0", 1, 4095, 32, 8, 128),
        # a ragged chunk of a prompt over what is cached already
        _attention("attention_chunk333_f16", "F16", 333, 2777, 32, 8, 64),
        # a whole prompt
        _attention("attention_prompt2048_q8_0", "Q8_0", 2048, 0, 32, 8, 128),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    while True:
        if rng.random() < 0.3:
            kv_heads = rng.choice([1, 2, 4, 8])
            c = {"op": "attention", "cache": rng.choice(["F32", "F16", "Q8_0"]),
                 "tokens": 1 if rng.random() < 0.4 else _log(rng, 2, 2048),
                 "past": 0 if rng.random() < 0.2 else _log(rng, 1, 8192),
                 "heads": kv_heads * rng.choice([1, 2, 3, 4, 7, 8]), "kv_heads": kv_heads,
                 "head_dim": rng.choice([64, 128, 128, 256])}
            if work(c)["flops"] <= MAX_FLOPS / 3:  # products in fp32, so a third of the largest case's
                return c
            continue
        op = rng.choice(["linear", "linear", "residual", "gate_up", "shared"])
        wtype = rng.choice(list(TYPES))
        unit = 256 if wtype in ("Q4_K", "Q5_K", "Q6_K", "Q8_0_RS") else 32 if rng.random() < 0.3 else 256
        m = 1 if rng.random() < 0.25 else _log(rng, 2, 2048)
        n = _log(rng, 256, 32768)
        if rng.random() < 0.7:
            n = (n + 63) // 64 * 64
        if op == "shared":
            n = n // 4 * 4
        k = unit * max(1, _log(rng, 512, 14336) // unit)
        c = {"op": op, "type": wtype, "m": m, "n": n, "k": k,
             "scratch": rng.choice(["kept", "kept", "library"]) if op != "shared" else "kept"}
        if work(c)["flops"] <= MAX_FLOPS and work(c)["bytes"] <= 3.5e8:
            return c


# ---- weights: GGUF rows of normal values -------------------------------------------------------

def _half(t):
    return t.to(torch.float16).to(torch.float32)


def _safe(t):
    return torch.where(t == 0, torch.ones_like(t), t)


def _fields(wtype, w):
    """The quantized fields of rows w [n, k], by the plain nearest-level rule of each format."""
    n, k = w.shape
    if wtype in ("Q8_0", "Q8_0_RS"):
        b = w.view(n, k // 32, 32)
        d = _half(b.abs().amax(-1, keepdim=True) / 127)
        return {"d": d, "q": (b / _safe(d)).round().clamp(-127, 127)}
    if wtype == "Q4_0":
        b = w.view(n, k // 32, 32)
        top = b.gather(-1, b.abs().argmax(-1, keepdim=True))
        d = _half(top / -8)
        return {"d": d, "q": (b / _safe(d)).round().clamp(-8, 7)}
    if wtype == "Q6_K":
        b = w.view(n, k // 256, 16, 16)
        s = b.abs().amax(-1, keepdim=True) / 31
        d = _half(s.amax(-2, keepdim=True) / 127)
        sc = (s / _safe(d)).round().clamp(0, 127)
        # a group's scale takes either sign, as the format's quantizers write it
        sc = sc * torch.where(b.sum(-1, keepdim=True) < 0, -1.0, 1.0)
        return {"d": d, "sc": sc, "q": (b / _safe(d * sc)).round().clamp(-32, 31)}
    levels = 15 if wtype == "Q4_K" else 31
    b = w.view(n, k // 256, 8, 32)
    lo = b.amin(-1, keepdim=True).clamp(max=0)
    s = (b.amax(-1, keepdim=True) - lo) / levels
    d, dmin = _half(s.amax(-2, keepdim=True) / 63), _half((-lo).amax(-2, keepdim=True) / 63)
    sc, mn = (s / _safe(d)).round().clamp(0, 63), (-lo / _safe(dmin)).round().clamp(0, 63)
    return {"d": d, "dmin": dmin, "sc": sc, "mn": mn, "q": ((b + dmin * mn) / _safe(d * sc)).round().clamp(0, levels)}


def _values(wtype, f):
    """What the fields stand for, in 64 bits [n, k]."""
    v = f["q"].double() * f["d"].double()
    if "sc" in f:
        v = v * f["sc"].double()
    if "dmin" in f:
        v = v - f["dmin"].double() * f["mn"].double()
    return v.reshape(v.shape[0], -1)


def _bytes_of(t, dtype):
    return t.to(dtype).contiguous().view(torch.uint8)


def _pack(wtype, f):
    """The fields as rows of the GGUF format, uint8 [n, row bytes]."""
    n = f["d"].shape[0]
    d = _bytes_of(f["d"].flatten(2), torch.float16)
    u8 = torch.uint8
    if wtype in ("Q8_0", "Q8_0_RS"):
        return torch.cat([d, _bytes_of(f["q"], torch.int8)], -1).reshape(n, -1)
    if wtype == "Q4_0":
        q = (f["q"] + 8).to(u8)
        return torch.cat([d, q[..., :16] | (q[..., 16:] << 4)], -1).reshape(n, -1)
    if wtype == "Q6_K":
        q = (f["q"] + 32).to(u8).reshape(n, -1, 2, 4, 32)  # half, quarter, element
        low, high = q & 15, q >> 4
        ql = torch.cat([low[..., 0, :] | (low[..., 2, :] << 4), low[..., 1, :] | (low[..., 3, :] << 4)], -1)
        qh = high[..., 0, :] | (high[..., 1, :] << 2) | (high[..., 2, :] << 4) | (high[..., 3, :] << 6)
        return torch.cat([ql.flatten(2), qh.flatten(2), _bytes_of(f["sc"].flatten(2), torch.int8), d], -1).reshape(n, -1)
    sc, mn = f["sc"].flatten(2).to(u8), f["mn"].flatten(2).to(u8)
    scales = torch.cat([sc[..., :4] | ((sc[..., 4:] >> 4) << 6), mn[..., :4] | ((mn[..., 4:] >> 4) << 6),
                        (sc[..., 4:] & 15) | ((mn[..., 4:] & 15) << 4)], -1)
    q = f["q"].to(u8)
    nibbles = ((q[..., 0::2, :] & 15) | ((q[..., 1::2, :] & 15) << 4)).flatten(2)
    parts = [d, _bytes_of(f["dmin"].flatten(2), torch.float16), scales]
    if wtype == "Q5_K":
        bit = torch.arange(8, device=q.device, dtype=u8).view(8, 1)
        parts.append(((q >> 4) << bit).sum(-2, dtype=torch.int32).to(u8))
    return torch.cat(parts + [nibbles], -1).reshape(n, -1)


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _weight_parts(wtype, n, k, seed):
    """The fields of a [n, k] weight, some rows at a time."""
    g = _generator(seed)
    rows = max(1, (1 << 26) // k)
    for r in range(0, n, rows):
        yield _fields(wtype, torch.randn((min(rows, n - r), k), generator=g, device="cuda") * 0.02)


def _weight(wtype, n, k, seed):
    w = torch.cat([_pack(wtype, f) for f in _weight_parts(wtype, n, k, seed)])
    if wtype == "Q8_0_RS":  # a weight loaded once into the library's own row layout
        w = dc.repack_weights(dc.TYPE_Q8_0, w, n, k, dc.TYPE_Q8_0_RS)
    return w


def _shapes(case):
    """(rows, seed offset) of the weights that a case reads."""
    n = case["n"]
    return {"gate_up": [(n, 1), (n, 2)], "shared": [(n, 1), (n // 4, 2), (n // 4, 3)]}.get(case["op"], [(n, 1)])


def _activation(m, k, seed):
    g = _generator(seed)
    x = torch.randn((m, k), generator=g, device="cuda")
    x[:, torch.randperm(k, generator=g, device="cuda")[: max(1, k // 128)]] *= 10
    return x


# ---- a case's state and its pass ---------------------------------------------------------------

def _attention_inputs(case, seed):
    g = _generator(8 * seed)

    def normal(rows, cols, std=1.0):
        return torch.randn((rows, cols), generator=g, device="cuda") * std

    t, p, hd, row = case["tokens"], case["past"], case["head_dim"], case["kv_heads"] * case["head_dim"]
    blocks = (p + t + 15) // 16
    table = torch.randperm(blocks, generator=g, device="cuda").to(torch.int32)
    return {"q": normal(t, case["heads"] * hd, 2.0), "k": normal(t, row), "v": normal(t, row), "k_past": normal(p, row),
            "v_past": normal(p, row), "table": table, "blocks": blocks}


def prepare(case, seed):
    if case["op"] == "attention":
        i = _attention_inputs(case, seed)
        cache = dc.PagedKVCache(CACHE_TYPES[case["cache"]], i["blocks"], LAYERS, case["kv_heads"], case["head_dim"])
        if case["past"]:
            cache.write("k", LAYER, i["table"], 0, i["k_past"])
            cache.write("v", LAYER, i["table"], 0, i["v_past"])
        need = dc.kv_attention_workspace_size(case["heads"], case["kv_heads"], case["head_dim"], case["tokens"],
                                              case["past"])
        return {"case": case, "cache": cache, "table": i["table"], "q": i["q"], "k": i["k"], "v": i["v"],
                "out": torch.empty_like(i["q"]), "scale": 1 / math.sqrt(case["head_dim"]),
                "workspace": torch.empty(need, dtype=torch.uint8, device="cuda") if need else None}
    wtype, m, n, k = case["type"], case["m"], case["n"], case["k"]
    t = TYPES[wtype]
    s = {"case": case, "type": t, "x": _activation(m, k, 8 * seed),
         "w": [_weight(wtype, rows, k, 8 * seed + o) for rows, o in _shapes(case)],
         "y": [torch.empty((m, rows), device="cuda") for rows, _ in _shapes(case)[: 1 if case["op"] == "gate_up" else 3]],
         "workspace": None}
    if case["op"] == "residual":
        s["r"] = torch.randn((m, n), generator=_generator(8 * seed + 4), device="cuda")
    if case["scratch"] == "kept":
        size = {"gate_up": lambda: dc.ffn_gate_up_workspace_size(t, m, n, k),
                "residual": lambda: dc.mul_mat_add_workspace_size(t, m, n, k)}.get(
                    case["op"], lambda: dc.mul_mat_workspace_size(t, m, k))()
        s["workspace"] = torch.empty(size, dtype=torch.uint8, device="cuda")
    return s


def run(s):
    c = s["case"]
    if c["op"] == "attention":
        cache, past = s["cache"], c["past"]
        cache.write("k", LAYER, s["table"], past, s["k"])
        cache.write("v", LAYER, s["table"], past, s["v"])
        out = cache.attention(LAYER, s["table"], s["q"], s["k"], s["v"], past, s["scale"], out=s["out"],
                              workspace=s["workspace"])
        return [out, cache.k, cache.v]
    t, n, k, x, y, ws = s["type"], c["n"], c["k"], s["x"], s["y"], s["workspace"]
    if c["op"] == "linear":
        return [dc.mul_mat(t, s["w"][0], n, k, x, y=y[0], workspace=ws)]
    if c["op"] == "residual":
        return [dc.mul_mat_add(t, s["w"][0], n, k, x, s["r"], y=y[0], workspace=ws)]
    if c["op"] == "gate_up":
        return [dc.ffn_gate_up(t, s["w"][0], s["w"][1], n, k, x, y=y[0], workspace=ws)]
    dc.quantize_src1(t, x, ws)
    return [dc.mul_mat_q(t, w, o.shape[1], k, ws, c["m"], y=o) for w, o in zip(s["w"], y)]


def work(case):
    if case["op"] == "attention":
        t, p, hd = case["tokens"], case["past"], case["head_dim"]
        row = case["kv_heads"] * hd
        cached = CACHE_ROW[case["cache"]]
        # q and out, the step's k and v (read, and written to the cache), the history
        return {"bytes": 8 * t * case["heads"] * hd + 2 * t * row * (4 + cached) + 2 * p * row * cached,
                "flops": 4 * case["heads"] * hd * (t * p + t * (t + 1) // 2)}
    size, block = ROW_BYTES[case["type"]]
    m, k = case["m"], case["k"]
    rows = sum(r for r, _ in _shapes(case))
    outs = case["n"] if case["op"] == "gate_up" else rows
    out_bytes = 4 * m * outs * (2 if case["op"] == "residual" else 1)
    return {"bytes": rows * (k // block) * size + 4 * m * k + out_bytes, "flops": 2 * m * k * rows}


def tolerance(case):
    # fp32 sums in another order, of products that cancel: four times the distance from the same
    # products summed in 64 bits
    if case["op"] == "attention":
        return {"rel": 4e-6}
    return {"rel": 1e-6}


# ---- the same in 64 bits -----------------------------------------------------------------------

def _over(a, b):
    """a / b correctly rounded (with a number on either side torch multiplies by a reciprocal)."""
    return torch.full_like(b, a) / b if torch.is_tensor(b) else a / torch.full_like(a, b)


def _quantized_activation(wtype, x):
    """The values of the activation after the format's own quantization (fp32 steps, as defined)."""
    m, k = x.shape
    if wtype in ("Q8_0", "Q8_0_RS", "Q4_0"):
        b = x.view(m, k // 32, 32)
        amax = b.abs().amax(-1, keepdim=True)
        q = (b * _over(127.0, _safe(amax))).round()
        return (q.double() * _half(_over(amax, 127.0)).double()).view(m, k)
    b = x.view(m, k // 256, 256)
    top = b.gather(-1, b.abs().argmax(-1, keepdim=True))
    scale = _over(-127.0, _safe(top))
    return ((scale * b).round().clamp(max=127).double() * _over(1.0, scale).double()).view(m, k)


def _cached(kind, rows):
    """Rows as the cache holds them, in 64 bits."""
    if kind == "F32":
        return rows.double()
    if kind == "F16":
        return rows.half().double()
    b = rows.view(rows.shape[0], rows.shape[1] // 32, 32)
    d = _over(b.abs().amax(-1, keepdim=True), 127.0)
    q = b * _over(1.0, _safe(d))
    q = torch.where(q < 0, -1.0, 1.0) * (q.abs() + 0.5).floor()
    return (q.double() * _half(d).double()).view(rows.shape)


def _exact_attention(case, seed):
    i = _attention_inputs(case, seed)
    t, p, hd = case["tokens"], case["past"], case["head_dim"]
    group = case["heads"] // case["kv_heads"]
    k_all = torch.cat([_cached(case["cache"], i["k_past"]), i["k"].double()])
    v_all = torch.cat([_cached(case["cache"], i["v_past"]), i["v"].double()])
    hidden = torch.arange(p + t, device="cuda").view(1, -1) > torch.arange(p, p + t, device="cuda").view(-1, 1)
    out = torch.empty_like(i["q"], dtype=torch.float64)
    scale = torch.tensor(1 / math.sqrt(hd), dtype=torch.float32).double().item()
    for h in range(case["heads"]):
        one, kv = slice(h * hd, (h + 1) * hd), slice(h // group * hd, (h // group + 1) * hd)
        scores = (i["q"][:, one].double() @ k_all[:, kv].t().contiguous()) * scale
        out[:, one] = torch.softmax(scores.masked_fill(hidden, -math.inf), -1) @ v_all[:, kv].contiguous()
    return [out, None, None]


def exact(case, seed):
    if case["op"] == "attention":
        return _exact_attention(case, seed)
    wtype, k = case["type"], case["k"]
    x = _quantized_activation(wtype, _activation(case["m"], k, 8 * seed)).t().contiguous()
    y = [torch.cat([_values(wtype, f) @ x for f in _weight_parts(wtype, rows, k, 8 * seed + o)]).t()
         for rows, o in _shapes(case)]
    if case["op"] == "residual":
        return [y[0] + torch.randn((case["m"], case["n"]), generator=_generator(8 * seed + 4), device="cuda").double()]
    if case["op"] == "gate_up":
        return [torch.nn.functional.silu(y[0]) * y[1]]
    return y
