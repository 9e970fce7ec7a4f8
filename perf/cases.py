"""The work that a program using this library has it do, as measurable cases.

Single layers go through the C entry points on device buffers, the way an
engine that binds the library calls them; two whole calls go through the
model layer and return logits. Inputs are made on the GPU from the seed.

  linear  : one projection (prana_matmul: quantize the activations, multiply)
            in every weight format the loader keeps, one token to a prompt
  softmax : probabilities over a vocabulary (prana_softmax, temperature sampling)
  prefill : causal attention over a prompt's f32 K/V (prana_attention_prefill)
  cache   : exact attention of a decode row or a verify batch over an f16
            cache (prana_attention_decode / _verify)
  splitk  : split-K decode attention of independent sequences
  model   : "step" = one forward over a filled cache, "prompt" = a prefill and
            the forward of its last token, "verify" = a forward_batch
"""
import ctypes as C
import math

import numpy as np
import torch

import prana_amd as P

F32, Q4_0, Q8_0, Q4_K, Q6_K = P.F32, P.Q4_0, P.Q8_0, P.Q4_K, P.Q6_K
TYPES = {"f32": F32, "q8_0": Q8_0, "q4_0": Q4_0, "q4_k": Q4_K, "q6_k": Q6_K, "q8": None}
BYTES = {"f32": 4.0, "q8_0": 34 / 32, "q4_0": 18 / 32, "q4_k": 144 / 256, "q6_k": 210 / 256, "q8": 36 / 32}

# Model shapes: the 15M llama shape (Q8_0) and the first four layers of the
# qwen2-0.5B shape (Q4_0 with Q8_0 / Q6_K parts, biases, tied head).
MODELS = {
    "15m": dict(dim=288, hidden_dim=768, n_layers=6, n_heads=6, n_kv_heads=6, vocab_size=32000, seq_len=256,
                head_dim=48, rope_theta=1e4, norm_eps=1e-5, emb_scale=1.0, rope_neox=0, act=0),
    "0.5b": dict(dim=896, hidden_dim=4864, n_layers=4, n_heads=14, n_kv_heads=2, vocab_size=151936, seq_len=4096,
                 head_dim=64, rope_theta=1e6, norm_eps=1e-6, emb_scale=1.0, rope_neox=1, act=0),
}
# (query heads, KV heads, head width) of the shapes above, of the 7B shape, and of other widths the entry points take
HEADS = ((6, 6, 48), (14, 2, 64), (32, 8, 128), (8, 1, 256), (16, 16, 80), (12, 4, 96))


def listed():
    return [
        # the head of a dense (f32) 15M checkpoint, one decoded token
        {"name": "dense_token", "op": "linear", "type": "f32", "rows": 32000, "cols": 288, "tokens": 1},
        # a dense projection over a prompt (an F32 / F16 checkpoint kept at full precision)
        {"name": "dense_prompt", "op": "linear", "type": "f32", "rows": 2048, "cols": 2048, "tokens": 301},
        # the down projection of the 7B shape, one decoded token
        {"name": "q4_0_token", "op": "linear", "type": "q4_0", "rows": 4096, "cols": 14336, "tokens": 1},
        # a gate projection over a verify batch
        {"name": "q8_0_verify", "op": "linear", "type": "q8_0", "rows": 14336, "cols": 4096, "tokens": 9},
        # the gate projection of the 7B shape over a prompt
        {"name": "q4_0_prompt", "op": "linear", "type": "q4_0", "rows": 14336, "cols": 4096, "tokens": 511},
        # the down projection of the 0.5B shape over a long prompt
        {"name": "q6_k_prompt", "op": "linear", "type": "q6_k", "rows": 896, "cols": 4864, "tokens": 2047},
        # temperature sampling over the 0.5B shape's vocabulary
        {"name": "vocab_softmax", "op": "softmax", "rows": 1, "cols": 151936},
        # one layer's attention of the 0.5B shape over a long prompt
        {"name": "prefill_attention", "op": "prefill", "seq": 3001, "heads": 14, "kv_heads": 2, "width": 64},
        # the 7B shape's attention for one decoded token over a long cache
        {"name": "cache_attention", "op": "cache", "first": 4099, "rows": 1, "heads": 32, "kv_heads": 8,
         "width": 128},
        # a serving batch: eight sequences of different lengths
        {"name": "splitk_attention", "op": "splitk", "seqs": 8, "longest": 32768, "heads": 32, "kv_heads": 8,
         "width": 128},
        # the smallest whole call: one token through the 15M shape
        {"name": "model_step", "op": "model", "mode": "step", "shape": "15m", "past": 100, "tokens": 1},
        # a long prompt through the 0.5B shape, to its last token's logits
        {"name": "model_prompt", "op": "model", "mode": "prompt", "shape": "0.5b", "past": 0, "tokens": 2500},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(("linear", "linear", "linear", "linear", "softmax", "prefill", "prefill", "cache", "cache",
                     "splitk", "model"))
    if op == "linear":
        kind = rng.choice(("f32", "f32", "q8_0", "q4_0", "q4_0", "q4_k", "q6_k", "q8"))
        tokens = rng.choice((1, 1, rng.randint(2, 16), _log(rng, 2, 600)))
        unit = {"f32": 1, "q4_k": 256, "q6_k": 256}.get(kind, 32)
        cols = max(1, _log(rng, 256, 14336) // unit) * unit
        most = min(32000, 2048 * 2048 * 301 // (cols * tokens))
        return {"op": op, "type": kind, "rows": _log(rng, 64, max(most, 65)), "cols": cols, "tokens": tokens}
    if op == "softmax":
        cols = _log(rng, 500, 151936)
        return {"op": op, "rows": rng.randint(1, max(1, 600000 // cols) if cols > 5000 else 100), "cols": cols}
    if op == "model":
        shape = rng.choice(sorted(MODELS))
        mode = rng.choice(("step", "prompt", "verify"))
        past = 0 if mode == "prompt" else _log(rng, 4, 200 if shape == "15m" else 2600)
        tokens = {"step": 1, "verify": rng.randint(2, 9)}.get(mode) or _log(rng, 4, 240 if shape == "15m" else 2400)
        return {"op": op, "mode": mode, "shape": shape, "past": past, "tokens": tokens}
    heads, kv_heads, width = rng.choice(HEADS)
    case = {"op": op, "heads": heads, "kv_heads": kv_heads, "width": width}
    if op == "prefill":
        most = math.isqrt(14 * 64 * 3001 * 3001 // (heads * width))
        case["seq"] = _log(rng, 16, most)
    elif op == "cache":
        case["rows"] = rng.choice((1, 1, rng.randint(2, 9)))
        case["first"] = _log(rng, 8, 16384)
    else:
        case["seqs"] = rng.randint(1, 8)
        case["longest"] = _log(rng, 64, 32768)
    return case


# ------------------------------------------------------------------ weights
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _normal(g, *shape, sigma=1.0):
    return torch.randn(*shape, device="cuda", generator=g) * sigma


def _halves(x):
    """f32 -> f16 bits as bytes, and the value they stand for."""
    h = x.to(torch.float16)
    return h.view(torch.uint8).reshape(*x.shape, 2), h.float()


def _encode(kind, w):
    """Weights [rows, cols] in a stored format: (bytes or parts, value of every weight in 64 bits as a function)."""
    rows, cols = w.shape
    if kind == "f32":
        return w.contiguous(), lambda: w.double()
    if kind in ("q8_0", "q8"):
        b = w.reshape(rows, -1, 32)
        d = b.abs().amax(-1) / 127
        raw_d, d16 = _halves(d)
        d = d16 if kind == "q8_0" else d
        q = torch.clamp(torch.round(b / torch.where(d > 0, d, 1.0)[..., None]), -127, 127)
        if kind == "q8":
            parts = (q.to(torch.int8).reshape(rows, cols), d)
        else:
            parts = torch.cat([raw_d, q.to(torch.int8).view(torch.uint8)], -1)
        return parts, lambda: (q.double() * d.double()[..., None]).reshape(rows, cols)
    if kind == "q4_0":
        b = w.reshape(rows, -1, 32)
        top = b.gather(-1, b.abs().argmax(-1, keepdim=True))
        raw_d, d = _halves(top[..., 0] / -8)
        q = torch.clamp(torch.floor(b / torch.where(d != 0, d, 1.0)[..., None] + 8.5), 0, 15).to(torch.uint8)
        raw = torch.cat([raw_d, q[..., :16] | (q[..., 16:] << 4)], -1)
        return raw, lambda: ((q.double() - 8) * d.double()[..., None]).reshape(rows, cols)
    b = w.reshape(rows, -1, 256)
    if kind == "q4_k":
        s = b.reshape(rows, -1, 8, 32)
        low = torch.clamp(-s.amin(-1), min=0)
        step = (s.amax(-1) + low) / 15
        raw_d, d = _halves(step.amax(-1) / 63)
        raw_m, dm = _halves(low.amax(-1) / 63)
        ls = torch.clamp(torch.round(step / torch.where(d > 0, d, 1.0)[..., None]), 0, 63)
        lm = torch.clamp(torch.round(low / torch.where(dm > 0, dm, 1.0)[..., None]), 0, 63)
        scale, least = d[..., None] * ls, dm[..., None] * lm
        q = torch.round((s + least[..., None]) / torch.where(scale > 0, scale, 1.0)[..., None])
        q = torch.clamp(q, 0, 15).to(torch.uint8)
        a, m = ls.to(torch.uint8), lm.to(torch.uint8)
        packed = torch.cat([a[..., :4] | ((a[..., 4:] >> 4) << 6), m[..., :4] | ((m[..., 4:] >> 4) << 6),
                            (a[..., 4:] & 15) | ((m[..., 4:] & 15) << 4)], -1)
        pairs = q.reshape(rows, -1, 4, 2, 32)
        body = (pairs[..., 0, :] | (pairs[..., 1, :] << 4)).reshape(rows, -1, 128)
        raw = torch.cat([raw_d, raw_m, packed, body], -1)
        return raw, lambda: (scale.double()[..., None] * q.double() - least.double()[..., None]).reshape(rows, cols)
    s = b.reshape(rows, -1, 16, 16)
    step = s.abs().amax(-1) / 32
    raw_d, d = _halves(step.amax(-1) / 127)
    sc = torch.clamp(torch.round(step / torch.where(d > 0, d, 1.0)[..., None]), 0, 127)
    scale = d[..., None] * sc
    q = torch.clamp(torch.round(s / torch.where(scale > 0, scale, 1.0)[..., None]), -32, 31)
    u = (q + 32).to(torch.uint8).reshape(rows, -1, 2, 4, 32)  # [half][quarter][32]
    low, high = u & 15, u >> 4
    ql = torch.cat([low[..., 0, :] | (low[..., 2, :] << 4), low[..., 1, :] | (low[..., 3, :] << 4)], -1)
    qh = high[..., 0, :] | (high[..., 1, :] << 2) | (high[..., 2, :] << 4) | (high[..., 3, :] << 6)
    raw = torch.cat([ql.reshape(rows, -1, 128), qh.reshape(rows, -1, 64), sc.to(torch.int8).view(torch.uint8), raw_d],
                    -1)
    return raw, lambda: (scale.double()[..., None] * q.double()).reshape(rows, cols)


def _matrix(kind, rows, cols, encoded):
    if kind == "q8":
        return P.Matrix.q8_parts(encoded[0].cpu().numpy(), encoded[1].cpu().numpy())
    return P.Matrix(TYPES[kind], rows, cols, encoded.cpu().numpy())


def _quantized(x):
    """What the activations are after quantization to 8 bits in blocks of 32 (amax / 127, ties away from zero)."""
    b = x.float().cpu().reshape(*x.shape[:-1], -1, 32)
    amax = b.abs().amax(-1, keepdim=True)
    scale = torch.where(amax > 0, amax / 127, torch.ones_like(amax))
    t = b * (1.0 / scale)
    q = torch.sign(t) * torch.floor(t.abs() + 0.5)
    return (q.double() * scale.double()).reshape(x.shape).cuda()


# ------------------------------------------------------------------ models
_models = {}


def _kind_of(shape, name, cols):
    if shape == "15m":
        return "q8_0"
    six = name.endswith("attn_v.weight") or name.endswith("ffn_down.weight")
    if cols % 256 == 0:
        return "q6_k" if six else "q4_k"
    return "q8_0" if six else "q4_0"


def _tensors(shape):
    """Every tensor of a model: name -> (kind, weights), from the shape alone."""
    c = MODELS[shape]
    d, h, q, kv = c["dim"], c["hidden_dim"], c["n_heads"] * c["head_dim"], c["n_kv_heads"] * c["head_dim"]
    g = _gen(17)
    mats = [("token_embd.weight", d, c["vocab_size"])]
    for i in range(c["n_layers"]):
        b = "blk.%d." % i
        mats += [(b + "attn_q.weight", d, q), (b + "attn_k.weight", d, kv), (b + "attn_v.weight", d, kv),
                 (b + "attn_output.weight", q, d), (b + "ffn_gate.weight", d, h), (b + "ffn_up.weight", d, h),
                 (b + "ffn_down.weight", h, d)]
    if shape == "15m":
        mats.append(("output.weight", d, c["vocab_size"]))
    for name, cols, rows in mats:
        yield name, _kind_of(shape, name, cols), _normal(g, rows, cols, sigma=0.02)
    for i in range(c["n_layers"]):
        b = "blk.%d." % i
        yield b + "attn_norm.weight", "vec", 1 + _normal(g, d, sigma=0.05)
        yield b + "ffn_norm.weight", "vec", 1 + _normal(g, d, sigma=0.05)
        if shape != "15m":
            for name, n in (("attn_q.bias", q), ("attn_k.bias", kv), ("attn_v.bias", kv)):
                yield b + name, "vec", _normal(g, n, sigma=0.02)
    yield "output_norm.weight", "vec", 1 + _normal(g, d, sigma=0.05)


def _model(shape):
    if shape not in _models:  # a program loads its weights once, for all its sequences
        m = P.Model(MODELS[shape])
        for name, kind, w in _tensors(shape):
            if kind == "vec":
                m.set_tensor(name, F32, (w.numel(),), w.cpu().numpy())
            else:
                m.set_tensor(name, TYPES[kind], (w.shape[1], w.shape[0]), _encode(kind, w)[0].cpu().numpy())
        m.finalize()
        _models[shape] = m
    return _models[shape]


def _tokens(case, seed):
    n = case["past"] + case["tokens"]
    return np.random.default_rng(seed).integers(0, MODELS[case["shape"]]["vocab_size"], n).astype(np.uint32)


# ------------------------------------------------------------------ cases
def _lengths(case, seed):
    """Positions of a serving batch's sequences: the longest, and others between an eighth of it and all of it."""
    rng = np.random.default_rng(seed)
    n = [case["longest"]] + [int(case["longest"] * f) for f in rng.uniform(0.125, 1.0, case["seqs"] - 1)]
    return [max(0, x - 1) for x in n]


def _inputs(case, seed):
    g = _gen(seed)
    op = case["op"]
    if op == "linear":
        w = _normal(g, case["rows"], case["cols"], sigma=0.02)
        return {"weights": w, "x": _normal(g, case["tokens"], case["cols"])}
    if op == "softmax":
        return {"x": _normal(g, case["rows"], case["cols"], sigma=2.5)}
    h, kv, w = case["heads"], case["kv_heads"], case["width"]
    if op == "prefill":
        n = case["seq"]
        return {"q": _normal(g, n, h * w), "k": _normal(g, n, kv * w), "v": _normal(g, n, kv * w)}
    if op == "cache":
        n = case["first"] + case["rows"]
        return {"q": _normal(g, case["rows"], h * w), "k": _normal(g, n, kv * w).half(),
                "v": _normal(g, n, kv * w).half()}
    pos = _lengths(case, seed)
    return {"q": _normal(g, len(pos), h * w), "pos": pos,
            "k": [_normal(g, p + 1, kv * w).half() for p in pos],
            "v": [_normal(g, p + 1, kv * w).half() for p in pos]}


def prepare(case, seed):
    op = case["op"]
    P.init()
    if op == "model":
        m = _model(case["shape"])
        t = _tokens(case, seed)
        cache = m.cache(case["past"] + case["tokens"])
        if case["past"]:
            cache.prefill(t[:case["past"]])
        return {"case": case, "cache": cache, "tokens": t}
    s = _inputs(case, seed)
    s["case"] = case
    if op == "linear":
        s["matrix"] = _matrix(case["type"], case["rows"], case["cols"], _encode(case["type"], s.pop("weights"))[0])
        s["out"] = torch.empty(case["tokens"], case["rows"], device="cuda")
    elif op == "softmax":
        s["out"] = torch.empty_like(s["x"])
    else:
        s["out"] = torch.empty_like(s["q"])
    if op == "splitk":
        n = len(s["pos"])
        s["kp"] = (C.c_void_p * n)(*[k.data_ptr() for k in s["k"]])
        s["vp"] = (C.c_void_p * n)(*[v.data_ptr() for v in s["v"]])
        s["ps"] = (C.c_size_t * n)(*s["pos"])
    return s


def run(state):
    case, lib = state["case"], P.load()
    op = case["op"]
    if op == "model":
        cache, t, past = state["cache"], state["tokens"], case["past"]
        if case["mode"] == "verify":
            return cache.forward_batch(t[past:], past)
        if case["mode"] == "prompt":
            cache.prefill(t[:-1])
        return cache.forward(t[-1], len(t) - 1)
    out = state["out"]
    if op == "linear":
        P.check(lib.prana_matmul(state["matrix"].h, state["x"].data_ptr(), case["tokens"], out.data_ptr(), None))
        return out
    if op == "softmax":
        P.check(lib.prana_softmax(state["x"].data_ptr(), case["rows"], case["cols"], out.data_ptr(), None))
        return out
    heads = (case["heads"], case["kv_heads"], case["width"], out.data_ptr(), None)
    q = state["q"].data_ptr()
    if op == "splitk":
        P.check(lib.prana_attention_decode_splitk(q, state["kp"], state["vp"], state["ps"], case["seqs"], *heads))
        return out
    k, v = state["k"].data_ptr(), state["v"].data_ptr()
    if op == "prefill":
        P.check(lib.prana_attention_prefill(q, k, v, case["seq"], *heads))
    elif case["rows"] == 1:
        P.check(lib.prana_attention_decode(q, k, v, case["first"], *heads))
    else:
        P.check(lib.prana_attention_verify(q, k, v, case["first"], case["rows"], *heads))
    return out


def work(case):
    op = case["op"]
    if op == "linear":
        r, c, n = case["rows"], case["cols"], case["tokens"]
        return {"bytes": r * c * BYTES[case["type"]] + 4 * n * (r + c), "flops": 2 * r * c * n}
    if op == "softmax":
        return {"bytes": 8 * case["rows"] * case["cols"], "flops": 4 * case["rows"] * case["cols"]}
    if op == "model":
        c = MODELS[case["shape"]]
        d, h, kv = c["dim"], c["hidden_dim"], c["n_kv_heads"] * c["head_dim"]
        q = c["n_heads"] * c["head_dim"]
        layer = d * (2 * q + 2 * kv + 3 * h)
        n, last = case["tokens"], case["past"] + case["tokens"]
        heads = case["tokens"] if case["mode"] == "verify" else 1
        pairs = n * (case["past"] + (n + 1) / 2)
        weights = c["n_layers"] * layer + d * c["vocab_size"]
        each = 34 / 32 if case["shape"] == "15m" else 0.6
        return {"bytes": weights * each + c["n_layers"] * last * kv * 4 + heads * c["vocab_size"] * 4,
                "flops": 2 * n * c["n_layers"] * layer + 2 * heads * d * c["vocab_size"]
                + 4 * c["n_layers"] * pairs * q}
    h, kv, w = case["heads"], case["kv_heads"], case["width"]
    if op == "prefill":
        n = case["seq"]
        return {"bytes": 4 * n * w * (2 * h + 2 * kv), "flops": 4 * h * w * n * (n + 1) / 2}
    if op == "cache":
        n, rows = case["first"] + case["rows"], case["rows"]
        return {"bytes": 4 * n * kv * w + 8 * rows * h * w, "flops": 4 * h * w * rows * n}
    # the sequences other than the longest are 9/16 as long on average
    n = case["longest"] * (1 + (case["seqs"] - 1) * 9 / 16)
    return {"bytes": 4 * n * kv * w + 8 * case["seqs"] * h * w, "flops": 4 * h * w * n}


def tolerance(case):
    """About four times the distance from 64 bits that the library showed when these cases were written."""
    op = case["op"]
    if op == "model":  # a value that rounds to another 8-bit step in one layer moves all that follow
        return {"rel": 3e-2 if case["shape"] == "15m" else 8e-2}
    if op == "softmax":  # a left-to-right 32-bit sum drifts with its length
        return {"rel": 1e-6 + 3e-9 * case["cols"]}
    return {"rel": {"linear": 2e-6, "prefill": 6e-6, "cache": 1.2e-5, "splitk": 1e-6}[op]}


# ------------------------------------------------------------------ in 64 bits
def _attend(q, k, v, first, heads, kv_heads, width):
    """Causal attention of rows first.. over k and v, in 64 bits."""
    n, keys, group = q.shape[0], k.shape[0], heads // kv_heads
    out = torch.empty(n, heads * width, device="cuda", dtype=torch.float64)
    at = torch.arange(keys, device="cuda")
    for h in range(heads):
        kh = k[:, (h // group) * width:(h // group + 1) * width].double().contiguous()
        vh = v[:, (h // group) * width:(h // group + 1) * width].double().contiguous()
        for i in range(0, n, 1024):
            qh = q[i:i + 1024, h * width:(h + 1) * width].double().contiguous()
            s = (qh @ kh.t().contiguous()) / math.sqrt(width)
            rows = first + i + torch.arange(qh.shape[0], device="cuda")
            s.masked_fill_(at[None, :] > rows[:, None], -math.inf)
            out[i:i + 1024, h * width:(h + 1) * width] = torch.softmax(s, -1) @ vh
    return out


def _norm(x, w, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps) * w


def _rope(c, x, positions):
    n, hd = x.shape[0], c["head_dim"]
    m = torch.arange(hd // 2, device="cuda", dtype=torch.float64)
    freq = torch.tensor(c["rope_theta"], dtype=torch.float64) ** (-2 * m / hd)
    angle = positions[:, None, None].double() * freq
    x = x.reshape(n, -1, hd)
    a, b = (x[..., :hd // 2], x[..., hd // 2:]) if c["rope_neox"] else (x[..., ::2], x[..., 1::2])
    cos, sin = torch.cos(angle), torch.sin(angle)
    pair = (a * cos - b * sin, a * sin + b * cos)
    return (torch.cat(pair, -1) if c["rope_neox"] else torch.stack(pair, -1)).reshape(n, -1)


def _model_exact(case, seed):
    c = MODELS[case["shape"]]
    hd, nh, kvh = c["head_dim"], c["n_heads"], c["n_kv_heads"]
    w = {name: t.double() if kind == "vec" else _encode(kind, t)[1]() for name, kind, t in _tensors(case["shape"])}
    ids = torch.from_numpy(_tokens(case, seed).astype(np.int64)).cuda()
    n = ids.numel()
    # rows from here on attend over the f16 cache, those before it (a prefill) over the f32 rows
    cached = {"verify": case["past"]}.get(case["mode"], n - 1)
    at = torch.arange(n, device="cuda")
    x = w["token_embd.weight"][ids]
    for i in range(c["n_layers"]):
        b = "blk.%d." % i
        y = _quantized(_norm(x, w[b + "attn_norm.weight"], c["norm_eps"]))
        q, k, v = (y @ w[b + "attn_%s.weight" % s].t() + w.get(b + "attn_%s.bias" % s, 0.0) for s in "qkv")
        q, k = _rope(c, q, at), _rope(c, k, at)
        o = torch.empty_like(q)
        if cached:
            o[:cached] = _attend(q[:cached], k[:cached], v[:cached], 0, nh, kvh, hd)
        o[cached:] = _attend(q[cached:], k.half(), v.half(), cached, nh, kvh, hd)
        x = x + _quantized(o) @ w[b + "attn_output.weight"].t()
        y = _quantized(_norm(x, w[b + "ffn_norm.weight"], c["norm_eps"]))
        gate = y @ w[b + "ffn_gate.weight"].t()
        x = x + _quantized(gate * torch.sigmoid(gate) * (y @ w[b + "ffn_up.weight"].t())) @ w[b + "ffn_down.weight"].t()
    x = x[cached:]
    y = _norm(x, w["output_norm.weight"], c["norm_eps"])
    head = w.get("output.weight", w["token_embd.weight"])
    out = _quantized(y) @ head.t()
    return out if case["mode"] == "verify" else out[0]


def exact(case, seed):
    op = case["op"]
    if op == "model":
        return _model_exact(case, seed)
    s = _inputs(case, seed)
    if op == "linear":
        w = _encode(case["type"], s["weights"])[1]()
        return (s["x"].double() if case["type"] == "f32" else _quantized(s["x"])) @ w.t()
    if op == "softmax":
        return torch.softmax(s["x"].double(), -1)
    shape = (case["heads"], case["kv_heads"], case["width"])
    if op == "splitk":
        return torch.cat([_attend(s["q"][i:i + 1], s["k"][i], s["v"][i], p, *shape) for i, p in enumerate(s["pos"])])
    return _attend(s["q"], s["k"], s["v"], case.get("first", 0), *shape)
