"""Performance cases of the decode tier: the work its users have it do, from one
matvec to a whole model, through the package's public entry points.

Weights are GGUF payloads made on the GPU from the seed (codes and scales as
quantised N(0, 0.02) weights have them), activations are N(0, 1) and K/V rows
N(0, 1) as a norm leaves them.  ``exact`` repeats a case in 64 bits with torch
alone.
"""
from __future__ import annotations

import ctypes
import math

import numpy as np
import torch

import ramforge_amd as rf
from ramforge_amd import GGML, synthetic

# elements and bytes per block
GEOMETRY = {"F32": (1, 4), "Q4_0": (32, 18), "Q5_0": (32, 22), "Q8_0": (32, 34), "Q4_K": (256, 144),
            "Q5_K": (256, 176), "Q6_K": (256, 210)}
PACKED = ("Q8_0", "Q4_0", "Q4_K", "Q6_K")  # types with a device-native layout
EPS, THETA = 1e-5, 10000.0

# Llama-3-8B's and a 1.5B model's layer shapes (the second with six query heads per KV head)
SHAPE_8B = {"d": 4096, "heads": 32, "kv_heads": 8, "head_dim": 128, "ffn": 14336}
SHAPE_1B = {"d": 1536, "heads": 12, "kv_heads": 2, "head_dim": 128, "ffn": 8960}


def listed():
    return [
        # one small projection, as a host executor issues them one after the other: launch latency
        {"name": "matvec_small", "kind": "matvec", "type": "Q8_0", "out": 1536, "in": 1536},
        # the FFN down projection of an 8B model held as GGUF bytes
        {"name": "matvec_down", "kind": "matvec", "type": "Q4_K", "out": 4096, "in": 14336},
        # the output projection of the same model, the longest matvec of a token
        {"name": "matvec_output", "kind": "matvec", "type": "Q6_K", "out": 128256, "in": 4096},
        # a few prompt tokens (a short question, a ragged last chunk) through the Q/K/V rows
        {"name": "matmul_ragged", "kind": "matmul", "type": "Q8_0", "out": 6144, "in": 4096, "tokens": 37},
        # a prompt's worth of tokens through an FFN matrix
        {"name": "matmul_prompt", "kind": "matmul", "type": "Q4_K", "out": 14336, "in": 4096, "tokens": 512},
        # decode attention at a full context
        {"name": "attention_8k", "kind": "attention", "heads": 32, "kv_heads": 8, "head_dim": 128, "positions": 8192},
        # decode attention of a model with six query heads per KV head, in the middle of a document
        {"name": "attention_six", "kind": "attention", "heads": 12, "kv_heads": 2, "head_dim": 128, "positions": 1501},
        # one decoder layer of a token as the reference's executor runs it, call by call on GGUF bytes
        {"name": "layer_by_calls", "kind": "layer", "type": "Q4_K", "positions": 512, **SHAPE_8B},
        # a prompt through a model's layers (two of an 8B model's), then its logits
        {"name": "prompt_512", "kind": "prompt", "type": "Q8_0", "layers": 2, "vocab": 8192, "tokens": 512, **SHAPE_8B},
        # a long, ragged document: attention over thousands of positions joins the projections
        {"name": "prompt_long", "kind": "prompt", "type": "Q4_K", "layers": 1, "vocab": 8192, "tokens": 4001,
         **SHAPE_8B},
        # a turn of a chat with a small model whose tokens the host samples: prompt, then logits per token
        {"name": "chat_small", "kind": "chat", "type": "Q4_0", "layers": 8, "vocab": 32000, "tokens": 203, "steps": 6,
         **SHAPE_1B},
        # the whole 8B Q8_0 model: a short prompt, then greedy tokens chosen on the device
        {"name": "decode_8b", "kind": "decode", "type": "Q8_0", "tokens": 32, "steps": 16},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _heads(rng):
    """(query heads, KV heads, head_dim): one to eight query heads per KV head."""
    kv = rng.choice((1, 2, 3, 4, 5, 8))
    return {"heads": kv * rng.choice((1, 2, 3, 4, 4, 6, 7, 8)), "kv_heads": kv,
            "head_dim": rng.choice((64, 64, 128, 128, 128, 96, 256))}


def _model_heads(rng):
    kv, hd = rng.choice(((2, 128), (4, 64), (4, 128), (8, 64), (8, 128)))
    return {"heads": kv * rng.choice((1, 2, 3, 4, 4, 6, 7)), "kv_heads": kv, "head_dim": hd}


def draw(rng):
    kind = rng.choice(("matvec", "matvec", "packed", "matmul", "matmul", "attention", "attention", "layer", "prompt",
                       "prompt", "chat"))
    if kind in ("matvec", "packed", "matmul"):
        t = rng.choice(tuple(GEOMETRY) if kind == "matvec" else PACKED)
        qk = 256 if t.endswith("_K") else 32
        case = {"kind": kind, "type": t, "out": _log(rng, 64, 32768), "in": qk * max(1, _log(rng, 256, 16384) // qk)}
        if kind == "matmul":
            case["tokens"] = _log(rng, 2, 1024)
        return case
    if kind == "attention":
        return {"kind": kind, "positions": _log(rng, 16, 16384), **_heads(rng)}
    shape = {"d": 256 * rng.randint(3, 16), "ffn": 256 * rng.randint(6, 48)}
    if kind == "layer":
        return {"kind": kind, "type": rng.choice(("Q8_0", "Q4_0", "Q4_K", "Q5_K", "Q6_K")),
                "positions": _log(rng, 16, 8192), **shape, **_model_heads(rng)}
    case = {"kind": kind, "type": rng.choice(PACKED), "layers": rng.randint(1, 2), "vocab": 4096,
            "tokens": _log(rng, 5, 3000), **shape, **_model_heads(rng)}
    if kind == "chat":
        case.update(tokens=_log(rng, 5, 1500), steps=rng.randint(1, 8))
    return case


# ------------------------------------------------------------------ payloads

def _gen(seed, salt):
    return torch.Generator(device="cuda").manual_seed(int(seed) * 1000003 + salt)


def _half_bytes(v):
    """f16 values [n] as bytes [n, 2]"""
    return v.to(torch.float16).view(torch.uint8).reshape(-1, 2)


def _payload(t, out_dim, in_dim, seed, salt):
    """GGUF payload bytes [out_dim * blocks per row, block bytes] of a random matrix, on the GPU."""
    g = _gen(seed, salt)
    if t == "F32":
        return (torch.randn(out_dim * in_dim, generator=g, device="cuda") * 0.02).view(torch.uint8).reshape(-1, 4)
    qk, size = GEOMETRY[t]
    n = out_dim * in_dim // qk
    spread = 0.75 + 0.5 * torch.rand(n, generator=g, device="cuda")
    if t == "Q8_0":
        raw = torch.empty(n, size, dtype=torch.uint8, device="cuda")
        codes = torch.randn(n, 32, generator=g, device="cuda").mul_(42).round_().clamp_(-127, 127)
        raw[:, 2:] = codes.to(torch.int8).view(torch.uint8)
        raw[:, :2] = _half_bytes(spread * (0.02 / 42))
        return raw
    raw = torch.randint(0, 256, (n, size), generator=g, device="cuda", dtype=torch.uint8)
    if t in ("Q4_0", "Q5_0"):
        raw[:, :2] = _half_bytes(spread * (0.02 / (4.6 if t == "Q4_0" else 9.2)))
    elif t in ("Q4_K", "Q5_K"):
        # the min takes the codes' mean off (Q5_K's scale is a subnormal half, which counts half)
        d, mid = (8.5e-5, 7.5) if t == "Q4_K" else (4.7e-5, 7.75)
        raw[:, :2] = _half_bytes(spread * d)
        raw[:, 2:4] = _half_bytes(spread * (d * mid))
    else:  # Q6_K
        raw[:, 208:210] = _half_bytes(spread * 3e-5)
    return raw


def _half(b):
    """f16 bytes [..., 2] -> f64; a subnormal half counts half its value, as the format's decoder here defines it."""
    v = b.contiguous().view(torch.float16).squeeze(-1).double()
    return torch.where(v.abs() < 2.0 ** -14, v * 0.5, v)


def _k_scales(s):
    """The eight 6-bit scales and mins of 12 packed bytes [n, 12]."""
    s = s.long()
    lo, hi = s[:, 0:4], s[:, 4:8]
    sc = torch.cat([lo & 63, (s[:, 8:12] & 15) | (lo >> 6 << 4)], 1)
    m = torch.cat([hi & 63, (s[:, 8:12] >> 4) | (hi >> 6 << 4)], 1)
    return sc.double(), m.double()


def _decode(t, raw, in_dim):
    """The payload's weights [rows, in_dim] in f64."""
    n = raw.shape[0]
    if t == "F32":
        return raw.contiguous().view(torch.float32).double().reshape(-1, in_dim)
    if t == "Q8_0":
        w = raw[:, 2:].contiguous().view(torch.int8).double() * _half(raw[:, :2])[:, None]
    elif t in ("Q4_0", "Q5_0"):
        qs = raw[:, -16:].long()
        q = torch.cat([qs & 15, qs >> 4], 1)
        if t == "Q5_0":
            bits = torch.arange(8, device=raw.device)
            q = q | (raw[:, 2:6].long()[:, :, None] >> bits & 1).reshape(n, 32) << 4
        w = (q.double() - (8 if t == "Q4_0" else 16)) * _half(raw[:, :2])[:, None]
    elif t in ("Q4_K", "Q5_K"):
        sc, m = _k_scales(raw[:, 4:16])
        qs = raw[:, -128:].long().reshape(n, 4, 32)
        q = torch.stack([qs & 15, qs >> 4], 2).reshape(n, 8, 32)
        if t == "Q5_K":  # element l of sub-block s: bit s of byte 8 (s / 2) + l / 8
            s = torch.arange(8, device=raw.device)
            byte = (8 * (s // 2))[:, None] + torch.arange(4, device=raw.device)
            high = raw[:, 16:48].long()[:, byte] >> s[None, :, None] & 1
            q = q | high.repeat_interleave(8, 2) << 4
        w = (_half(raw[:, :2])[:, None] * sc)[:, :, None] * q - (_half(raw[:, 2:4])[:, None] * m)[:, :, None]
    else:  # Q6_K: halves of 128 elements in four 32-element quarters, a scale per 16
        ql, qh = raw[:, :128].long().reshape(n, 2, 2, 32), raw[:, 128:192].long().reshape(n, 2, 1, 32)
        low = torch.cat([ql & 15, ql >> 4], 2)
        two = torch.tensor([0, 2, 4, 6], device=raw.device)[None, None, :, None]
        q = (low | (qh >> two & 3) << 4).reshape(n, 16, 16).double() - 32
        scales = raw[:, 192:208].contiguous().view(torch.int8).double()
        w = q * (scales * _half(raw[:, 208:210])[:, None])[:, :, None]
    return w.reshape(-1, in_dim)


def _normal(seed, salt, *shape):
    return torch.randn(*shape, generator=_gen(seed, salt), device="cuda")


def _tokens(seed, salt, n, vocab):
    return torch.randint(0, vocab, (n,), generator=_gen(seed, salt), device="cuda").tolist()


# -------------------------------------------------------------------- shapes

def _dims(case):
    return case["heads"] * case["head_dim"], case["kv_heads"] * case["head_dim"]


def _projections(case):
    """(name, out, in) of a layer's matrices."""
    d, f = case["d"], case["ffn"]
    qd, kvd = _dims(case)
    return [("attn_q", qd, d), ("attn_k", kvd, d), ("attn_v", kvd, d), ("attn_output", d, qd), ("ffn_gate", f, d),
            ("ffn_up", f, d), ("ffn_down", d, f)]


def _model_tensors(case, seed):
    """(name, type, in, out, payload) of a model's tensors in turn: one matrix at a time is held."""
    t, d, qk = case["type"], case["d"], GEOMETRY[case["type"]][0]
    assert d % qk == 0
    yield "token_embd.weight", t, d, case["vocab"], _payload(t, case["vocab"], d, seed, 1)
    yield "output_norm.weight", "F32", d, 1, 1 + 0.1 * _normal(seed, 2, d)
    yield "output.weight", t, d, case["vocab"], _payload(t, case["vocab"], d, seed, 3)
    for i in range(case["layers"]):
        for k, name in enumerate(("attn_norm", "ffn_norm")):
            yield f"blk.{i}.{name}.weight", "F32", d, 1, 1 + 0.1 * _normal(seed, 100 * i + 10 + k, d)
        for k, (name, out_dim, in_dim) in enumerate(_projections(case)):
            yield f"blk.{i}.{name}.weight", t, in_dim, out_dim, _payload(t, out_dim, in_dim, seed, 100 * i + 20 + k)


# ------------------------------------------------------------------- prepare

_CTX = None


def _context():
    global _CTX
    if _CTX is None:
        _CTX = rf.Context(0)
    return _CTX


class _State:
    """What a pass needs.  A model has a context of its own (a context's ledger holds one model's charges); both are
    closed with the state."""

    def __init__(self, case):
        self.case, self.model = case, None
        self.ctx = rf.Context(0) if case["kind"] in ("prompt", "chat", "decode") else _context()

    def __del__(self):
        if self.model is not None:
            torch.cuda.synchronize()
            self.model.close()
            self.ctx.close()


def _config(case, context):
    return dict(vocab_size=case["vocab"], context_length=context, embedding_length=case["d"],
                block_count=case["layers"], feed_forward_length=case["ffn"], head_count=case["heads"],
                head_count_kv=case["kv_heads"], head_dim=case["head_dim"], rms_eps=EPS, rope_freq_base=THETA)


def prepare(case, seed):
    s, kind = _State(case), case["kind"]
    ctx = s.ctx
    if kind in ("matvec", "packed", "matmul"):
        n = case.get("tokens", 1)
        s.w = _payload(case["type"], case["out"], case["in"], seed, 1)
        s.x, s.y = _normal(seed, 2, n, case["in"]), torch.empty(n, case["out"], device="cuda")
        if kind != "matvec":
            raw, s.w = s.w, torch.empty_like(s.w)
            torch.cuda.synchronize()
            rf.pack_weights(ctx, getattr(GGML, case["type"]), raw.data_ptr(), case["out"], case["in"],
                            s.w.data_ptr(), raw_bytes=raw.numel())
            torch.cuda.synchronize()
    elif kind == "attention":
        qd, kvd = _dims(case)
        s.q, s.k, s.v = _normal(seed, 1, qd), _normal(seed, 2, kvd), _normal(seed, 3, kvd)
        s.kh, s.vh = _normal(seed, 4, case["positions"] - 1, kvd), _normal(seed, 5, case["positions"] - 1, kvd)
        s.out = torch.empty(qd, device="cuda")
    elif kind == "layer":
        qd, kvd = _dims(case)
        d, f = case["d"], case["ffn"]
        s.w = {name: _payload(case["type"], o, i, seed, 20 + k) for k, (name, o, i) in enumerate(_projections(case))}
        s.norms = [1 + 0.1 * _normal(seed, 10 + k, d) for k in range(2)]
        s.h = _normal(seed, 1, d)
        s.kh, s.vh = _normal(seed, 4, case["positions"] - 1, kvd), _normal(seed, 5, case["positions"] - 1, kvd)
        s.xn, s.q, s.k, s.v, s.a, s.o, s.h1, s.gate, s.up, s.act, s.h2 = (
            torch.empty(n, device="cuda") for n in (d, qd, kvd, kvd, qd, d, d, f, f, f, d))
    elif kind in ("prompt", "chat"):
        steps = case.get("steps", 0)
        s.tokens = _tokens(seed, 5, case["tokens"] + steps, case["vocab"])
        s.model = rf.GpuLlamaModel(ctx, _config(case, len(s.tokens)))
        for name, t, ne0, ne1, payload in _model_tensors(case, seed):
            s.model.set_tensor(name, getattr(GGML, t), ne0, ne1, payload.reshape(-1).view(torch.uint8).cpu().numpy())
    else:  # decode: the 8B model made in place by the package's generator
        cfg = dict(synthetic.CONFIG_8B)
        specs = synthetic.llama_specs(cfg, getattr(GGML, case["type"]), seed=seed)
        s.model = synthetic.build_device_model(ctx, cfg, specs, 512)
        s.model.use_graph(True)
        s.tokens = _tokens(seed, 5, case["tokens"], cfg["vocab_size"])
    torch.cuda.synchronize()  # the library's own stream does not wait for torch's
    return s


# ----------------------------------------------------------------------- run

def _run_layer(s):
    c, ctx, t = s.case, s.ctx, getattr(GGML, s.case["type"])
    shapes = {name: (o, i) for name, o, i in _projections(c)}
    d, f, n, kv, hd = c["d"], c["ffn"], c["heads"], c["kv_heads"], c["head_dim"]
    p = torch.Tensor.data_ptr

    def mv(name, x, y):
        rf.matvec(ctx, t, p(s.w[name]), shapes[name], p(x), p(y), w_bytes=s.w[name].numel())

    hist = c["positions"] - 1
    rf.rmsnorm(ctx, p(s.h), p(s.norms[0]), d, EPS, p(s.xn))
    mv("attn_q", s.xn, s.q)
    mv("attn_k", s.xn, s.k)
    mv("attn_v", s.xn, s.v)
    rf.apply_rope(ctx, p(s.q), p(s.k), hist, hd, n, kv, THETA)
    rf.attention_checked(ctx, p(s.q), p(s.kh), p(s.vh), p(s.k), p(s.v), hist, n, kv, hd, out=p(s.a))
    mv("attn_output", s.a, s.o)
    rf.add(ctx, p(s.h), p(s.o), d, p(s.h1))
    rf.rmsnorm(ctx, p(s.h1), p(s.norms[1]), d, EPS, p(s.xn))
    mv("ffn_gate", s.xn, s.gate)
    mv("ffn_up", s.xn, s.up)
    rf.swiglu(ctx, p(s.gate), p(s.up), f, p(s.act))
    mv("ffn_down", s.act, s.o)
    rf.add(ctx, p(s.h1), p(s.o), d, p(s.h2))
    return {"h": s.h2, "k": s.k, "v": s.v}


def run(s):
    c, ctx, kind = s.case, s.ctx, s.case["kind"]
    if kind in ("matvec", "packed", "matmul"):
        t, shape, n = getattr(GGML, c["type"]), (c["out"], c["in"]), s.w.numel()
        w, x, y = s.w.data_ptr(), s.x.data_ptr(), s.y.data_ptr()
        if kind == "matvec":
            rf.matvec(ctx, t, w, shape, x, y, w_bytes=n)
        elif kind == "packed":
            rf.matvec_packed(ctx, t, w, shape, x, y, w_bytes=n)
        else:
            rf.matmul_packed(ctx, t, w, shape, x, c["tokens"], y, w_bytes=n)
        return s.y
    if kind == "attention":
        rf.attention_checked(ctx, s.q.data_ptr(), s.kh.data_ptr(), s.vh.data_ptr(), s.k.data_ptr(), s.v.data_ptr(),
                             c["positions"] - 1, c["heads"], c["kv_heads"], c["head_dim"], out=s.out.data_ptr())
        return s.out
    if kind == "layer":
        return _run_layer(s)
    m = s.model
    m.reset()
    if kind == "prompt":
        return {"hidden": m.prefill(s.tokens, want_hidden=True), "logits": m.logits()}
    if kind == "chat":
        n = c["tokens"]
        m.prefill(s.tokens[:n])
        logits = [m.logits()]
        for pos in range(n, len(s.tokens)):
            m.forward(s.tokens[pos], pos)
            logits.append(m.logits())
        return logits
    m.prefill(s.tokens)
    m.decode_steps(c["steps"])
    return {"tokens": np.array(m.read_tokens(c["steps"]), np.int64), "logits": m.logits()}


# ----------------------------------------------------------- work, tolerance

def _matrix_bytes(t, out_dim, in_dim):
    qk, size = GEOMETRY[t]
    return out_dim * in_dim // qk * size


def _layer_work(c, tokens, before=0):
    """Bytes and operations of `tokens` tokens through one layer after `before` positions."""
    qd, kvd = _dims(c)
    rows = tokens * before + tokens * (tokens + 1) // 2  # (token, position) pairs
    weights = sum(_matrix_bytes(c["type"], o, i) for _, o, i in _projections(c))
    elements = sum(o * i for _, o, i in _projections(c))
    return {"bytes": weights + 8 * kvd * (before + tokens), "flops": 2 * elements * tokens + 4 * qd * rows}


def work(case):
    c, kind = case, case["kind"]
    if kind in ("matvec", "packed", "matmul"):
        n = c.get("tokens", 1)
        return {"bytes": _matrix_bytes(c["type"], c["out"], c["in"]) + 4 * n * (c["in"] + c["out"]),
                "flops": 2 * n * c["out"] * c["in"]}
    if kind == "attention":
        qd, kvd = _dims(c)
        return {"bytes": 8 * kvd * c["positions"] + 8 * qd, "flops": 4 * qd * c["positions"]}
    if kind == "layer":
        w = _layer_work(c, 1, c["positions"] - 1)
        return {"bytes": w["bytes"] + 8 * c["d"], "flops": w["flops"]}
    if kind == "decode":
        cfg = synthetic.CONFIG_8B
        c = dict(SHAPE_8B, type=c["type"], layers=cfg["block_count"], vocab=cfg["vocab_size"], tokens=c["tokens"],
                 steps=c["steps"])
    passes = [(c["tokens"], 0)] + [(1, c["tokens"] + k) for k in range(c.get("steps", 0))]
    total = {"bytes": 0, "flops": 0}
    for tokens, before in passes:
        w = _layer_work(c, tokens, before)
        total["bytes"] += c["layers"] * w["bytes"] + _matrix_bytes(c["type"], c["vocab"], c["d"]) + 4 * c["vocab"]
        total["flops"] += c["layers"] * w["flops"] + 2 * c["vocab"] * c["d"]
    return total


def tolerance(case):
    """f32 sums in another order: about four times the error measured against 64 bits.  A layer's steps, and a
    model's layers above all, carry a change of rounding on (the decode's is measured between two orders of its sums)."""
    return {"rel": {"matvec": 1e-6, "packed": 1e-6, "matmul": 1e-6, "attention": 4e-6, "layer": 4e-6, "prompt": 2e-5,
                    "chat": 2e-5, "decode": 5e-6}[case["kind"]]}


# --------------------------------------------------------------------- exact

def _libm(name, *args):
    f = getattr(ctypes.CDLL("libm.so.6"), name)
    f.restype, f.argtypes = ctypes.c_float, [ctypes.c_float] * len(args)
    return f(*args)


def _rope(x, positions, hd):
    """Half-split RoPE of x [tokens, heads, hd] f64; the angles are f32, theta ** (-2 i / hd) * position."""
    freq = np.array([_libm("powf", THETA, np.float32(-2.0) * np.float32(i) / np.float32(hd)) for i in range(hd // 2)],
                    np.float32)
    angle = torch.from_numpy((np.array(positions, np.float32)[:, None] * freq).astype(np.float64)).cuda()
    c, s = angle.cos()[:, None], angle.sin()[:, None]
    a, b = x[..., :hd // 2], x[..., hd // 2:]
    return torch.cat([a * c - b * s, a * s + b * c], -1)


def _attend(q, k, v, before):
    """q [tokens, heads, hd] at positions before.. over k, v [positions, kv heads, hd], causal, f64."""
    n, heads, hd = q.shape
    group = heads // k.shape[1]
    mask = torch.arange(k.shape[0], device="cuda")[None] > before + torch.arange(n, device="cuda")[:, None]
    out = torch.empty_like(q)
    for h in range(heads):
        kh, vh = k[:, h // group].contiguous(), v[:, h // group].contiguous()
        p = torch.softmax((q[:, h] @ kh.T / math.sqrt(hd)).masked_fill(mask, -math.inf), -1)
        out[:, h] = p @ vh
    return out


def _norm(x, w):
    return x / (x.square().mean(-1, keepdim=True) + EPS).sqrt() * w.double()


def _exact_layer(c, weight, norms, x, positions, kh, vh):
    """One layer over x [tokens, d]; kh, vh: [earlier positions, kv heads, hd].  Returns (x, new k, new v)."""
    n, kv, hd = c["heads"], c["kv_heads"], c["head_dim"]
    xn = _norm(x, norms[0])
    q = _rope((xn @ weight("attn_q").T).reshape(-1, n, hd), positions, hd)
    k = _rope((xn @ weight("attn_k").T).reshape(-1, kv, hd), positions, hd)
    v = (xn @ weight("attn_v").T).reshape(-1, kv, hd)
    a = _attend(q, torch.cat([kh, k]), torch.cat([vh, v]), kh.shape[0])
    x = x + a.reshape(-1, n * hd) @ weight("attn_output").T
    xn = _norm(x, norms[1])
    act = torch.nn.functional.silu(xn @ weight("ffn_gate").T) * (xn @ weight("ffn_up").T)
    return x + act @ weight("ffn_down").T, k, v


def exact(case, seed):
    c, kind = case, case["kind"]
    if kind == "decode":
        return None  # 32 layers of an 8B model in 64 bits
    if kind in ("matvec", "packed", "matmul"):
        raw = _payload(c["type"], c["out"], c["in"], seed, 1)
        x, per = _normal(seed, 2, c.get("tokens", 1), c["in"]).double(), raw.shape[0] // c["out"]
        return torch.cat([x @ _decode(c["type"], raw[r * per:(r + 8192) * per], c["in"]).T
                          for r in range(0, c["out"], 8192)], 1)
    if kind == "attention":
        n, kv, hd = c["heads"], c["kv_heads"], c["head_dim"]
        qd, kvd = _dims(c)
        rows = [torch.cat([_normal(seed, 4 + i, c["positions"] - 1, kvd), _normal(seed, 2 + i, kvd)[None]])
                for i in range(2)]
        k, v = (r.double().reshape(-1, kv, hd) for r in rows)
        return _attend(_normal(seed, 1, qd).double().reshape(1, n, hd), k, v, c["positions"] - 1).reshape(-1)
    kv, hd = c["kv_heads"], c["head_dim"]
    if kind == "layer":
        dims = {name: (k, o, i) for k, (name, o, i) in enumerate(_projections(c))}

        def weight(name):
            k, o, i = dims[name]
            return _decode(c["type"], _payload(c["type"], o, i, seed, 20 + k), i)

        norms = [1 + 0.1 * _normal(seed, 10 + k, c["d"]) for k in range(2)]
        kh, vh = (_normal(seed, s, c["positions"] - 1, kv * hd).double().reshape(-1, kv, hd) for s in (4, 5))
        h, k, v = _exact_layer(c, weight, norms, _normal(seed, 1, c["d"]).double()[None], [c["positions"] - 1], kh, vh)
        return {"h": h[0], "k": k.reshape(-1), "v": v.reshape(-1)}
    steps = c.get("steps", 0)
    tokens = _tokens(seed, 5, c["tokens"] + steps, c["vocab"])
    raws = {name: (t, ne0, raw) for name, t, ne0, _, raw in _model_tensors(c, seed)}

    def tensor(name):
        t, ne0, raw = raws[name + ".weight"]
        return raw if t == "F32" else _decode(t, raw, ne0)

    t, d, raw = raws["token_embd.weight"]
    per = raw.shape[0] // c["vocab"]
    x = _decode(t, raw.reshape(c["vocab"], per, -1)[torch.tensor(tokens, device="cuda")].flatten(0, 1), d)
    none = torch.empty(0, kv, hd, dtype=torch.float64, device="cuda")
    for i in range(c["layers"]):
        norms = [tensor(f"blk.{i}.{name}") for name in ("attn_norm", "ffn_norm")]
        x, _, _ = _exact_layer(c, lambda name: tensor(f"blk.{i}.{name}"), norms, x, range(len(tokens)), none, none)
    hidden = _norm(x[c["tokens"] - 1:], tensor("output_norm"))
    logits = hidden @ tensor("output").T
    return {"hidden": hidden[0], "logits": logits[0]} if kind == "prompt" else list(logits)
