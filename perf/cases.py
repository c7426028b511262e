"""The work that users of this package have it do, as cases that can be timed.

Three kinds, each through the public entry point its users call:

  attention  FASTMultiHeadAttention on (b, h, n, d) tensors, forward or forward + backward: the operator itself
  packed     qkv_attention on a fused (B, T, C) projection, forward + backward: one attention layer of a GPT block
  decode     ops.decode_step: one new token per head against the carried moment state
"""
import math

import torch

from fastmax_amd import FASTMultiHeadAttention, ops, qkv_attention

COEF = dict(normalize=True, temperature=1.0, a0=1.0, a1=1.0, a2=0.5, lim=1.0)
DTYPES = {"f32": torch.float32, "bf16": torch.bfloat16}


def _attention(name, dtype, b, h, n, d, mask, p, train, hkv=None, nk=None):
    case = dict(kind="attention", dtype=dtype, b=b, h=h, hkv=hkv or h, n=n, nk=nk or n, d=d, mask=mask, p=p, train=train)
    return dict(case, name=name) if name else case


def _packed(name, dtype, b, t, groups, q_per_kv, d, p):
    case = dict(kind="packed", dtype=dtype, b=b, h=groups * q_per_kv, hkv=groups, n=t, nk=t, d=d, mask=True, p=p, train=True)
    return dict(case, name=name) if name else case


def _decode(name, dtype, b, h, hkv, d, p):
    case = dict(kind="decode", dtype=dtype, b=b, h=h, hkv=hkv, n=1, nk=1, d=d, mask=True, p=p, train=False)
    return dict(case, name=name) if name else case


def listed():
    return [
        # a toy model or a unit test of a user's own: a handful of short heads of an odd size, where only launches
        # and host work count
        _attention("small-train-f32-d24", "f32", 2, 4, 61, 24, True, 2, True),
        # an encoder layer of moderate size: 8 x 8 heads x 1024 x 32, fp32, both directions
        _attention("encoder-train-f32-d32", "f32", 8, 8, 1024, 32, False, 2, True),
        # the same operator causal, over many short ragged sequences: 64 x 8 heads x 1000 x 32
        _attention("causal-train-f32-d32", "f32", 64, 8, 1000, 32, True, 2, True),
        # the headline: long causal fp32 sequences, 64 x 16 heads x 10000 x 64
        _attention("headline-train-f32-d64", "f32", 64, 16, 10000, 64, True, 2, True),
        # the headline shape at order 1
        _attention("headline-train-f32-d64-p1", "f32", 64, 16, 10000, 64, True, 1, True),
        # an encoder's forward pass without gradients: 64 x 8 heads x 1000 x 64, fp32
        _attention("encoder-eval-f32-d64", "f32", 64, 8, 1000, 64, False, 2, False),
        # long-context training in bf16: 16 x 32 heads x 16384 x 64
        _attention("long-train-bf16-d64", "bf16", 16, 32, 16384, 64, True, 2, True),
        # one attention layer of a GPT training step (batch 8 x 2048 tokens, 12 heads x 64, bf16) with RoPE on
        # the packed projection, at both orders
        _packed("gpt-layer-bf16-d64", "bf16", 8, 2048, 12, 1, 64, 2),
        _packed("gpt-layer-bf16-d64-p1", "bf16", 8, 2048, 12, 1, 64, 1),
        # a model with large heads and grouped keys and values, ragged length, training in bf16
        _attention("grouped-train-bf16-d128", "bf16", 2, 32, 2049, 128, True, 2, True, hkv=8),
        # the second piece of a prompt taken in two: 1000 new tokens behind 3000 earlier keys, no gradients
        _attention("prefill-piece-bf16-d64", "bf16", 4, 16, 1000, 64, True, 2, False, nk=4000),
        # serving: one token for each of 64 sequences, 16 heads x 64
        _decode("decode-f32-d64", "f32", 64, 16, 16, 64, 2),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _cost(case):
    """Seconds, roughly: a moment-form or score-form pass at the rates of the two element types."""
    w = work(case)
    flops = w["flops"]
    if case["d"] not in (32, 64) and case["p"] == 2:
        flops = _score_flops(case)   # these head dimensions take the form whose cost grows with n * nk
    return flops / (1.0e14 if case["dtype"] == "f32" else 4.0e14) + w["bytes"] / 2.0e12


def draw(rng):
    """A case of the ranges above: any kind, element type, direction, order and mask; 1 to 2048 heads, 1 to 16384
    tokens (from 16 with gradients: those of a single token are zero), head dimensions from 8 to 128."""
    top = max(_cost(c) for c in listed())
    while True:
        kind = rng.choice(["attention"] * 6 + ["packed"] * 2 + ["decode"])
        dtype = rng.choice(["f32", "bf16"])
        p = rng.choice([1, 2, 2])
        b = _log_int(rng, 1, 64)
        h = rng.choice([1, 2, 4, 8, 12, 16, 24, 32])
        hkv = rng.choice([h, h, h, max(1, h // 4)])
        if h % hkv:
            hkv = h
        d = rng.choice([32, 64, 64, 64, 64, rng.choice([8, 24, 40, 48, 80, 96, 128])])
        if kind == "decode":
            case = _decode(None, dtype, b, h, hkv, 32 if d < 64 else 64, p)
        elif kind == "packed":
            case = _packed(None, dtype, min(b, 16), _log_int(rng, 16, 8192), hkv, h // hkv, d, p)
        else:
            mask = rng.random() < 0.7
            train = rng.random() < 0.6
            n = _log_int(rng, 16 if train else 1, 16384)
            nk = n + _log_int(rng, 1, 4096) if mask and not train and rng.random() < 0.4 else n
            case = _attention(None, dtype, b, h, n, d, mask, p, train, hkv, nk)
        elements = b * h * max(case["n"], case["nk"]) * case["d"]
        if _cost(case) <= 0.6 * top and elements <= 64 * 16 * 10000 * 64:
            return case


class _State:
    pass


def prepare(case, seed):
    s = _State()
    s.case = dict(case)
    dtype, dev = DTYPES[case["dtype"]], torch.device("cuda")
    gen = torch.Generator(device=dev).manual_seed(seed)
    b, h, hkv, n, nk, d, p = (case[x] for x in ("b", "h", "hkv", "n", "nk", "d", "p"))

    def normal(*shape):
        return torch.randn(shape, generator=gen, device=dev, dtype=dtype)

    if case["kind"] == "attention":
        s.attention = FASTMultiHeadAttention()
        s.q, s.k, s.v = normal(b, h, n, d), normal(b, hkv, nk, d), normal(b, hkv, nk, d)
        if case["train"]:
            s.go = normal(b, h, n, d)
            s.inputs = [t.requires_grad_(True) for t in (s.q, s.k, s.v)]
    elif case["kind"] == "packed":
        s.groups, s.q_per_kv = hkv, h // hkv
        s.qkv = normal(b, n, hkv * (s.q_per_kv + 2) * d).requires_grad_(True)
        s.gy = normal(b, n, h * d)
        angle = torch.outer(torch.arange(n, device=dev, dtype=torch.float32),
                            10000.0 ** (-torch.arange(0, d, 2, device=dev, dtype=torch.float32) / d)).repeat(1, 2)
        s.cos, s.sin = angle.cos(), angle.sin()
    else:
        # every sequence has a few tokens behind it
        s.kw = dict(p=p)
        s.state = ops.new_state(b * hkv, d, p=p, dtype=dtype)
        for _ in range(8):
            s.q, s.k, s.v = 0.2 * normal(b * h, 1, d), 0.2 * normal(b * hkv, 1, d), normal(b * hkv, 1, d)
            ops.decode_step(s.state, s.q, s.k, s.v, **s.kw)
    return s


def run(s):
    case = s.case
    if case["kind"] == "attention":
        args = (None, case["mask"], 0.0, COEF["normalize"], COEF["temperature"], COEF["a0"], COEF["a1"], COEF["a2"],
                COEF["lim"], case["p"])
        if not case["train"]:
            with torch.no_grad():
                return s.attention(s.q, s.k, s.v, *args)
        o = s.attention(s.q, s.k, s.v, *args)
        dq, dk, dv = torch.autograd.grad(o, s.inputs, s.go)
        return {"o": o, "dq": dq, "dk": dk, "dv": dv}
    if case["kind"] == "packed":
        y = qkv_attention(s.qkv, s.cos, s.sin, s.groups, s.q_per_kv, case["d"], mask=True, p=case["p"], **COEF)
        dqkv, = torch.autograd.grad(y, [s.qkv], s.gy)
        return {"y": y, "dqkv": dqkv}
    o, den = ops.decode_step(s.state, s.q, s.k, s.v, **s.kw)
    return {"o": o, "den": den, "state": s.state}


def _score_flops(case):
    """Every visible score once: two products of length d forward, five backward."""
    lead = case["nk"] - case["n"]
    pairs = case["n"] * lead + case["n"] * (case["n"] + 1) // 2 if case["mask"] else case["n"] * case["nk"]
    return case["b"] * case["h"] * pairs * 2 * case["d"] * (7 if case["train"] else 2)


def work(case):
    """Flops: the cheaper of the score form and the moment form, whose features are 1, x_a and each unordered pair
    x_a x_b once, against d value columns and the denominator (one state build and one product forward; one more
    build and three products backward).  Bytes: each tensor once, a decode step's state in and out."""
    b, h, hkv, n, nk, d = (case[x] for x in ("b", "h", "hkv", "n", "nk", "d"))
    es = 4 if case["dtype"] == "f32" else 2
    feat = 1 + d + (d * (d + 1) // 2 if case["p"] == 2 else 0)
    if case["kind"] == "decode":
        state = b * hkv * feat * (d + 1)
        return {"bytes": 8 * state + es * b * d * (2 * h + 2 * hkv), "flops": 2 * state + 2 * b * h * feat * (d + 1)}
    query_side, key_side = (4, 4) if case["train"] else (2, 2)
    nbytes = es * b * d * (query_side * h * n + key_side * hkv * nk)
    builds = hkv * nk + (h * n if case["train"] else 0)
    products = h * n + (h * n + 2 * h * nk if case["train"] else 0)
    moments = b * 2 * feat * (d + 1) * (builds + products)
    return {"bytes": nbytes, "flops": min(moments, _score_flops(case))}


def tolerance(case):
    """Four times the largest error of any output (o, dq, dk, dv) of the listed cases against the same function in 64
    bits: relative 8.2e-7 and largest 8.3e-6 in fp32, 3.5e-3 and 0.22 in bf16 (8 bits of each output and of each
    score's polynomial; the largest error sits on gradients of the first positions' size against later rows')."""
    if case["dtype"] == "bf16":
        return {"rel": 1.4e-2, "max": 0.9}
    return {"rel": 3.3e-6, "max": 3.3e-5}
