"""The calls a program makes on this framework, as measurable cases.

Every case is one call (or, for `decoder`, one request) through the public
entry points of `catena_amd`, on inputs already resident on the device:

  runtime      Runtime.exec("matmul-2x2-via-mem"), output read back: the
               reference's own way in, a synchronous call of a small program
  f32_matmul   gemm_f32_exact: the stdlib matmul in the reference's order
  bf16_gemm    gemm_bf16: projections, from one decode row to whole prompts
  attn_decode  attn_decode_bf16: one query per (sequence, head) over a cache
  attn_causal  attn_causal_bf16: prompts, whole or after a cached prefix
  rows         softmax_f32 / rmsnorm_f32 / sum_f32 over many rows
  decoder      Decoder.prefill, the prompt's logits kept, Decoder.generate

`listed()` names the cases, `draw(rng)` gives more of the same ranges.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "catena-lang_amd"))
import catena_amd as ca  # noqa: E402

MATMUL_DECL = """
(def program matmul-2x2-via-mem :
  ([n m k.] {(cap.ref mem) (cap.ref mem) ({[.n] u64} :) ({[.m] u64} :) ({[.k] u64} :)
             ({({[.n] [.k]} *) u64} :) ({({[.k] [.m]} *) u64} :) ({({[.n] [.m]} *) u64} :)})
  -> ([n m k.] (cap.own mem)) = native)
"""


def listed():
    return [
        # the smallest call: a reference program on 256^3, synchronous, read back
        {"name": "runtime_matmul_256", "op": "runtime", "n": 256, "m": 256, "k": 256},
        # the stdlib matmul at an ordinary large size
        {"name": "f32_matmul_2048", "op": "f32_matmul", "n": 2048, "m": 2048, "k": 2048},
        # the same on sizes no tile divides
        {"name": "f32_matmul_ragged", "op": "f32_matmul", "n": 1000, "m": 1531, "k": 771},
        # the headline bf16 product
        {"name": "bf16_gemm_4096", "op": "bf16_gemm", "n": 4096, "m": 4096, "k": 4096, "out": "bf16"},
        # a prompt of 1000 tokens through a q / k / v projection (f32 out, as the decoder takes it)
        {"name": "bf16_gemm_ragged", "op": "bf16_gemm", "n": 1000, "m": 6144, "k": 2048, "out": "f32"},
        # one decode step of 8 sequences through a 4096 x 11008 projection
        {"name": "bf16_gemm_decode", "op": "bf16_gemm", "n": 8, "m": 11008, "k": 4096, "out": "bf16"},
        # one decode step of 64 sequences through the way back
        {"name": "bf16_gemm_batch64", "op": "bf16_gemm", "n": 64, "m": 4096, "k": 11008, "out": "bf16"},
        # decode attention of a full serving batch over 4096 cached positions
        {"name": "attn_decode_4096", "op": "attn_decode", "batch": 32, "heads": 32, "max_len": 4096, "ragged": False},
        # prompt attention of 8 x 512 tokens into a 640-position cache
        {"name": "attn_prefill_512", "op": "attn_causal", "batch": 8, "tq": 512, "heads": 16, "max_len": 640, "prefix": 0, "out": "bf16"},
        # one long prompt, a length no block divides
        {"name": "attn_prefill_2000", "op": "attn_causal", "batch": 1, "tq": 2000, "heads": 16, "max_len": 2048, "prefix": 0, "out": "bf16"},
        # attention-score rows through nn.softmax
        {"name": "softmax_rows", "op": "rows", "fold": "softmax", "rows": 4096, "n": 2048},
        # a request of three 333-token prompts and 16 greedy tokens each
        {"name": "decoder_request", "op": "decoder", "heads": 16, "ffn": 5632, "layers": 1, "vocab": 32000, "batch": 3, "t": 333, "steps": 16, "max_len": 640},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _size(rng, lo, hi, step):
    """Log-uniform in [lo, hi]; half of the draws on a multiple of `step`."""
    v = _log(rng, lo, hi)
    if rng.random() < 0.5:
        v = max(step, (v + step // 2) // step * step)
    return v


def draw(rng):
    op = rng.choice(["runtime", "f32_matmul", "bf16_gemm", "bf16_gemm", "attn_decode", "attn_causal", "rows", "decoder"])
    if op == "runtime":
        return {"op": op, **{s: _size(rng, 16, 512, 16) for s in ("n", "m", "k")}}
    if op == "f32_matmul":
        return {"op": op, **{s: _size(rng, 64, 2048, 64) for s in ("n", "m", "k")}}
    if op == "bf16_gemm":
        # rows: anything from one to whole prompts; widths: of a model, or any
        while True:
            n = _size(rng, 1, 4096, 16)
            m, k = ((128 * _log(rng, 2, 86) if rng.random() < 0.7 else _size(rng, 200, 11008, 8)) for _ in range(2))
            if n * m * k <= 4096**3:
                return {"op": op, "n": n, "m": m, "k": k, "out": rng.choice(["bf16", "f32"])}
    if op == "attn_decode":
        while True:
            c = {"op": op, "batch": _log(rng, 1, 64), "heads": rng.choice([4, 8, 16, 32]), "max_len": _size(rng, 64, 8192, 64), "ragged": rng.random() < 0.5}
            if c["batch"] * c["heads"] * c["max_len"] <= 32 * 32 * 4096:
                return c
    if op == "attn_causal":
        while True:
            tq = _log(rng, 2, 2000)
            prefix = rng.choice([0, 0, _log(rng, 16, 1024)])
            room = rng.choice([0, 48, 128])
            c = {"op": op, "batch": _log(rng, 1, 8), "tq": tq, "heads": rng.choice([4, 8, 16, 32]), "max_len": tq + prefix + room, "prefix": prefix, "out": rng.choice(["bf16", "f32"])}
            if c["batch"] * c["heads"] * tq * (tq + 2 * prefix) <= 16 * 2000 * 2000:
                return c
    if op == "rows":
        fold = rng.choice(["softmax", "rmsnorm", "sum"])
        while True:
            rows, n = _log(rng, 1, 16384), _size(rng, 32, 8192, 32)
            n = (n + 3) // 4 * 4 if fold == "rmsnorm" else n
            if rows * n <= 4096 * 2048:
                return {"op": op, "fold": fold, "rows": rows, "n": n}
    t, steps = _size(rng, 8, 600, 16), rng.choice([0, 4, 16])
    while True:
        batch = _log(rng, 1, 32)
        if batch * t <= 2048:
            break
    return {"op": op, "heads": rng.choice([4, 8, 16]), "ffn": 64 * rng.randint(8, 88), "layers": rng.choice([1, 1, 2]), "vocab": 8 * _log(rng, 128, 4000), "batch": batch, "t": t, "steps": steps,
            "max_len": t + steps + rng.choice([0, 24, 128])}


# ------------------------------------------------------------------ inputs

def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _normal(g, *shape, dtype=torch.float32, scale=1.0):
    return torch.randn(*shape, generator=g, device="cuda", dtype=torch.float32).mul_(scale).to(dtype)


def _lens(case, g):
    """Valid positions per sequence: the whole cache, or anything from one on."""
    if case["op"] == "attn_causal":
        lens = torch.full((case["batch"],), case["tq"] + case["prefix"], device="cuda", dtype=torch.int64)
    elif case["ragged"]:
        lens = torch.randint(1, case["max_len"] + 1, (case["batch"],), generator=g, device="cuda")
    else:
        lens = torch.full((case["batch"],), case["max_len"], device="cuda", dtype=torch.int64)
    return lens


def _inputs(case, seed):
    """The case's inputs as torch tensors on the device, from the seed alone."""
    g, op = _gen(seed), case["op"]
    bf16 = torch.bfloat16
    if op in ("runtime", "f32_matmul"):
        return {"a": _normal(g, case["n"], case["k"]), "b": _normal(g, case["k"], case["m"], scale=case["k"] ** -0.5)}
    if op == "bf16_gemm":
        # normalized activations against weights of a 0.02 spread
        return {"a": _normal(g, case["n"], case["k"], dtype=bf16), "b": _normal(g, case["k"], case["m"], dtype=bf16, scale=0.02)}
    if op in ("attn_decode", "attn_causal"):
        b, h, l = case["batch"], case["heads"], case["max_len"]
        return {"q": _normal(g, b, case.get("tq", 1), h, 128, dtype=bf16), "k": _normal(g, b, h, l, 128, dtype=bf16),
                "v": _normal(g, b, h, l, 128, dtype=bf16), "lens": _lens(case, g)}
    if op == "rows":
        return {"x": _normal(g, case["rows"], case["n"], scale=3.0 if case["fold"] == "softmax" else 1.0)}
    d, f, v = 128 * case["heads"], case["ffn"], case["vocab"]
    w = {"tokens": torch.randint(0, v, (case["batch"], case["t"]), generator=g, device="cuda"),
         "embed": _normal(g, v, d, dtype=bf16, scale=0.02), "lm": _normal(g, d, v, dtype=bf16, scale=0.02)}
    for i in range(case["layers"]):
        for name, shape in (("qkv", (d, 3 * d)), ("o", (d, d)), ("gu", (d, 2 * f)), ("down", (f, d))):
            w["%s%d" % (name, i)] = _normal(g, *shape, dtype=bf16, scale=0.02)
    return w


def _load(dst, t):
    """Checkpoint tensor `t` into a decoder tensor."""
    assert dst.len == t.numel() * t.element_size() and dst.len % 16 == 0
    ca.copy_bytes(dst.data, t.data_ptr(), dst.len)


def prepare(case, seed):
    ca.init(0)
    x, op = _inputs(case, seed), case["op"]
    if op == "runtime":
        a, b = (ca.Buffer.from_array(x[s].cpu().numpy()) for s in "ab")
        n, m, k = case["n"], case["m"], case["k"]
        args = [ca.Value.mem(a.mem), ca.Value.mem(b.mem)] + [ca.Value.u64(v) for v in (n, m, k, n * k, k * m, n * m)]
        return {"case": case, "rt": ca.Runtime([MATMUL_DECL]), "args": args, "held": (a, b)}
    s = {"case": case, **x}
    dev = {"device": "cuda"}
    if op == "f32_matmul":
        s["out"] = torch.zeros(case["n"], case["m"], **dev)
    elif op == "bf16_gemm":
        s["out"] = torch.zeros(case["n"], case["m"], dtype=torch.float32 if case["out"] == "f32" else torch.bfloat16, **dev)
    elif op in ("attn_decode", "attn_causal"):
        s["lens"] = x["lens"].to(torch.int32)
        s["out"] = torch.zeros(x["q"].shape, dtype=torch.bfloat16 if case.get("out") == "bf16" else torch.float32, **dev)
    elif op == "rows":
        s["out"] = torch.zeros((case["rows"],) if case["fold"] == "sum" else x["x"].shape, **dev)
    else:
        b = case["batch"]
        dec = ca.Decoder(128 * case["heads"], case["heads"], case["ffn"], case["layers"], case["vocab"], b, case["max_len"])
        torch.cuda.synchronize()
        _load(dec.tensor(ca.DEC_EMBED), x["embed"])
        _load(dec.tensor(ca.DEC_W_LM), x["lm"])
        for i in range(case["layers"]):
            for which, name in ((ca.DEC_W_QKV, "qkv"), (ca.DEC_W_O, "o"), (ca.DEC_W_GU, "gu"), (ca.DEC_W_DOWN, "down")):
                _load(dec.tensor(which, i), x["%s%d" % (name, i)])
        ca.synchronize()
        logits = 2 if case["steps"] else 1
        s = {"case": case, "dec": dec, "tokens": x["tokens"].to(torch.int32), "next": torch.zeros(b, dtype=torch.int32, **dev),
             "out": torch.zeros(case["steps"], b, dtype=torch.int32, **dev), "logits": torch.zeros(logits, b, case["vocab"], **dev)}
    torch.cuda.synchronize()
    return s


# ------------------------------------------------------------------ the calls

def run(s):
    c = s["case"]
    op = c["op"]
    if op == "runtime":
        [res] = s["rt"].exec("matmul-2x2-via-mem", s["args"], 1)
        out = ca.mem_to_array(res.get(), np.float32)
        ca.mem_free(res.get())
        return out
    if op == "f32_matmul":
        ca.gemm_f32_exact(s["a"].data_ptr(), s["b"].data_ptr(), s["out"].data_ptr(), c["n"], c["m"], c["k"])
    elif op == "bf16_gemm":
        ca.gemm_bf16(s["a"].data_ptr(), s["b"].data_ptr(), s["out"].data_ptr(), c["n"], c["m"], c["k"], c["out"] == "f32")
    elif op == "attn_decode":
        ca.attn_decode_bf16(s["q"].data_ptr(), s["k"].data_ptr(), s["v"].data_ptr(), s["lens"].data_ptr(), s["out"].data_ptr(),
                            c["batch"], c["heads"], c["max_len"], 128, 128**-0.5)
    elif op == "attn_causal":
        ca.attn_causal_bf16(s["q"].data_ptr(), s["k"].data_ptr(), s["v"].data_ptr(), s["lens"].data_ptr(), s["out"].data_ptr(),
                            c["batch"], c["tq"], c["heads"], c["max_len"], 128, 128**-0.5, c["out"] == "f32")
    elif op == "rows":
        {"softmax": ca.softmax_f32, "rmsnorm": ca.rmsnorm_f32, "sum": ca.sum_f32}[c["fold"]](s["x"].data_ptr(), s["out"].data_ptr(), c["rows"], c["n"])
    else:
        dec, logits = s["dec"], s["logits"]
        nbytes = logits[0].numel() * 4
        dec.prefill(s["tokens"].data_ptr(), c["batch"], c["t"], s["next"].data_ptr())
        ca.copy_bytes(logits.data_ptr(), dec.tensor(ca.DEC_LOGITS).data, nbytes)
        if not c["steps"]:
            return {"prompt_logits": logits[0], "next": s["next"]}
        dec.generate(c["steps"], s["out"].data_ptr())
        ca.copy_bytes(logits.data_ptr() + nbytes, dec.tensor(ca.DEC_LOGITS).data, nbytes)
        return {"prompt_logits": logits[0], "next": s["next"], "logits": logits[1], "out": s["out"]}
    return s["out"]


# ------------------------------------------------------------------ what a call cannot do without

def _positions(case):
    """Total (query, key) pairs of one head of one sequence, and cached rows read."""
    tq, n = case["tq"], case["tq"] + case["prefix"]
    return tq * n - tq * (tq - 1) // 2, n


def work(case):
    op = case["op"]
    if op in ("runtime", "f32_matmul"):
        n, m, k = case["n"], case["m"], case["k"]
        return {"bytes": 4 * (n * k + k * m + n * m), "flops": 2 * n * m * k}
    if op == "bf16_gemm":
        n, m, k = case["n"], case["m"], case["k"]
        return {"bytes": 2 * (n * k + k * m) + (4 if case["out"] == "f32" else 2) * n * m, "flops": 2 * n * m * k}
    if op == "attn_decode":
        pairs, share = case["batch"] * case["heads"], 0.5 if case["ragged"] else 1.0  # ragged lengths: half the cache on average
        rows = pairs * case["max_len"] * share
        return {"bytes": int(rows * 512 + pairs * 128 * 6), "flops": int(rows * 512)}
    if op == "attn_causal":
        bh = case["batch"] * case["heads"]
        pairs, rows = _positions(case)
        return {"bytes": bh * (rows * 512 + case["tq"] * 128 * (2 + (2 if case["out"] == "bf16" else 4))), "flops": bh * pairs * 512}
    if op == "rows":
        x = 4 * case["rows"] * case["n"]
        return {"bytes": x + 4 * case["rows"] if case["fold"] == "sum" else 2 * x, "flops": 0}
    d, f, v, b, t, steps = 128 * case["heads"], case["ffn"], case["vocab"], case["batch"], case["t"], case["steps"]
    block = 4 * d * d + 3 * d * f
    weights = 2 * (case["layers"] * block + d * v)
    rows = b * (t + steps)
    cache = case["layers"] * b * case["heads"] * 512 * sum(range(t + 1, t + steps + 1))
    attn = case["layers"] * b * case["heads"] * 512 * (t * (t + 1) // 2 + sum(range(t + 1, t + steps + 1)))
    return {"bytes": (1 + steps) * (weights + 4 * b * v) + cache, "flops": 2 * case["layers"] * rows * block + 2 * b * (1 + steps) * d * v + attn}


def tolerance(case):
    """The f32 programs and the attention are defined bit by bit (one order of
    one operation after the other), so they do not move at all.  A bf16
    product is a sum in some order with one rounding at the end."""
    if case["op"] == "bf16_gemm":
        return {"rel": 7e-3, "max": 0.02} if case["out"] == "bf16" else {"rel": 2e-6, "max": 3e-5}
    if case["op"] == "decoder":
        return {"rel": 0.02, "max": 0.2, "differ": 0.0}
    return "exact"


# ------------------------------------------------------------------ the same in 64 bits

def _bits(x):
    return float(np.array([x], np.uint32).view(np.float32)[0])


# math.exp-approx and math.sqrt of the stdlib are what they are by definition, a
# cubic with its own coefficients after a range reduction (2e-3 from e^x) and six
# Newton steps (not converged for small arguments): in 64 bits here, with the
# stdlib's constants.
_C0, _C1, _C2, _C3 = (_bits(x) for x in (0x3F7FF8FC, 0x3F809C7E, 0x3EEF1187, 0x3E738A8B))
_INV_LN2, _LN2 = _bits(0x3FB8AA3B), _bits(0x3F317200) + _bits(0x35BFBE8E)
_RMS_EPS = _bits(0x3727C5AC)


def _exp(x):
    m = x.abs().clamp(max=200.0)  # beyond it f32 has only 0 and infinity
    k = torch.round(m * _INV_LN2)
    r = m - k * _LN2
    y = torch.ldexp(_C0 + r * (_C1 + r * (_C2 + r * _C3)), k)
    return torch.where(x < 0, 1 / y, y)


def _sqrt(x):
    g = x.clamp(min=1.0)
    for _ in range(6):
        g = (g + x / g) * 0.5
    return g


def _softmax(x):
    e = _exp(x - x.amax(-1, keepdim=True))
    return e / e.sum(-1, keepdim=True)


def _rms(x):
    return x / _sqrt(x.square().mean(-1, keepdim=True) + _RMS_EPS)


def _attention(q, k, v, lens, causal_tq):
    """q [tq][128], k / v [L][128] of one head in 64 bits; query i sees lens - (tq - 1 - i) positions."""
    n = int(lens)
    s = (q @ k[:n].T.contiguous()) * 128**-0.5
    if causal_tq > 1:
        i, j = torch.arange(causal_tq, device="cuda")[:, None], torch.arange(n, device="cuda")[None]
        s.masked_fill_(j >= n - (causal_tq - 1 - i), -math.inf)
    return _softmax(s) @ v[:n]


def _prompt_logits(case, x):
    """The decoder's prefill without its roundings: the logits of each prompt's last token."""
    b, t, h, d, f = case["batch"], case["t"], case["heads"], 128 * case["heads"], case["ffn"]
    w = {name: v.double() for name, v in x.items() if name != "tokens"}
    r = w["embed"][x["tokens"].reshape(-1)]
    freq = 10000.0 ** (-torch.arange(64, device="cuda", dtype=torch.float64) / 64)
    theta = torch.arange(t, device="cuda", dtype=torch.float64)[:, None] * freq
    cos, sin = theta.cos()[None, :, None], theta.sin()[None, :, None]

    def rope(y):
        y1, y2 = y[..., :64], y[..., 64:]
        return torch.cat([y1 * cos - y2 * sin, y2 * cos + y1 * sin], -1)

    for i in range(case["layers"]):
        q, k, v = (_rms(r) @ w["qkv%d" % i]).view(b, t, 3, h, 128).unbind(2)
        q, k = rope(q), rope(k)
        o = torch.stack([torch.stack([_attention(q[s, :, j], k[s, :, j], v[s, :, j], t, t) for j in range(h)], 1) for s in range(b)])
        r = r + o.reshape(b * t, d) @ w["o%d" % i]
        gu = (_rms(r) @ w["gu%d" % i]).view(b * t, f // 64, 2, 64)
        r = r + (gu[:, :, 0] / (1 + _exp(-gu[:, :, 0])) * gu[:, :, 1]).reshape(b * t, f) @ w["down%d" % i]
    return _rms(r.view(b, t, d)[:, -1]) @ w["lm"]


def exact(case, seed):
    x, op = _inputs(case, seed), case["op"]
    if op in ("runtime", "f32_matmul", "bf16_gemm"):
        y = x["a"].double() @ x["b"].double()
        return y.reshape(-1).cpu().numpy() if op == "runtime" else y
    if op in ("attn_decode", "attn_causal"):
        q, tq, out = x["q"], x["q"].shape[1], torch.zeros(x["q"].shape, device="cuda", dtype=torch.float64)
        for b in range(case["batch"]):
            for h in range(case["heads"]):
                out[b, :, h] = _attention(q[b, :, h].double(), x["k"][b, h].double(), x["v"][b, h].double(), x["lens"][b], tq)
        return out
    if op == "rows":
        v = x["x"].double()
        return _softmax(v) if case["fold"] == "softmax" else _rms(v) if case["fold"] == "rmsnorm" else v.sum(-1)
    logits = _prompt_logits(case, x)
    # what follows the first greedy choice depends on it, and has no value of its own
    return {"prompt_logits": logits, "next": None, **({"logits": None, "out": None} if case["steps"] else {})}
