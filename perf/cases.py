"""Performance cases of the quantized-matmul library: what a program that uses
it calls, from one GEMV of a decode step to a long prompt through a decoder
block. Each case goes through the Python mirror (``smegemm``) on device
tensors, on torch's current stream.

A case is a dict: ``op`` (the call), its sizes, and the options that matter to
it. ``listed()`` names the fixed ones, ``draw()`` gives others of the same
ranges, ``prepare`` makes a program's state (weights packed once, inputs,
outputs), ``run`` is one pass, ``exact`` the same result in 64 bits.
"""
import math
import os
import sys

import numpy as np
import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "sme-gemm_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import smegemm as smg  # noqa: E402

DEV = "cuda:0"

# The decoder layer of the block cases: Llama-style, grouped-query attention,
# SwiGLU, RMSNorm, NeoX RoPE.
BLOCK = dict(d=4096, heads=32, kv_heads=8, hd=128, ffn=14336)
THETA, EPS = 10000.0, 1e-5


def listed():
    return [
        # A projection of a small model (K = 384 to 1536 outputs), one token:
        # the smallest call, all latency.
        dict(name="q4_decode_small", op="q4", m=1, n=1536, k=384, bf16=False, affine=False, ep="none"),
        # A 4096-wide model's square projection, one token.
        dict(name="q4_decode", op="q4", m=1, n=4096, k=4096, bf16=False, affine=False, ep="none"),
        # A 1-bit model's up projection with bias and activation, one token.
        dict(name="q1_decode", op="lowbit", bits=1, m=1, n=14336, k=4096, ep="bias_silu"),
        # One generated token through a whole decoder layer, 4096 tokens in.
        dict(name="block_decode", op="block", rows=1, past=4096, **BLOCK),
        # A long prompt through the same layer, from an empty cache.
        dict(name="block_prefill", op="block", rows=2048, past=0, **BLOCK),
        # A prompt's up projection: Q4 weights, column scale, bias, activation.
        dict(name="q4_prefill", op="q4", m=512, n=14336, k=4096, bf16=False, affine=False, ep="scale_bias_silu"),
        # A batch of sequences decoding together, or a short prompt: bf16
        # activations, Q4_1 weights, ragged rows and columns.
        dict(name="q4_batch", op="q4", m=77, n=11003, k=4096, bf16=True, affine=True, ep="bias_silu"),
        # A 2-bit (ternary) model's prompt on the bit-exact int8 path.
        dict(name="q2_prefill", op="lowbit", bits=2, m=512, n=11008, k=4096, ep="none"),
        # A 1-bit model's prompt on the f16-weight path.
        dict(name="q1_mopa_prefill", op="mopa", bits=1, m=512, n=14336, k=4096, ep="bias_silu"),
        # A dense layer prepacked once, through the builder.
        dict(name="gemm_packed", op="packed", m=4096, n=4096, k=4096, bf16=False, ep="bias_gelu"),
        # An ordinary strided GEMM call: column-major B, added into C.
        dict(name="gemm_strided", op="strided", m=1000, n=3000, k=2000, bf16=True, bcol=True, alpha=0.5),
        # A prompt chunk's attention after 4096 cached tokens.
        dict(name="attend_causal", op="attend", rows=512, start=4096, heads=32, kv_heads=8, hd=128),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _width(rng, lo, hi, odd):
    """A layer width: a multiple of 128 as models have, or (odd) any size."""
    x = _log(rng, lo, hi)
    return x if odd else max(128, x // 128 * 128)


# The most a drawn case costs (operations): under the largest listed one.
_MOST = 6e11


def draw(rng):
    op = rng.choice(["q4", "q4", "lowbit", "lowbit", "mopa", "packed", "strided", "attend", "block"])
    while True:
        odd = rng.random() < 0.35
        if op == "q4":
            c = dict(op=op, m=rng.choice([1, 1, _log(rng, 2, 32), _log(rng, 33, 4096), _log(rng, 33, 4096)]),
                     n=_width(rng, 384, 32768, odd), k=max(32, _width(rng, 256, 14336, odd) // 32 * 32),
                     bf16=rng.random() < 0.4, affine=rng.random() < 0.4,
                     ep=rng.choice(["none", "bias_silu", "scale_bias_silu"]))
        elif op == "lowbit":
            c = dict(op=op, bits=rng.choice([1, 2]), m=rng.choice([1, _log(rng, 2, 8), _log(rng, 9, 1024),
                                                                   _log(rng, 9, 1024)]),
                     n=_width(rng, 512, 16384, odd), k=_width(rng, 512, 8192, odd),
                     ep=rng.choice(["none", "bias_silu"]))
        elif op == "mopa":
            c = dict(op=op, bits=rng.choice([1, 2]), m=_log(rng, 16, 2048), n=_width(rng, 512, 16384, odd),
                     k=_width(rng, 512, 8192, odd), ep=rng.choice(["none", "bias_silu"]))
        elif op == "packed":
            c = dict(op=op, m=_log(rng, 32, 4096), n=_width(rng, 256, 8192, odd), k=_width(rng, 256, 8192, odd),
                     bf16=rng.random() < 0.5, ep=rng.choice(["none", "bias_gelu"]))
        elif op == "strided":
            c = dict(op=op, m=_log(rng, 32, 4096), n=_width(rng, 256, 4096, odd), k=_width(rng, 256, 4096, odd),
                     bf16=rng.random() < 0.5, bcol=rng.random() < 0.5, alpha=rng.choice([0.0, 0.5]))
        elif op == "attend":
            h, kvh, hd = rng.choice([(32, 8, 128), (12, 12, 64), (16, 8, 128), (20, 20, 64), (32, 32, 128)])
            c = dict(op=op, rows=rng.choice([1, _log(rng, 2, 31), _log(rng, 32, 2048), _log(rng, 32, 2048)]),
                     start=rng.choice([0, _log(rng, 16, 8192)]), heads=h, kv_heads=kvh, hd=hd)
        else:
            d, h, kvh, hd, ffn = rng.choice([(2048, 16, 8, 128, 6144), (4096, 32, 8, 128, 14336),
                                             (1024, 16, 4, 64, 2816)])
            c = dict(op=op, rows=rng.choice([1, _log(rng, 2, 31), _log(rng, 32, 1024)]),
                     past=rng.choice([0, _log(rng, 16, 8192)]), d=d, heads=h, kv_heads=kvh, hd=hd, ffn=ffn)
        if work(c)["flops"] <= _MOST:
            return c


# ---- inputs -------------------------------------------------------------------

class _Rng:
    """Seeded inputs, made on the GPU."""

    def __init__(self, seed):
        self.g = torch.Generator(device=DEV).manual_seed(seed)

    def normal(self, *shape):
        return torch.randn(shape, generator=self.g, device=DEV)

    def uniform(self, lo, hi, *shape):
        return torch.rand(shape, generator=self.g, device=DEV) * (hi - lo) + lo

    def ints(self, hi, *shape):
        return torch.randint(0, hi, shape, generator=self.g, device=DEV, dtype=torch.uint8)


def _half(x, bf16=False):
    return x.to(torch.bfloat16 if bf16 else torch.float16)


def _np16(x):
    return x.cpu().view(torch.int16).numpy().view(np.uint16)


def _nbk(k, block):
    return -(-k // block)


def _q4_arrays(r, n, k, affine, lo=0.005, hi=0.02):
    """Codes (two a byte, row-major k x n, low nibble first), a scale and
    perhaps a min for each column's block of 32."""
    q = r.ints(256, (k * n + 1) // 2)
    sc = _half(r.uniform(lo, hi, n, _nbk(k, 32)))
    mn = _half(r.uniform(-0.1, 0.1, n, _nbk(k, 32))) if affine else None
    return q, sc, mn


def _q4_weights(arrays, n, k):
    q, sc, mn = arrays
    if mn is None:
        return smg.Q4Weights(q.cpu().numpy(), _np16(sc), n, k)
    return smg.Q4Weights.with_params(q.cpu().numpy(), _np16(sc), _np16(mn), n, k, smg.Q4Params(32).affine())


def _q4_dense(arrays, n, k):
    """The weights in 64 bits, k x n."""
    q, sc, mn = arrays
    nib = torch.stack([q & 15, q >> 4], 1).reshape(-1)[: k * n].to(torch.int8)
    w = torch.where(nib < 8, nib, nib - 16).double().reshape(k, n)
    rep = lambda s: s.double().t().repeat_interleave(32, 0)[:k]  # noqa: E731
    w *= rep(sc)
    if mn is not None:
        w += rep(mn)
    return w


def _lowbit_arrays(r, bits, n, k):
    """Ternary codes (four a byte, row-major k x n) or signs (eight a byte,
    each output's K together), a scale for each column's block of 128."""
    sc = _half(r.uniform(0.01, 0.05, n, _nbk(k, 128)))
    if bits == 1:
        return r.ints(256, (k * n + 7) // 8), sc
    c = r.ints(3, -(-k * n // 4), 4)
    return c[:, 0] | (c[:, 1] << 2) | (c[:, 2] << 4) | (c[:, 3] << 6), sc


def _lowbit_weights(arrays, bits, n, k):
    q, sc = arrays
    if bits == 1:
        return smg.Q1Weights(q.cpu().numpy(), _np16(sc), smg.WeightLayout.OutIn, n, k, 128)
    return smg.Q2Weights(q.cpu().numpy(), _np16(sc), n, k, smg.Q2Params(128))


def _lowbit_codes(q, bits, n, k):
    """The codes' values in 64 bits, k x n."""
    if bits == 1:
        b = torch.stack([(q >> i) & 1 for i in range(8)], 1).reshape(-1)[: k * n]
        return (2.0 * b.double() - 1.0).reshape(n, k).t()
    c = torch.stack([(q >> (2 * i)) & 3 for i in range(4)], 1).reshape(-1)[: k * n]
    return torch.tensor([-1.0, 0.0, 1.0, 0.0], device=DEV, dtype=torch.float64)[c.long()].reshape(k, n)


def _ep_arrays(r, ep, n, bf16):
    s = _half(r.uniform(0.5, 1.5, n), bf16) if "scale" in ep else None
    b = _half(0.1 * r.normal(n), bf16) if "bias" in ep else None
    return s, b


def _ep_build(target, ep, arrays):
    s, b = arrays
    if s is not None:
        target = target.mul_col(s)
    if b is not None:
        target = target.add_col(b)
    if ep.endswith("silu"):
        target = target.silu()
    elif ep.endswith("gelu"):
        target = target.gelu()
    return target


def _ep_exact(x, ep, arrays):
    s, b = arrays
    if s is not None:
        x = x * s.double()
    if b is not None:
        x = x + b.double()
    if ep.endswith("silu"):
        x = x * torch.sigmoid(x)
    elif ep.endswith("gelu"):
        x = torch.nn.functional.gelu(x, approximate="tanh")
    return x


def _inputs(case, seed):
    """Everything `case` is computed from: the same for prepare and exact."""
    r, op, i = _Rng(seed), case["op"], {}
    if op in ("q4", "lowbit", "mopa"):
        m, n, k, bf16 = case["m"], case["n"], case["k"], case.get("bf16", False)
        i["w"] = _q4_arrays(r, n, k, case["affine"]) if op == "q4" else _lowbit_arrays(r, case["bits"], n, k)
        i["a"] = _half(r.normal(m, k), bf16)
        i["ep"] = _ep_arrays(r, case["ep"], n, bf16)
    elif op == "packed":
        m, n, k, bf16 = case["m"], case["n"], case["k"], case["bf16"]
        i["a"] = _half(r.normal(m, k), bf16)
        i["b"] = _half(r.normal(k, n) / math.sqrt(k), bf16)
        i["ep"] = _ep_arrays(r, case["ep"], n, bf16)
    elif op == "strided":
        m, n, k, bf16 = case["m"], case["n"], case["k"], case["bf16"]
        i["a"] = _half(r.normal(m, k), bf16)
        i["b"] = _half(r.normal(n, k) / math.sqrt(k) if case["bcol"] else r.normal(k, n) / math.sqrt(k), bf16)
        i["c"] = _half(r.normal(m, n), bf16)
    elif op == "attend":
        ql, ld, ln = case["heads"] * case["hd"], case["kv_heads"] * case["hd"], case["start"] + case["rows"]
        i["q"] = r.normal(case["rows"], ql)
        i["k"], i["v"] = _half(r.normal(ln, ld)), _half(r.normal(ln, ld))
    else:
        d, ffn, hd = case["d"], case["ffn"], case["hd"]
        ql, ld = case["heads"] * hd, case["kv_heads"] * hd
        for name, n, k in (("qkv", ql + 2 * ld, d), ("out", d, ql), ("gate", ffn, d), ("up", ffn, d), ("down", d, ffn)):
            i[name] = _q4_arrays(r, n, k, False, 0.0025, 0.0075)
        i["n1"], i["n2"] = r.uniform(0.9, 1.1, d), r.uniform(0.9, 1.1, d)
        i["k"], i["v"] = _half(r.normal(case["past"], ld)), _half(r.normal(case["past"], ld))
        i["x"] = r.normal(case["rows"], d)
    return i


def prepare(case, seed):
    i, op = _inputs(case, seed), case["op"]
    s = dict(case=case)
    if op in ("q4", "lowbit", "mopa"):
        m, n, k = case["m"], case["n"], case["k"]
        s["w"] = _q4_weights(i["w"], n, k) if op == "q4" else _lowbit_weights(i["w"], case["bits"], n, k)
        s["a"], s["c"] = i["a"], torch.empty(m, n, dtype=i["a"].dtype, device=DEV)
        s["ep"] = _ep_build(smg.Epilogue(case.get("bf16", False)), case["ep"], i["ep"])
    elif op == "packed":
        pack = smg.prepack_bf16 if case["bf16"] else smg.prepack_f16
        s["w"] = pack(_np16(i["b"]), case["n"], case["k"])
        s["a"], s["c"] = i["a"], torch.empty(case["m"], case["n"], dtype=i["a"].dtype, device=DEV)
        s["ep"] = i["ep"]
    elif op == "strided":
        s.update(i)
    elif op == "attend":
        cache = smg.KvCache(case["heads"], case["kv_heads"], case["hd"], case["start"] + case["rows"])
        cache.extend(i["k"], i["v"])
        s["cache"], s["q"], s["out"] = cache, i["q"], torch.empty_like(i["q"])
    else:
        d, ffn, heads, kvh, hd = (case[x] for x in ("d", "ffn", "heads", "kv_heads", "hd"))
        lin = lambda x, n, k: smg.Linear(_q4_weights(i[x], n, k))  # noqa: E731
        attn = smg.SelfAttention(lin("qkv", (heads + 2 * kvh) * hd, d), lin("out", d, heads * hd), heads, kvh, hd,
                                 THETA)
        up = smg.GatedLinear.from_q4(_q4_weights(i["gate"], ffn, d), _q4_weights(i["up"], ffn, d), smg.Gate.Silu)
        s["block"] = smg.Block(smg.Norm.rms(i["n1"].cpu().numpy(), EPS), attn, smg.Norm.rms(i["n2"].cpu().numpy(), EPS),
                               smg.Mlp.gated(up, lin("down", d, ffn)))
        s["cache"] = s["block"].cache(case["past"] + case["rows"])
        if case["past"]:
            s["cache"].extend(i["k"], i["v"])
        s["x0"], s["x"] = i["x"], torch.empty_like(i["x"])
    return s


def run(s):
    case = s["case"]
    op = case["op"]
    if op == "q4":
        f = smg.matmul_q4_bf16_ep if case["bf16"] else smg.matmul_q4_ep
        return f(s["a"], s["w"], s["c"], case["m"], s["ep"])
    if op == "lowbit":
        f = smg.matmul_q1_ep if case["bits"] == 1 else smg.matmul_q2_ep
        return f(s["a"], s["w"], s["c"], case["m"], s["ep"])
    if op == "mopa":
        f = smg.matmul_q1_mopa_ep if case["bits"] == 1 else smg.matmul_q2_mopa_ep
        return f(s["a"], s["w"], s["c"], case["m"], s["ep"])
    if op == "packed":
        return _ep_build(smg.Gemm(s["a"], s["w"], case["m"]), case["ep"], s["ep"]).run(s["c"])
    if op == "strided":
        m, n, k = case["m"], case["n"], case["k"]
        f = smg.gemm_bf16 if case["bf16"] else smg.gemm_f16
        b_rs, b_cs = (1, k) if case["bcol"] else (n, 1)
        return f(m, n, k, s["c"], n, 1, s["a"], k, 1, s["b"], b_rs, b_cs, case["alpha"], 1.0)
    if op == "attend":
        if case["rows"] == 1:
            return s["cache"].attend(s["q"], s["out"])
        return s["cache"].attend_causal(s["q"], case["rows"], s["out"])
    # a layer's input arrives in the residual stream; its positions follow the
    # cached ones
    s["cache"].truncate(case["past"])
    s["x"].copy_(s["x0"])
    return s["block"].accumulate(s["x"], s["cache"], case["rows"])


# ---- what a pass cannot do without --------------------------------------------

def _q4_size(n, k, affine=False):
    return k * n / 2 + 2 * n * _nbk(k, 32) * (2 if affine else 1)


def work(case):
    op = case["op"]
    if op in ("q4", "lowbit", "mopa"):
        m, n, k = case["m"], case["n"], case["k"]
        w = _q4_size(n, k, case["affine"]) if op == "q4" else k * n * case["bits"] / 8 + 2 * n * _nbk(k, 128)
        vec = 2 * n * (("scale" in case["ep"]) + ("bias" in case["ep"]))
        return {"bytes": w + 2 * m * k + 2 * m * n + vec, "flops": 2 * m * n * k}
    if op == "packed":
        m, n, k = case["m"], case["n"], case["k"]
        return {"bytes": 2 * (m * k + k * n + m * n) + 2 * n * ("bias" in case["ep"]), "flops": 2 * m * n * k}
    if op == "strided":
        m, n, k = case["m"], case["n"], case["k"]
        return {"bytes": 2 * (m * k + k * n + m * n * (2 if case["alpha"] else 1)), "flops": 2 * m * n * k}
    rows, heads, kvh, hd = case["rows"], case["heads"], case["kv_heads"], case["hd"]
    past = case["start"] if op == "attend" else case["past"]
    pairs = rows * past + rows * (rows + 1) / 2  # (query, key) pairs a head multiplies
    attn = 4 * pairs * heads * hd
    kv = 4 * (past + rows) * kvh * hd
    if op == "attend":
        return {"bytes": kv + 8 * rows * heads * hd, "flops": attn}
    d, ffn = case["d"], case["ffn"]
    shapes = (((heads + 2 * kvh) * hd, d), (d, heads * hd), (2 * ffn, d), (d, ffn))
    # weights once, the cache once (its new rows are written), the residual in and out
    return {"bytes": sum(_q4_size(n, k) for n, k in shapes) + kv + 8 * rows * d + 8 * d,
            "flops": attn + sum(2 * rows * n * k for n, k in shapes)}


def tolerance(case):
    op = case["op"]
    if op == "lowbit":
        return "exact"  # the int8 path's contract: the reference's bits
    # rel: the 16-bit output's rounding, where sums in another order fall on
    # the other side of it; the block's and attention's come from f16
    # roundings between their stages
    if op in ("q4", "mopa", "packed", "strided"):
        return {"rel": 4e-3, "max": 3e-2} if case.get("bf16") else {"rel": 5e-4, "max": 4e-3}
    if op == "attend":
        return {"rel": 1e-3, "max": 2e-2}
    return {"rel": 2e-3, "max": 4e-2}


# ---- the same in 64 bits -------------------------------------------------------

def _attend64(q, k, v, past, heads, kv_heads, hd):
    """Causal softmax attention: q [rows][heads*hd], k / v [past + rows][kv_heads*hd]."""
    rows, ln = q.shape[0], k.shape[0]
    out = torch.empty_like(q)
    mask = torch.arange(ln, device=DEV)[None, :] > past + torch.arange(rows, device=DEV)[:, None]
    for h in range(heads):
        j = h // (heads // kv_heads)
        p = q[:, h * hd:(h + 1) * hd] @ k[:, j * hd:(j + 1) * hd].t().contiguous() / math.sqrt(hd)
        p = torch.softmax(p.masked_fill_(mask, -math.inf), 1)
        out[:, h * hd:(h + 1) * hd] = p @ v[:, j * hd:(j + 1) * hd].contiguous()
    return out


def _rms64(x, w):
    return x / torch.sqrt((x * x).mean(1, keepdim=True) + EPS) * w.double()


def _rope64(x, pos, hd):
    inv = THETA ** (-torch.arange(0, hd, 2, device=DEV, dtype=torch.float64) / hd)
    ang = pos[:, None].double() * inv[None, :]
    c, s = ang.cos()[:, None, :], ang.sin()[:, None, :]
    x = x.reshape(x.shape[0], -1, 2, hd // 2)
    a, b = x[:, :, 0], x[:, :, 1]
    return torch.stack([a * c - b * s, b * c + a * s], 2).reshape(x.shape[0], -1)


def exact(case, seed):
    i, op = _inputs(case, seed), case["op"]
    if op == "q4":
        return _ep_exact(i["a"].double() @ _q4_dense(i["w"], case["n"], case["k"]), case["ep"], i["ep"])
    if op == "mopa":
        q, sc = i["w"]
        w = _lowbit_codes(q, case["bits"], case["n"], case["k"])
        w = w * sc.double().t().repeat_interleave(128, 0)[: case["k"]]
        return _ep_exact(i["a"].double() @ w, case["ep"], i["ep"])
    if op == "lowbit":
        # activations as int8 with a scale a row and block of 128 (part of
        # what is asked: the quantized product), the rest in 64 bits
        q, sc = i["w"]
        codes = _lowbit_codes(q, case["bits"], case["n"], case["k"])
        total = torch.zeros(case["m"], case["n"], dtype=torch.float64, device=DEV)
        for b in range(_nbk(case["k"], 128)):
            a = i["a"][:, 128 * b:128 * (b + 1)].float()
            amax = a.abs().amax(1, keepdim=True)
            inv = torch.where(amax > 0, 127.0 / amax, torch.zeros_like(amax))
            total += (torch.round(a * inv).double() @ codes[128 * b:128 * (b + 1)].contiguous()
                      * (amax.double() / 127.0) * sc[:, b].double())
        return _ep_exact(total, case["ep"], i["ep"])
    if op == "packed":
        return _ep_exact(i["a"].double() @ i["b"].double(), case["ep"], i["ep"])
    if op == "strided":
        b = i["b"].double()
        r = i["a"].double() @ (b.t().contiguous() if case["bcol"] else b)
        return r + case["alpha"] * i["c"].double()
    if op == "attend":
        return _attend64(i["q"].double(), i["k"].double(), i["v"].double(), case["start"], case["heads"],
                         case["kv_heads"], case["hd"])
    heads, kvh, hd, d, ffn, past = (case[x] for x in ("heads", "kv_heads", "hd", "d", "ffn", "past"))
    ql, ld = heads * hd, kvh * hd
    x = i["x"].double()
    qkv = _rms64(x, i["n1"]) @ _q4_dense(i["qkv"], ql + 2 * ld, d)
    pos = past + torch.arange(case["rows"], device=DEV)
    k = torch.cat([i["k"].double(), _rope64(qkv[:, ql:ql + ld], pos, hd)])
    v = torch.cat([i["v"].double(), qkv[:, ql + ld:]])
    x = x + _attend64(_rope64(qkv[:, :ql], pos, hd), k, v, past, heads, kvh, hd) @ _q4_dense(i["out"], d, ql)
    h = _rms64(x, i["n2"])
    g = h @ _q4_dense(i["gate"], ffn, d)
    h = g * torch.sigmoid(g) * (h @ _q4_dense(i["up"], ffn, d))
    return x + h @ _q4_dense(i["down"], d, ffn)
