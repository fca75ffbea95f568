"""The work that users of this package have it do, as cases that can be timed and checked.

Three whole calls of the decode engine (a greedy step, a prompt, a multi-token
verify pass) on a Phi-4-shaped model, and the weight formats' GEMVs through
``asdsl.kernels``, one layer matrix at a time.  Weights, activations and caches
are synthetic and drawn on the device from a seed: W ~ N(0, 0.02) quantized in
the format's own way, x ~ N(0, 1), cached K/V rows ~ N(0, 1).
"""

from __future__ import annotations

import math
import sys
from pathlib import Path

import numpy as np
import torch

_PKG = str(Path.cwd() / "asdsl-framework_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

PHI = {"heads": 24, "kv_heads": 8, "ffn": 8192, "vocab": 200064}  # DecodeConfig's defaults


def listed():
    return [
        # One token of generation through the whole 32-layer model, a
        # thousand tokens into a conversation: what serving spends its time on.
        {"name": "decode_step", "kind": "decode", **PHI, "layers": 32, "ctx": 1000, "kv": "fp16"},
        # A speculative-decoding step: eight drafted tokens checked at once.
        {"name": "verify_8", "kind": "verify", **PHI, "layers": 32, "ctx": 1000, "tokens": 8, "kv": "fp16"},
        # A chat turn's prompt (an odd length) before its first token.
        {"name": "prefill_517", "kind": "prefill", **PHI, "layers": 8, "tokens": 517, "kv": "fp16"},
        # A long document as the prompt, with the reference's int8 KV cache.
        {"name": "prefill_2300_int8", "kind": "prefill", **PHI, "layers": 4, "tokens": 2300, "kv": "int8"},
        # One attention output projection: the smallest matrix of a layer.
        {"name": "gemv_o_proj", "kind": "preq2", "m": 3072, "k": 3072, "gs": 32},
        # The output projection over the vocabulary, the largest single GEMV,
        # in the asymmetric format and in the 66-byte blocks of the
        # reference engine's tied lm_head.
        {"name": "gemv_lm_head_g128", "kind": "preq2", "m": 200064, "k": 3072, "gs": 128},
        {"name": "gemv_lm_head_q4_128", "kind": "q4_128", "m": 200064, "k": 3072},
        # The MLP's gate and up rows in the K-quant superblock format.
        {"name": "gemv_gate_up_q4k", "kind": "q4k", "m": 16384, "k": 3072},
        # The same rows with fp32 scales and biases and an fp32 activation:
        # the weight store's own format, before any repacking.
        {"name": "gemv_gate_up_fp32", "kind": "fp32", "m": 16384, "k": 3072, "gs": 32},
        # Many activation columns against one matrix: a prompt chunk on the
        # kernel API (a ragged column count), and the fp32 batch of 16.
        {"name": "batch_gate_up_45", "kind": "preq2_batch", "m": 16384, "k": 3072, "gs": 32, "n": 45},
        {"name": "batch_fp32_gate_up_16", "kind": "fp32_batch", "m": 16384, "k": 3072, "gs": 32, "n": 16},
        # The down projection after FATReLU: a fifth of the rows are active.
        {"name": "sparse_down_80", "kind": "sparse_down", "rows": 8192, "out": 3072, "gs": 128, "zeros": 0.8},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["decode", "verify", "prefill", "preq2", "q4_128", "q4k", "fp32", "preq2_batch", "fp32_batch",
                       "sparse_down"])
    if kind in ("decode", "verify", "prefill"):
        c = {"kind": kind, **rng.choice([
            PHI, {"heads": 16, "kv_heads": 4, "ffn": 128 * rng.randint(24, 64), "vocab": 32000 + rng.randint(0, 3)},
            {"heads": 8, "kv_heads": 4, "ffn": 128 * rng.randint(12, 32), "vocab": 32000 + rng.randint(0, 3)}])}
        c["kv"] = rng.choice(["fp16", "int8"])
        if kind == "prefill":
            c["layers"] = rng.randint(1, 4)
            c["tokens"] = _log_int(rng, 3, 2300)
        else:
            c["layers"] = _log_int(rng, 1, 32)
            c["ctx"] = _log_int(rng, 16, 4000)
            if kind == "verify":
                c["tokens"] = rng.randint(2, 16)
        return c
    if kind == "sparse_down":
        return {"kind": kind, "rows": 32 * rng.randint(64, 256), "out": 128 * rng.randint(8, 32), "gs": 128,
                "zeros": round(rng.uniform(0.5, 0.95), 3)}
    c = {"kind": kind, "m": _log_int(rng, 1000, 60000 if kind in ("preq2", "q4_128", "q4k") else 16384)}
    if kind == "q4k":
        c["k"] = 256 * rng.randint(4, 32)
    elif kind == "q4_128":
        c["k"] = 128 * rng.randint(8, 64)
    else:
        c["gs"] = rng.choice([32, 128] if kind.startswith("preq2") else [32, 64, 128])
        c["k"] = 128 * rng.randint(8, 64 if not kind.endswith("batch") else 24)
    if kind.endswith("batch"):
        c["n"] = _log_int(rng, 2, 64 if kind == "preq2_batch" else 32)
    return c


# ------------------------------------------------------------------ inputs
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _randn(gen, *shape):
    return torch.randn(shape, generator=gen, device="cuda", dtype=torch.float32)


def _preq2(gen, m, k, gs):
    from asdsl.quantization.synthetic import preq2_from_weights_torch

    return preq2_from_weights_torch(_randn(gen, m, k) * 0.02, gs)


def _affine(gen, m, k, gs):
    """Packed nibbles with fp32 (scale, bias) per group: the asymmetric store, w = q * s + b."""
    w = (_randn(gen, m, k) * 0.02).reshape(m, k // gs, gs)
    lo = w.amin(dim=2, keepdim=True)
    s = torch.clamp_min(w.amax(dim=2, keepdim=True) - lo, 1e-5) / 15.0
    q = torch.clamp(torch.round((w - lo) / s), 0, 15).to(torch.uint8).reshape(m, k)
    return ((q[:, 0::2] | (q[:, 1::2] << 4)).contiguous().reshape(-1), s.reshape(-1).contiguous(),
            lo.reshape(-1).contiguous())


def _q4k(gen, m, k):
    """144-byte superblocks: fp16 d, fp16 dmin, 16 6-bit fields (8 scales, 8 mins; LSB first), 128 nibble bytes."""
    nb = m * (k // 256)
    fields = torch.randint(20, 64, (nb, 16), generator=gen, device="cuda", dtype=torch.int64)
    words = torch.zeros((nb, 12), device="cuda", dtype=torch.int64)
    for i in range(16):
        bit = 6 * i
        v = fields[:, i] << (bit % 8)
        words[:, bit // 8] |= v & 0xFF
        if bit % 8 > 2:
            words[:, bit // 8 + 1] |= v >> 8
    d = (0.02 / 4.6 / 40 * (1.0 + 0.1 * torch.rand(nb, generator=gen, device="cuda"))).half()
    dmin = (d.float() * 7.5).half()
    out = torch.empty((nb, 144), device="cuda", dtype=torch.uint8)
    out[:, 0:2] = d.view(torch.int16).reshape(-1, 1).view(torch.uint8)
    out[:, 2:4] = dmin.view(torch.int16).reshape(-1, 1).view(torch.uint8)
    out[:, 4:16] = words.to(torch.uint8)
    q = torch.clamp(torch.round(_randn(gen, nb, 256) * 2.5 + 7.5), 0, 15).to(torch.uint8)
    out[:, 16:] = q[:, 0::2] | (q[:, 1::2] << 4)
    return out.reshape(-1)


def _engine(case, gen):
    """A model as a user's program holds it: weights laid out, caches of the length it serves."""
    from asdsl.engine import DecodeConfig, DecodeEngine, kv_quantize_int8

    hidden = case["heads"] * 128
    ctx = case.get("ctx", 0)
    cfg = DecodeConfig(hidden=hidden, ffn=case["ffn"], vocab=case["vocab"], n_layers=case["layers"],
                       n_heads=case["heads"], n_kv_heads=case["kv_heads"],
                       max_seq=(ctx + case.get("tokens", 1) + 319) // 64 * 64, kv_format=case["kv"])
    dtype = torch.int8 if cfg.kv_format == "int8" else torch.float16
    shape = (cfg.n_layers, cfg.n_kv_heads, cfg.max_seq, 128)
    cache = {n: torch.zeros(shape, dtype=dtype, device="cuda") for n in ("k_cache", "v_cache")}
    if cfg.kv_format == "int8":
        cache |= {n: torch.ones(shape[:3] + (2,), device="cuda") for n in ("k_scale", "v_scale")}
    for n in ("k", "v"):
        if ctx:
            rows = _randn(gen, *shape[:2], ctx, 128)
            if cfg.kv_format == "int8":
                cache[n + "_cache"][:, :, :ctx], cache[n + "_scale"][:, :, :ctx] = kv_quantize_int8(rows)
            else:
                cache[n + "_cache"][:, :, :ctx] = rows.half()
    layers = []
    for i in range(cfg.n_layers):
        layers.append({"qkv": _preq2(gen, cfg.qkv_dim, hidden, 32), "o": _preq2(gen, hidden, hidden, 32),
                       "gu": _preq2(gen, 2 * cfg.ffn, hidden, 128), "down": _preq2(gen, hidden, cfg.ffn, 128),
                       "rms_att": 1.0 + 0.1 * _randn(gen, hidden), "rms_ffn": 1.0 + 0.1 * _randn(gen, hidden),
                       **{n: t[i] for n, t in cache.items()}})
    embed = _randn(gen, cfg.vocab, hidden).half()
    lm_meta, lm_quant = _preq2(gen, cfg.vocab, hidden, 128)
    eng = DecodeEngine(cfg, layers, embed, 1.0 + 0.1 * _randn(gen, hidden), lm_meta, lm_quant)
    return eng, cache


def prepare(case, seed):
    from asdsl.kernels import _native_gemv  # noqa: F401  (a program has its kernels loaded)

    gen, kind = _gen(seed), case["kind"]
    if kind in ("decode", "verify", "prefill"):
        eng, cache = _engine(case, gen)
        n = case.get("tokens", 1)
        toks = torch.randint(0, case["vocab"], (n,), generator=gen, device="cuda").tolist()
        return {"kind": kind, "eng": eng, "cache": cache, "tokens": toks, "ctx": case.get("ctx", 0)}
    s = {"kind": kind, **{n: case[n] for n in ("m", "k", "gs", "n", "rows", "out") if n in case}}
    if kind == "sparse_down":
        rows, out, gs = case["rows"], case["out"], case["gs"]
        s["w"], s["s"], s["b"] = _affine(gen, rows, out, gs)
        x = _randn(gen, rows)
        x[torch.rand(rows, generator=gen, device="cuda") < case["zeros"]] = 0.0
        s["x"], s["active"] = x, torch.nonzero(x).reshape(-1).to(torch.int32)
        return s
    m, k = case["m"], case["k"]
    s["x"] = _randn(gen, case["n"], k) if "n" in case else _randn(gen, k)
    s["y"] = torch.empty(((case["n"], m) if "n" in case else (m,)), device="cuda")
    if kind in ("preq2", "preq2_batch"):
        s["meta"], s["quant"] = _preq2(gen, m, k, case["gs"])
    elif kind == "q4_128":
        from asdsl.quantization.synthetic import q4_128_from_weights_torch

        s["w"] = q4_128_from_weights_torch(_randn(gen, m, k) * 0.02)
    elif kind == "q4k":
        s["w"] = _q4k(gen, m, k)
    else:
        s["w"], s["s"], s["b"] = _affine(gen, m, k, case["gs"])
    return s


def run(st):
    from asdsl.kernels import _native_gemv as ng

    kind = st["kind"]
    if kind in ("decode", "verify", "prefill"):
        eng = st["eng"]
        if kind == "decode":
            logits = eng.forward_token(st["tokens"][0], st["ctx"])
        elif kind == "verify":
            logits = eng.forward_batch_all_logits(st["tokens"], st["ctx"])
        else:
            eng.prefill(st["tokens"])
            logits = eng.logits
        return {"logits": logits, **st["cache"]}
    if kind in ("preq2", "preq2_batch"):
        ng.gemv_preq2_fused_avx2(st["meta"], st["quant"], st["x"], st["y"], st["m"], st["k"], st["gs"])
    elif kind == "q4_128":
        ng.gemv_q4_128_fused(st["w"], st["x"], st["y"], st["m"], st["k"], 128)
    elif kind == "q4k":
        ng.gemv_q4km_q8_avx2(st["w"], st["x"], st["y"], st["m"], st["k"])
    elif kind == "fp32":
        return ng.gemv_q4_packed(st["w"], st["x"], st["s"], st["b"], st["m"], st["k"], st["gs"])
    elif kind == "fp32_batch":
        ng.matmul_batch_q4(st["w"], st["s"], st["b"], st["x"], st["y"], st["m"], st["k"], st["n"], st["gs"])
    else:
        from asdsl.kernels import _native_sparse_gemv as sg

        return sg.sparse_down_proj_T(st["w"], st["s"], st["b"], st["x"], st["active"], st["rows"], st["out"],
                                     st["gs"])
    return st["y"]


# ------------------------------------------------------------- what it takes
def _model_work(c):
    h, ffn, kvd = c["heads"] * 128, c["ffn"], c["kv_heads"] * 128
    per = {32: (4 + 16) / 32, 128: (4 + 64) / 128}  # bytes per weight
    attn_w, mlp_w = (h + 2 * kvd) * h + h * h, 3 * ffn * h
    n, ctx = c.get("tokens", 1), c.get("ctx", 0)
    row = 2 * kvd * (2.0 if c["kv"] == "fp16" else 1.0 + 4 / 64)  # a position's K and V
    seen = sum(ctx + i + 1 for i in range(n))
    out_cols = n if c["kind"] == "verify" else 1
    nbytes = c["layers"] * (attn_w * per[32] + mlp_w * per[128] + 8 * h + row * (ctx + 2 * n)) \
        + c["vocab"] * h * per[128] + 4 * h + 2 * h * n + 4 * c["vocab"] * out_cols
    flops = c["layers"] * (2 * (attn_w + mlp_w) * n + 4 * h * seen) + 2 * c["vocab"] * h * out_cols
    return {"bytes": nbytes, "flops": flops}


def work(c):
    kind = c["kind"]
    if kind in ("decode", "verify", "prefill"):
        return _model_work(c)
    if kind == "sparse_down":
        live = c["rows"] * (1.0 - c["zeros"])
        return {"bytes": live * (c["out"] / 2 + 8 * c["out"] / c["gs"] + 4) + 4 * c["rows"] + 4 * c["out"],
                "flops": 2 * live * c["out"]}
    m, k, n = c["m"], c["k"], c.get("n", 1)
    if kind in ("preq2", "preq2_batch"):
        w = m * (k // 2 + 4 * (k // c["gs"]))
    elif kind == "q4_128":
        w = m * (k // 128) * 66
    elif kind == "q4k":
        w = m * (k // 256) * 144
    else:
        w = m * (k // 2 + 8 * (k // c["gs"]))
    return {"bytes": w + 4 * n * (k + m), "flops": 2 * m * k * n}


# A GEMV's sums are 32-bit (its int8 activation codes are part of what it
# computes): four times the largest distance from the same sums in 64 bits
# (4e-7 for the fp32 activations, 1.5e-7 for the integer formats).
#
# A whole model is another matter: a change of rounding moves an int8
# activation code by one here and there and travels through every later
# layer.  Four times what is measured when each projection takes its sums in
# another order (the multi-token pass's own-order form, the step's factored
# norm): logits 0.0049 at 2 layers, 0.017-0.025 at 4, 0.024-0.037 at 8,
# 0.051-0.066 at 32; largest single value about six times that.
def tolerance(c):
    if c["kind"] in ("decode", "verify", "prefill"):
        rel = 4 * 0.012 * math.sqrt(c["layers"])
        return {"rel": rel, "max": min(0.9, 6 * rel), "differ": 0.5}
    return {"rel": 1.6e-6 if c["kind"] in ("fp32", "fp32_batch") else 6e-7, "max": 1e-5}


# ------------------------------------------------------------------ 64 bits
def _codes(x, gs, away=False):
    """The int8 activation codes and fp32 scales that the integer formats
    define (x: (n, k)): per group, scale = amax / 127 and code = x * (127 /
    amax) rounded to nearest even (Q4_K: away from zero at ties)."""
    n, k = x.shape
    g = x.reshape(n, k // gs, gs)
    amax = g.abs().amax(dim=2)
    inv = torch.where(amax < 1e-9, torch.zeros_like(amax), 127.0 / amax)
    v = g * inv[:, :, None]
    q = torch.sign(v) * torch.floor(v.abs() + 0.5) if away else torch.round(v)
    q = torch.clamp(q, -127 if away else -128, 127)
    scale = amax * float(np.float32(1.0 / 127.0))
    return q.double(), scale.double()


def _nibbles(b):
    return torch.stack((b & 15, b >> 4), dim=-1).reshape(*b.shape[:-1], -1).double()


def _rows(m, k, step=1 << 26):
    r = max(4, step // k // 4 * 4)
    return [(a, min(a + r, m)) for a in range(0, m, r)]


def exact(c, seed):
    kind = c["kind"]
    if kind in ("decode", "verify", "prefill"):
        return None
    st = prepare(c, seed)
    if kind == "sparse_down":
        rows, out, gs = c["rows"], c["out"], c["gs"]
        w = _nibbles(st["w"].reshape(rows, out // 2)).reshape(rows, out // gs, gs)
        w = w * st["s"].reshape(rows, -1, 1).double() + st["b"].reshape(rows, -1, 1).double()
        return st["x"].double() @ w.reshape(rows, out)
    m, k = c["m"], c["k"]
    x = st["x"].reshape(-1, k)
    y = torch.empty((x.shape[0], m), device="cuda", dtype=torch.float64)
    if kind in ("preq2", "preq2_batch", "q4_128", "q4k"):
        gs = {"q4_128": 128, "q4k": 32}.get(kind, c.get("gs"))
        q, s = _codes(x, gs, away=kind == "q4k")
        xd = (q * s[:, :, None]).reshape(-1, k)
    else:
        xd = x.double()
    for a, b in _rows(m, k):
        r = b - a
        if kind in ("preq2", "preq2_batch"):
            gs = c["gs"]
            G = k // gs
            meta = st["meta"].view(torch.float16).reshape(m, G, 2)[a:b].double()
            bands = (r + 3) // 4
            qb = st["quant"].reshape(-1, G, 4, gs // 2)[a // 4:a // 4 + bands].permute(0, 2, 1, 3)
            w = _nibbles(qb.reshape(bands * 4, G, gs // 2)[:r])
            w = (w - meta[:, :, 1:2]) * meta[:, :, 0:1]
        elif kind == "q4_128":
            blk = st["w"].reshape(m, k // 128, 66)[a:b]
            d = blk[:, :, 0:2].contiguous().view(torch.float16).double()
            w = (_nibbles(blk[:, :, 2:]) - 8.0) * d
        elif kind == "q4k":
            blk = st["w"].reshape(m, k // 256, 144)[a:b]
            d = blk[:, :, 0:4].contiguous().view(torch.float16).double()
            bits = blk[:, :, 4:16].to(torch.int64)
            f = torch.stack([((bits[:, :, 6 * i // 8] | (bits[:, :, min(11, 6 * i // 8 + 1)] << 8)) >> (6 * i % 8)) & 63
                             for i in range(16)], dim=-1).double()
            w = _nibbles(blk[:, :, 16:]).reshape(r, k // 256, 8, 32)
            w = (d[:, :, 0:1] * f[:, :, :8])[..., None] * w - (d[:, :, 1:2] * f[:, :, 8:])[..., None]
        else:
            gs = c["gs"]
            w = _nibbles(st["w"].reshape(m, k // 2)[a:b]).reshape(r, k // gs, gs)
            w = w * st["s"].reshape(m, -1, 1)[a:b].double() + st["b"].reshape(m, -1, 1)[a:b].double()
        y[:, a:b] = xd @ w.reshape(r, k).T
    return y if "n" in c else y[0]
