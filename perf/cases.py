"""The work this library is timed and compared on: quantized linears, the dense strategy, weight
quantization, the MoE feed-forward, attention, and whole decoder passes, each through the entry point a
program calls. Weights are GGML blocks made here from seeded normal values (a plain min/max fit), so that
`exact` can decode the same blocks without the library and form the results in 64 bits. The activations'
own quantization (Q8_K / Q8_0) is part of what a quantized matmul computes, so `exact` applies it too.
"""
import ctypes
import math

import numpy as np
import torch

from inference_amd import qmm
from inference_amd.llama_decode import DecodeSession, LlamaConfig, LlamaWeights
from inference_amd.qmm import GgmlDType, MatmulStrategy, QLinear, QMatMul, QTensor, QuantizedLinear

DEV = torch.device("cuda", 0)
TYPES = {"q4k": GgmlDType.Q4K, "q6k": GgmlDType.Q6K, "q8_0": GgmlDType.Q8_0}
DENSE = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
BLOCK = {"q4k": (256, 144), "q6k": (256, 210), "q8_0": (32, 34)}  # elements, bytes
PARTS = ("q", "k", "v", "o", "gate", "up", "down")


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------

def listed():
    return [
        # the smallest projection of a decode step (a kv head group): one row, latency and launch cost
        {"name": "linear_q4k_m1", "kind": "linear", "type": "q4k", "m": 1, "n": 1024, "k": 4096, "x": "f32"},
        # a few sequences decoded together through the Q6_K down projection
        {"name": "linear_q6k_m5", "kind": "linear", "type": "q6k", "m": 5, "n": 4096, "k": 14336, "x": "f32"},
        # prompt processing through the widest projection
        {"name": "linear_q4k_m512", "kind": "linear", "type": "q4k", "m": 512, "n": 14336, "k": 4096, "x": "f32"},
        # an 8-bit layer of a bf16 model, with its bias, over a ragged prompt
        {"name": "linear_q8_0_m333", "kind": "linear", "type": "q8_0", "m": 333, "n": 4096, "k": 4096, "x": "bf16"},
        # the media models' default strategy: the weight dequantized for a dense product
        {"name": "dense_q8_0_m256", "kind": "dense", "type": "q8_0", "m": 256, "n": 14336, "k": 4096, "x": "bf16"},
        # loading a dense checkpoint into a 4-bit projection, and reading it back
        {"name": "quantize_q4k", "kind": "quantize", "type": "q4k", "n": 4096, "k": 4096, "x": "f32"},
        # mixture of experts, batched decode
        {"name": "moe_t8", "kind": "moe", "tokens": 8, "experts": 8, "topk": 2, "hidden": 4096, "ffn": 14336,
         "shared": 0},
        # mixture of experts, prompt
        {"name": "moe_t512", "kind": "moe", "tokens": 512, "experts": 8, "topk": 2, "hidden": 4096, "ffn": 14336,
         "shared": 0},
        # causal attention over a long prompt
        {"name": "prefill_attention_1999", "kind": "prefill_attention", "first": 0, "count": 1999, "heads": 32,
         "kv_heads": 8, "head_dim": 128},
        # one token's attention deep in a conversation
        {"name": "decode_attention_3000", "kind": "decode_attention", "pos": 3000, "heads": 32, "kv_heads": 8,
         "head_dim": 128},
        # time to the first token: a prompt through some of the 8B-shaped layers and the head
        {"name": "model_prefill_700", "kind": "model_prefill", "tokens": 700, "layers": 3},
        # token steps of the same model, the tokens given (as a scorer or a draft checker runs it)
        {"name": "model_decode_16", "kind": "model_decode", "tokens": 16, "layers": 3},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _mult(rng, lo, hi, step):
    return max(lo // step, min(hi // step, int(round(_log(rng, lo, hi) / step)))) * step


HEADS = ((32, 8, 128), (16, 16, 128), (32, 4, 128), (8, 2, 64), (8, 1, 64), (16, 2, 256))


def draw(rng):
    kind = rng.choice(("linear", "linear", "dense", "quantize", "moe", "prefill_attention", "decode_attention",
                       "model_prefill", "model_decode"))
    t = rng.choice(("q4k", "q6k", "q8_0"))
    step = BLOCK[t][0]
    if kind == "linear":
        # one row as often as a few or many: decode, batched decode and prompts
        m = rng.choice((1, rng.randint(2, 8), _log(rng, 9, 512)))
        return {"kind": kind, "type": t, "m": m, "n": _log(rng, 256, 14336), "k": _mult(rng, 512, 14336, step),
                "x": rng.choice(("f32", "f32", "bf16", "f16"))}
    if kind == "dense":
        return {"kind": kind, "type": t, "m": _log(rng, 1, 512), "n": _log(rng, 512, 14336),
                "k": _mult(rng, 512, 8192, step), "x": rng.choice(("bf16", "f16"))}
    if kind == "quantize":
        return {"kind": kind, "type": rng.choice(("q4k", "q8_0")), "n": _log(rng, 256, 4096),
                "k": _mult(rng, 512, 4096, 256), "x": rng.choice(("f32", "bf16"))}
    if kind == "moe":
        experts = rng.choice((4, 8, 16, 64))
        hidden = _mult(rng, 512, 4096, 256)
        ffn = _mult(rng, 512, 14336 * 8 // max(8, experts), 256)
        return {"kind": kind, "tokens": _log(rng, 1, 512), "experts": experts,
                "topk": rng.choice((1, 2, 4) if experts < 64 else (6, 8)), "hidden": hidden, "ffn": ffn,
                "shared": rng.choice((0, 0, 1024))}
    if kind in ("prefill_attention", "decode_attention"):
        h, kv, hd = rng.choice(HEADS)
        geom = {"heads": h, "kv_heads": kv, "head_dim": hd}
        if kind == "decode_attention":
            return {"kind": kind, "pos": _log(rng, 1, 8191), **geom}
        return {"kind": kind, "first": rng.choice((0, rng.randint(1, 1000))), "count": _log(rng, 9, 1900), **geom}
    if kind == "model_prefill":
        return {"kind": kind, "tokens": _log(rng, 10, 700), "layers": rng.randint(1, 3)}
    return {"kind": kind, "tokens": rng.randint(4, 16), "layers": rng.randint(1, 3)}


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------

def _gen(seed, tag):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed * 1009 + tag)
    return g


def _randn(seed, tag, shape, std=1.0):
    return torch.randn(shape, generator=_gen(seed, tag), device=DEV, dtype=torch.float32) * std


def _f16_bytes(t):
    return t.to(torch.float16).contiguous().view(torch.uint8)


def _blocks(w, kind):
    """GGML blocks (uint8 [rows, blocks, bytes]) of dense f32 rows: a min/max fit per sub-block."""
    n, k = w.shape
    if kind == "q8_0":
        b = w.view(n, k // 32, 32)
        d = (b.abs().amax(-1, keepdim=True) / 127).to(torch.float16)
        q = (b / d.float().clamp_min(1e-8)).round().clamp(-127, 127).to(torch.int8)
        return torch.cat([_f16_bytes(d), q.view(torch.uint8)], -1)
    if kind == "q6k":
        b = w.view(n, k // 256, 16, 16)
        s = b.abs().amax(-1) / 31
        d = (s.amax(-1, keepdim=True) / 127).to(torch.float16)
        sc = (s / d.float().clamp_min(1e-8)).round().clamp(1, 127)
        q = (b / (d.float() * sc).clamp_min(1e-12).unsqueeze(-1)).round().clamp(-32, 31).to(torch.int32) + 32
        q = q.view(n, k // 256, 2, 4, 32)
        low, high = q & 15, q >> 4
        ql = torch.cat([low[..., 0, :] | low[..., 2, :] << 4, low[..., 1, :] | low[..., 3, :] << 4], -1)
        qh = high[..., 0, :] | high[..., 1, :] << 2 | high[..., 2, :] << 4 | high[..., 3, :] << 6
        return torch.cat([ql.flatten(-2).to(torch.uint8), qh.flatten(-2).to(torch.uint8),
                          sc.to(torch.int8).view(torch.uint8), _f16_bytes(d)], -1)
    b = w.view(n, k // 256, 8, 32)
    low = (-b.amin(-1)).clamp_min(0)
    s = (b.amax(-1) + low) / 15
    d = (s.amax(-1, keepdim=True) / 63).to(torch.float16)
    dm = (low.amax(-1, keepdim=True) / 63).to(torch.float16)
    sc = (s / d.float().clamp_min(1e-8)).round().clamp(1, 63)
    mn = (low / dm.float().clamp_min(1e-8)).round().clamp(0, 63)
    q = (b + (dm.float() * mn).unsqueeze(-1)) / (d.float() * sc).clamp_min(1e-12).unsqueeze(-1)
    q = q.round().clamp(0, 15).to(torch.uint8).view(n, k // 256, 4, 2, 32)
    qs = (q[..., 0, :] | q[..., 1, :] << 4).flatten(-2)
    sc, mn = sc.to(torch.uint8), mn.to(torch.uint8)
    s0 = (sc[..., :4] & 63) | (sc[..., 4:] >> 4) << 6
    s1 = (mn[..., :4] & 63) | (mn[..., 4:] >> 4) << 6
    s2 = (sc[..., 4:] & 15) | (mn[..., 4:] & 15) << 4
    return torch.cat([_f16_bytes(d), _f16_bytes(dm), s0, s1, s2, qs], -1)


def _weight(kind, n, k, seed, tag, std=0.02):
    """GGML bytes [n, row bytes] of an [n, k] weight drawn from N(0, std^2)."""
    e, size = BLOCK[kind]
    out = torch.empty((n, k // e * size), dtype=torch.uint8, device=DEV)
    g = _gen(seed, tag)
    rows = max(1, (1 << 25) // k)
    for r in range(0, n, rows):
        w = torch.randn((min(rows, n - r), k), generator=g, device=DEV, dtype=torch.float32) * std
        out[r:r + rows] = _blocks(w, kind).flatten(1)
    return out


def _tensor(kind, n, k, seed, tag, std=0.02):
    return QTensor.from_ggml(_weight(kind, n, k, seed, tag, std).view(-1), TYPES[kind], (n, k))


def _config(case):
    return LlamaConfig(layers=case["layers"])


def _part(cfg, name):
    return "q4k" if cfg.dtypes[name] == GgmlDType.Q4K else "q6k"


def _norm(seed, tag, n):
    return 1 + 0.1 * _randn(seed, tag, (n,))


def _embed(cfg, seed):
    return _randn(seed, 7000, (cfg.vocab, cfg.hidden))


def _std(cfg, name):
    """The projections into the residual stream are scaled down by the depth, so that a layer adds a part of
    the stream and does not replace it."""
    return 0.02 / 8 if name in ("o", "down") else 0.02


def _prompt(case, cfg, seed):
    r = np.random.RandomState(seed % (1 << 31))
    return [int(t) for t in r.randint(0, cfg.vocab, case["tokens"])]


def _max_seq(case):
    return -(-(case["tokens"] + 1) // 256) * 256


def _session(case, seed):
    cfg = _config(case)
    sh = cfg.shapes()
    layers = [{p: _tensor(_part(cfg, p), *sh[p], seed, 16 * li + j, _std(cfg, p)) for j, p in enumerate(PARTS)}
              for li in range(cfg.layers)]
    head = _tensor(_part(cfg, "head"), *sh["head"], seed, 6000)
    w = LlamaWeights(cfg, layers, head, _embed(cfg, seed),
                     [_norm(seed, 8000 + li, cfg.hidden) for li in range(cfg.layers)],
                     [_norm(seed, 8100 + li, cfg.hidden) for li in range(cfg.layers)],
                     _norm(seed, 8200, cfg.hidden))
    return DecodeSession(w, _max_seq(case))


def _attention_inputs(case, seed, rows, max_seq):
    h, kv, hd = case["heads"], case["kv_heads"], case["head_dim"]
    return (_randn(seed, 1, (rows, h * hd)), _randn(seed, 2, (kv, max_seq, hd)), _randn(seed, 3, (kv, max_seq, hd)))


def _angles(max_seq, hd):
    inv = 1.0 / (500000.0 ** (np.arange(0, hd, 2, dtype=np.float64) / hd))
    a = np.arange(max_seq, dtype=np.float64)[:, None] * np.concatenate([inv, inv])[None, :]
    return (torch.from_numpy(np.cos(a).astype(np.float32)).to(DEV),
            torch.from_numpy(np.sin(a).astype(np.float32)).to(DEV))


def _span(case):
    """Cache positions an attention case's program holds: what it needs, rounded up."""
    need = case["pos"] + 1 if case["kind"] == "decode_attention" else case["first"] + case["count"]
    return -(-need // 256) * 256


def prepare(case, seed):
    kind = case["kind"]
    s = {"kind": kind}
    if kind in ("linear", "dense"):
        n, k, dt = case["n"], case["k"], DENSE[case["x"]]
        qt = _tensor(case["type"], n, k, seed, 1)
        s["x"] = _randn(seed, 2, (case["m"], k)).to(dt)
        if kind == "dense":
            bias = _randn(seed, 3, (n,)).to(dt)
            s["layer"] = QLinear(qt, bias, MatmulStrategy.DEQUANT_DENSE)
        elif case["x"] == "f32":
            s["layer"] = QMatMul.from_qtensor(qt)
        else:
            s["layer"] = QuantizedLinear(QMatMul.from_qtensor(qt), _randn(seed, 3, (n,)).to(dt))
    elif kind == "quantize":
        s["w"] = _randn(seed, 1, (case["n"], case["k"]), 0.02).to(DENSE[case["x"]])
        s["type"] = TYPES[case["type"]]
    elif kind == "moe":
        e, h, f = case["experts"], case["hidden"], case["ffn"]
        s["gate"], s["up"] = (_tensor("q4k", e * f, h, seed, t) for t in (1, 2))
        s["down"] = _tensor("q6k", e * h, f, seed, 3)
        s["x"] = _randn(seed, 4, (case["tokens"], h))
        s["logits"] = _randn(seed, 5, (case["tokens"], e))
        s["topk"], s["shared"], s["shared_gate"] = case["topk"], None, None
        if case["shared"]:
            fs = case["shared"]
            s["shared"] = (_tensor("q4k", fs, h, seed, 6), _tensor("q4k", fs, h, seed, 7),
                           _tensor("q6k", h, fs, seed, 8))
            s["shared_gate"] = _randn(seed, 9, (h,), 0.02)
    elif kind == "prefill_attention":
        span = _span(case)
        s["q"], s["kc"], s["vc"] = _attention_inputs(case, seed, case["count"], span)
        s["out"] = torch.empty_like(s["q"])
        s["args"] = (case["first"], case["count"], case["heads"], case["kv_heads"], case["head_dim"], span)
    elif kind == "decode_attention":
        span = _span(case)
        h, kv, hd = case["heads"], case["kv_heads"], case["head_dim"]
        s["q"], s["kc"], s["vc"] = _attention_inputs(case, seed, 1, span)
        s["k"], s["v"] = _randn(seed, 4, (kv, hd)), _randn(seed, 5, (kv, hd))
        s["cos"], s["sin"] = _angles(span, hd)
        s["pos"] = torch.full((1,), case["pos"], dtype=torch.int32, device=DEV)
        s["out"] = torch.empty((h, hd), dtype=torch.float32, device=DEV)
        s["ws"] = torch.zeros(int(qmm.lib().qmm_decode_attention_workspace_size(h, kv, hd, span)), dtype=torch.uint8,
                              device=DEV)
        s["args"] = (h, kv, hd, span)
        s["at"] = case["pos"]
    else:
        s["session"] = _session(case, seed)
        s["prompt"] = _prompt(case, s["session"].cfg, seed)
        steps = 1 if kind == "model_prefill" else case["tokens"]
        s["logits"] = torch.empty((steps, s["session"].cfg.vocab), dtype=torch.float32, device=DEV)
    return s


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------

def _call(status):
    if status != qmm.QMM_OK:
        raise qmm.QmmError(status, qmm.last_error())


def run(s):
    kind = s["kind"]
    if kind in ("linear", "dense"):
        return s["layer"].forward(s["x"])
    if kind == "quantize":
        return QuantizedLinear.quantize(s["w"], s["type"]).inner.qtensor.dequantize()
    if kind == "moe":
        return qmm.moe_ffn(s["x"], s["logits"], s["gate"], s["up"], s["down"], s["topk"], shared=s["shared"],
                           shared_gate=s["shared_gate"])
    if kind == "prefill_attention":
        first, count, h, kv, hd, span = s["args"]
        stream = ctypes.c_void_p(torch.cuda.current_stream(DEV).cuda_stream)
        _call(qmm.lib().qmm_prefill_attention(s["q"].data_ptr(), h * hd, s["kc"].data_ptr(), s["vc"].data_ptr(), first,
                                              count, s["out"].data_ptr(), h * hd, h, kv, hd, span,
                                              ctypes.c_float(hd ** -0.5), stream))
        return s["out"]
    if kind == "decode_attention":
        h, kv, hd, span = s["args"]
        stream = ctypes.c_void_p(torch.cuda.current_stream(DEV).cuda_stream)
        _call(qmm.lib().qmm_decode_rope_attention(
            s["q"].data_ptr(), s["k"].data_ptr(), s["v"].data_ptr(), s["cos"].data_ptr(), s["sin"].data_ptr(),
            s["pos"].data_ptr(), s["kc"].data_ptr(), s["vc"].data_ptr(), s["out"].data_ptr(), h, kv, hd, span,
            ctypes.c_float(hd ** -0.5), s["ws"].data_ptr(), s["ws"].numel(), stream))
        return {"out": s["out"], "k": s["kc"][:, s["at"]], "v": s["vc"][:, s["at"]]}
    ses = s["session"]
    ses.reset(s["prompt"])
    if kind == "model_prefill":
        ses.prefill()
    ses.run(s["logits"].shape[0], history=s["logits"])
    return {"logits": s["logits"], "k": ses.kcache, "v": ses.vcache}


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------

def _wbytes(kind, n, k):
    e, size = BLOCK[kind]
    return n * (k // e) * size


def work(case):
    kind = case["kind"]
    if kind in ("linear", "dense"):
        m, n, k = case["m"], case["n"], case["k"]
        el = 4 if case["x"] == "f32" else 2
        bias = 0 if kind == "linear" and case["x"] == "f32" else el * n
        return {"bytes": _wbytes(case["type"], n, k) + el * m * (n + k) + bias, "flops": 2 * m * n * k}
    if kind == "quantize":
        n, k = case["n"], case["k"]
        # the dense weight read, the blocks written, the f32 values written back
        return {"bytes": n * k * ((4 if case["x"] == "f32" else 2) + 4) + _wbytes(case["type"], n, k), "flops": n * k}
    if kind == "moe":
        t, e, h, f, k = (case[x] for x in ("tokens", "experts", "hidden", "ffn", "topk"))
        active = e * (1 - (1 - k / e) ** t)  # experts that some token is sent to, on average
        b = active * (2 * _wbytes("q4k", f, h) + _wbytes("q6k", h, f)) + 8 * t * h + 4 * t * e
        fl = 2 * t * k * 3 * h * f
        if case["shared"]:
            fs = case["shared"]
            b += 2 * _wbytes("q4k", fs, h) + _wbytes("q6k", h, fs) + 4 * h
            fl += 2 * t * 3 * h * fs
        return {"bytes": b, "flops": fl}
    if kind == "prefill_attention":
        first, c, h, kv, hd = (case[x] for x in ("first", "count", "heads", "kv_heads", "head_dim"))
        pairs = c * first + c * (c + 1) // 2
        return {"bytes": 8 * c * h * hd + 8 * (first + c) * kv * hd, "flops": 4 * pairs * h * hd}
    if kind == "decode_attention":
        p, h, kv, hd = (case[x] for x in ("pos", "heads", "kv_heads", "head_dim"))
        return {"bytes": 8 * h * hd + 8 * (p + 1) * kv * hd + 8 * kv * hd + 8 * hd, "flops": 4 * (p + 1) * h * hd}
    cfg = _config(case)
    sh = cfg.shapes()
    layer = sum(_wbytes(_part(cfg, p), *sh[p]) for p in PARTS)
    lfl = sum(2 * a * b for a, b in (sh[p] for p in PARTS))
    head = _wbytes(_part(cfg, "head"), *sh["head"])
    t, kvd = case["tokens"], cfg.kv_heads * cfg.head_dim
    # the caches as reset clears them, the rows' keys and values, the embedding rows and the logits
    cache = 8 * cfg.layers * kvd * _max_seq(case)
    att = cfg.layers * 4 * (t * (t + 1) // 2) * cfg.heads * cfg.head_dim
    if kind == "model_prefill":
        b = cfg.layers * layer + head + cache + 8 * cfg.layers * kvd * t + 4 * t * cfg.hidden + 4 * cfg.vocab
        return {"bytes": b, "flops": t * cfg.layers * lfl + att + 2 * cfg.vocab * cfg.hidden}
    b = t * (cfg.layers * layer + head + 4 * cfg.hidden + 12 * cfg.vocab) + cache
    return {"bytes": b, "flops": t * (cfg.layers * lfl + 2 * cfg.vocab * cfg.hidden) + att}


def tolerance(case):
    """About four times what the same pass differs by when its 32-bit sums are taken in another order (or in
    64 bits). Where an intermediate is quantized again, a last-bit change moves a few of its 8-bit codes by
    one, and a decoder passes that on from layer to layer. 16-bit outputs may round the other way."""
    kind = case["kind"]
    if kind == "quantize":
        return "exact"
    if kind in ("linear", "dense") and case["x"] != "f32":
        return {"rel": 1.2e-3 if case["x"] == "f16" else 1e-2}
    if kind == "moe":
        return {"rel": 4e-4, "max": 2e-2}
    if kind.startswith("model"):
        return {"rel": 3e-2, "max": 0.3}
    return {"rel": 2e-6 if kind.endswith("attention") else 1e-6, "max": 1e-4}


# ---------------------------------------------------------------------------
# the results in 64 bits
# ---------------------------------------------------------------------------

def _dequantize(b, kind, n, k):
    """f64 [n, k] of GGML bytes [n, row bytes]."""
    e, size = BLOCK[kind]
    b = b.view(n, k // e, size)

    def half(lo):
        return b[..., lo:lo + 2].contiguous().view(torch.float16).double()

    if kind == "q8_0":
        return (half(0) * b[..., 2:].contiguous().view(torch.int8).double()).view(n, k)
    if kind == "q6k":
        ql = b[..., :128].reshape(n, k // 256, 2, 2, 32)
        qh = b[..., 128:192].reshape(n, k // 256, 2, 1, 32)
        shift = torch.tensor([0, 2, 4, 6], dtype=torch.uint8, device=b.device).view(4, 1)
        q = torch.cat([ql & 15, ql >> 4], 3) | ((qh >> shift) & 3) << 4  # [..., half, 4, 32]
        sc = b[..., 192:208].contiguous().view(torch.int8).double().unsqueeze(-1)
        return (half(208).unsqueeze(-1) * sc * (q.double() - 32).view(n, k // 256, 16, 16)).view(n, k)
    s = b[..., 4:16].to(torch.int32)
    s0, s1, s2 = s[..., :4], s[..., 4:8], s[..., 8:]
    sc = torch.cat([s0 & 63, (s2 & 15) | (s0 >> 6) << 4], -1).double().unsqueeze(-1)
    mn = torch.cat([s1 & 63, (s2 >> 4) | (s1 >> 6) << 4], -1).double().unsqueeze(-1)
    qs = b[..., 16:].reshape(n, k // 256, 4, 1, 32)
    q = torch.cat([qs & 15, qs >> 4], 3).reshape(n, k // 256, 8, 32).double()
    return (half(0).unsqueeze(-1) * sc * q - half(2).unsqueeze(-1) * mn).view(n, k)


def _quantized(x, kind):
    """f64 values of f32 rows after the quantization a `kind` weight multiplies against."""
    m, k = x.shape
    if kind == "q8_0":
        b = x.float().view(m, k // 32, 32)
        d = b.abs().amax(-1, keepdim=True) / torch.tensor(127.0, device=x.device)
        inv = torch.where(d > 0, 1.0 / d, torch.zeros_like(d))
        v = (b * inv).double()
        scale = d.half().double()
    else:
        b = x.float().view(m, k // 256, 256)
        at = b.abs().argmax(-1, keepdim=True)
        mx = b.gather(-1, at)
        inv = torch.where(mx != 0, -128.0 / mx, torch.zeros_like(mx))
        v = (inv * b).double()
        scale = torch.where(mx != 0, 1.0 / inv, torch.zeros_like(mx)).double()
    q = torch.sign(v) * torch.floor(v.abs() + 0.5)  # ties away from zero
    return (q.clamp(-128, 127) * scale).view(m, k)


def _matmul(x, kind, n, k, seed, tag, std=0.02):
    """x @ W^T in f64 over the quantized rows, a slice of the weight's rows at a time."""
    b = _weight(kind, n, k, seed, tag, std)
    xq = _quantized(x, kind)
    rows = max(1, (1 << 26) // k)
    return torch.cat([xq @ _dequantize(b[r:r + rows], kind, min(rows, n - r), k).t() for r in range(0, n, rows)], 1)


def _silu(v):
    return v / (1 + torch.exp(-v))


def _exact_moe(case, seed):
    t, e, h, f, k = (case[x] for x in ("tokens", "experts", "hidden", "ffn", "topk"))
    x, logits = _randn(seed, 4, (t, h)), _randn(seed, 5, (t, e)).double()
    p = torch.softmax(logits, -1)
    top, at = torch.topk(p, k, dim=-1)
    top = top / top.sum(-1, keepdim=True)
    gate, up = (_weight("q4k", e * f, h, seed, i) for i in (1, 2))
    down = _weight("q6k", e * h, f, seed, 3)
    out = torch.zeros((t, h), dtype=torch.float64, device=DEV)
    for i in range(e):
        tok, slot = torch.nonzero(at == i, as_tuple=True)
        if not tok.numel():
            continue
        xq = _quantized(x[tok], "q4k")
        g = xq @ _dequantize(gate[i * f:(i + 1) * f], "q4k", f, h).t()
        u = xq @ _dequantize(up[i * f:(i + 1) * f], "q4k", f, h).t()
        y = _quantized(_silu(g) * u, "q6k") @ _dequantize(down[i * h:(i + 1) * h], "q6k", h, f).t()
        out.index_add_(0, tok, y * top[tok, slot].unsqueeze(-1))
    if case["shared"]:
        fs = case["shared"]
        g, u = (_matmul(x, "q4k", fs, h, seed, i) for i in (6, 7))
        y = _matmul(_silu(g) * u, "q6k", h, fs, seed, 8)
        out += y * torch.sigmoid(x.double() @ _randn(seed, 9, (h,), 0.02).double()).unsqueeze(-1)
    return out


def _exact_attention(q, kc, vc, first, kv_heads, hd):
    """Causal attention of rows at positions first.. against the caches, f64, a few heads at a time."""
    rows = q.shape[0]
    heads = q.shape[1] // hd
    last = first + rows
    mask = torch.arange(last, device=q.device).unsqueeze(0) > torch.arange(first, last, device=q.device).unsqueeze(1)
    out = torch.empty((rows, heads, hd), dtype=torch.float64, device=q.device)
    for h in range(heads):
        g = h // (heads // kv_heads)
        sc = q.view(rows, heads, hd)[:, h].double() @ kc[g, :last].double().t() * hd ** -0.5
        out[:, h] = torch.softmax(sc.masked_fill(mask, -math.inf), -1) @ vc[g, :last].double()
    return out.view(rows, heads * hd)


def _rotate(x, cos, sin):
    half = x.shape[-1] // 2
    return x * cos + torch.cat([-x[..., half:], x[..., :half]], -1) * sin


def _model_angles(cfg, rows):
    """cos / sin [rows, 1, head_dim] of the scaled rotary frequencies, the angles in f32 as the model has them."""
    f = np.float32
    inv = np.empty(cfg.head_dim // 2, dtype=f)
    low, high = f(cfg.rope_orig_ctx) / f(cfg.rope_low), f(cfg.rope_orig_ctx) / f(cfg.rope_high)
    for i in range(inv.size):
        v = f(1) / np.power(f(cfg.rope_theta), f(2 * i) / f(cfg.head_dim), dtype=f)
        length = f(2) * f(math.pi) / v
        if length > low:
            v = v / f(cfg.rope_factor)
        elif length >= high:
            a = (f(cfg.rope_orig_ctx) / length - f(cfg.rope_low)) / (f(cfg.rope_high) - f(cfg.rope_low))
            v = (f(1) - a) * v / f(cfg.rope_factor) + a * v
        inv[i] = v
    a = np.arange(rows, dtype=f)[:, None] * inv[None, :]
    a = torch.from_numpy(np.concatenate([a, a], 1).astype(f)).to(DEV).double()
    return torch.cos(a).float().double().unsqueeze(1), torch.sin(a).float().double().unsqueeze(1)


def _exact_model(case, seed):
    cfg = _config(case)
    sh = cfg.shapes()
    rows, hd = case["tokens"], cfg.head_dim
    x = _embed(cfg, seed)[torch.tensor(_prompt(case, cfg, seed), device=DEV)].double()
    cos, sin = _model_angles(cfg, rows)
    cache = torch.zeros((2, cfg.layers, cfg.kv_heads, _max_seq(case), hd), dtype=torch.float64, device=DEV)

    def norm(v, w):
        return v / torch.sqrt((v * v).mean(-1, keepdim=True) + cfg.eps) * w.double()

    for li in range(cfg.layers):
        def mm(v, p):
            return _matmul(v, _part(cfg, p), *sh[p], seed, 16 * li + PARTS.index(p), _std(cfg, p))

        n = norm(x, _norm(seed, 8000 + li, cfg.hidden))
        q = _rotate(mm(n, "q").view(rows, cfg.heads, hd), cos, sin)
        k = _rotate(mm(n, "k").view(rows, cfg.kv_heads, hd), cos, sin)
        v = mm(n, "v").view(rows, cfg.kv_heads, hd)
        cache[0, li, :, :rows], cache[1, li, :, :rows] = k.transpose(0, 1), v.transpose(0, 1)
        att = _exact_attention(q.reshape(rows, -1), cache[0, li], cache[1, li], 0, cfg.kv_heads, hd)
        x = x + mm(att, "o")
        n = norm(x, _norm(seed, 8100 + li, cfg.hidden))
        x = x + mm(_silu(mm(n, "gate")) * mm(n, "up"), "down")
    if case["kind"] == "model_prefill":
        x = x[-1:]
    n = norm(x, _norm(seed, 8200, cfg.hidden))
    return {"logits": _matmul(n, _part(cfg, "head"), *sh["head"], seed, 6000), "k": cache[0], "v": cache[1]}


def exact(case, seed):
    kind = case["kind"]
    if kind == "quantize":
        return None  # a search over codes and scales: it has no value in 64 bits
    if kind == "moe":
        return _exact_moe(case, seed)
    if kind == "prefill_attention":
        q, kc, vc = _attention_inputs(case, seed, case["count"], _span(case))
        return _exact_attention(q, kc, vc, case["first"], case["kv_heads"], case["head_dim"])
    if kind == "decode_attention":
        kv, hd, p = case["kv_heads"], case["head_dim"], case["pos"]
        q, kc, vc = (t.double() for t in _attention_inputs(case, seed, 1, _span(case)))
        cos, sin = (t[p].double() for t in _angles(_span(case), hd))
        k, v = _rotate(_randn(seed, 4, (kv, hd)).double(), cos, sin), _randn(seed, 5, (kv, hd)).double()
        kc[:, p], vc[:, p] = k, v
        q = _rotate(q.view(-1, hd), cos, sin).view(1, -1)
        return {"out": _exact_attention(q, kc, vc, p, kv, hd).view(-1, hd), "k": k, "v": v}
    if kind.startswith("model"):
        return _exact_model(case, seed)
    n, k = case["n"], case["k"]
    x, dt = _randn(seed, 2, (case["m"], k)).to(DENSE[case["x"]]), DENSE[case["x"]]
    if kind == "dense":
        w = _dequantize(_weight(case["type"], n, k, seed, 1), case["type"], n, k).to(dt).double()
        return x.double() @ w.t() + _randn(seed, 3, (n,)).to(dt).double()
    y = _matmul(x.float(), case["type"], n, k, seed, 1)
    return y if case["x"] == "f32" else y + _randn(seed, 3, (n,)).to(dt).double()
