"""The work that a user of the library has it do, as cases that can be timed.

Each case is one pass through the public Python entry points on an MI355X:
whole cache sessions (prefill, attention over the prompt, decode steps),
decode steps over long and ragged caches, the cache codec in both directions,
prefill attention, the core vector codec and the QJL estimator.  `listed()`
holds the fixed cases, `draw()` gives more of the same ranges, `exact()` the
same results in 64-bit arithmetic from plain torch.

Shapes follow the configurations that bench.py and the tests use: 16 query
heads over 8 KV heads of 128 elements and 32 over 8, codes of 2 to 4 bits,
contexts up to 32,768 tokens (twice that where few heads keep it small).
"""
import math

import numpy as np
import torch

import turboquant_amd as tq

DTYPES = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}
ROT_SEED, QJL_SEED = 42, 12345  # the caches' default seeds


def listed():
    return [
        # a short chat turn: latency and launches (2 of a model's layers)
        {"name": "chat_pqo3", "kind": "chat", "mode": "pqo", "bits": 3, "dim": 128, "heads": 16, "kv_heads": 8,
         "prompt": 77, "steps": 4, "layers": 2, "dtype": "bf16"},
        # the same through a TqCache with small heads and more query heads per KV head
        {"name": "chat_tq4_d64", "kind": "chat", "mode": "tq", "bits": 4, "dim": 64, "heads": 8, "kv_heads": 2,
         "prompt": 150, "steps": 4, "layers": 2, "dtype": "f16"},
        # one token over 8 layers' full 32K contexts, batch 1
        {"name": "decode_pqo3_32k", "kind": "decode", "mode": "pqo", "bits": 3, "dim": 128, "heads": 16,
         "kv_heads": 8, "batch": 1, "ctx": 32768, "ragged": False, "layers": 8, "dtype": "bf16"},
        # a serving batch of 16 sequences of different lengths
        {"name": "decode_pqo4_batch16", "kind": "decode", "mode": "pqo", "bits": 4, "dim": 128, "heads": 32,
         "kv_heads": 8, "batch": 16, "ctx": 16384, "ragged": True, "layers": 1, "dtype": "bf16"},
        # TQ records (with the QJL correction of the logits), a small ragged batch
        {"name": "decode_tq3_batch3", "kind": "decode", "mode": "tq", "bits": 3, "dim": 128, "heads": 32,
         "kv_heads": 8, "batch": 3, "ctx": 6001, "ragged": True, "layers": 2, "dtype": "bf16"},
        # a 28-layer model's 4,096-token prompt into records
        {"name": "quantize_pqo3", "kind": "quantize", "mode": "pqo", "bits": 3, "dim": 128, "n": 1835008,
         "dtype": "bf16"},
        # records back to activations (the contract of a later prefill)
        {"name": "dequantize_pqo4", "kind": "dequantize", "mode": "pqo", "bits": 4, "dim": 128, "n": 300001,
         "dtype": "f16"},
        # a whole prompt's causal attention straight over the records
        {"name": "prefill_pqo3_4096", "kind": "prefill", "mode": "pqo", "bits": 3, "dim": 128, "heads": 16,
         "kv_heads": 8, "q_len": 4096, "ctx": 4096, "causal": True, "dtype": "bf16"},
        # a ragged chunk of a prompt at the end of a long TQ context
        {"name": "prefill_tq3_chunk", "kind": "prefill", "mode": "tq", "bits": 3, "dim": 128, "heads": 32,
         "kv_heads": 8, "q_len": 500, "ctx": 20001, "causal": True, "dtype": "f16"},
        # two prompt chunks into a TqCache: records, sketch, logit bias, dequantized layer
        {"name": "extend_tq3", "kind": "extend", "mode": "tq", "bits": 3, "dim": 128, "heads": 16, "kv_heads": 8,
         "first": 1024, "second": 513, "dtype": "bf16"},
        # the QJL estimator as attention: sketch keys and values, 64 queries' scores, softmax, weighted values
        {"name": "qjl_8192x64", "kind": "qjl", "bits": 3, "dim": 128, "keys": 8192, "queries": 64},
        # the core vector codec, both directions
        {"name": "codec_10000", "kind": "codec", "bits": 3, "dim": 128, "n": 10000},
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.4)))))))


def draw(rng):
    kind = rng.choice(["chat", "decode", "decode", "quantize", "dequantize", "prefill", "prefill", "extend", "qjl",
                       "codec"])
    mode = rng.choice(["pqo", "pqo", "pq", "tq"])
    bits, dim, dtype = rng.choice([3, 4]), rng.choice([64, 128, 128, 256]), rng.choice(["bf16", "bf16", "f16", "f32"])
    kv_heads, group = rng.choice([1, 2, 4, 8]), rng.choice([1, 2, 4, 8])
    case = {"kind": kind, "mode": mode, "bits": bits, "dim": dim, "heads": kv_heads * group, "kv_heads": kv_heads}
    if kind == "chat":
        return {**case, "prompt": _log(rng, 1, 1500), "steps": rng.randint(1, 6), "layers": rng.randint(1, 3),
                "dtype": dtype}
    if kind == "decode":
        batch = _log(rng, 1, 16)
        most = 32768 * 8 * 128 // (batch * kv_heads * dim)
        return {**case, "batch": batch, "ctx": _log(rng, 64, min(65536, most)), "ragged": rng.random() < 0.5,
                "layers": rng.randint(1, 3), "dtype": dtype}
    if kind in ("quantize", "dequantize"):
        dim = rng.choice([64, 96, 128, 256])
        most = {"quantize": 1800000, "dequantize": 900000}[kind] * 64 // dim
        return {"kind": kind, "mode": "pqo" if mode == "tq" else mode, "bits": bits, "dim": dim,
                "n": _log(rng, 1, most), "dtype": dtype}
    if kind == "prefill":
        group = rng.choice([1, 2, 4])
        ctx = _log(rng, 64, 16384)
        return {**case, "dim": 128, "heads": kv_heads * group, "ctx": ctx,
                "q_len": _log(rng, 2, min(ctx, 300000000 // (ctx * kv_heads * group))),
                "causal": rng.random() < 0.8, "dtype": dtype}
    if kind == "extend":
        return {**case, "mode": "pqo" if mode == "pq" else mode, "first": _log(rng, 16, 1200),
                "second": _log(rng, 1, 600), "dtype": dtype}
    if kind == "qjl":
        return {"kind": kind, "bits": bits, "dim": rng.choice([32, 64, 128, 128]), "keys": _log(rng, 1, 16384),
                "queries": _log(rng, 1, 64)}
    dim = rng.choice([32, 64, 128, 256])
    return {"kind": kind, "bits": rng.choice([2, 3, 4]), "dim": dim, "n": _log(rng, 1, 6400000 // dim)}


# ---------------------------------------------------------------- inputs

def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _kv(gen, heads, tokens, dim, dtype):
    """N(0,1) keys or values with four channels a head eight times as large, as key caches have them."""
    x = torch.randn((heads, tokens, dim), generator=gen, device="cuda")
    ch = torch.rand((heads, dim), generator=gen, device="cuda").argsort(1)[:, :4]
    m = torch.ones((heads, dim), device="cuda").scatter_(1, ch, 8.0)
    return (x * m[:, None, :]).to(DTYPES[dtype])


def _lengths(case, seed):
    b, ctx = case["batch"], case["ctx"]
    if not case["ragged"]:
        return [ctx] * b
    return np.random.default_rng(seed).integers(max(1, ctx // 4), ctx + 1, size=b).tolist()


def _outliers(mode):
    return tq.cache.OUTLIER_ALL if mode == "pqo" else 0


def _cache(case, layers):
    config = tq.CacheConfig(bits=case["bits"], head_dim=case["dim"], num_kv_heads=case["kv_heads"],
                            num_layers=layers, outlier_blocks=_outliers(case["mode"]))
    return (tq.TqCache if case["mode"] == "tq" else tq.PqoCache)(config)


def _queries(gen, shape, dtype):
    return torch.randn(shape, generator=gen, device="cuda").to(DTYPES[dtype])


def _chat_inputs(case, seed):
    """Per layer: prompt K, V, q, then one (K, V, q) per step."""
    g, c = _gen(seed), case
    layers = []
    for _ in range(c["layers"]):
        k, v = (_kv(g, c["kv_heads"], c["prompt"] + c["steps"], c["dim"], c["dtype"])[None] for _ in range(2))
        q = _queries(g, (1, c["heads"], c["prompt"] + c["steps"], c["dim"]), c["dtype"])
        cut = [c["prompt"]] + [1] * c["steps"]
        layers.append([tuple(t.contiguous() for t in p) for p in
                       zip(k.split(cut, 2), v.split(cut, 2), q.split(cut, 2))])
    return layers


def _extend_inputs(case, seed):
    g, c = _gen(seed), case
    return [(_kv(g, c["kv_heads"], t, c["dim"], c["dtype"])[None], _kv(g, c["kv_heads"], t, c["dim"], c["dtype"])[None],
             _queries(g, (1, c["heads"], t, c["dim"]), c["dtype"])) for t in (c["first"], c["second"])]


def _decode_inputs(case, seed):
    """Per layer: queries and the K and V of each sequence, one (sequence, layer) at a time."""
    g, c = _gen(seed), case
    lens = _lengths(c, seed)
    for layer in range(c["layers"]):
        q = _queries(g, (c["batch"], c["heads"], c["dim"]), c["dtype"])
        for b in range(c["batch"]):
            yield layer, b, lens[b], q, *(_kv(g, c["kv_heads"], lens[b], c["dim"], "bf16") for _ in range(2))


def _prefill_inputs(case, seed):
    g, c = _gen(seed), case
    return (_queries(g, (c["heads"], c["q_len"], c["dim"]), c["dtype"]),
            *(_kv(g, c["kv_heads"], c["ctx"], c["dim"], "bf16") for _ in range(2)))


def _attends(case):
    """Whether attention over a prompt can be had straight from the records."""
    return case["dim"] == 128 and case["heads"] // case["kv_heads"] in (1, 2, 4)


def prepare(case, seed):
    c, kind = case, case["kind"]
    state = {"case": c}
    if kind == "chat":
        state.update(cache=_cache(c, c["layers"]), layers=_chat_inputs(c, seed))
    elif kind == "extend":
        state.update(cache=_cache(c, 1), chunks=_extend_inputs(c, seed))
    elif kind == "decode":
        bsz, hk, d, cap, bits = c["batch"], c["kv_heads"], c["dim"], c["ctx"], c["bits"]
        layers = []
        for layer, b, t, q, k, v in _decode_inputs(c, seed):
            if b == 0:
                idx = [torch.zeros((bsz, hk, cap, d * bits // 8), dtype=torch.uint8, device="cuda") for _ in range(2)]
                sc = [torch.zeros((bsz, hk, cap, d // 32), dtype=torch.int16, device="cuda") for _ in range(2)]
                sg = torch.zeros((bsz, hk, cap, d // 8), dtype=torch.uint8, device="cuda")
                nm = torch.zeros((bsz, hk, cap), dtype=torch.int16, device="cuda")
                layers.append((q, idx, sc, sg, nm))
            for i, x in enumerate((k, v)):
                r = _encode(x, bits, c["mode"])
                idx[i][b, :, :t], sc[i][b, :, :t] = r["packed"], r["scales"]
                if i == 0 and c["mode"] == "tq":
                    sg[b, :, :t], nm[b, :, :t] = _sketch(x, r)
        lens = torch.tensor(_lengths(c, seed), dtype=torch.int32, device="cuda")
        state.update(layers=layers, lens=lens, ws=tq.AttentionWorkspace(bsz, c["heads"], hk, d, cap),
                     rmat=tq.qjl_sign_matrix(d, QJL_SEED) if c["mode"] == "tq" else None)
    elif kind == "quantize":
        state.update(x=_kv(_gen(seed), 1, c["n"], c["dim"], c["dtype"])[0])
    elif kind == "dequantize":
        r = _encode(_kv(_gen(seed), 1, c["n"], c["dim"], "bf16"), c["bits"], c["mode"])
        state.update(packed=r["packed"][0], scales=r["scales"][0])
    elif kind == "prefill":
        q, k, v = _prefill_inputs(c, seed)
        rk, rv = _encode(k, c["bits"], c["mode"]), _encode(v, c["bits"], c["mode"])
        sg, nm = _sketch(k, rk) if c["mode"] == "tq" else (None, None)
        state.update(q=q, recs=(rk["packed"], rk["scales"], rv["packed"], rv["scales"]), sg=sg, nm=nm,
                     rmat=tq.qjl_sign_matrix(c["dim"], QJL_SEED) if c["mode"] == "tq" else None)
    elif kind == "qjl":
        g = _gen(seed)
        state.update(zip(("k", "v", "q"), (torch.randn((n, c["dim"]), generator=g, device="cuda")
                                           for n in (c["keys"], c["keys"], c["queries"]))))
    else:
        state.update(x=torch.randn((c["n"], c["dim"]), generator=_gen(seed), device="cuda"))
    return state


# ---------------------------------------------------------------- one pass

def run(state):
    return globals()["_run_" + state["case"]["kind"]](state, state["case"])


def _run_chat(s, c):
    cache, scale = s["cache"], c["dim"] ** -0.5
    cfg = tq.AttendConfig(scale, c["heads"] // c["kv_heads"])
    cache.reset()
    out = []
    for step in range(c["steps"] + 1):
        for layer, parts in enumerate(s["layers"]):
            k, v, q = parts[step]
            if step:
                out.append(cache.decode(layer, k, v, q, cfg))
                continue
            r = cache.prefill(layer, k, v, q)
            if _attends(c):
                out.append(cache.attend_prefill(layer, q, scale))
            elif r.logit_bias is not None:
                out.append(r.logit_bias)
    return out


def _run_extend(s, c):
    s["cache"].reset()
    first, second = (s["cache"].prefill(0, *chunk) for chunk in s["chunks"])
    out = {"k": second.k, "v": second.v}
    if c["mode"] == "tq":
        out.update(bias1=first.logit_bias, bias2=second.logit_bias)
    return out


def _run_decode(s, c):
    out, cap = [], c["ctx"]
    for q, (ki, vi), (ks, vs), sg, nm in s["layers"]:
        args = (q, ki, ks, vi, vs, s["lens"], c["kv_heads"], c["bits"], cap, cap, c["kv_heads"] * cap,
                c["dim"] ** -0.5, s["ws"])
        if c["mode"] == "pqo":
            out.append(tq.pqo_decode_attention(*args))
        elif c["mode"] == "pq":
            out.append(tq.cache_decode_attention(*args, 0))
        else:
            out.append(tq.cache_decode_attention(*args, 0, None, sg, nm, qjl_sign_matrix=s["rmat"]))
    return out


def _run_quantize(s, c):
    return tq.polar_quantize(s["x"], c["bits"], _outliers(c["mode"]))


def _run_dequantize(s, c):
    return tq.polar_dequantize(s["packed"], s["scales"], c["bits"], c["dim"], _outliers(c["mode"]),
                               out_dtype=DTYPES[c["dtype"]])


def _run_prefill(s, c):
    rq = None
    if c["mode"] == "tq":
        rq = tq.qjl_project(s["q"].view(-1, c["dim"]), s["rmat"]).view(s["q"].shape)
    return tq.cache_prefill_attention(s["q"], *s["recs"], c["kv_heads"], c["bits"], c["ctx"], c["ctx"],
                                      c["dim"] ** -0.5, _outliers(c["mode"]), c["causal"], rq, s["sg"], s["nm"],
                                      out_dtype=DTYPES[c["dtype"]])


def _run_qjl(s, c):
    b, d = c["bits"], c["dim"]
    kr = tq.qjl_quantize_batch(s["k"], b, ROT_SEED, QJL_SEED)
    vr = tq.qjl_quantize_batch(s["v"], b, ROT_SEED, QJL_SEED)
    ctx = tq.qjl_query_context(s["q"], ROT_SEED, QJL_SEED)
    scores = tq.qjl_scores(ctx, *kr, b - 1, ROT_SEED)
    probs = tq.softmax_rows(scores, d ** -0.5)
    out = tq.qjl_weighted_values(vr[0], vr[1], probs, b - 1, d, ROT_SEED)
    return {"keys": kr, "values": vr, "ctx": ctx, "scores": scores, "probs": probs, "out": out}


def _run_codec(s, c):
    packed, scales = tq.quantize_vec_batch(s["x"], c["bits"], ROT_SEED)
    back = tq.dequantize_vec_batch(packed, scales, c["bits"], c["dim"], ROT_SEED)
    return {"packed": packed, "scales": scales, "back": back,
            "rotated": tq.dequantize_rotated_batch(packed, scales, c["bits"], c["dim"])}


# ---------------------------------------------------------------- what a pass cannot do without

def work(case):
    c, kind = case, case["kind"]
    size = {"f32": 4, "bf16": 2, "f16": 2}[c.get("dtype", "f32")]
    d = c["dim"]
    rec = d * c["bits"] // 8 + 2 * (d // 32)          # bytes of one stored vector
    krec = rec + (d // 8 + 2 if c.get("mode") == "tq" else 0)
    if kind == "quantize" or kind == "dequantize":
        return {"bytes": c["n"] * (d * size + rec), "flops": c["n"] * d * 6}
    if kind == "codec":
        n, packed = c["n"], d * c["bits"] // 8 + 2
        return {"bytes": n * (3 * 4 * d + 3 * packed), "flops": n * d * (2 * math.log2(d) + 6)}
    if kind == "qjl":
        n, q = c["keys"], c["queries"]
        row = d * (c["bits"] - 1) // 8 + 2 + d // 8 + 2
        return {"bytes": 2 * n * (4 * d + row) + n * (2 * row - d // 8 - 2) + q * (8 * n + 4 * d * 4),
                "flops": 2 * n * 2 * d * d + 2 * d * d * q + 6 * q * n * d + 6 * q * n}
    hq, hk = c["heads"], c["kv_heads"]
    if kind == "decode":
        tokens = c["layers"] * sum(_lengths(c, 0))
        return {"bytes": tokens * hk * (krec + rec) + c["layers"] * c["batch"] * hq * d * (size + 4),
                "flops": tokens * hq * d * (6 if c["mode"] == "tq" else 4)}
    if kind == "prefill":
        ql, t = c["q_len"], c["ctx"]
        pairs = ql * (t - ql) + ql * (ql + 1) // 2 if c["causal"] else ql * t
        return {"bytes": t * hk * (krec + rec) + 2 * hq * ql * d * size,
                "flops": pairs * hq * d * (6 if c["mode"] == "tq" else 4)}
    if kind == "chat":
        p, n = c["prompt"], c["steps"]
        tokens = p + n
        read = sum(p + 1 + i for i in range(n)) * hk * (krec + rec)
        b = tokens * hk * (2 * d * size + krec + rec) + read + (tokens + n) * hq * d * size
        f = sum(p + 1 + i for i in range(n)) * hq * d * 4 + p * p * hq * d * 2
        return {"bytes": c["layers"] * b, "flops": c["layers"] * f}
    one, two = c["first"], c["second"]
    total = one + two
    b = total * hk * (2 * d * size + krec + rec) + total * hk * (rec + rec + 2 * d * size)
    f = 0
    if c["mode"] == "tq":
        b += total * hq * d * size + (one * one + two * total) * hq * size + total * hk * (d // 8 + 2)
        f = 2 * d * hq * (one * one + two * total) + 2 * d * d * total * (hk + hq)
    return {"bytes": b, "flops": f + total * hk * d * 24}


def tolerance(case):
    """About four times the distance from `exact()` that was measured.  Codes, scales, signs and norms are fixed by the
    format; f32 results carry the order of f32 sums and products of 22 significant bits; 16-bit results one rounding of
    the output; decoding 4-bit PQO records, whose codes are contracted before their offset is taken off, 1.1e-3."""
    kind, dtype = case["kind"], case.get("dtype", "f32")
    if kind in ("quantize", "codec"):
        return "exact"
    if kind == "qjl":
        return {"rel": 2e-6}
    grid = kind in ("chat", "decode") and case["mode"] == "pqo" and case["bits"] == 4
    if kind == "decode" or dtype == "f32":
        return {"rel": 5e-3 if grid else 1e-5 if kind in ("chat", "decode", "prefill") else 2e-6}
    if dtype == "bf16":
        return {"rel": 8e-3 if grid else 7e-3}
    return {"rel": 5e-3 if grid else 1.2e-3}


# ---------------------------------------------------------------- the same in 64 bits
# The stored formats are defined in 32-bit arithmetic (the order of the
# rotation's butterflies, the sums of squares and the sketch's sums), so codes
# and signs are formed that way; everything computed from them is 64-bit.

SIGNS = 0xB1A6D4B2  # bit j: element j of a rotated block is negated
OUTLIER3 = ([-2.1573, -1.3336, -0.7434, -0.2428, 0.2428, 0.7434, 1.3336, 2.1573],
            [-1.7455, -1.0385, -0.4931, 0.0, 0.4931, 1.0385, 1.7455])
OUTLIER2 = ([-2.1573, -0.7434, 0.7434, 2.1573], [-1.0385, 0.0, 1.0385])


def _codebook(bits):
    """Centroids and boundaries of the cache's `bits`-bit codebook, f32 values."""
    if bits < 4:
        c, b = OUTLIER3 if bits == 3 else OUTLIER2
        return np.array(c, np.float32), np.array(b, np.float32)
    r, n = np.float32(2.1573), np.arange(16, dtype=np.float32)
    step = np.float32(np.float32(2) * r) / np.float32(15)
    return -r + n * step, -r + (n[:15] + np.float32(0.5)) * step


def _dev(a, dtype=torch.float32):
    return torch.as_tensor(np.ascontiguousarray(a), device="cuda").to(dtype)


def _signs32():
    return _dev([-1.0 if (SIGNS >> j) & 1 else 1.0 for j in range(32)])


def _butterfly(x):
    """Unnormalized Walsh-Hadamard transform of the last axis, stages from the closest pairs up, in x's type."""
    n, shape = x.shape[-1], x.shape
    h = 1
    while h < n:
        y = x.reshape(-1, n // (2 * h), 2, h)
        a, b = y[:, :, 0], y[:, :, 1]
        x = torch.stack((a + b, a - b), 2)
        h *= 2
    return x.reshape(shape)


def _pack(codes, bits):
    """Codes [..., d] as a little-endian bitstream [..., d * bits / 8]."""
    c = codes.reshape(-1, 8).to(torch.int64)
    w = sum(c[:, i] << (bits * i) for i in range(8))
    b = torch.stack([(w >> (8 * i)) & 255 for i in range(bits)], 1).to(torch.uint8)
    return b.reshape(*codes.shape[:-1], codes.shape[-1] * bits // 8)


def _f16_bits(x):
    return x.to(torch.float16).view(torch.int16)


def _bucket(v, bounds):
    return sum((v > float(b)).to(torch.uint8) for b in bounds)


def _encode(x, bits, mode):
    """Cache records of x [H, T, d]: packed codes, f16 scale bits, the codes and the scales."""
    heads, t, d = x.shape
    cent, bounds = _codebook(bits if mode == "pqo" else bits - 1)
    f = _signs32() * float(np.float32(1) / np.sqrt(np.float32(32)))
    r = _butterfly(x.float().reshape(-1, 32)) * f
    outer = np.float32(_codebook(bits)[0].max())
    s = (r.abs().amax(1) * float(np.float32(1.0 / float(outer)))).clamp_min(float(np.float32(1e-10)))
    codes = _bucket(r / s[:, None], bounds).reshape(heads, t, d)
    half = s.to(torch.float16)
    sign = -1.0 if mode == "pqo" else 1.0
    return {"packed": _pack(codes, bits), "scales": _f16_bits(half * sign).reshape(heads, t, d // 32), "codes": codes,
            "s": half.reshape(heads, t, d // 32), "cent": cent}


def _decoded(r, dtype=torch.float64):
    """The vectors that records stand for, [H, T, d]."""
    z = _dev(r["cent"])[r["codes"].long()].to(dtype)
    shape = z.shape
    if dtype == torch.float32:  # the record format's own steps
        inv = np.float32(1) / np.sqrt(np.float32(32))
        y = _butterfly(z.reshape(-1, 32) * (_signs32() * float(inv * np.sqrt(np.float32(32))))) * float(inv)
        return (y * r["s"].reshape(-1, 1).float()).reshape(shape)
    y = _butterfly(z.reshape(-1, 32) * _signs32().double()) / math.sqrt(32.0)
    return (y * r["s"].reshape(-1, 1).double()).reshape(shape)


def _rademacher(dim, seed=QJL_SEED):
    """The +-1 matrix of the sketch: a SplitMix64 finalizer per entry."""
    with np.errstate(over="ignore"):
        u = np.uint64
        j = np.arange(dim, dtype=u)
        m = u(seed) * u(0x517CC1B727220A95) + j
        row = m ^ (m >> u(32)) ^ u(0x6C62272E07BB0142)
        z = (row + j * u(0x9E3779B97F4A7C15))[:, None] + j[None, :]
        z = (z ^ (z >> u(30))) * u(0xBF58476D1CE4E5B9)
        z = (z ^ (z >> u(27))) * u(0x94D049BB133111EB)
        z ^= z >> u(31)
    return np.where(z & u(1), -1.0, 1.0)


def _inv_sqrt(d):
    return float(np.float32(1) / np.sqrt(np.float32(d)))


def _sketch_of(r):
    """Sign bits [N, d] and f16 norms [N] of residuals r [N, d], summed in element order."""
    n, d = r.shape
    ss, p = torch.zeros(n, device="cuda"), torch.zeros((n, d), device="cuda")
    m = _dev(_rademacher(d))
    for c in range(d):
        col = r[:, c].contiguous()
        ss = ss + col * col
        p = p + col[:, None] * m[:, c][None, :]
    return (p * _inv_sqrt(d) >= 0).to(torch.uint8), ss.sqrt().to(torch.float16)


def _sketch(x, r):
    heads, t, d = x.shape
    bits, norms = _sketch_of((x.float() - _decoded(r, torch.float32)).reshape(-1, d))
    return _pack(bits, 1).reshape(heads, t, d // 8), _f16_bits(norms).reshape(heads, t)


def _correction(q, signs, norms):
    """Logit correction of queries [H, L, d] against sketched keys ([Hk, T, d/8] bits, [Hk, T] f16 bits)."""
    heads, ql, d = q.shape
    rq = q.double().reshape(-1, d) @ _dev(_rademacher(d), torch.float64).T / math.sqrt(d)
    b = (signs[..., None] >> torch.arange(8, dtype=torch.uint8, device="cuda")) & 1
    b = b.reshape(*signs.shape[:-1], d).double() * 2 - 1
    c = norms.view(torch.float16).double() * (math.sqrt(math.pi / 2) / math.sqrt(d))
    hk = signs.shape[0]
    return (rq.reshape(hk, -1, d) @ b.transpose(1, 2) * c[:, None, :]).reshape(heads, ql, -1)


def _attention(q, k, v, scale, bias=None, causal=False):
    """softmax(scale (q k + bias)) v in f64; q [H, L, d], k and v [Hk, T, d]; queries at the last L positions."""
    heads, ql, d = q.shape
    hk, t, _ = k.shape
    out = torch.empty((heads, ql, d), dtype=torch.float64, device="cuda")
    for h in range(heads):
        g = h // (heads // hk)
        for lo in range(0, ql, 1024):
            qs = q[h, lo:lo + 1024].double()
            x = qs @ k[g].T
            if bias is not None:
                x += bias[h, lo:lo + 1024]
            x *= scale
            if causal:
                pos = torch.arange(lo, lo + qs.shape[0], device="cuda")[:, None] + (t - ql)
                x.masked_fill_(torch.arange(t, device="cuda")[None, :] > pos, -math.inf)
            out[h, lo:lo + 1024] = torch.softmax(x, 1) @ v[g]
    return out


def _layer(case, k, v, q):
    """(keys, values, correction or None) in f64 of stored k, v [Hk, T, d] for queries q [H, L, d]."""
    rk, rv = _encode(k, case["bits"], case["mode"]), _encode(v, case["bits"], case["mode"])
    bias = _correction(q, *_sketch(k, rk)) if case["mode"] == "tq" else None
    return _decoded(rk), _decoded(rv), bias


def exact(case, seed):
    return globals()["_exact_" + case["kind"]](case, seed)


def _exact_chat(c, seed):
    scale, out = c["dim"] ** -0.5, []
    layers = _chat_inputs(c, seed)
    for step in range(c["steps"] + 1):
        for parts in layers:
            k, v = (torch.cat([p[i][0] for p in parts[:step + 1]], 1) for i in (0, 1))
            q = parts[step][2][0]
            kd, vd, bias = _layer(c, k, v, q)
            if step or _attends(c):
                out.append(_attention(q, kd, vd, scale, bias, causal=not step)[None])
            elif bias is not None:
                out.append(bias[None])
    return out


def _exact_extend(c, seed):
    (k0, v0, q0), (k1, v1, q1) = _extend_inputs(c, seed)
    k, v = torch.cat((k0, k1), 2)[0], torch.cat((v0, v1), 2)[0]
    kd, vd, bias = _layer(c, k, v, q1[0])
    out = {"k": kd[None], "v": vd[None]}
    if c["mode"] == "tq":
        out.update(bias1=_layer(c, k0[0], v0[0], q0[0])[2][None], bias2=bias[None])
    return out


def _exact_decode(c, seed):
    rows = {}
    for layer, b, t, q, k, v in _decode_inputs(c, seed):
        kd, vd, bias = _layer(c, k, v, q[b][:, None, :])
        rows.setdefault(layer, []).append(_attention(q[b][:, None, :], kd, vd, c["dim"] ** -0.5, bias)[:, 0])
    return [torch.stack(r) for r in rows.values()]


def _exact_quantize(c, seed):
    return None  # codes and scale bits: whole numbers


def _exact_dequantize(c, seed):
    return _decoded(_encode(_kv(_gen(seed), 1, c["n"], c["dim"], "bf16"), c["bits"], c["mode"]))[0]


def _exact_prefill(c, seed):
    q, k, v = _prefill_inputs(c, seed)
    kd, vd, bias = _layer(c, k, v, q)
    return _attention(q, kd, vd, c["dim"] ** -0.5, bias, c["causal"])


# The core codec's positive centroids and boundaries, by (bits, dim): the
# Lloyd-Max quantizer of a rotated unit vector's elements.
CORE = {
    (2, 32): ([0.07980195923950428, 0.2633194690486460], [0.1715607141440753]),
    (2, 64): ([0.05651489047635316, 0.18749689292196107], [0.12200589169915712]),
    (2, 128): ([0.03999160906335884, 0.13304154846077333], [0.08651657876206609]),
    (2, 256): ([0.02828860721372156, 0.09423779913129649], [0.06126320317250903]),
    (3, 32): ([0.04285157006670087, 0.1317562436100486, 0.23246076086351817, 0.3662684197149948],
              [0.08730390683837475, 0.1821085022367834, 0.299364590289256]),
    (3, 64): ([0.03046922045737837, 0.0938323758441605, 0.16616801009118487, 0.26391407457137683],
              [0.06215079815076943, 0.13000019296767268, 0.21504104233128085]),
    (3, 128): ([0.02160433847349997, 0.06658568378325364, 0.11813986946554235, 0.18839728518004373],
               [0.0440950111283768, 0.09236277662439799, 0.15326857732279303]),
    (3, 256): ([0.01529750782483941, 0.04716676527922715, 0.0837655314597689, 0.13385436276083063],
               [0.03123213655203328, 0.06546614836949802, 0.10880994711029976]),
    (4, 32): ([0.02235501645565882, 0.06749924527967028, 0.1140141752861917, 0.16307095286109712, 0.2163621312970216,
               0.2767423715764117, 0.3500919292405678, 0.4535648440640392],
              [0.04492713086766455, 0.090756710282931, 0.1385425640736444, 0.18971654207905935, 0.24655225143671666,
               0.3134171504084897, 0.401828386652303]),
    (4, 64): ([0.0159419303520814, 0.04815672368589858, 0.08141753279040376, 0.11662310388676207, 0.15508179062990365,
               0.19901983361887085, 0.25307088610074774, 0.33092994168409773],
              [0.03204932701898999, 0.06478712823815116, 0.09902031833858291, 0.13585244725833287,
               0.17705081212438725, 0.22604535985980928, 0.2920004138924227]),
    (4, 128): ([0.01132093590150223, 0.03420549908335103, 0.05785765497830671, 0.08293881469006784,
                0.11041538921898804, 0.14193912272806147, 0.18096588552769086, 0.23777655506958537],
               [0.02276321749242663, 0.04603157703082887, 0.07039823483418728, 0.09667710195452794,
                0.12617725597352475, 0.16145250412787615, 0.2093712202986381]),
    (4, 256): ([0.00802245010411462, 0.02424206232116148, 0.04101444098641885, 0.05881658417438018,
                0.07834675699488723, 0.10080108457584613, 0.12868871755030106, 0.16949853314441155],
               [0.01613225621263805, 0.03262825165379016, 0.04991551258039952, 0.06858167058463371,
                0.08957392078536669, 0.1147449010630736, 0.14909362534735632]),
}


def _core(x, bits):
    """The core codec on rows x [N, d]: codes, centroids, f16 norms (ROT_SEED is even: signs +, -, +, ...)."""
    n, d = x.shape
    ss = torch.zeros(n, device="cuda")
    for c in range(d):
        col = x[:, c].contiguous()
        ss = ss + col * col
    norm = ss.sqrt()
    alt = _dev([1.0, -1.0] * (d // 2))
    r = _butterfly(x * (1.0 / norm)[:, None] * alt) * _inv_sqrt(d)
    pos, cut = CORE[bits, d]
    codes = _bucket(r.double(), [-b for b in reversed(cut)] + [0.0] + list(cut))
    return codes, np.array([-p for p in reversed(pos)] + list(pos), np.float32), norm.to(torch.float16)


def _core_decoded(codes, cent, norm, dtype=torch.float64, rotate=True):
    z = _dev(cent)[codes.long()].to(dtype)
    d = z.shape[1]
    if rotate:
        alt = _dev([1.0, -1.0] * (d // 2), dtype)
        z = _butterfly(z) * (_inv_sqrt(d) if dtype == torch.float32 else 1 / math.sqrt(d)) * alt
    return z * norm.to(dtype)[:, None]


def _exact_qjl(c, seed):
    g = _gen(seed)
    k, v, q = (torch.randn((n, c["dim"]), generator=g, device="cuda") for n in (c["keys"], c["keys"], c["queries"]))
    d = c["dim"]
    codes, cent, norm = _core(k, c["bits"] - 1)
    bits, rn = _sketch_of(k - _core_decoded(codes, cent, norm, torch.float32))
    rq = q.double() @ _dev(_rademacher(d), torch.float64).T / math.sqrt(d)
    alt = _dev([1.0, -1.0] * (d // 2), torch.float64)
    qt = _butterfly(q.double() * alt) / math.sqrt(d)
    est = q.double() @ _core_decoded(codes, cent, norm).T
    est += rq @ (bits.double() * 2 - 1).T * (rn.double() * (math.sqrt(math.pi / 2) / math.sqrt(d)))[None, :]
    probs = torch.softmax(est * d ** -0.5, 1)
    none = [None] * 4
    return {"keys": none, "values": none, "ctx": torch.cat((qt, rq), 1), "scores": est, "probs": probs,
            "out": probs @ _core_decoded(*_core(v, c["bits"] - 1))}


def _exact_codec(c, seed):
    r = _core(torch.randn((c["n"], c["dim"]), generator=_gen(seed), device="cuda"), c["bits"])
    return {"packed": None, "scales": None, "back": _core_decoded(*r), "rotated": _core_decoded(*r, rotate=False)}
