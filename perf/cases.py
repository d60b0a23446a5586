"""Performance cases: what a program does with this framework, through its public entry points.

Every case is TinyLlama-1.1B-shape (22 layers, hidden 2048, 32 query / 4 KV heads of 64, FFN 5632, vocabulary
32000, 2048 positions), the configuration of bench.py and of the full-size tests, with random N(0, 0.02) weights
quantized per output channel.  Layer cases use an engine of one layer, whole calls all 22.

Ranges (`draw` spreads over them):
  decode_layer  one token through one layer, 0 .. 2047 cached rows
  layer_rows    2 .. 2048 consecutive tokens of one sequence through one layer, behind 0 .. 2046 cached rows
  lm_head       one row through the final RMSNorm, an LM head of 1024 .. 32000 ids and the argmax, logits out
  score         a prompt of 2 .. 640 tokens through all layers, logits of every position out
  generate      a prompt of 1 .. 512 tokens scored, then 1 .. 64 greedy tokens
  batch         2 .. 128 sequences with 0 .. 2000 cached rows each (ragged), 2 .. 32 greedy steps together
  gemm          INT8 GEMM + dequantization (+ residual) of 2 .. 2048 rows by one projection's weights
  linear_f32    one float32 projection of 1 .. 640 rows (the float model of the analysis report)

The INT8 path fixes every rounding and every order of summation (per-row INT8 activations, exact INT32 sums,
float32 steps without contraction, softmax sums per 64-key block), so its results are the same bits in any correct
implementation: tolerance "exact".  The float32 projection has no fixed order of summation.
"""
from __future__ import annotations

import ctypes
import math
import random

import numpy as np
import torch

from __graft_entry__ import load_package

lpta = load_package()

D, F, V, HEADS, KV_HEADS, HD, MAX_POS, LAYERS = 2048, 5632, 32000, 32, 4, 64, 2048, 22
KVD = KV_HEADS * HD
QKV = D + 2 * KVD
EPS = np.float32(1e-5)
# [N, K] of the projections: Q|K|V, O, gate (and up), down
ROLES = {"qkv": (QKV, D), "o": (D, D), "gate": (F, D), "down": (D, F)}
LAYER_SHAPES = [(D, D), (KVD, D), (KVD, D), (D, D), (F, D), (F, D), (D, F)]   # q, k, v, o, gate, up, down
LAYER_WEIGHTS = sum(n * k for n, k in LAYER_SHAPES)


def listed():
    return [
        # one decoder layer for one token of a running conversation (512 cached rows with its own)
        {"name": "decode_layer_511", "kind": "decode_layer", "pos": 511},
        # the head on the last hidden row of a program that samples from the logits itself
        {"name": "lm_head_row", "kind": "lm_head", "vocab": V},
        # a few tokens at once in the middle of a conversation (a short user turn, a draft to verify)
        {"name": "layer_rows_5", "kind": "layer_rows", "rows": 5, "pos0": 300},
        # a short prompt: fewer rows than the large tiles take
        {"name": "layer_rows_45", "kind": "layer_rows", "rows": 45, "pos0": 0},
        # a ragged chunk of a long prompt behind earlier chunks
        {"name": "layer_rows_333", "kind": "layer_rows", "rows": 333, "pos0": 701},
        # a prompt that fills the context
        {"name": "layer_rows_2048", "kind": "layer_rows", "rows": 2048, "pos0": 0},
        # the benchmark's 512-token prefill with the logits of every position (scoring a text)
        {"name": "score_512", "kind": "score", "n": 512},
        # one user's request: the prompt, then greedy tokens one by one
        {"name": "generate_100_48", "kind": "generate", "n": 100, "new": 48},
        # serving near the end of the context (the benchmark's batch)
        {"name": "batch_32x1984", "kind": "batch", "seqs": 32, "ctx": 1984, "steps": 24},
        # serving more, shorter conversations than one 32-row tile holds
        {"name": "batch_90x260", "kind": "batch", "seqs": 90, "ctx": 260, "steps": 16},
        # the projection operator on the rows of a long prompt (ragged)
        {"name": "gemm_1000_gate", "kind": "gemm", "m": 1000, "role": "gate", "residual": False},
        # the float32 model beside the INT8 one in the analysis report
        {"name": "linear_f32_100_gate", "kind": "linear_f32", "m": 100, "role": "gate", "bias": False,
         "residual": False},
    ]


def _log_int(rng: random.Random, lo: int, hi: int) -> int:
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["decode_layer", "layer_rows", "layer_rows", "layer_rows", "lm_head", "score", "generate",
                       "batch", "batch", "gemm", "gemm", "linear_f32"])
    if kind == "decode_layer":
        return {"kind": kind, "pos": _log_int(rng, 1, MAX_POS) - 1}
    if kind == "layer_rows":
        rows = _log_int(rng, 2, MAX_POS)
        return {"kind": kind, "rows": rows, "pos0": rng.choice([0, rng.randint(0, MAX_POS - rows)])}
    if kind == "lm_head":
        return {"kind": kind, "vocab": 64 * _log_int(rng, 16, V // 64)}
    if kind == "score":
        return {"kind": kind, "n": _log_int(rng, 2, 640)}
    if kind == "generate":
        return {"kind": kind, "n": _log_int(rng, 1, 512), "new": _log_int(rng, 1, 64)}
    if kind == "batch":
        seqs = _log_int(rng, 2, 128)
        steps = rng.randint(2, 24 if seqs <= 32 else 16)
        # no more cached rows over the batch than the largest listed case has
        return {"kind": kind, "seqs": seqs, "ctx": rng.randint(0, min(2000, 32 * 1984 // seqs)), "steps": steps}
    role = rng.choice(sorted(ROLES))
    if kind == "gemm":
        return {"kind": kind, "m": _log_int(rng, 2, 2048), "role": role, "residual": rng.random() < 0.5}
    return {"kind": kind, "m": _log_int(rng, 1, 640), "role": role, "bias": rng.random() < 0.3,
            "residual": rng.random() < 0.3}


# ---- inputs -----------------------------------------------------------------------------------------------------

def _gen(seed: int, part: int) -> torch.Generator:
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) * 1000003 + part)
    return g


def _quant_rows(w):
    """INT8 per output channel: scale max|w| / 127 in float32, round to nearest even."""
    s = (w.abs().amax(dim=1).double() / 127.0).float()
    return torch.clamp(torch.round(w / s[:, None]), -127, 127).to(torch.int8), s


def _weight(g, n, k):
    return _quant_rows(torch.randn(n, k, generator=g, device="cuda") * 0.02)


def _gain(g):
    return 1.0 + 0.02 * torch.randn(D, generator=g, device="cuda")


def _layer(seed: int, layer: int) -> dict:
    g = _gen(seed, 10 + layer)
    w, s = zip(*[_weight(g, n, k) for n, k in LAYER_SHAPES])
    return {"w": list(w), "s": list(s), "g_in": _gain(g), "g_post": _gain(g)}


def _head(seed: int, vocab: int = V):
    g = _gen(seed, 1)
    w, s = _weight(g, vocab, D)
    return w, s, _gain(g)


def _embedding(seed: int):
    return _weight(_gen(seed, 2), V, D)


def _rope_table():
    """cos and sin [position][64] float32, the two halves of a head alike."""
    inv = 1.0 / 10000.0 ** (np.arange(0, HD, 2, dtype=np.float32) / np.float32(HD))
    ang = np.outer(np.arange(MAX_POS, dtype=np.float32), inv.astype(np.float32)).astype(np.float32)
    ang = np.concatenate([ang, ang], axis=1)
    return np.cos(ang), np.sin(ang)


def _kv_scales(seed: int, layers: int):
    rng = np.random.default_rng([seed, 3])
    return (rng.uniform(0.02, 0.06, (layers, KV_HEADS)).astype(np.float32),
            rng.uniform(0.02, 0.06, (layers, KV_HEADS)).astype(np.float32))


def _hidden(seed: int, rows: int):
    """Rows of the residual stream: each row with a magnitude of its own."""
    g = _gen(seed, 4)
    x = torch.randn(rows, D, generator=g, device="cuda")
    return x * torch.exp(0.5 * torch.randn(rows, 1, generator=g, device="cuda"))


def _kv_rows(seed: int, heads: int, n: int):
    """Cached K (or V) rows [heads][n][64] int8: normal, about 22 steps of the scale."""
    rng = np.random.default_rng([seed, 5])
    pool = np.clip(np.rint(rng.standard_normal((65536, HD), np.float32) * 22.0), -127, 127).astype(np.int8)
    at = rng.integers(0, pool.shape[0] - max(n, 1), heads)
    return [pool[a:a + n] for a in at]


def _tokens(seed: int, n: int):
    return np.random.default_rng([seed, 6]).integers(0, V, n).astype(np.int32)


def _cfg(layers: int, vocab: int) -> dict:
    return dict(hidden=D, intermediate=F, n_layers=layers, n_heads=HEADS, n_kv_heads=KV_HEADS, head_dim=HD,
                vocab=vocab, max_pos=MAX_POS, rms_eps=EPS, rope_theta=10000.0)


def _engine(seed: int, layers: int, whole: bool, max_seqs: int = 1):
    eng = lpta.Engine(_cfg(layers, V if whole else 64), max_seqs=max_seqs)
    for i in range(layers):
        eng.load_layer(i, _layer(seed, i))
    if whole:
        eng.load_lm_head(*_head(seed))
        eng.load_embedding(*_embedding(seed))
    eng.set_kv_scales(*_kv_scales(seed, layers))
    eng.set_rope_table(*_rope_table())
    return eng


def _cached(seed: int, seqs: int, layers: int, n: int):
    """(seq, layer, head, K rows, V rows) of every plane that holds cached rows."""
    if n == 0:
        return
    planes = seqs * layers * KV_HEADS
    k, v = _kv_rows(seed, planes, n), _kv_rows(seed + 7919, planes, n)
    for i in range(planes):
        yield i // (layers * KV_HEADS), i // KV_HEADS % layers, i % KV_HEADS, k[i], v[i]


def _starts(case, seed):
    """Ragged context lengths of a batch: each sequence within 25 rows below the longest."""
    return (case["ctx"] - np.random.default_rng([seed, 8]).integers(0, min(25, case["ctx"]) + 1,
                                                                    case["seqs"])).astype(np.int32)


def prepare(case, seed):
    kind = case["kind"]
    st = {"case": case}
    if kind in ("decode_layer", "layer_rows"):
        pos0 = case["pos"] if kind == "decode_layer" else case["pos0"]
        st["eng"] = _engine(seed, 1, False)
        for s, l, h, k, v in _cached(seed, 1, 1, pos0):
            st["eng"].kv_write(s, l, h, 0, k, v)
        st["x"] = _hidden(seed, case.get("rows", 1))
    elif kind == "lm_head":
        st["eng"] = lpta.Engine(_cfg(1, case["vocab"]))
        st["eng"].load_lm_head(*_head(seed, case["vocab"]))
        st["x"] = _hidden(seed, 1)
        st["logits"] = torch.empty(case["vocab"], device="cuda")
    elif kind in ("score", "generate"):
        st["eng"] = _engine(seed, LAYERS, True)
        st["tokens"] = _tokens(seed, case["n"])
        st["logits"] = torch.empty(case["n"], V, device="cuda")
    elif kind == "batch":
        st["eng"] = _engine(seed, LAYERS, True, case["seqs"])
        for s, l, h, k, v in _cached(seed, case["seqs"], LAYERS, case["ctx"]):
            st["eng"].kv_write(s, l, h, 0, k, v)
        st["tokens"] = _tokens(seed, case["seqs"])
        st["start"] = _starts(case, seed)
    elif kind == "gemm":
        n, k = ROLES[case["role"]]
        st["eng"] = lpta.Engine(_cfg(1, 64))
        st["w"], st["ws"] = _weight(_gen(seed, 10), n, k)
        st["a"], st["as"] = _gemm_rows(seed, case["m"], k)
        st["residual"] = _residual(case, seed, n)
        st["y"] = torch.empty(case["m"], n, device="cuda")
    else:
        n, k = ROLES[case["role"]]
        st["eng"] = lpta.Engine(_cfg(1, 64))
        st["x"], st["w"], st["b"] = _float_inputs(case, seed, n, k)
        st["residual"] = _residual(case, seed, n)
        st["y"] = torch.empty(case["m"], n, device="cuda")
    torch.cuda.synchronize()
    return st


def _gemm_rows(seed, m, k):
    """INT8 rows with their float64 scales, as the row quantizer leaves them."""
    x = torch.randn(m, k, generator=_gen(seed, 4), device="cuda")
    s = x.abs().amax(dim=1).double() / 127.0
    return torch.clamp(torch.round(x / s.float()[:, None]), -127, 127).to(torch.int8), s


def _float_inputs(case, seed, n, k):
    g = _gen(seed, 10)
    x = torch.randn(case["m"], k, generator=g, device="cuda")
    w = torch.randn(k, n, generator=g, device="cuda") * 0.02
    b = torch.randn(n, generator=g, device="cuda") * 0.1 if case["bias"] else None
    return x, w, b


def _residual(case, seed, n):
    return torch.randn(case["m"], n, generator=_gen(seed, 9), device="cuda") if case["residual"] else None


# ---- one pass ---------------------------------------------------------------------------------------------------

def run(state):
    case, eng = state["case"], state["eng"]
    kind = case["kind"]
    if kind == "decode_layer":
        # the layer works in place: the program keeps its input row
        x = state["x"].clone()
        eng.decode_layer(x, 0, case["pos"])
        return x
    if kind == "layer_rows":
        x = state["x"].clone()
        eng.rt.call("tl_layer_rows", 0, 0, case["pos0"], case["rows"], x)
        return x
    if kind == "lm_head":
        token, logit = ctypes.c_int32(), ctypes.c_float()
        eng.rt.call("tl_lm_head_argmax", state["x"], token, logit, state["logits"])
        return {"token": token.value, "logit": logit.value, "logits": state["logits"]}
    if kind == "score":
        eng.rt.call("tl_prefill_logits", 0, state["tokens"], case["n"], state["logits"])
        return state["logits"]
    if kind == "generate":
        eng.rt.call("tl_prefill_logits", 0, state["tokens"], case["n"], state["logits"])
        tokens, _ = eng.decode(case["new"])
        return {"logits": state["logits"], "tokens": tokens}
    if kind == "batch":
        tokens = eng.decode_batch(state["tokens"], state["start"], case["steps"])
        # beside the ids, which are all that the call returns: the K/V rows that the last layer appended for KV head 0
        # of every sequence
        rows = [eng.kv_read(b, LAYERS - 1, 0, int(s), case["steps"]) for b, s in enumerate(state["start"])]
        return {"tokens": tokens, "k": np.stack([r[0] for r in rows]), "v": np.stack([r[1] for r in rows])}
    n, k = ROLES[case["role"]]
    if kind == "gemm":
        eng.rt.call("tl_gemm_i8_dequant", state["a"], state["as"], state["w"], state["ws"], case["m"], n, k,
                    state["residual"], state["y"])
    else:
        eng.rt.call("tl_linear_f32", state["x"], state["w"], state["b"], state["residual"], case["m"], n, k,
                    state["y"])
    return state["y"]


# ---- what a pass cannot do without ------------------------------------------------------------------------------

def _layer_work(rows, keys):
    """One layer over `rows` rows with `keys` (row, key) pairs in its attention, weights and cache apart."""
    return 2.0 * rows * LAYER_WEIGHTS + 4.0 * keys * D


def _causal(pos0, rows):
    return rows * pos0 + rows * (rows + 1) // 2


def work(case):
    kind = case["kind"]
    scales = 4 * sum(n for n, _ in LAYER_SHAPES) + 8 * D
    layer_bytes = LAYER_WEIGHTS + scales
    head_bytes = V * D + 4 * V + 4 * D
    if kind in ("decode_layer", "layer_rows"):
        rows, pos0 = case.get("rows", 1), case.get("pos0", case.get("pos"))
        # weights, rows in and out, cached rows in, new ones out
        return {"bytes": layer_bytes + 8 * rows * D + 2 * KVD * (pos0 + rows),
                "flops": _layer_work(rows, _causal(pos0, rows))}
    if kind == "lm_head":
        v = case["vocab"]
        return {"bytes": v * D + 8 * v + 8 * D, "flops": 2.0 * v * D}
    if kind in ("score", "generate"):
        n, new = case["n"], case.get("new", 0)
        # the prompt's rows once, then one pass over weights and cache per token; the next token after the prompt
        # comes from the last row's logits
        by = LAYERS * (layer_bytes + 2 * KVD * n) + head_bytes + n * D + 4 * n * V
        fl = LAYERS * _layer_work(n, _causal(0, n)) + 2.0 * n * V * D
        by += new * (LAYERS * layer_bytes + head_bytes) + LAYERS * 2 * KVD * sum(n + i + 1 for i in range(new))
        fl += LAYERS * sum(_layer_work(1, n + i + 1) for i in range(new)) + new * 2.0 * V * D
        return {"bytes": by, "flops": fl}
    if kind == "batch":
        b, steps = case["seqs"], case["steps"]
        keys = [max(case["ctx"] - 12, 0) + i + 1 for i in range(steps)]
        by = steps * (LAYERS * layer_bytes + head_bytes) + LAYERS * 2 * KVD * b * sum(keys) + steps * b * D
        fl = sum(LAYERS * _layer_work(b, b * t) + 2.0 * b * V * D for t in keys)
        return {"bytes": by, "flops": fl}
    n, k = ROLES[case["role"]]
    m = case["m"]
    extra = 4 * m * n if case["residual"] else 0
    if kind == "gemm":
        return {"bytes": m * k + 8 * m + n * k + 4 * n + 4 * m * n + extra, "flops": 2.0 * m * n * k}
    return {"bytes": 4 * (m * k + n * k + m * n) + extra, "flops": 2.0 * m * n * k}


def tolerance(case):
    # float32 sums of 2048 or 5632 products in another order: about four times the 8e-7 (K = 2048) to 1.3e-6 that
    # sequential sums measure against 64 bits
    return {"rel": 5e-6} if case["kind"] == "linear_f32" else "exact"


# ---- the same in 64 bits ----------------------------------------------------------------------------------------

def _q64(x):
    """INT8 per row: values and scales."""
    s = x.abs().amax(dim=-1, keepdim=True) / 127.0
    s = torch.where(s == 0, torch.ones_like(s), s)
    return torch.clamp(torch.round(x / s), -127, 127), s


def _norm64(x, g):
    return x / torch.sqrt((x * x).mean(dim=-1, keepdim=True) + float(EPS)) * g.double()


def _linear64(q, s, w, ws):
    return (q @ w.double().t()) * (s * ws.double())


def _rope64(x, cos, sin):
    """x [rows][heads][64], tables [rows][64]."""
    half = torch.cat([-x[..., HD // 2:], x[..., :HD // 2]], dim=-1)
    return x * cos[:, None, :] + half * sin[:, None, :]


def _layer64(x, L, sk, sv, cached_k, cached_v, pos0, cos, sin):
    """One decoder layer over rows at pos0 ..; cached_k / cached_v [heads][pos0][64] int8."""
    rows = x.shape[0]
    q, s = _q64(_norm64(x, L["g_in"]))
    c, sn = cos[pos0:pos0 + rows], sin[pos0:pos0 + rows]
    qr = _rope64(_linear64(q, s, L["w"][0], L["s"][0]).view(rows, HEADS, HD), c, sn)
    kr = _rope64(_linear64(q, s, L["w"][1], L["s"][1]).view(rows, KV_HEADS, HD), c, sn)
    vr = _linear64(q, s, L["w"][2], L["s"][2]).view(rows, KV_HEADS, HD)
    q8, qs = _q64(qr.reshape(rows, D))
    q8 = q8.view(rows, HEADS, HD)
    mask = torch.arange(pos0 + rows, device=x.device)[None, :] > (pos0 + torch.arange(rows, device=x.device))[:, None]
    out = torch.empty(rows, HEADS, HD, dtype=torch.float64, device=x.device)
    for h in range(KV_HEADS):
        k8 = torch.clamp(torch.round(kr[:, h] / float(sk[h])), -127, 127)
        v8 = torch.clamp(torch.round(vr[:, h] / float(sv[h])), -127, 127)
        if pos0:
            k8, v8 = torch.cat([cached_k[h].double(), k8]), torch.cat([cached_v[h].double(), v8])
        for hq in range(h * HEADS // KV_HEADS, (h + 1) * HEADS // KV_HEADS):
            sc = (q8[:, hq] @ k8.t()) * (qs * float(sk[h]) * 0.125)
            p = torch.softmax(sc.masked_fill(mask, -math.inf), dim=-1)
            out[:, hq] = (torch.round(p * 127.0) @ v8) * (float(sv[h]) / 127.0)
    q, s = _q64(out.reshape(rows, D))
    x = x + _linear64(q, s, L["w"][3], L["s"][3])
    q, s = _q64(_norm64(x, L["g_post"]))
    gate = _linear64(q, s, L["w"][4], L["s"][4])
    q, s = _q64(gate * torch.sigmoid(gate) * _linear64(q, s, L["w"][5], L["s"][5]))
    return x + _linear64(q, s, L["w"][6], L["s"][6])


def _tables():
    return tuple(torch.from_numpy(t).cuda().double() for t in _rope_table())


def exact(case, seed):
    kind = case["kind"]
    if kind in ("batch", "score", "generate"):
        # An INT8 rounding that falls the other way in one layer moves every layer after it: 22 layers in 64 bits end
        # 8 to 13 % away from the float32 contract.  The layer and head cases hold the comparison.
        return None
    if kind in ("decode_layer", "layer_rows"):
        pos0 = case["pos"] if kind == "decode_layer" else case["pos0"]
        sk, sv = _kv_scales(seed, 1)
        planes = list(_cached(seed, 1, 1, pos0))
        ck = [torch.from_numpy(p[3]).cuda() for p in planes]
        cv = [torch.from_numpy(p[4]).cuda() for p in planes]
        return _layer64(_hidden(seed, case.get("rows", 1)).double(), _layer(seed, 0), sk[0], sv[0], ck, cv, pos0,
                        *_tables())
    if kind == "lm_head":
        w, s, g = _head(seed, case["vocab"])
        logits = _linear64(*_q64(_norm64(_hidden(seed, 1).double(), g)), w, s)[0]
        return {"token": None, "logit": float(logits.max()), "logits": logits}
    n, k = ROLES[case["role"]]
    res = _residual(case, seed, n)
    if kind == "gemm":
        w, ws = _weight(_gen(seed, 10), n, k)
        a, s = _gemm_rows(seed, case["m"], k)
        y = _linear64(a.double(), s[:, None], w, ws)
    else:
        x, w, b = _float_inputs(case, seed, n, k)
        y = x.double() @ w.double()
        if b is not None:
            y = y + b.double()
    return y if res is None else res.double() + y
