"""The work this library is measured on: decode and prefill attention and the cache writer in
front of them, called through ``brasa_amd.Kernels`` on device memory that torch holds.

One case is one pass of a user's program: a decode step over the layers of a model, one batched
decode, one prefill chunk of one layer, one QK-norm + RoPE + cache write. Shapes are the ones the
benchmark and the tests use: the Qwen3-4B heads (32 query, 8 KV, head_dim 128, 36 layers), and
the other GQA groups the decode and prefill kernels are compiled for. Queries and keys are
N(0, 1) through a per-head RMS norm (what the attention sees behind QK-norm), values N(0, 1).
"""
from __future__ import annotations

import math
import random

import torch

from brasa_amd import (AttnShape, Kernels, KvType, OutDType, PrefillPrecision, decode_partials_len,
                       rope_table)

DIM = 128
EPS = 1e-6
THETA = 1e6
KV = {"f32": KvType.F32, "f16": KvType.F16, "q8_0": KvType.Q8_0}
ROW = {"f32": 512, "f16": 256, "q8_0": 136}
PRECISION = {"f16": PrefillPrecision.F16, "f16_pf32": PrefillPrecision.F16_PF32,
             "f32": PrefillPrecision.F32}


def listed():
    return [
        # the first reply token of a short chat: one layer's call, bound by launch and latency
        {"name": "decode_f16_257", "op": "decode", "kv": "f16", "hq": 32, "hkv": 8, "lk": 257,
         "layers": 1, "write": False},
        # a decode step at an ordinary context, with the cache write of the new token in front
        # of each layer's attention, as the model's step issues them
        {"name": "decode_step_f16_4k", "op": "decode", "kv": "f16", "hq": 32, "hkv": 8,
         "lk": 4097, "layers": 36, "write": True},
        # the benchmark's decode step: 36 layers at 16K context, a cache of its own per layer
        {"name": "decode_f16_16k", "op": "decode", "kv": "f16", "hq": 32, "hkv": 8, "lk": 16384,
         "layers": 36, "write": False},
        # the same step on the quantised cache, at a length that is no multiple of anything
        {"name": "decode_q8_0_16k", "op": "decode", "kv": "q8_0", "hq": 32, "hkv": 8,
         "lk": 16001, "layers": 36, "write": False},
        # the exact cache type, at the benchmark's shorter context
        {"name": "decode_f32_2k", "op": "decode", "kv": "f32", "hq": 32, "hkv": 8, "lk": 2048,
         "layers": 36, "write": False},
        # a server's batch: eight sequences of mixed lengths in one call
        {"name": "decode_batch8_f16", "op": "batch", "kv": "f16", "hq": 32, "hkv": 8, "n": 8,
         "lk_min": 1024, "lk_max": 16384, "lens": 12345},
        # the benchmark's prompt of 2K tokens
        {"name": "prefill_f16_2k", "op": "prefill", "kv": "f16", "precision": "f16", "hq": 32,
         "hkv": 8, "tokens": 2048, "pos0": 0},
        # the largest: an 8K prompt in one call
        {"name": "prefill_f16_8k", "op": "prefill", "kv": "f16", "precision": "f16", "hq": 32,
         "hkv": 8, "tokens": 8192, "pos0": 0},
        # one 512-token chunk of a long prompt, on the quantised cache
        {"name": "prefill_q8_0_chunk", "op": "prefill", "kv": "q8_0", "precision": "f16",
         "hq": 32, "hkv": 8, "tokens": 512, "pos0": 16384},
        # a short user turn in a long conversation: few queries, many cached keys
        {"name": "prefill_f16_turn", "op": "prefill", "kv": "f16", "precision": "f16", "hq": 32,
         "hkv": 8, "tokens": 45, "pos0": 7001},
        # the exact variant, on the exact cache: an odd prompt of about 1K
        {"name": "prefill_f32_1k", "op": "prefill", "kv": "f32", "precision": "f32", "hq": 32,
         "hkv": 8, "tokens": 1000, "pos0": 0},
        # the producer of a 2K prompt's queries and cache rows
        {"name": "store_f16_2k", "op": "store", "kv": "f16", "hq": 32, "hkv": 8, "tokens": 2048,
         "pos0": 0},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["decode", "decode", "batch", "prefill", "prefill", "prefill", "store"])
    kv = rng.choice(["f16", "f16", "q8_0", "q8_0", "f32"])
    hq, hkv = rng.choice([(32, 8), (32, 8), (32, 8), (16, 8), (32, 4), (32, 32)])
    if op == "decode":
        lk = _log(rng, 129, 32768)
        # a step's caches: no more bytes than the 36 layers of 16K fp16 positions
        most = 36 * 16384 * 8 * 256 // (lk * hkv * ROW[kv])
        return {"op": op, "kv": kv, "hq": hq, "hkv": hkv, "lk": lk,
                "layers": max(1, min(36, most, rng.choice([1, 4, 12, 36]))),
                "write": rng.random() < 0.3}
    if op == "batch":
        n = rng.randint(2, 16)
        lo = _log(rng, 64, 1024)
        return {"op": op, "kv": kv, "hq": hq, "hkv": hkv, "n": n, "lk_min": lo,
                "lk_max": _log(rng, 2 * lo, 16384 * 8 // max(n, 8)), "lens": rng.randrange(1 << 16)}
    if op == "store":
        return {"op": op, "kv": kv, "hq": hq, "hkv": hkv, "tokens": _log(rng, 1, 4096),
                "pos0": rng.choice([0, _log(rng, 1, 16384)])}
    precision = rng.choice(["f16", "f16", "f16", "f16_pf32", "f32"])
    tokens = _log(rng, 8, 4096)
    pos0 = rng.choice([0, _log(rng, 16, 16384)])
    # (query, key) pairs: those of the 8K prompt at most; an eighth where every product is exact
    most = 16 << 20 if precision == "f16" else 4 << 20
    pos0 = max(0, min(pos0, most // tokens - tokens))
    return {"op": op, "kv": kv, "precision": precision, "hq": hq, "hkv": hkv, "tokens": tokens,
            "pos0": pos0}


# ---- inputs ------------------------------------------------------------------------------------
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _normed(g, *shape):
    x = torch.randn(*shape, generator=g, device="cuda")
    return x.mul_(torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS))


def _quantise(x):
    """[rows, 128] f32 -> q8_0 rows of 136 bytes: 128 codes, then four f16 scales."""
    b = x.reshape(-1, 4, 32)
    d = (b.abs().amax(-1) / 127.0).half()
    s = d.float().unsqueeze(-1)
    codes = torch.where(s != 0, (b / s).round().clamp(-127, 127), torch.zeros_like(b))
    codes = codes.to(torch.int8).reshape(-1, DIM).view(torch.uint8)
    return torch.cat([codes, d.view(torch.uint8).reshape(-1, 8)], 1).contiguous()


def _cache(kv, x):
    """f32 [rows, hkv, 128] -> the cache rows of that type, one per position and head."""
    x = x.reshape(-1, DIM)
    return x if kv == "f32" else x.half() if kv == "f16" else _quantise(x)


def _seen(kv, cache, hkv):
    """The values a cache holds, [rows, hkv, 128] in 64 bits."""
    if kv != "q8_0":
        return cache.double().reshape(-1, hkv, DIM)
    codes = cache[:, :DIM].contiguous().view(torch.int8).double().reshape(-1, 4, 32)
    scale = cache[:, DIM:].contiguous().view(torch.float16).double().reshape(-1, 4, 1)
    return (codes * scale).reshape(-1, hkv, DIM)


def _lens(case):
    r = random.Random(case["lens"])
    return [r.randint(case["lk_min"], case["lk_max"]) for _ in range(case["n"])]


def _pair(g, kv, rows, hkv, used=None):
    """K and V caches of `rows` positions; positions from `used` on are zero."""
    k, v = _normed(g, rows, hkv, DIM), torch.randn(rows, hkv, DIM, generator=g, device="cuda")
    if used is not None:
        k[used:] = 0
        v[used:] = 0
    return _cache(kv, k), _cache(kv, v)


def _table(pos, rows=1):
    cos, sin = rope_table(THETA, DIM, pos + rows)
    return torch.from_numpy(cos).cuda(), torch.from_numpy(sin).cuda()


class _Table:
    """A rope table in torch memory, as ``Kernels`` takes it."""

    def __init__(self, cos, sin):
        from brasa_amd._lib import RopeTableC
        self.cos, self.sin = cos, sin
        self._c = RopeTableC(cos.data_ptr(), sin.data_ptr(), DIM, cos.shape[0])

    def c(self):
        return self._c


def _inputs(case, seed):
    """What the case reads, from the seed alone."""
    g = _gen(seed)
    op, hq, hkv, kv = case["op"], case["hq"], case["hkv"], case["kv"]
    if op == "decode":
        n, lk = case["layers"], case["lk"]
        # one K and one V buffer for all layers, as the model's cache is laid out
        first = _pair(g, kv, lk, hkv)
        all_k, all_v = (c.new_empty(n, *c.shape) for c in first)
        for i in range(n):
            all_k[i], all_v[i] = first if i == 0 else _pair(g, kv, lk, hkv)
        x = {"all_k": all_k, "all_v": all_v, "caches": list(zip(all_k, all_v)),
             "q": _normed(g, n, hq, DIM)}
        if case["write"]:
            x["q"] = torch.randn(n, hq, DIM, generator=g, device="cuda")
            x["k"] = torch.randn(n, hkv, DIM, generator=g, device="cuda")
            x["v"] = torch.randn(n, hkv, DIM, generator=g, device="cuda")
            x["qn"] = 1 + 0.1 * torch.randn(DIM, generator=g, device="cuda")
            x["kn"] = 1 + 0.1 * torch.randn(DIM, generator=g, device="cuda")
        return x
    if op == "batch":
        return {"caches": [_pair(g, kv, lk, hkv) for lk in _lens(case)],
                "q": _normed(g, case["n"], hq, DIM)}
    t, pos0 = case["tokens"], case["pos0"]
    if op == "prefill":
        rows = (pos0 + t + 63) // 64 * 64
        return {"caches": [_pair(g, kv, rows, hkv, pos0 + t)], "q": _normed(g, t, hq, DIM)}
    return {"q": torch.randn(t, hq, DIM, generator=g, device="cuda"),
            "k": torch.randn(t, hkv, DIM, generator=g, device="cuda"),
            "v": torch.randn(t, hkv, DIM, generator=g, device="cuda"),
            "qn": 1 + 0.1 * torch.randn(DIM, generator=g, device="cuda"),
            "kn": 1 + 0.1 * torch.randn(DIM, generator=g, device="cuda")}


_kernels = None


def prepare(case, seed):
    global _kernels
    if _kernels is None:
        _kernels = Kernels()
    s = dict(case, **_inputs(case, seed))
    op, kv, hq, hkv = s["op"], s["kv"], s["hq"], s["hkv"]
    s["type"] = KV[kv]
    if op == "decode":
        s["o"] = torch.empty(s["layers"], hq, DIM, device="cuda")
        s["plen"] = decode_partials_len(hq, s["lk"])
        s["part"] = torch.empty(s["plen"], device="cuda")
        # a program keeps its layers' addresses
        row = (s["lk"] - 1) * hkv * ROW[kv]
        s["at"] = [(s["q"][i].data_ptr(), k.data_ptr(), v.data_ptr(), s["o"][i].data_ptr())
                   for i, (k, v) in enumerate(s["caches"])]
        if s["write"]:
            s["table"] = _Table(*_table(s["lk"]))
            s["new"] = [(s["k"][i].data_ptr(), s["v"][i].data_ptr(), k.data_ptr() + row,
                         v.data_ptr() + row) for i, (k, v) in enumerate(s["caches"])]
    elif op == "batch":
        s["lks"] = _lens(case)
        s["o"] = torch.empty(s["n"], hq, DIM, device="cuda")
        s["plen"] = sum(decode_partials_len(hq, lk) for lk in s["lks"])
        s["part"] = torch.empty(s["plen"], device="cuda")
    elif op == "prefill":
        s["o"] = torch.empty(s["tokens"], hq, DIM, device="cuda",
                             dtype=torch.float32 if s["precision"] == "f32" else torch.float16)
    else:
        s["table"] = _Table(*_table(s["pos0"], s["tokens"]))
        n = s["tokens"] * hkv
        kind = {"f32": torch.float32, "f16": torch.float16, "q8_0": torch.uint8}[kv]
        width = ROW[kv] if kv == "q8_0" else DIM
        s["kc"] = torch.empty(n, width, dtype=kind, device="cuda")
        s["vc"] = torch.empty(n, width, dtype=kind, device="cuda")
    return s


def run(s):
    stream = torch.cuda.current_stream().cuda_stream
    op, kv, hq, hkv = s["op"], s["type"], s["hq"], s["hkv"]
    if op == "decode":
        shape = AttnShape(1, hq, hkv, DIM, s["lk"] - 1, kv)
        part, plen = s["part"].data_ptr(), s["plen"]
        if not s["write"]:
            for q, k, v, o in s["at"]:
                _kernels.decode_attention_lanes(q, k, v, part, o, shape, OutDType.F32, stream, plen)
            return s["o"]
        norms = s["qn"].data_ptr(), s["kn"].data_ptr()
        for (q, k, v, o), (nk, nv, kd, vd) in zip(s["at"], s["new"]):
            _kernels.qk_norm_rope_store(kv, (q, nk, nv), norms, EPS, s["table"], (kd, vd), shape,
                                        stream)
            _kernels.decode_attention_lanes(q, k, v, part, o, shape, OutDType.F32, stream, plen)
        # the step's updates: the rotated q and k, and each layer's new cache rows
        return {"o": s["o"], "q": s["q"], "k": s["k"], "k_rows": s["all_k"][:, -hkv:],
                "v_rows": s["all_v"][:, -hkv:]}
    if op == "batch":
        _kernels.decode_attention_batch(s["q"].data_ptr(), [k.data_ptr() for k, _ in s["caches"]],
                                        [v.data_ptr() for _, v in s["caches"]], s["lks"],
                                        s["part"].data_ptr(), s["o"].data_ptr(), hq, hkv, kv,
                                        OutDType.F32, stream, s["plen"])
        return s["o"]
    shape = AttnShape(s["tokens"], hq, hkv, DIM, s["pos0"], kv)
    if op == "prefill":
        (k, v), = s["caches"]
        _kernels.flash_attention_with(s["q"].data_ptr(), k.data_ptr(), v.data_ptr(),
                                      s["o"].data_ptr(), shape, PRECISION[s["precision"]], stream)
        return s["o"]
    _kernels.qk_norm_rope_store(kv, (s["q"].data_ptr(), s["k"].data_ptr(), s["v"].data_ptr()),
                                (s["qn"].data_ptr(), s["kn"].data_ptr()), EPS, s["table"],
                                (s["kc"].data_ptr(), s["vc"].data_ptr()), shape, stream)
    return {"q": s["q"], "k": s["k"], "kc": s["kc"], "vc": s["vc"]}


def work(case):
    op, hq, hkv, row = case["op"], case["hq"], case["hkv"], ROW[case["kv"]]
    if op in ("decode", "batch"):
        lks = [case["lk"]] * case["layers"] if op == "decode" else _lens(case)
        b = sum(2 * lk * hkv * row + 2 * hq * DIM * 4 for lk in lks)
        if case.get("write"):
            b += len(lks) * ((2 * hq + 3 * hkv) * DIM * 4 + 2 * hkv * row)
        return {"bytes": b, "flops": sum(4 * hq * DIM * lk for lk in lks)}
    t, pos0 = case["tokens"], case["pos0"]
    if op == "prefill":
        return {"bytes": 2 * (pos0 + t) * hkv * row
                + t * hq * DIM * (8 if case["precision"] == "f32" else 6),
                "flops": 4 * hq * DIM * (t * pos0 + t * (t + 1) / 2)}
    # q and k are read and written in place, v is read, the cache rows and the table's rows
    return {"bytes": t * ((2 * hq + 3 * hkv) * DIM * 4 + 2 * hkv * row + DIM * 4),
            "flops": 8 * t * (hq + hkv) * DIM}


def tolerance(case):
    if case["op"] == "prefill" and case["precision"] != "f32":
        # the f16 output's own rounding is 2.1e-4. P in f16 beside it, and, on a q8_0 cache, its
        # values in f16; a chunk's sums over many keys come to less than that
        return {"rel": 1e-3 if case["precision"] == "f16_pf32" else 2e-3}
    # sums in 32 bits; bytes of a q8_0 cache stay as they are
    return {"rel": 2e-6}


# ---- the same in 64 bits -----------------------------------------------------------------------
def _rope(x, cos, sin):
    a, b = x[..., :64], x[..., 64:]
    return torch.cat([a * cos - b * sin, b * cos + a * sin], -1)


def _angles(pos0, t):
    inv = THETA ** (-torch.arange(0, DIM, 2, dtype=torch.float64, device="cuda") / DIM)
    ang = torch.arange(pos0, pos0 + t, dtype=torch.float64, device="cuda")[:, None, None] * inv
    return ang.cos(), ang.sin()


def _norm64(x, w):
    x = x.double()
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * w.double()


def _attend(q, k, v, pos0):
    """q [t, hq, 128] over k, v [lk, hkv, 128]: causal from position pos0, one head at a time."""
    t, hq, _ = q.shape
    lk, hkv = k.shape[0], k.shape[1]
    out = torch.empty(t, hq, DIM, dtype=torch.float64, device="cuda")
    ahead = None
    if t > 1:
        ahead = torch.arange(lk, device="cuda")[None] > pos0 + torch.arange(t, device="cuda")[:, None]
    for kh in range(hkv):
        kt, vh = k[:, kh].t().contiguous(), v[:, kh].contiguous()
        for h in range(kh * (hq // hkv), (kh + 1) * (hq // hkv)):
            s = (q[:, h].double().contiguous() @ kt) / math.sqrt(DIM)
            if ahead is not None:
                s.masked_fill_(ahead, -math.inf)
            out[:, h] = torch.softmax(s, -1) @ vh
    return out


def exact(case, seed):
    x = _inputs(case, seed)
    op, kv, hkv = case["op"], case["kv"], case["hkv"]
    if op == "batch":
        return torch.cat([_attend(x["q"][i:i + 1], _seen(kv, k, hkv), _seen(kv, v, hkv), 0)
                          for i, (k, v) in enumerate(x["caches"])])
    if op == "prefill":
        (k, v), = x["caches"]
        lk = case["pos0"] + case["tokens"]
        return _attend(x["q"], _seen(kv, k, hkv)[:lk], _seen(kv, v, hkv)[:lk], case["pos0"])
    if op == "decode":
        q = x["q"].double()
        if case["write"]:
            cos, sin = _angles(case["lk"] - 1, 1)
            q, nk = _rope(_norm64(x["q"], x["qn"]), cos, sin), _rope(_norm64(x["k"], x["kn"]), cos, sin)
            for i, (k, v) in enumerate(x["caches"]):
                k[-hkv:] = _cache(kv, nk[i].float())
                v[-hkv:] = _cache(kv, x["v"][i])
        o = torch.cat([_attend(q[i:i + 1], _seen(kv, k, hkv), _seen(kv, v, hkv), 0)
                       for i, (k, v) in enumerate(x["caches"])])
        if not case["write"]:
            return o
        new = (None, None) if kv == "q8_0" else (nk, x["v"].double())
        return {"o": o, "q": q, "k": nk, "k_rows": new[0], "v_rows": new[1]}
    cos, sin = _angles(case["pos0"], case["tokens"])
    q, k = _rope(_norm64(x["q"], x["qn"]), cos, sin), _rope(_norm64(x["k"], x["kn"]), cos, sin)
    v = x["v"].double()
    return {"q": q, "k": k, "kc": None if kv == "q8_0" else k.reshape(-1, DIM),
            "vc": None if kv == "q8_0" else v.reshape(-1, DIM)}
