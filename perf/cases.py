"""The work whose speed this repository is measured by.

A case is one call sequence of an attention layer (or of its cache) as a
generate loop makes it, through the public cache classes and
``scaled_dot_product_attention``:

  layer   append L new tokens to a cache that holds ``tokens`` already, attend
          with L query rows per head over all of them, and take the tokens back
          again (``trim``), so that the pass can be repeated.  L = 1 is a decode
          step, 2..8 a speculative verify, more a prefill chunk.  ``cache`` is
          "turbo" (packed) or "plain" (the fp16 layers of the mixed-precision
          split); ``window`` > 0 brings the boolean sliding-window mask.
  batch   decode over a left-padded continuous-batching cache, whose rows hold
          ``shortest`` .. ``tokens`` tokens.
  append  quantize a prompt of L tokens into a reserved cache.
  codec   the same, then ``dequantize`` all of it to f32.

Keys and values are N(0, 1) times a log-normal scale per channel, queries
N(0, 1): the distributions of the repository's benchmark.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from kaplumba_amd import (BatchTurboQuantKVCache, KVCache, TurboQuantKVCache,
                          scaled_dot_product_attention)

DTYPES = {"f16": torch.float16, "bf16": torch.bfloat16, "f32": torch.float32}

BASE = dict(kind="layer", cache="turbo", B=1, Hq=32, Hkv=8, D=128, Dv=128, tokens=0, shortest=0,
            L=1, kb=3, vb=3, rotation="auto", dtype="bf16", norm="f32", window=0)


def listed():
    c = lambda name, **kw: dict(BASE, name=name, **kw)  # noqa: E731
    return [
        # the first steps of a chat: latency and launches, hardly any data
        c("decode_short", tokens=511),
        # one layer of the headline benchmark: one token against 32k cached ones
        c("decode_32k", tokens=32767),
        # a server's batch of 32 requests of unlike length, head dim 256, K4/V2, dense rotation
        c("decode_ragged_d256", kind="batch", B=32, Hq=16, D=256, Dv=256, kb=4, vb=2,
          rotation="dense", tokens=8192, shortest=2048),
        # a model whose head dim is no power of two (dense rotation), eight requests
        c("decode_d96", B=8, D=96, Dv=96, kb=4, vb=4, tokens=6000),
        # four drafts verified in each of four long sequences, K2/V1
        c("verify_131k", B=4, tokens=131072, L=4, kb=2, vb=1),
        # a chunk of a long prompt through a packed layer
        c("prefill_d128", tokens=7936, L=256),
        # the same at head dim 64: two prompts, odd lengths, 3.5 bits, f16 norms as the reference stores them
        c("prefill_d64", B=2, D=64, Dv=64, tokens=3597, L=500, kb=3, vb=4, dtype="f16", norm="f16"),
        # the same at head dim 256, K4/V2, dense rotation: how the ragged batch's requests come in
        c("prefill_d256", Hq=16, D=256, Dv=256, tokens=3584, L=512, kb=4, vb=2, rotation="dense"),
        # a chunk through a sliding-window layer (boolean array mask)
        c("prefill_window", tokens=7680, L=512, window=4096),
        # a chunk through one of the fp16 layers of the mixed-precision split
        c("prefill_plain", cache="plain", tokens=7680, L=512),
        # a whole 8192-token prompt quantized into one layer, dense rotation
        c("append_dense", kind="append", Hq=8, L=8192, rotation="dense"),
        # quantize 4096 tokens of f16 and reconstruct them
        c("quantize_dequantize", kind="codec", Hq=8, L=4096, dtype="f16"),
    ]


# what a drawn case may cost: as much as the largest listed one does
MOST_PAIRS = 32 * 512 * 8192 * 256     # query-head rows x tokens x (Dk + Dv), prefill
MOST_PAIRS_OTHER = MOST_PAIRS // 2     # the same where the head dim is no power of two
MOST_CACHE = 32 * 131072 * 256         # kv-head tokens x (Dk + Dv) of a packed cache
MOST_INPUT = 8 * 16384 * 256           # kv-head tokens x (Dk + Dv) appended at once


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    c = dict(BASE)
    c["kind"] = rng.choice(["layer"] * 7 + ["batch", "append", "codec"])
    c["D"], c["Dv"] = rng.choice([(64, 64), (128, 128), (128, 128), (256, 256), (80, 80), (96, 96), (192, 128)])
    pow2 = c["D"] in (64, 128, 256) and c["Dv"] in (64, 128, 256)
    c["Hkv"] = rng.choice([2, 4, 8, 8, 16])
    c["Hq"] = c["Hkv"] * rng.choice([1, 2, 4, 4, 7, 8])
    c["kb"], c["vb"] = rng.choice([(3, 3), (3, 3), (4, 4), (3, 4), (2, 2), (4, 2), (2, 1)])
    c["rotation"] = rng.choice(["auto", "auto", "dense"])
    c["dtype"] = rng.choice(["bf16", "bf16", "f16"])
    c["norm"] = rng.choice(["f32", "f32", "f16"])
    per = c["D"] + c["Dv"]
    if c["kind"] in ("append", "codec"):
        c["B"] = rng.choice([1, 1, 2, 4])
        most = MOST_INPUT // (2 if c["kind"] == "codec" else 1) // (1 if pow2 else 4)
        c["L"] = _log_int(rng, 16, max(17, most // (c["B"] * c["Hkv"] * per)))
        return c
    if c["kind"] == "batch":
        c["B"] = _log_int(rng, 2, 48)
        most = MOST_CACHE // (1 if pow2 else 4) // (c["B"] * c["Hkv"] * per)
        c["tokens"] = _log_int(rng, 64, max(65, min(16384, most)))
        c["shortest"] = max(1, int(c["tokens"] * rng.uniform(0.1, 1.0)))
        return c
    c["cache"] = rng.choice(["turbo"] * 5 + ["plain"])
    mode = rng.choice(["decode", "decode", "verify", "prefill", "prefill"])
    c["B"] = _log_int(rng, 1, 4 if mode == "prefill" else 16)
    c["L"] = {"decode": 1, "verify": rng.randint(2, 8), "prefill": _log_int(rng, 16, 1024)}[mode]
    rows = c["Hq"] * c["L"]
    if rng.random() < 0.2:
        c["window"] = rng.choice([512, 1024, 4096])
    most = MOST_CACHE // (1 if pow2 and not c["window"] else 8) // (c["B"] * c["Hkv"] * per)
    if mode != "decode":
        most = min(most, (MOST_PAIRS if pow2 else MOST_PAIRS_OTHER) // (c["B"] * rows * per))
    most = min(most, 131072, MOST_CACHE // 8 // (c["B"] * c["Hkv"] * per) if c["cache"] == "plain" else most)
    c["tokens"] = _log_int(rng, 32, max(33, most - c["L"]))
    return c


def _kv(g, shape, dtype):
    """Keys or values: N(0, 1) times a log-normal scale per (kv head, channel)."""
    scale = torch.exp(torch.randn(1, shape[1], 1, shape[3], device="cuda", generator=g) * 0.5)
    return (torch.randn(shape, device="cuda", generator=g) * scale).to(dtype)


def _lengths(case):
    """Tokens of each row of a batch, from ``shortest`` to ``tokens`` in mixed order; one row has all."""
    B, lo, hi = case["B"], case["shortest"], case["tokens"]
    return [hi - (hi - lo) * ((7 * b) % B) // max(B - 1, 1) for b in range(B)]


def prepare(case, seed):
    g = torch.Generator(device="cuda").manual_seed(int(seed))
    dtype = DTYPES[case["dtype"]]
    B, H, L, n = case["B"], case["Hkv"], case["L"], case["tokens"]
    D, Dv = case["D"], case["Dv"]
    turbo = dict(bits=max(case["kb"], case["vb"]), key_bits=case["kb"], val_bits=case["vb"],
                 rotation=case["rotation"], norm_dtype=DTYPES[case["norm"]])
    mask = None
    if case["kind"] == "batch":
        cache = BatchTurboQuantKVCache([n - m for m in _lengths(case)], **turbo)
    elif case["cache"] == "plain":
        cache = KVCache()
    else:
        cache = TurboQuantKVCache(**turbo)
        cache.reserve(n + L, B, H, D, Dv, torch.device("cuda"))
    if n:
        cache.update_and_fetch(_kv(g, (B, H, n, D), dtype), _kv(g, (B, H, n, Dv), dtype))
    state = {"case": case, "cache": cache, "scale": 1.0 / math.sqrt(D)}
    if case["kind"] != "batch":
        if case["window"]:
            mask = cache.make_mask(L, window_size=case["window"]).to("cuda")
        elif L > 1:
            mask = "causal"
        state["k"], state["v"] = _kv(g, (B, H, L, D), dtype), _kv(g, (B, H, L, Dv), dtype)
        if case["cache"] == "plain" and n:
            # the buffer grows in steps: let the append that needs more room happen before
            cache.update_and_fetch(state["k"], state["v"])
            cache.trim(L)
    state["mask"] = mask
    if case["kind"] in ("layer", "batch"):
        state["q"] = torch.randn(B, case["Hq"], L, D, device="cuda", generator=g).to(dtype)
    return state


def _words(st):
    """A packed state's norms and rows, the rows' words as the signed integers that torch can compare."""
    return st.norms, st.indices.view(torch.int32)


def run(state):
    case, cache = state["case"], state["cache"]
    if case["kind"] == "batch":
        ks, vs = cache.state[:2]
        return {"out": scaled_dot_product_attention(state["q"], ks, vs, cache, state["scale"], None)}
    ks, vs = cache.update_and_fetch(state["k"], state["v"])
    if case["kind"] == "layer":
        out = scaled_dot_product_attention(state["q"], ks, vs, cache, state["scale"], state["mask"])
        cache.trim(case["L"])
        if case["cache"] == "plain":
            return {"out": out, "keys": ks, "values": vs}
        return {"out": out, "keys": _words(ks), "values": _words(vs)}
    got = {"keys": _words(ks), "values": _words(vs)}
    if case["kind"] == "codec":
        got["k"], got["v"] = cache.dequantize(ks, vs)
    cache.trim(case["L"])
    return got


def _dense(case, dim):
    """Whether a side of this head dim takes the dense rotation ("auto": where it is no power of two)."""
    return case["rotation"] == "dense" or dim & (dim - 1) != 0


def _row_bytes(case):
    """Bytes of one kv head's cached token, keys and values."""
    if case["cache"] == "plain" and case["kind"] == "layer":
        return 2 * (case["D"] + case["Dv"])
    words = (case["D"] * case["kb"] + 31) // 32 + (case["Dv"] * case["vb"] + 31) // 32
    return 4 * words + 2 * DTYPES[case["norm"]].itemsize


def work(case):
    B, L, D, Dv = case["B"], case["L"], case["D"], case["Dv"]
    heads, item = B * case["Hkv"], DTYPES[case["dtype"]].itemsize
    io = B * case["Hq"] * L * (D + Dv) * item      # queries in, attention out
    new = heads * L * (D + Dv) * item              # keys and values to append
    if case["kind"] == "batch":
        n = sum(_lengths(case))
        return {"bytes": case["Hkv"] * n * _row_bytes(case) + io, "flops": 2 * case["Hq"] * n * (D + Dv)}
    rotate = 2 * heads * L * sum(d * d for d in (D, Dv) if _dense(case, d))
    if case["kind"] in ("append", "codec"):
        # packed rows written once; read once more and f32 written when dequantized
        back = heads * L * (_row_bytes(case) + 4 * (D + Dv)) if case["kind"] == "codec" else 0
        return {"bytes": new + heads * L * _row_bytes(case) + back,
                "flops": rotate * (2 if case["kind"] == "codec" else 1)}
    n = case["tokens"]
    seen = [min(n + i + 1, case["window"] or n + L) for i in range(L)]  # tokens that query i sees
    first = max(0, n + 1 - case["window"]) if case["window"] else 0     # the first token any of them sees
    return {"bytes": heads * (n + L - first) * _row_bytes(case) + heads * L * _row_bytes(case) + new + io,
            "flops": 2 * B * case["Hq"] * sum(seen) * (D + Dv) + (rotate if case["cache"] == "turbo" else 0)}


def tolerance(case):
    # Measured against exact(): bf16 results are 1.7e-3 off, f16 ones 2e-4 to 3e-4 (the rounding of the
    # result and of the weights), norms 3e-8.  A dense rotation may put a coordinate that lies within an
    # ulp of a codebook midpoint on either side of it: two or three of 8 million, each in a word of its
    # own, and each moves a 4-million-value reconstruction by 2.5e-4.
    tie = 0.0
    if _dense(case, case["D"]) or _dense(case, case["Dv"]):
        words = case["B"] * case["Hkv"] * (case["tokens"] + case["L"]) * min(
            (case["D"] * case["kb"] + 31) // 32, (case["Dv"] * case["vb"] + 31) // 32)
        tie = min(0.01, 4e-5 + 1.5 / words)
    if case["kind"] == "append":
        return {"rel": 1e-6, "differ": tie} if tie else "exact"
    if case["kind"] == "codec":
        return {"rel": 3e-3, "max": 0.3, "differ": tie} if tie else {"rel": 1e-6, "max": 2e-5}
    bf16 = case["dtype"] == "bf16"
    return {"rel": 7e-3 if bf16 else 1e-3, "max": 0.06 if bf16 else 0.02, "differ": tie}


# ------------------------------------------------------ the same in 64 bits ---
def _rotation64(codec):
    """The rotation M (y = M x) of a codec, from its signs or its matrix."""
    r = torch.from_numpy(np.array(codec.rot_host)).double().cuda()
    if r.dim() == 2:
        return r
    h = torch.ones(1, 1, dtype=torch.float64, device="cuda")
    while h.shape[0] < r.shape[0]:
        h = torch.cat([torch.cat([h, h], 1), torch.cat([h, -h], 1)], 0)
    return h * r[None, :] / math.sqrt(r.shape[0])


def _levels64(words, bits, dim, codebook):
    """Codebook levels (..., dim) of packed rows (..., words): an LSB-first bit stream."""
    w = words.to(torch.int64)
    w = torch.cat([w, torch.zeros_like(w[..., :1])], -1)
    at = torch.arange(dim, device="cuda") * bits
    lo = w[..., at // 32] >> (at % 32)
    hi = torch.where(at % 32 + bits > 32, w[..., at // 32 + 1] << (32 - at % 32), torch.zeros_like(at))
    return codebook[(lo | hi) & ((1 << bits) - 1)]


def _quantized64(x, codec, norm_dtype):
    """(norms, rotated and quantized unit vectors) of x in 64 bits."""
    x = x.double()
    n = x.norm(dim=-1)
    y = (x / n.clamp_min(1e-6)[..., None]) @ _rotation64(codec).T
    cb = torch.from_numpy(codec.codebook.copy()).double().cuda()
    return n.to(norm_dtype).double() if norm_dtype == torch.float16 else n, \
        cb[torch.bucketize(y, (cb[1:] + cb[:-1]) / 2)]


def exact(case, seed):
    state = prepare(case, seed)
    cache, turbo = state["cache"], not (case["cache"] == "plain" and case["kind"] == "layer")
    norm_dtype = DTYPES[case["norm"]]
    if turbo:
        codecs = cache.key_codec, cache.value_codec
        rot = [_rotation64(c) for c in codecs]
    if case["kind"] in ("append", "codec"):
        got = {}
        for side, name, c, m in (("k", "keys", codecs[0], 0), ("v", "values", codecs[1], 1)):
            n, y = _quantized64(state[side], c, norm_dtype)
            got[name] = (n, None)
            if case["kind"] == "codec":
                got[side] = n[..., None] * (y @ rot[m])
        return got
    # scaled queries are rounded to their type: that is how the reference defines the scores
    q = state["q"] * torch.tensor(state["scale"], dtype=state["q"].dtype)
    q = q.double()
    B, Hq, L, _ = q.shape
    R = Hq // case["Hkv"]
    new = None
    if not turbo:
        ks, vs = (torch.cat([old, x], 2) for old, x in zip(cache.state, (state["k"], state["v"])))
    else:
        ks, vs = cache.state[:2]
        if case["kind"] == "layer":
            new = [_quantized64(state[s], c, norm_dtype) for s, c in zip("kv", codecs)]
    lengths = _lengths(case) if case["kind"] == "batch" else None
    out = torch.empty(B, Hq, L, case["Dv"], dtype=torch.float64, device="cuda")
    for b in range(B):
        for h in range(case["Hkv"]):
            rows = q[b, h * R:(h + 1) * R].reshape(R * L, -1)
            if not turbo:
                k, v = ks[b, h].double(), vs[b, h].double()
            else:
                rows = rows @ rot[0].T
                kv = []
                for i, (st, c) in enumerate(zip((ks, vs), codecs)):
                    cb = torch.from_numpy(c.codebook.copy()).double().cuda()
                    x = st[0][b, h].double()[:, None] * _levels64(st[1][b, h], c.bits, c.dim, cb)
                    if new is not None:
                        x = torch.cat([x, new[i][0][b, h][:, None] * new[i][1][b, h]], 0)
                    kv.append(x)
                k, v = kv
                if lengths:
                    k, v = k[-lengths[b]:], v[-lengths[b]:]
            s = (rows @ k.T).reshape(R, L, -1)
            if L > 1 or case["window"]:
                i = torch.arange(case["tokens"], case["tokens"] + L, device="cuda")[:, None]
                t = torch.arange(s.shape[-1], device="cuda")[None, :]
                keep = (t <= i) & ((i < t + case["window"]) if case["window"] else True)
                s = s.masked_fill(~keep, -math.inf)
            o = torch.softmax(s, -1).reshape(R * L, -1) @ v
            out[b, h * R:(h + 1) * R] = (o @ rot[1] if turbo else o).reshape(R, L, -1)
    if not turbo:
        return {"out": out, "keys": ks.double(), "values": vs.double()}
    return {"out": out} if case["kind"] == "batch" else {"out": out, "keys": (None, None), "values": (None, None)}
