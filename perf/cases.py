"""The work that a user of pagedkv has it do, as measurable cases.

Every case is one call (or one layer's call) of the public entry points at a
shape that this repository's configurations, tests or benchmark use, or a
generic one of the same range: decode steps from a handful of sequences to a
full batch, whole prompts and chunks of prompts, a step that carries both,
the prefill glue with the rotary embedding, copy-on-write block copies and
token selection.

What a user's program has in hand before a call is built by `prepare`: the
pool with the sequences' keys and values in it, block tables, lengths, the
rotary tables and the projections of the step.  Lengths belong to the case
(they set its work); values and block placement come from the seed.
"""
import math
import os
import random
import sys

import torch

sys.path.insert(0, os.path.join(os.getcwd(), "ai-engine_amd"))
import pagedkv  # noqa: E402

DT = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
DEV = "cuda"


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------
def _decode(name, model, dtype, batch, lo, hi, lens, rope=False, block=16):
    h, kv, hd = model
    return {"name": name, "kind": "decode", "dtype": dtype, "heads": h, "kv_heads": kv,
            "head_dim": hd, "block": block, "batch": batch, "ctx_lo": lo, "ctx_hi": hi,
            "lens": lens, "rope": rope}


def _prefill(name, model, dtype, seqs, q_lo, q_hi, prior_lo, prior_hi, lens, block=16):
    h, kv, hd = model
    return {"name": name, "kind": "prefill", "dtype": dtype, "heads": h, "kv_heads": kv,
            "head_dim": hd, "block": block, "seqs": seqs, "q_lo": q_lo, "q_hi": q_hi,
            "prior_lo": prior_lo, "prior_hi": prior_hi, "lens": lens}


LLAMA_1B = (32, 8, 64)
TINYLLAMA = (32, 4, 64)
LLAMA_8B = (32, 8, 128)
LLAMA_70B = (64, 8, 128)
QWEN_05B = (14, 2, 64)


def listed():
    return [
        # A chat server at low load: 8 sequences of up to a thousand tokens on
        # the smallest Llama (f16): latency of one layer's decode step.
        _decode("decode_1b_8", LLAMA_1B, "f16", 8, 128, 1024, 11),
        # The headline batch: 256 sequences of 512 to 4096 tokens, Llama-3-8B.
        _decode("decode_8b_256", LLAMA_8B, "bf16", 256, 512, 4096, 12),
        # A few long conversations on the 70B shape, the engine's f32
        # projections rotated inside the decode call.
        _decode("decode_70b_long", LLAMA_70B, "bf16", 3, 9000, 32000, 13, rope=True),
        # The reference's own pool type and parity model: f32, ratio 7.
        _decode("decode_qwen_f32", QWEN_05B, "f32", 24, 100, 1000, 14, rope=True),
        # Whole prompts of 3 to 4 thousand tokens (a document and a question),
        # stored and attended in one call.
        _prefill("prefill_8b_prompt", LLAMA_8B, "bf16", 2, 2900, 4096, 0, 0, 15),
        # Chunked prefill: 256-token chunks over priors of up to a thousand.
        _prefill("prefill_tiny_chunks", TINYLLAMA, "f16", 8, 256, 256, 0, 1024, 16),
        # Short prompts of any length into the reference's f32 pool.
        _prefill("prefill_qwen_f32", QWEN_05B, "f32", 6, 30, 900, 0, 0, 17),
        # One layer of a continuous-batching step: chunks and decodes together.
        {"name": "mixed_tiny", "kind": "mixed", "dtype": "f16", "heads": 32, "kv_heads": 4,
         "head_dim": 64, "block": 16, "seqs": 8, "q_lo": 256, "q_hi": 256, "prior_lo": 0,
         "prior_hi": 1024, "batch": 56, "ctx_lo": 256, "ctx_hi": 2048, "lens": 18},
        # Prefill glue of a layer: 2048 prompt tokens' q and k rotated, k and v
        # stored, from the engine's f32 projections.
        {"name": "append_rope_8b", "kind": "append_rope", "dtype": "bf16", "heads": 32,
         "kv_heads": 8, "head_dim": 128, "block": 16, "tokens": 2048, "lens": 19},
        # Copy-on-write after forks: 300 blocks of every layer of an 8B stage.
        {"name": "fork_copy_8b", "kind": "copy", "dtype": "bf16", "kv_heads": 8,
         "head_dim": 128, "block": 16, "layers": 16, "blocks": 1024, "copies": 300},
        # Token selection of a step's rows: f32 logits of 8 sequences ...
        {"name": "sample_f32_8", "kind": "sample", "dtype": "f32", "batch": 8,
         "vocab": 128256},
        # ... and a full batch of bf16 logits, some rows greedy.
        {"name": "sample_bf16_256", "kind": "sample", "dtype": "bf16", "batch": 256,
         "vocab": 128256},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """A case of the listed ranges: any of the models, types and options, sizes
    spread over their logarithm."""
    kind = rng.choice(["decode", "decode", "decode", "prefill", "prefill", "prefill", "mixed",
                       "append_rope", "copy", "sample", "sample"])
    h, kv, hd = rng.choice([LLAMA_1B, TINYLLAMA, LLAMA_8B, LLAMA_70B, QWEN_05B])
    dtype = rng.choice(["bf16", "bf16", "f16", "f16", "f32"])
    block = rng.choice([16, 16, 16, 32])
    lens = rng.randrange(1 << 20)
    row = kv * hd * 2 * (4 if dtype == "f32" else 2)  # K and V bytes of a token
    if kind == "decode":
        batch = _log(rng, 1, 256)
        hi = _log(rng, 40, max(41, min(32768, 1_200_000_000 // (row * batch))))
        c = _decode("", (h, kv, hd), dtype, batch, max(1, int(hi * rng.uniform(0.1, 1.0))), hi,
                    lens, rng.random() < 0.4, block)
    elif kind == "prefill":
        prior = 0 if rng.random() < 0.5 else _log(rng, 16, 8192)
        seqs = _log(rng, 1, 16)
        # (query, key) pairs x heads x head_dim below the largest listed case
        most = 9e10 * (0.04 if dtype == "f32" else 1.0) / (h * hd * 4 * seqs)
        q = _log(rng, 5, 4096)
        while q * (prior + q / 2) > most and q > 5:
            q = max(5, q * 3 // 4)
            prior = prior * 3 // 4
        c = _prefill("", (h, kv, hd), dtype, seqs, max(1, int(q * rng.uniform(0.3, 1.0))), q,
                     int(prior * rng.uniform(0.0, 1.0)), prior, lens, block)
    elif kind == "mixed":
        c = {"kind": "mixed", "dtype": dtype if dtype != "f32" else "bf16", "heads": h,
             "kv_heads": kv, "head_dim": hd, "block": block, "seqs": _log(rng, 1, 8),
             "q_lo": 16, "q_hi": _log(rng, 17, 512), "prior_lo": 0,
             "prior_hi": _log(rng, 16, 2048), "batch": _log(rng, 1, 64), "ctx_lo": 16,
             "ctx_hi": _log(rng, 100, 2048), "lens": lens}
    elif kind == "append_rope":
        c = {"kind": "append_rope", "dtype": dtype, "heads": h, "kv_heads": kv, "head_dim": hd,
             "block": block, "tokens": _log(rng, 1, 8192), "lens": lens}
    elif kind == "copy":
        blocks = _log(rng, 64, 1024)
        c = {"kind": "copy", "dtype": "bf16", "kv_heads": kv, "head_dim": hd, "block": 16,
             "layers": rng.choice([8, 16, 22]), "blocks": blocks,
             "copies": _log(rng, 1, blocks // 2)}
    else:
        c = {"kind": "sample", "dtype": rng.choice(["f32", "bf16", "f16"]),
             "batch": _log(rng, 1, 256), "vocab": rng.choice([32000, 128256, _log(rng, 1000, 150000)])}
    c.pop("name", None)
    return c


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _ints(case, salt, n, lo, hi):
    r = random.Random(case["lens"] * 131 + salt)
    return [r.randint(lo, hi) for _ in range(n)]


def _decode_lens(case):
    """Tokens cached per sequence before the step."""
    return _ints(case, 1, case["batch"], case["ctx_lo"], case["ctx_hi"])


def _prefill_lens(case):
    """(prior, chunk) tokens per sequence."""
    return (_ints(case, 2, case["seqs"], case["prior_lo"], case["prior_hi"]),
            _ints(case, 3, case["seqs"], case["q_lo"], case["q_hi"]))


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _normal(g, shape, dtype):
    return torch.randn(shape, generator=g, device=DEV, dtype=torch.float32).to(dtype)


def _pool_values(g, n, kv, hd, dtype):
    """n tokens' rows, drawn in pieces (no f32 copy of a whole large pool)."""
    out = torch.empty((n, kv, hd), dtype=dtype, device=DEV)
    for i in range(0, n, 1 << 16):
        m = min(n - i, 1 << 16)
        out[i:i + m] = _normal(g, (m, kv, hd), dtype)
    return out


def _tables(g, totals, bs, spare=1.2):
    """Block tables of sequences of `totals` tokens over a shuffled pool."""
    need = [-(-t // bs) for t in totals]
    nb = max(int(math.ceil(sum(need) * spare)), sum(need) + 1)
    perm = torch.randperm(nb, generator=g, device=DEV).to(torch.int32)
    tables = torch.zeros((len(totals), max(need)), dtype=torch.int32, device=DEV)
    at = 0
    for i, n in enumerate(need):
        tables[i, :n] = perm[at:at + n]
        at += n
    return tables, nb


def _inputs(case, seed):
    """Plain tensors of a case: what `prepare` gives to the library and `exact`
    computes from."""
    g = _gen(seed)
    d = {}
    if case["kind"] == "sample":
        b, v = case["batch"], case["vocab"]
        x = _normal(g, (b, v), torch.float32) * 2.5
        at = torch.randint(0, v, (b, 24), generator=g, device=DEV)  # likely tokens stand out
        x.scatter_add_(1, at, torch.rand((b, 24), generator=g, device=DEV) * 12.0)
        d["logits"] = x.to(DT[case["dtype"]])
        t = torch.rand(b, generator=g, device=DEV) * 0.9 + 0.4
        if b > 4:
            t[:: 8] = 0.0  # greedy requests
        d["temps"] = t
        return d
    dt, kv, hd, bs = DT[case["dtype"]], case["kv_heads"], case["head_dim"], case["block"]
    if case["kind"] == "copy":
        perm = torch.randperm(case["blocks"], generator=g, device=DEV).to(torch.int32)
        n = case["copies"]
        d["src"], d["dst"] = perm[:n].contiguous(), perm[n:2 * n].contiguous()
        d["slab"] = torch.empty((case["layers"], 2, case["blocks"] * bs, kv, hd), dtype=dt,
                                device=DEV)
        for l in range(case["layers"]):
            for w in range(2):
                d["slab"][l, w] = _pool_values(g, case["blocks"] * bs, kv, hd, dt)
        return d
    h = case["heads"]
    if case["kind"] == "append_rope":
        n = case["tokens"]
        nb = -(-n // bs) * 2
        blocks = torch.randperm(nb, generator=g, device=DEV)[:-(-n // bs)]
        pos = torch.arange(n, device=DEV)
        d["slots"] = (blocks[pos // bs] * bs + pos % bs).to(torch.int32)
        d["positions"] = pos.to(torch.int32)
        d["num_blocks"] = nb
        for k, rows in (("q", h), ("k", kv), ("v", kv)):
            d[k] = _normal(g, (n, rows, hd), torch.float32)
        return d
    totals = []
    if case["kind"] in ("prefill", "mixed"):
        prior, chunk = _prefill_lens(case)
        totals += [p + c for p, c in zip(prior, chunk)]
    if case["kind"] in ("decode", "mixed"):
        totals += [c + 1 for c in _decode_lens(case)]
    d["tables"], d["num_blocks"] = _tables(g, totals, bs)
    d["k"] = _pool_values(g, d["num_blocks"] * bs, kv, hd, dt)
    d["v"] = _pool_values(g, d["num_blocks"] * bs, kv, hd, dt)
    if case["kind"] in ("prefill", "mixed"):
        n = sum(chunk)
        d["cu"] = torch.tensor([sum(chunk[:i]) for i in range(len(chunk) + 1)],
                               dtype=torch.int32, device=DEV)
        d["p_lens"] = torch.tensor([p + c for p, c in zip(prior, chunk)], dtype=torch.int32,
                                   device=DEV)
        d["p_q"], d["p_k"], d["p_v"] = (_normal(g, (n, r, hd), dt) for r in (h, kv, kv))
    if case["kind"] in ("decode", "mixed"):
        ctx = _decode_lens(case)
        proj = torch.float32 if case.get("rope") else dt
        d["d_lens"] = torch.tensor([c + 1 for c in ctx], dtype=torch.int32, device=DEV)
        d["d_q"], d["d_k"], d["d_v"] = (_normal(g, (len(ctx), r, hd), proj) for r in (h, kv, kv))
    return d


class _Memory:
    """Device memory of a pool as an array interface; holds the pool, so that a
    tensor over it never outlives it."""

    def __init__(self, cache, ptr, n, item):
        self.cache = cache
        self.__cuda_array_interface__ = {"shape": (n,), "typestr": {2: "<i2", 4: "<f4"}[item],
                                         "data": (ptr, False), "version": 2}


def _pool_view(cache, layer, which, shape):
    """A tensor over the pool's own K (0) or V (1) memory."""
    import ctypes
    k, v = ctypes.c_void_p(), ctypes.c_void_p()
    pagedkv.lib().pkv_pool_layer_ptrs(cache.handle, layer, ctypes.byref(k), ctypes.byref(v))
    item = cache.dtype.itemsize
    t = torch.as_tensor(_Memory(cache, (k, v)[which].value, math.prod(shape), item), device=DEV)
    return t.view(cache.dtype).view(shape)


def prepare(case, seed):
    d = _inputs(case, seed)
    s = {"kind": case["kind"]}
    if case["kind"] == "sample":
        s.update(logits=d["logits"], temps=d["temps"])
        return s
    dt, kv, hd, bs = DT[case["dtype"]], case["kv_heads"], case["head_dim"], case["block"]
    if case["kind"] == "copy":
        nb = case["blocks"]
        cache = pagedkv.PagedKvCache(case["layers"], nb, bs, kv, hd, dt)
        for l in range(case["layers"]):
            slots = torch.arange(nb * bs, dtype=torch.int32, device=DEV)
            cache.layer(l).append(d["slab"][l, 0], d["slab"][l, 1], slots)
        slab = _pool_view(cache, 0, 0, (case["layers"], 2, nb * bs, kv, hd))
        torch.cuda.synchronize()
        s.update(cache=cache, src=d["src"], dst=d["dst"], slab=slab)
        return s
    nb = d["num_blocks"]
    cache = pagedkv.PagedKvCache(1, nb, bs, kv, hd, dt)
    layer = cache.layer(0)
    shape = (nb * bs, kv, hd)
    s.update(cache=cache, layer=layer, pool_k=_pool_view(cache, 0, 0, shape),
             pool_v=_pool_view(cache, 0, 1, shape))
    if case["kind"] == "append_rope":
        s["rope"] = pagedkv.Rope(hd, 500000.0, case["tokens"] + 1)
        s.update({k: d[k] for k in ("q", "k", "v", "slots", "positions")})
        return s
    layer.append(d["k"], d["v"], torch.arange(nb * bs, dtype=torch.int32, device=DEV))
    n_p = case.get("seqs", 0)
    if "p_q" in d:
        prior, chunk = _prefill_lens(case)
        s["prefill"] = dict(q=d["p_q"], cu_q_lens=d["cu"], context_lens=d["p_lens"],
                            block_tables=d["tables"][:n_p].contiguous(), max_q_len=max(chunk),
                            max_context_len=max(p + c for p, c in zip(prior, chunk)),
                            k_new=d["p_k"], v_new=d["p_v"])
    if "d_q" in d:
        s["decode"] = dict(q=d["d_q"], context_lens=d["d_lens"],
                           block_tables=d["tables"][n_p:].contiguous(),
                           max_context_len=max(_decode_lens(case)) + 1, k_new=d["d_k"],
                           v_new=d["d_v"])
        if case.get("rope"):
            s["decode"]["rope"] = pagedkv.Rope(hd, 500000.0, case["ctx_hi"] + 2)
            s["decode"]["out_dtype"] = torch.float32
    torch.cuda.synchronize()
    return s


def run(s):
    kind = s["kind"]
    if kind == "sample":
        return pagedkv.sample(s["logits"], s["temps"])
    if kind == "copy":
        s["cache"].copy_blocks(s["src"], s["dst"])
        return s["slab"]
    layer = s["layer"]
    if kind == "append_rope":
        q = layer.append_rope(s["rope"], s["k"], s["v"], s["slots"], s["positions"], q=s["q"])
        return {"q": q, "k": s["pool_k"], "v": s["pool_v"]}
    if kind == "decode":
        out = layer.decode_attention(**s["decode"])
    elif kind == "prefill":
        out = layer.prefill_attention(**s["prefill"])
    else:
        out = layer.mixed_attention(s["prefill"], s["decode"])
    return {"out": out, "k": s["pool_k"], "v": s["pool_v"]}


# ---------------------------------------------------------------------------
# work, tolerance, 64-bit results
# ---------------------------------------------------------------------------
def work(case):
    kind = case["kind"]
    e = 4 if case["dtype"] == "f32" else 2
    if kind == "sample":
        b, v = case["batch"], case["vocab"]
        return {"bytes": b * v * e + 8 * b, "flops": 0}
    kv, hd, bs = case["kv_heads"], case["head_dim"], case["block"]
    row = kv * hd * e
    if kind == "copy":
        return {"bytes": 2 * 2 * case["layers"] * case["copies"] * bs * row, "flops": 0}
    h = case["heads"]
    if kind == "append_rope":
        n = case["tokens"]
        return {"bytes": n * (h + 2 * kv) * hd * (4 + e) + 8 * n, "flops": 0}
    b = f = 0
    if kind in ("decode", "mixed"):
        x = 4 if case.get("rope") else e  # projections and results
        for c in _decode_lens(case):
            b += 2 * c * row + 2 * kv * hd * (x + e) + 2 * h * hd * x + 4 * -(-(c + 1) // bs) + 4
            f += 4 * (c + 1) * h * hd
    if kind in ("prefill", "mixed"):
        for p, c in zip(*_prefill_lens(case)):
            b += 2 * p * row + 4 * c * row + 2 * c * h * hd * e + 4 * -(-(p + c) // bs) + 8
            f += 4 * h * hd * (c * p + c * (c + 1) // 2)
    return {"bytes": b, "flops": f}


def tolerance(case):
    if case["kind"] in ("sample", "copy"):
        return "exact"
    # Four times the error against 64 bits: f32 sums 4.1e-7 at most over drawn
    # cases, 16-bit results 2.9e-4 (f16) and 1.7e-3 (bf16), f32 results of
    # rotated rows 2.2e-5 (a rotated element that rounds the other way).
    if case.get("rope") and case["dtype"] != "f32":
        return {"rel": 1e-4}
    return {"rel": {"f32": 1.6e-6, "f16": 1.2e-3, "bf16": 6.8e-3}[case["dtype"]]}


def _rope64(x, pos, hd):
    """Rotate-half rope: f32 angles as the tables define them, cos and sin and
    the products in 64 bits."""
    i = torch.arange(hd // 2, device=DEV, dtype=torch.float64)
    power = torch.pow(torch.tensor(500000.0, device=DEV, dtype=torch.float64), 2.0 * i / hd)
    theta = 1.0 / power.to(torch.float32)
    a = (pos.to(torch.float32)[:, None] * theta[None, :]).double()
    c, s = a.cos()[:, None, :], a.sin()[:, None, :]
    x = x.double()
    x1, x2 = x[..., : hd // 2], x[..., hd // 2:]
    return torch.cat([x1 * c - x2 * s, x1 * s + x2 * c], dim=-1)


def _slots(table, lo, hi, bs):
    p = torch.arange(lo, hi, device=DEV)
    return table[p // bs].long() * bs + p % bs


def exact(case, seed):
    kind = case["kind"]
    if kind in ("sample", "copy"):  # whole numbers and bytes
        return None
    d = _inputs(case, seed)
    dt, kv, hd, bs, h = (DT[case["dtype"]], case["kv_heads"], case["head_dim"], case["block"],
                         case["heads"])
    if kind == "append_rope":
        nb = d["num_blocks"]
        pk = torch.zeros((nb * bs, kv, hd), dtype=torch.float64, device=DEV)
        pv = torch.zeros_like(pk)
        pk[d["slots"].long()] = _rope64(d["k"], d["positions"], hd)
        pv[d["slots"].long()] = d["v"].double()
        return {"q": _rope64(d["q"], d["positions"], hd), "k": pk, "v": pv}
    pk, pv = d["k"], d["v"]
    scale, g = 1.0 / math.sqrt(hd), h // kv
    outs = []
    at = 0
    if "p_q" in d:
        prior, chunk = _prefill_lens(case)
        out = torch.empty((sum(chunk), h, hd), dtype=torch.float64, device=DEV)
        for i, (p, c) in enumerate(zip(prior, chunk)):
            new = _slots(d["tables"][i], p, p + c, bs)
            pk[new], pv[new] = d["p_k"][at:at + c], d["p_v"][at:at + c]
            sl = _slots(d["tables"][i], 0, p + c, bs)
            for j in range(kv):
                kk, vv = pk[sl, j].double(), pv[sl, j].double()
                for r in range(0, c, 512):
                    m = min(512, c - r)
                    n = p + r + m  # keys that these queries can see
                    q = d["p_q"][at + r:at + r + m, j * g:(j + 1) * g].double()
                    sc = (q.reshape(m * g, hd) @ kk[:n].t()).view(m, g, n) * scale
                    far = torch.arange(n, device=DEV)[None, :] > (p + r + torch.arange(
                        m, device=DEV))[:, None]
                    sc.masked_fill_(far[:, None, :], -math.inf)
                    w = torch.softmax(sc, dim=-1).view(m * g, n)
                    out[at + r:at + r + m, j * g:(j + 1) * g] = (w @ vv[:n]).view(m, g, hd)
            at += c
        outs.append(out.view(at, h * hd))
    if "d_q" in d:
        ctx = _decode_lens(case)
        q, kn, vn = d["d_q"].double(), d["d_k"].double(), d["d_v"].double()
        if case.get("rope"):
            pos = torch.tensor(ctx, device=DEV)
            q, kn = _rope64(d["d_q"], pos, hd), _rope64(d["d_k"], pos, hd)
            q = q.to(torch.float32).to(dt).double()  # rotated rows are of the pool's type
        kn, vn = kn.to(torch.float32).to(dt), vn.to(torch.float32).to(dt)
        out = torch.empty((len(ctx), h, hd), dtype=torch.float64, device=DEV)
        for i, c in enumerate(ctx):
            t = d["tables"][case.get("seqs", 0) + i]
            sl = _slots(t, 0, c + 1, bs)
            pk[sl[-1]], pv[sl[-1]] = kn[i], vn[i]
            kk, vv = pk[sl].double(), pv[sl].double()
            for j in range(kv):
                w = torch.softmax(q[i, j * g:(j + 1) * g] @ kk[:, j].t() * scale, dim=-1)
                out[i, j * g:(j + 1) * g] = w @ vv[:, j]
        outs.append(out.view(len(ctx), h * hd))
    return {"out": outs[0] if kind != "mixed" else tuple(outs), "k": pk.double(),
            "v": pv.double()}
