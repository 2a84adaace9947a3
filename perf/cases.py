"""The work a user of this framework has it do, as cases that can be timed and compared.

listed() are the cases, draw() gives more of the same ranges; prepare() makes what a
user's program holds before the call, run() is one pass through the public entry points,
work() the bytes and operations the pass cannot do without, tolerance() how far another
correct implementation's results may lie, exact() the results in 64 bits from plain torch.

A case's "kind" names the path:
  decode         one new token's attention over [sink | INT4 middle | recent window] of
                 `layers` layers (ops.decode_attention): eager, or captured in a HIP graph
                 once and replayed for every token, as DecodeGraph does
  pack           the append: quantize + pack a run of tokens into the INT4 block pool
                 (ops.pack_tokens)
  compress       KVCompressor.compress and decompress of a KV tensor
  gather         HeteroKVManager.decompress_dram_chunks: every INT4 token of a layer back
                 as fp16 K and V
  prefill        one prompt chunk's attention over [sink | INT4 middle | recent window] and,
                 causally, itself (ops.prefill_attention)
  fused_decode   fused_dequant_attn_decode on codes, scales and zero points in the
                 unpacked layout KVCompressor returns
  fused_forward  fused_dequant_attn_forward on the same layout
"""
import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "hetero-kvcache-optimizer_amd"))

D = 128            # head_dim of every kernel
BLOCK = 16         # tokens of one INT4 block record
OUTLIERS = [7, 31, 64, 100]   # key channels with 8 times the others' magnitude
TYPES = {"fp16": torch.float16, "bf16": torch.bfloat16}
DEV = "cuda"


def listed():
    return [
        # -- decode: one token per step and sequence
        # the first tokens of a chat turn: nothing evicted yet, one layer called eagerly
        {"name": "decode_short", "kind": "decode", "batch": 1, "hq": 32, "hkv": 8, "sink": 64, "mid": 0,
         "recent": 443, "spread": 0.0, "dtype": "fp16", "layers": 1, "graph": False},
        # a 32K context (the repository's headline decode): 64 + 28608 INT4 + 4096 recent tokens
        {"name": "decode_32k", "kind": "decode", "batch": 1, "hq": 32, "hkv": 8, "sink": 64, "mid": 28608,
         "recent": 4096, "spread": 0.0, "dtype": "fp16", "layers": 8, "graph": True},
        # a 128K context of the 28-layer, 28/4-head bf16 decoder
        {"name": "decode_128k", "kind": "decode", "batch": 1, "hq": 28, "hkv": 4, "sink": 64, "mid": 126912,
         "recent": 4096, "spread": 0.0, "dtype": "bf16", "layers": 4, "graph": True},
        # paged serving of 16 sequences with contexts from 8K to 32K, blocks anywhere in the pool
        {"name": "decode_batch16", "kind": "decode", "batch": 16, "hq": 32, "hkv": 8, "sink": 64, "mid": 28608,
         "recent": 4096, "spread": 0.857, "dtype": "fp16", "layers": 1, "graph": True},
        # -- append and the way back
        # a prefill chunk's evicted tokens (K and V, 4096 tokens of 8 heads)
        {"name": "pack_4k", "kind": "pack", "batch": 1, "hkv": 8, "tokens": 4096, "start": 0, "dtype": "fp16"},
        # the compressor's round trip on one [1, 8, 4096, 128] tensor
        {"name": "compress_4k", "kind": "compress", "batch": 1, "hkv": 8, "tokens": 4096, "dtype": "fp16"},
        # a layer's whole INT4 middle at 32K dequantized for an attention of the user's own
        {"name": "gather_28k", "kind": "gather", "hkv": 8, "tokens": 28608, "dtype": "fp16"},
        # -- prefill: one prompt chunk
        # the last 2048-token chunk of a 128K prompt that attends every evicted token
        {"name": "prefill_128k", "kind": "prefill", "batch": 1, "hq": 32, "hkv": 8, "queries": 2048, "sink": 64,
         "mid": 131072, "recent": 4096, "chunk": True, "dtype": "fp16"},
        # the same chunk as ChunkedPrefillEngine has it attended (sink, recent window, itself)
        # in the 28/4-head bf16 decoder
        {"name": "prefill_chunk", "kind": "prefill", "batch": 1, "hq": 28, "hkv": 4, "queries": 2048, "sink": 64,
         "mid": 0, "recent": 4096, "chunk": True, "dtype": "bf16"},
        # a follow-up question of a conversation: a short, odd chunk against a 32K history
        {"name": "prefill_turn", "kind": "prefill", "batch": 1, "hq": 32, "hkv": 8, "queries": 203, "sink": 64,
         "mid": 28597, "recent": 4096, "chunk": True, "dtype": "fp16"},
        # -- the reference's fused kernels' own signature (32 heads x 16K tokens is the size its
        # resilience benchmark decodes)
        {"name": "fused_decode_16k", "kind": "fused_decode", "batch": 1, "hq": 32, "hkv": 32, "tokens": 16384,
         "dtype": "fp16"},
        {"name": "fused_forward_4k", "kind": "fused_forward", "batch": 1, "hq": 32, "hkv": 32, "queries": 512,
         "tokens": 4096, "dtype": "fp16"},
    ]


# (query heads, kv heads): grouped-query decoders of the repository's configurations and
# tests, and multi-head attention
HEADS = [(32, 8), (32, 8), (28, 4), (16, 2), (32, 32), (24, 8)]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "decode", "pack", "compress", "gather", "prefill", "prefill", "prefill",
                       "fused_decode", "fused_forward"])
    dtype = rng.choice(["fp16", "bf16"])
    hq, hkv = rng.choice(HEADS)
    if kind == "decode":
        batch = rng.choice([1, 1, 1, 2, 3, 5, 8, 16, 24, 48])
        c = {"kind": kind, "batch": batch, "hq": hq, "hkv": hkv, "sink": rng.choice([0, 16, 64]),
             "mid": rng.choice([0, 1, 1, 1, 1]) * _log(rng, 40, 131072), "recent": _log(rng, 16, 4160),
             "spread": 0.0 if batch == 1 else rng.choice([0.0, 0.5, 0.9]), "dtype": dtype, "layers": 1,
             "graph": rng.choice([False, True, True])}
        while work(c)["bytes"] > 6e8:
            c["mid"], c["recent"] = c["mid"] * 2 // 3, max(16, c["recent"] * 4 // 5)
        if c["graph"]:   # as many layers as keep a step's records out of the caches
            c["layers"] = max(1, min(8, int(3.2e8 / work(c)["bytes"])))
        return c
    if kind == "pack":
        t = _log(rng, 1, 16384)
        return {"kind": kind, "batch": rng.choice([1, 1, 2, 4]), "hkv": hkv, "tokens": t,
                "start": rng.choice([0, 0, 16 * rng.randrange(64), rng.randrange(1024)]), "dtype": dtype}
    if kind == "compress":
        return {"kind": kind, "batch": rng.choice([1, 1, 2]), "hkv": hkv, "tokens": _log(rng, 16, 16384),
                "dtype": dtype}
    if kind == "gather":
        return {"kind": kind, "hkv": hkv, "tokens": _log(rng, 100, 65536 * 8 // hkv), "dtype": dtype}
    if kind == "prefill":
        c = {"kind": kind, "batch": rng.choice([1, 1, 1, 2, 4]), "hq": hq, "hkv": hkv, "queries": _log(rng, 16, 2048),
             "sink": rng.choice([0, 64]), "mid": rng.choice([0, 1, 1]) * _log(rng, 100, 131072),
             "recent": rng.choice([0, 1, 1, 1]) * _log(rng, 16, 4160), "chunk": rng.choice([True, True, False]),
             "dtype": dtype}
        if c["mid"] + c["recent"] == 0:
            c["chunk"] = True
        while work(c)["flops"] > 1.5e12 or work(c)["bytes"] > 6e8:
            c["mid"] = c["mid"] * 2 // 3
        return c
    c = {"kind": kind, "batch": rng.choice([1, 1, 1, 2, 4]), "hq": hq, "hkv": hkv}
    if kind == "fused_decode":
        c.update(tokens=_log(rng, 64, 32768))
    else:
        c.update(queries=_log(rng, 16, 2048), tokens=_log(rng, 64, 16384))
    c["dtype"] = dtype
    while work(c)["bytes"] > 4e8 or work(c)["flops"] > 1e12:
        c["tokens"] = c["tokens"] * 2 // 3
    return c


def _mids(c):
    """INT4 tokens of every sequence: from mid * (1 - spread) to mid, in no order."""
    b = c["batch"]
    if b == 1 or not c["spread"]:
        return [c["mid"]] * b
    step = next(s for s in (7, 5, 3, 1) if math.gcd(s, b) == 1)
    return [int(c["mid"] * (1 - c["spread"] * ((i * step) % b) / (b - 1))) for i in range(b)]


# ------------------------------------------------------------------------------- inputs
def _gen(seed, *more):
    s = int(seed)
    for m in more:
        s = (s * 1000003 + m + 1) % (1 << 62)
    return torch.Generator(device=DEV).manual_seed(s)


def _keys(g, shape, dtype):
    k = torch.randn(shape, generator=g, device=DEV, dtype=torch.float32)
    k[..., OUTLIERS] *= 8
    return k.to(dtype)


def _values(g, shape, dtype):
    return torch.randn(shape, generator=g, device=DEV, dtype=torch.float32).to(dtype)


def _layer(c, seed, layer):
    """K and V of one decode layer: per sequence the INT4 tokens, then sink and recent."""
    g, dt, h = _gen(seed, 1, layer), TYPES[c["dtype"]], c["hkv"]
    mids = [(_keys(g, (h, m, D), dt), _values(g, (h, m, D), dt)) for m in _mids(c)]
    zones = [(_keys(g, (c["batch"], h, n, D), dt), _values(g, (c["batch"], h, n, D), dt))
             for n in (c["sink"], c["recent"])]
    q = _values(g, (c["batch"], c["hq"], D), dt)
    return mids, zones, q


def _quantize(x):
    """One INT4 group per 128-value row: codes, scales and zero points as KVCompressor gives
    them, from plain torch in 32 bits."""
    f = x.float()
    mn, mx = f.amin(-1, keepdim=True), f.amax(-1, keepdim=True)
    # a tensor divisor: torch multiplies by the rounded reciprocal of a Python number, which
    # moves scales by an ulp and with them the codes of values halfway between two steps
    scale = ((mx - mn) / torch.full_like(mx, 15.0)).clamp(min=1e-8)
    zp = (-mn / scale).round().clamp(0, 15)
    codes = (f / scale + zp).round().clamp(0, 15).to(torch.uint8)
    return codes, scale.squeeze(-1), zp.squeeze(-1).to(torch.uint8)


def _dequantize64(codes, scale, zp):
    return (codes.double() - zp.double().unsqueeze(-1)) * scale.double().unsqueeze(-1)


def _table(g, counts):
    """Block table of sequences with `counts` blocks each, blocks anywhere in the pool."""
    total, width = sum(counts), max(counts)
    perm = torch.randperm(total, generator=g, device=DEV).to(torch.int32)
    bt = torch.zeros((len(counts), width), dtype=torch.int32, device=DEV)
    off = 0
    for b, n in enumerate(counts):
        bt[b, :n] = perm[off:off + n]
        off += n
    return bt


def _fill(zone_kv, batch, heads):
    from heterokv import ops
    zones = []
    for k, v in zone_kv:
        n = k.shape[2]
        if n:
            z = ops.F16Zone(batch, heads, n, DEV)
            z.write(k, v, 0)
            zones.append((z, None, n))
    return zones


def prepare(case, seed):
    from heterokv import HeteroKVManager, ops
    c, kind = case, case["kind"]
    dt, h = TYPES[c["dtype"]], c["hkv"]
    if kind == "decode":
        lens = _mids(c)
        calls = []
        ws = ops.DecodeWorkspace(DEV)
        for layer in range(c["layers"]):
            mids, zone_kv, q = _layer(c, seed, layer)
            kw = {"zones": _fill(zone_kv, c["batch"], h), "workspace": ws}
            if max(lens):
                counts = [(m + BLOCK - 1) // BLOCK for m in lens]
                pool = ops.Int4Pool(sum(counts), h, DEV)
                bt = _table(_gen(seed, 2, layer), counts)
                for b, (k, v) in enumerate(mids):
                    if lens[b]:
                        ops.pack_tokens(pool, k[None], v[None], 0, bt[b:b + 1])
                kw.update(pool=pool, block_table=bt, int4_max_len=max(lens),
                          int4_lens=torch.tensor(lens, dtype=torch.int32, device=DEV) if c["spread"] else None)
            calls.append((q, kw))
        state = {"kind": kind, "calls": calls, "graph": None}
        if c["graph"]:
            outs = [torch.empty_like(q) for q, _ in calls]
            for (q, kw), o in zip(calls, outs):
                ops.decode_attention(q, out=o, **kw)   # the workspace and the library are there before the capture
            torch.cuda.synchronize()
            graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(graph):
                for (q, kw), o in zip(calls, outs):
                    ops.decode_attention(q, out=o, **kw)
            state.update(graph=graph, outs=outs)
        return state
    if kind == "pack":
        g = _gen(seed, 3)
        shape = (c["batch"], h, c["tokens"], D)
        nb = (c["start"] + c["tokens"] + BLOCK - 1) // BLOCK
        return {"kind": kind, "k": _keys(g, shape, dt), "v": _values(g, shape, dt), "start": c["start"],
                "pool": ops.Int4Pool(nb * c["batch"], h, DEV), "bt": _table(g, [nb] * c["batch"])}
    if kind == "compress":
        from heterokv import KVCompressor
        return {"kind": kind, "x": _keys(_gen(seed, 4), (c["batch"], h, c["tokens"], D), dt),
                "comp": KVCompressor(), "dtype": dt}
    if kind == "gather":
        g = _gen(seed, 5)
        # sink and recent window of 16 tokens each beside the evicted ones
        k, v = _keys(g, (1, h, c["tokens"] + 32, D), dt), _values(g, (1, h, c["tokens"] + 32, D), dt)
        mgr = HeteroKVManager(1, sink_tokens=16, hbm_budget_tokens=32, device=DEV)
        mgr.update(0, k, v, "prefill", 0)
        return {"kind": kind, "mgr": mgr}
    if kind == "prefill":
        (mk, mv), zone_kv, q, ck, cv = _prefill_inputs(c, seed)
        kw = {"zones": _fill(zone_kv, c["batch"], h)}
        if c["mid"]:
            nb = (c["mid"] + BLOCK - 1) // BLOCK
            kw.update(pool=ops.Int4Pool(nb * c["batch"], h, DEV), block_table=_table(_gen(seed, 6), [nb] * c["batch"]),
                      int4_max_len=c["mid"])
            ops.pack_tokens(kw["pool"], mk, mv, 0, kw["block_table"])
        if c["chunk"]:
            kw.update(chunk_k=ck, chunk_v=cv)
        return {"kind": kind, "q": q, "kw": kw}
    k, v, q = _fused_inputs(c, seed)
    return {"kind": kind, "args": (q,) + _quantize(k) + _quantize(v)}


def _prefill_inputs(c, seed):
    g, dt, h, b = _gen(seed, 7), TYPES[c["dtype"]], c["hkv"], c["batch"]
    mid = _keys(g, (b, h, c["mid"], D), dt), _values(g, (b, h, c["mid"], D), dt)
    zones = [(_keys(g, (b, h, n, D), dt), _values(g, (b, h, n, D), dt)) for n in (c["sink"], c["recent"])]
    q = _values(g, (b, c["hq"], c["queries"], D), dt)
    return mid, zones, q, _keys(g, (b, h, c["queries"], D), dt), _values(g, (b, h, c["queries"], D), dt)


def _fused_inputs(c, seed):
    g, dt = _gen(seed, 8), TYPES[c["dtype"]]
    kv = (c["batch"], c["hkv"], c["tokens"], D)
    q = _values(g, (c["batch"], c["hq"], c.get("queries", 1), D), dt)
    return _keys(g, kv, dt), _values(g, kv, dt), q


def run(state):
    from heterokv import fused_dequant_attn_decode, fused_dequant_attn_forward, ops
    kind = state["kind"]
    if kind == "decode":
        if state["graph"] is not None:
            state["graph"].replay()
            return state["outs"]
        return [ops.decode_attention(q, **kw) for q, kw in state["calls"]]
    if kind == "pack":
        ops.pack_tokens(state["pool"], state["k"], state["v"], state["start"], state["bt"])
        return state["pool"].data
    if kind == "compress":
        codes, scales, zps = state["comp"].compress(state["x"])
        return codes, scales, zps, state["comp"].decompress(codes, scales, zps, target_dtype=state["dtype"])
    if kind == "gather":
        return state["mgr"].decompress_dram_chunks(0)
    if kind == "prefill":
        return ops.prefill_attention(state["q"], **state["kw"])
    if kind == "fused_decode":
        return fused_dequant_attn_decode(*state["args"])
    return fused_dequant_attn_forward(*state["args"])


# ------------------------------------------------------------------------- work, results
def work(case):
    c, kind, h = case, case["kind"], case["hkv"]
    if kind == "decode":
        mids = _mids(c)
        mid, f16 = sum(mids), c["batch"] * (c["sink"] + c["recent"])
        blocks = sum((m + BLOCK - 1) // BLOCK for m in mids)
        return {"bytes": c["layers"] * (h * (138 * mid + 512 * f16) + 4 * blocks + 2 * c["batch"] * c["hq"] * 256),
                "flops": c["layers"] * 4 * D * c["hq"] * (mid + f16)}
    if kind == "pack":
        return {"bytes": 2 * c["batch"] * h * c["tokens"] * (256 + 69), "flops": 0}
    if kind == "compress":
        return {"bytes": c["batch"] * h * c["tokens"] * 2 * (256 + 128 + 5), "flops": 0}
    if kind == "gather":
        return {"bytes": 2 * h * c["tokens"] * (69 + 256), "flops": 0}
    if kind == "prefill":
        f16, sq = c["sink"] + c["recent"], c["queries"]
        seen = sq * (c["mid"] + f16) + (sq * (sq + 1) // 2 if c["chunk"] else 0)
        return {"bytes": c["batch"] * (h * (138 * c["mid"] + 512 * (f16 + (sq if c["chunk"] else 0))) +
                                       c["hq"] * sq * 512),
                "flops": c["batch"] * 4 * D * c["hq"] * seen}
    sq = c.get("queries", 1)
    return {"bytes": c["batch"] * (2 * h * c["tokens"] * (128 + 5) + c["hq"] * sq * 512),
            "flops": c["batch"] * 4 * D * c["hq"] * sq * c["tokens"]}


def tolerance(case):
    if case["kind"] in ("pack", "compress", "gather"):
        return "exact"
    # about four times what the paths are off exact(): decode 3e-4 in fp16 and 1.7e-3 in bf16
    # (the output's own rounding), prefill 1.7e-3 to 2.5e-3 in both (fp16 operands)
    if case["kind"] in ("decode", "fused_decode"):
        return {"rel": 1.2e-3} if case["dtype"] == "fp16" else {"rel": 7e-3}
    return {"rel": 1e-2}


def _attend64(q, k, v, causal=False):
    """softmax(q k^T / sqrt(D)) v in 64 bits: q [G, S, D] of one kv head, k / v [T, D]; with
    `causal` the last S of the T tokens are the queries' own."""
    out = []
    s, t = q.shape[1], k.shape[0]
    for i in range(0, s, 512):
        qi = q[:, i:i + 512]
        n = qi.shape[1]
        w = (qi.reshape(-1, D) @ k.t()).view(q.shape[0], n, t) / math.sqrt(D)
        if causal:
            row = torch.arange(i, i + n, device=DEV)[:, None]
            w[:, :, t - s:].masked_fill_(torch.arange(s, device=DEV)[None, :] > row, float("-inf"))
        out.append((torch.softmax(w, -1).view(-1, t) @ v).view(q.shape[0], n, D))
    return torch.cat(out, 1)


def exact(case, seed):
    c, kind, h = case, case["kind"], case["hkv"]
    if kind == "pack":
        return None      # bytes of the block records: compared as they are
    if kind == "compress":
        codes, scales, zps = _quantize(_keys(_gen(seed, 4), (c["batch"], h, c["tokens"], D), TYPES[c["dtype"]]))
        return codes, scales.reshape(-1).double(), zps.reshape(-1), _dequantize64(codes, scales, zps)
    if kind == "gather":
        g, dt, n = _gen(seed, 5), TYPES[c["dtype"]], c["tokens"]
        k, v = _keys(g, (1, h, n + 32, D), dt), _values(g, (1, h, n + 32, D), dt)
        return _dequantize64(*_quantize(k[:, :, 16:16 + n])), _dequantize64(*_quantize(v[:, :, 16:16 + n])), n
    rep = c["hq"] // h
    if kind == "decode":
        outs = []
        for layer in range(c["layers"]):
            mids, zones, q = _layer(c, seed, layer)
            out = torch.empty((c["batch"], c["hq"], D), dtype=torch.float64, device=DEV)
            for b, (mk, mv) in enumerate(mids):
                for i in range(h):
                    k = torch.cat([_dequantize64(*_quantize(mk[i]))] + [z[0][b, i].double() for z in zones])
                    v = torch.cat([_dequantize64(*_quantize(mv[i]))] + [z[1][b, i].double() for z in zones])
                    out[b, i * rep:(i + 1) * rep] = _attend64(q[b, i * rep:(i + 1) * rep, None].double(), k, v)[:, 0]
            outs.append(out)
        return outs
    if kind == "prefill":
        (mk, mv), zones, q, ck, cv = _prefill_inputs(c, seed)
        out = torch.empty(q.shape, dtype=torch.float64, device=DEV)
        for b in range(c["batch"]):
            for i in range(h):
                k, v = [_dequantize64(*_quantize(mk[b, i]))], [_dequantize64(*_quantize(mv[b, i]))]
                for zk, zv in zones + ([(ck, cv)] if c["chunk"] else []):
                    k.append(zk[b, i].double())
                    v.append(zv[b, i].double())
                out[b, i * rep:(i + 1) * rep] = _attend64(q[b, i * rep:(i + 1) * rep].double(), torch.cat(k),
                                                          torch.cat(v), c["chunk"])
        return out
    k, v, q = _fused_inputs(c, seed)
    out = torch.empty(q.shape, dtype=torch.float64, device=DEV)
    for b in range(c["batch"]):
        for i in range(h):
            out[b, i * rep:(i + 1) * rep] = _attend64(q[b, i * rep:(i + 1) * rep].double(),
                                                      _dequantize64(*_quantize(k[b, i])),
                                                      _dequantize64(*_quantize(v[b, i])))
    return out
