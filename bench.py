"""INT4-KV hot-path benchmark on one MI355X.

    python bench.py [--steps K] [--warmup W] [--gpus 1] [--legs c1,c3,c4,c5] [--workload ...]

Headline (`value`): single-layer decode attention, batch 1, 32 query heads / 8 kv heads
(GQA), head_dim 128, context 32768 = 64 fp16 sink tokens + 28608 INT4 tokens (16-token
blocks) + 4096 fp16 recent tokens; q ~ N(0,1)/sqrt(128) fp16; K, V ~ N(0,1) fp16 with K
channels 7/31/64/100 scaled x8; seeded, synthetic.  One step = one launch of the split-K
decode kernel; eight copies of the KV are rotated (8 x 48.6 MB > the 256 MB Infinity
Cache) and the K timed launches are replayed from a HIP graph.  value = algorithmic bytes
x K / elapsed (GB/s).

The same JSON line carries one block per other configuration (each with its own roofline,
CPU baseline and parity figure; their step counts are fixed, not --steps):
  c1_quant      quantize+pack of K, V [1, 8, 4096, 128] fp16 and the round trip to fp16
  c3_paged      batch-16 paged decode, contexts 8K-32K, random-permutation block table
  c4_prefill    2048-query chunked prefill over 64 + 131072 INT4 + 4096 tokens (MFMA bound)
  offload_128k  end-to-end 28-layer bf16 decode at 131072 tokens with 75% of the INT4 KV
                in pinned host memory: full and windowed retrieval tok/s, prefetch stall
CPU baselines are the reference's path restated in float32 torch (oracle/torch_ref.py) on
the host cores (threads: the affinity mask capped by OMP_NUM_THREADS), on bounded samples
that each block names.
"""
import argparse
import json
import math
import os
import statistics
import sys
import time

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, os.path.join(ROOT, "hetero-kvcache-optimizer_amd"))

METRIC = "INT4-KV decode-attn GB/s (% HBM peak) at 32K ctx; tok/s at 128K w/ offload"
HBM_PEAK_GBS = 8000.0
B, HQ, HKV, D = 1, 32, 8, 128
SINK, MID, RECENT = 64, 28608, 4096
CTX = SINK + MID + RECENT
OUTLIERS = [7, 31, 64, 100]
# Algorithmic bytes per step: packed INT4 codes + per-token fp32 scale / u8 zp for K and V,
# the fp16 sink + recent K and V, the fp16 query and the fp16 output.
BYTES_CODES = 2 * HKV * MID * (D // 2)
BYTES_META = 2 * HKV * MID * 5
BYTES_F16 = 2 * HKV * (SINK + RECENT) * D * 2
BYTES_QO = 2 * B * HQ * D * 2
STEP_BYTES = BYTES_CODES + BYTES_META + BYTES_F16 + BYTES_QO  # 48,638,976
TRAFFIC_FILE = os.path.join(ROOT, "profiles", "decode_attn_c2_traffic.txt")


def make_inputs(torch, seed=2):
    g = torch.Generator().manual_seed(seed)
    K = torch.randn((B, HKV, CTX, D), generator=g)
    K[..., OUTLIERS] *= 8
    V = torch.randn((B, HKV, CTX, D), generator=g)
    q = torch.randn((B, HQ, D), generator=g) / math.sqrt(D)
    return q.half(), K.half(), V.half()


def build_copy(torch, ops, q, K, V, dev, bt=None):
    """One KV copy of the 32K decode workload; `bt` is a block table to share between
    copies (the layers of a decode step read one table)."""
    sink = ops.F16Zone(B, HKV, SINK, dev)
    sink.write(K[:, :, :SINK].to(dev), V[:, :, :SINK].to(dev), [0])
    rec = ops.F16Zone(B, HKV, RECENT, dev)
    rec.write(K[:, :, SINK + MID:].to(dev), V[:, :, SINK + MID:].to(dev), [0])
    nb = (MID + 15) // 16
    pool = ops.Int4Pool(nb, HKV, dev)
    if bt is None:
        bt = torch.arange(nb, dtype=torch.int32, device=dev)[None]
    ops.pack_tokens(pool, K[:, :, SINK:SINK + MID].to(dev), V[:, :, SINK:SINK + MID].to(dev),
                    torch.zeros(1, dtype=torch.int32, device=dev), bt)
    pool.check_errors()
    return dict(zones=[(sink, None, SINK), (rec, None, RECENT)], pool=pool, bt=bt)


def read_traffic():
    """HBM bytes per launch measured with rocprofv3 --pmc (committed summary), or None."""
    try:
        with open(TRAFFIC_FILE) as f:
            for ln in f:
                if ln.startswith("traffic_bytes_per_launch:"):
                    return float(ln.split(":", 1)[1])
    except OSError:
        pass
    return None


def cpu_threads(torch):
    """Host threads for the CPU baselines: the affinity mask, capped by OMP_NUM_THREADS
    (the box's CPU share), set on torch; returned as the `cores` figure."""
    n = len(os.sched_getaffinity(0))
    env = os.environ.get("OMP_NUM_THREADS", "")
    if env.isdigit() and int(env) > 0:
        n = min(n, int(env))
    torch.set_num_threads(n)
    return n


def time_cpu(fn, budget_s, max_reps=50):
    """One warmup call, then calls until `budget_s` is spent; median seconds per call."""
    out = fn()
    times = []
    t_end = time.perf_counter() + budget_s
    while True:
        t0 = time.perf_counter()
        out = fn()
        times.append(time.perf_counter() - t0)
        if time.perf_counter() >= t_end or len(times) >= max_reps:
            break
    return statistics.median(times), len(times), out


def cpu_baseline_c2(torch, q, K, V, budget_s):
    """The reference's decode step on the host cores in float32 torch (oracle/torch_ref.py):
    Path C dequantizes the 28608 INT4 tokens of the 8 kv heads to fp16 and concatenates them
    before the sink and recent tokens (manager.py:779-821), then softmax(q K^T / sqrt(d)) V
    with GQA (fused_dequant_attn.py:242-247)."""
    from oracle import torch_ref as tr
    n = cpu_threads(torch)
    kc, ks, kz = tr.compress(K[0, :, SINK:SINK + MID], 128)
    vc, vs, vz = tr.compress(V[0, :, SINK:SINK + MID], 128)
    zk = [K[0, :, :SINK], K[0, :, SINK + MID:]]
    zv = [V[0, :, :SINK], V[0, :, SINK + MID:]]
    q3 = q[0][:, None].float()

    def step():
        return tr.attend(q3, tr.path_c_keys(kc, ks, kz, zk), tr.path_c_keys(vc, vs, vz, zv))

    t, reps, out = time_cpu(step, budget_s)
    return out[:, 0], dict(value=STEP_BYTES / t / 1e9, unit="GB/s", cores=n, kind="port",
                           sample="%d full C2 decode steps (float32 torch: Path C dequant of 28608 INT4 tokens "
                                  "to fp16 + attention), median %.1f ms" % (reps, t * 1e3))


def read_profile(name, key):
    """A "key: value" figure from a committed rocprofv3 summary under profiles/, or None."""
    try:
        with open(os.path.join(ROOT, "profiles", name)) as f:
            for ln in f:
                if ln.startswith(key + ":"):
                    return float(ln.split(":", 1)[1])
    except (OSError, ValueError):
        pass
    return None


def event_time_ms(torch, fn, n, stream=None):
    """Average ms per call of fn over n calls, HIP events on the launch stream."""
    stream = stream or torch.cuda.current_stream()
    e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    e0.record(stream)
    for i in range(n):
        fn(i)
    e1.record(stream)
    e1.synchronize()
    return e0.elapsed_time(e1) / n


LEAD_CYCLES = 1_000_000   # ~0.4 ms of spinning at the shader clock


def lead_in(torch, stream):
    """Enqueues a short spin kernel on `stream` ahead of a timed region, so that the GPU is
    still busy while the host submits the timed graph: the region then holds the timed
    launches back to back, without the host's submission latency in front of the first."""
    with torch.cuda.stream(stream):
        torch.cuda._sleep(LEAD_CYCLES)


def graph_time_ms(torch, launch, n, warmup, dev):
    """Average ms per launch of n launches replayed from one captured HIP graph (launch(i)
    enqueues one kernel), HIP events on the graph's stream."""
    stream = torch.cuda.Stream(device=dev)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=stream):
        for i in range(n):
            launch(i)
    for _ in range(max(warmup, 1)):
        g.replay()
    torch.cuda.synchronize()
    e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    lead_in(torch, stream)
    with torch.cuda.stream(stream):
        e0.record(stream)
        g.replay()
        e1.record(stream)
    e1.synchronize()
    torch.cuda.synchronize()
    return e0.elapsed_time(e1) / n


# ------------------------------------------------------------------------------ C4 prefill
P_SQ, P_SINK, P_MID, P_RECENT = 2048, 64, 131072, 4096
P_HIST = P_SINK + P_MID + P_RECENT
# 4*Hq*D per (query, visible key): history fully visible, the chunk causally
P_FLOPS = 4 * HQ * D * P_SQ * P_HIST + 4 * HQ * D * (P_SQ * (P_SQ + 1) // 2)
MFMA_PEAK_TFLOPS = 2500.0
P_ROWS = list(range(0, 32)) + list(range(P_SQ - 32, P_SQ))   # CPU sample / parity rows


def leg_c4(torch, ops, args):
    """Chunked prefill (one hkv_prefill_attn call: the chunk rewrite into the zone layout, the
    attention kernel over the fp16 zones and the chunk, then over the INT4 tiles, which merges the
    first one's softmax states into its own; all three inside the timed call): 2048 fp16
    queries, 32 q / 8 kv heads, over 64 fp16 sink + 131072 INT4 + 4096 fp16 recent tokens plus the
    chunk itself, causally."""
    from oracle import torch_ref as tr
    dev = torch.device("cuda:0")
    g = torch.Generator().manual_seed(4)
    K = torch.randn((HKV, P_HIST, D), generator=g)
    K[..., OUTLIERS] *= 8
    K = K.half()
    V = torch.randn((HKV, P_HIST, D), generator=g).half()
    CK = torch.randn((HKV, P_SQ, D), generator=g).half()
    CV = torch.randn((HKV, P_SQ, D), generator=g).half()
    q = (torch.randn((HQ, P_SQ, D), generator=g) / math.sqrt(D)).half()
    sink = ops.F16Zone(1, HKV, P_SINK, dev)
    sink.write(K[None, :, :P_SINK].to(dev), V[None, :, :P_SINK].to(dev), 0)
    rec = ops.F16Zone(1, HKV, P_RECENT, dev)
    rec.write(K[None, :, P_SINK + P_MID:].to(dev), V[None, :, P_SINK + P_MID:].to(dev), 0)
    nb = P_MID // 16
    pool = ops.Int4Pool(nb, HKV, dev)
    bt = torch.arange(nb, dtype=torch.int32, device=dev)[None]
    ops.pack_tokens(pool, K[None, :, P_SINK:P_SINK + P_MID].to(dev), V[None, :, P_SINK:P_SINK + P_MID].to(dev),
                    torch.zeros(1, dtype=torch.int32, device=dev), bt)
    qd, ckd, cvd = q[None].to(dev), CK[None].to(dev), CV[None].to(dev)
    out = torch.empty((1, HQ, P_SQ, D), dtype=torch.float16, device=dev)
    zones = [(sink, None, P_SINK), (rec, None, P_RECENT)]

    def launch(i):
        ops.prefill_attention(qd, zones=zones, pool=pool, block_table=bt, int4_max_len=P_MID,
                              chunk_k=ckd, chunk_v=cvd, out=out)

    for i in range(10):
        launch(i)
    torch.cuda.synchronize()
    pool.check_errors()
    ms = event_time_ms(torch, launch, 50)
    tflops = P_FLOPS / (ms * 1e-3) / 1e12
    got = out[0][:, P_ROWS].float().cpu()
    blk = {"workload": "chunked prefill: 2048 fp16 queries, 32 q / 8 kv heads, head_dim 128, over 64 fp16 sink "
                       "+ 131072 INT4 + 4096 fp16 recent + the chunk causally (one hkv_prefill_attn call, two kernels)",
           "value": round(tflops, 2), "unit": "TFLOP/s", "ms_per_step": round(ms, 4), "steps": 50,
           "flops_per_step": P_FLOPS,
           "roofline": {"bound": "mfma", "achieved": round(tflops, 2), "peak": MFMA_PEAK_TFLOPS, "unit": "TFLOP/s",
                        "frac": round(tflops / MFMA_PEAK_TFLOPS, 4),
                        "traffic": read_profile("prefill_attn_c4_traffic.txt", "traffic_bytes_per_call"),
                        "mfma_busy_frac": read_profile("prefill_attn_c4_mfma_busy.txt", "mfma_busy_fraction")}}
    del pool, sink, rec, qd, ckd, cvd
    if args.no_cpu_baseline:
        return blk
    n = cpu_threads(torch)
    kc, ks, kz = tr.compress(K[:, P_SINK:P_SINK + P_MID], 128)
    vc, vs, vz = tr.compress(V[:, P_SINK:P_SINK + P_MID], 128)
    zk = [K[:, :P_SINK], K[:, P_SINK + P_MID:], CK]
    zv = [V[:, :P_SINK], V[:, P_SINK + P_MID:], CV]

    rows = torch.tensor(P_ROWS)
    qr = q[:, rows]

    def step():
        keys = tr.path_c_keys(kc, ks, kz, zk)
        vals = tr.path_c_keys(vc, vs, vz, zv)
        return tr.attend(qr, keys, vals, causal_from=P_HIST, rows=rows)

    t, reps, ref = time_cpu(step, args.cpu_budget, max_reps=5)
    flops = sum(4 * HQ * D * (P_HIST + r + 1) for r in P_ROWS)
    blk["cpu_baseline"] = {"value": round(flops / t / 1e12, 5), "unit": "TFLOP/s", "cores": n, "kind": "port",
                           "sample": "Path C dequant of the 131072 INT4 tokens to fp16 plus float32 attention "
                                     "of 64 query rows (0-31, 2016-2047) x 32 heads, %d rep(s), median %.2f s"
                                     % (reps, t)}
    blk["parity"] = {"rows_checked": len(P_ROWS) * HQ,
                     "max_abs_err_vs_cpu": round(float((got - ref).abs().max()), 6), "tolerance": 2e-3}
    return blk


# ------------------------------------------------------------------------------ C3 paged decode
C3_B, C3_SAMPLE = 16, 2


def leg_c3(torch, ops, args):
    """Batched paged decode: 16 sequences, contexts uniform in [8192, 32768] (seeded), 32 q / 8 kv
    heads, each context = 64 fp16 sink + INT4 middle + 4096 fp16 recent; the INT4 middle lives
    in 16-token blocks of one pool addressed through a seeded random-permutation block table."""
    from oracle import torch_ref as tr
    dev = torch.device("cuda:0")
    gen = torch.Generator().manual_seed(7)
    ctx = torch.randint(8192, 32769, (C3_B,), generator=gen)
    mids = (ctx - SINK - RECENT).tolist()
    nbs = [(m + 15) // 16 for m in mids]
    nbmax, total = max(nbs), sum(nbs)
    perm = torch.randperm(total, generator=gen).to(torch.int32)
    bt = torch.zeros((C3_B, nbmax), dtype=torch.int32)
    off = 0
    for b, nb in enumerate(nbs):
        bt[b, :nb] = perm[off:off + nb]
        off += nb
    g = torch.Generator(device=dev).manual_seed(8)
    pool = ops.Int4Pool(total, HKV, dev)
    bt_d = bt.to(dev)
    keep = []
    for b in range(C3_B):
        Kb = torch.randn((1, HKV, mids[b], D), generator=g, device=dev)
        Kb[..., OUTLIERS] *= 8
        Kb = Kb.half()
        Vb = torch.randn((1, HKV, mids[b], D), generator=g, device=dev).half()
        ops.pack_tokens(pool, Kb, Vb, torch.zeros(1, dtype=torch.int32, device=dev), bt_d[b:b + 1])
        if b < C3_SAMPLE:
            keep.append((Kb[0].cpu(), Vb[0].cpu()))
    pool.check_errors()
    sk = torch.randn((C3_B, HKV, SINK, D), generator=g, device=dev).half()
    sv = torch.randn((C3_B, HKV, SINK, D), generator=g, device=dev).half()
    rk = torch.randn((C3_B, HKV, RECENT, D), generator=g, device=dev).half()
    rv = torch.randn((C3_B, HKV, RECENT, D), generator=g, device=dev).half()
    sink = ops.F16Zone(C3_B, HKV, SINK, dev)
    rec = ops.F16Zone(C3_B, HKV, RECENT, dev)
    sink.write(sk, sv, 0)
    rec.write(rk, rv, 0)
    q = (torch.randn((C3_B, HQ, D), generator=g, device=dev) / math.sqrt(D)).half()
    lens = torch.tensor(mids, dtype=torch.int32, device=dev)
    out = torch.empty((C3_B, HQ, D), dtype=torch.float16, device=dev)
    ws = ops.DecodeWorkspace(dev)
    err = ops.ErrorWord(dev)

    def launch(i):
        ops.decode_attention(q, zones=[(sink, None, SINK), (rec, None, RECENT)], pool=pool, block_table=bt_d,
                             int4_lens=lens, int4_max_len=max(mids), workspace=ws, out=out, err=err)

    for i in range(3):
        launch(i)
    torch.cuda.synchronize()
    ms = graph_time_ms(torch, launch, 40, 2, dev)
    err.check()
    step_bytes = sum(2 * HKV * (m * (D // 2 + 5) + (SINK + RECENT) * D * 2) for m in mids) + \
        2 * C3_B * HQ * D * 2 + 4 * total
    gbs = step_bytes / (ms * 1e-3) / 1e9
    traffic = read_profile("decode_attn_c3_traffic.txt", "traffic_bytes_per_launch")
    launch(0)
    got = out[:C3_SAMPLE].float().cpu()
    blk = {"workload": "batched paged decode: batch 16, contexts uniform in [8192, 32768] (64 fp16 sink + INT4 "
                       "middle + 4096 fp16 recent), 32 q / 8 kv heads, head_dim 128, INT4 blocks through a "
                       "random-permutation block table (%d blocks, one pool)" % total,
           "contexts": ctx.tolist(), "bytes_per_step": step_bytes,
           "value": round(gbs, 2), "unit": "GB/s", "ms_per_step": round(ms, 6), "steps": 40, "launch": "hip graph",
           "roofline": {"bound": "hbm", "achieved": round(gbs, 2), "peak": HBM_PEAK_GBS, "unit": "GB/s",
                        "frac": round(gbs / HBM_PEAK_GBS, 4), "traffic": traffic}}
    if args.no_cpu_baseline:
        return blk
    n = cpu_threads(torch)
    # the sampled sequences' INT4 data as the reference keeps it (codes per token row), in
    # 16-token blocks of a host pool at the same random-permutation positions
    cpu_pool_k = torch.zeros((total, HKV, 16, D), dtype=torch.uint8)
    cpu_pool_v = torch.zeros_like(cpu_pool_k)
    meta = torch.zeros((total, 4, HKV, 16), dtype=torch.float32)
    for b, (Kb, Vb) in enumerate(keep):
        nb, m = nbs[b], mids[b]
        ids = bt[b, :nb].long()
        for pool_c, X, mi in ((cpu_pool_k, Kb, 0), (cpu_pool_v, Vb, 2)):
            c, s_, z = tr.compress(X, 128)
            cp = torch.zeros((HKV, nb * 16, D), dtype=torch.uint8)
            cp[:, :m] = c
            pool_c[ids] = cp.view(HKV, nb, 16, D).transpose(0, 1)
            sp = torch.zeros((HKV, nb * 16))
            zp = torch.zeros((HKV, nb * 16))
            sp[:, :m] = s_.view(HKV, m)
            zp[:, :m] = z.view(HKV, m).float()
            meta[ids, mi] = sp.view(HKV, nb, 16).transpose(0, 1)
            meta[ids, mi + 1] = zp.view(HKV, nb, 16).transpose(0, 1)
    skc, svc, rkc, rvc, qc = sk[:C3_SAMPLE].cpu(), sv[:C3_SAMPLE].cpu(), rk[:C3_SAMPLE].cpu(), rv[:C3_SAMPLE].cpu(), \
        q[:C3_SAMPLE].cpu()

    def one(b, pool_c, mi, zones):
        nb, m = nbs[b], mids[b]
        ids = bt[b, :nb].long()
        codes = pool_c.index_select(0, ids).transpose(0, 1).reshape(HKV, nb * 16, D)[:, :m]
        md = meta.index_select(0, ids)[:, mi:mi + 2].permute(1, 2, 0, 3).reshape(2, HKV, nb * 16)[:, :, :m]
        return tr.path_c_keys(codes, md[0].reshape(-1).contiguous(), md[1].reshape(-1).to(torch.uint8), zones)

    def step():
        outs = []
        for b in range(C3_SAMPLE):
            keys = one(b, cpu_pool_k, 0, [skc[b], rkc[b]])
            vals = one(b, cpu_pool_v, 2, [svc[b], rvc[b]])
            outs.append(tr.attend(qc[b][:, None].float(), keys, vals)[:, 0])
        return torch.stack(outs)

    t, reps, ref = time_cpu(step, args.cpu_budget)
    sb = sum(2 * HKV * (mids[b] * (D // 2 + 5) + (SINK + RECENT) * D * 2) + 2 * HQ * D * 2 for b in range(C3_SAMPLE))
    blk["cpu_baseline"] = {"value": round(sb / t / 1e9, 4), "unit": "GB/s", "cores": n, "kind": "port",
                           "sample": "sequences 0-%d of the batch (contexts %s): block-table gather of the INT4 "
                                     "rows, Path C dequant to fp16, float32 attention; %d rep(s), median %.1f ms"
                                     % (C3_SAMPLE - 1, ctx[:C3_SAMPLE].tolist(), reps, t * 1e3)}
    blk["parity"] = {"sequences_checked": C3_SAMPLE,
                     "max_abs_err_vs_cpu": round(float((got - ref).abs().max()), 6), "tolerance": 2e-3}
    return blk


# ------------------------------------------------------------------------------ C1 quantize+pack
C1_BYTES = 2 * 8 * 4096 * 128 * 2 + 2 * (8 * 4096 * 64 + 8 * 4096 * 4 + 8 * 4096)   # 21,299,200


def leg_c1(torch, ops, args):
    """Quantize+pack K, V [1, 8, 4096, 128] fp16 (group 128 = one token row, 4 outlier K channels
    x8): hkv_pack_tokens writes the INT4 block records; back to fp16 by the Path C route
    (hkv_unpack_tokens + hkv_dequantize_groups).  21,299,200 algorithmic bytes per K+V call;
    16 rotated copies keep the inputs out of the 256 MB Infinity Cache."""
    from heterokv.kv_compressor import KVCompressor
    from oracle import torch_ref as tr
    dev = torch.device("cuda:0")
    g = torch.Generator().manual_seed(0)
    K = torch.randn((1, 8, 4096, 128), generator=g)
    K[..., OUTLIERS] *= 8
    V = torch.randn((1, 8, 4096, 128), generator=g)
    K16, V16 = K.half(), V.half()
    R = 16
    ks = [K16.to(dev) for _ in range(R)]
    vs = [V16.to(dev) for _ in range(R)]
    pools = [ops.Int4Pool(256, 8, dev) for _ in range(R)]
    bt = torch.arange(256, dtype=torch.int32, device=dev)[None]
    # the start slot as the manager's append passes it: a host value, which goes to the
    # kernel by value (HkvPackArgs.start_base)
    start = [0]

    def quant(i):
        ops.pack_tokens(pools[i % R], ks[i % R], vs[i % R], start, bt)

    def roundtrip(i):
        for which in (0, 1):
            c, s_, z = ops.unpack_tokens(pools[i % R], bt[0], 4096, which)
            ops.dequantize_groups(c, s_, z)

    for i in range(2 * R):
        quant(i)
        roundtrip(i)
    torch.cuda.synchronize()
    us_q = graph_time_ms(torch, quant, 64, 2, dev) * 1e3
    us_rt = event_time_ms(torch, roundtrip, 64) * 1e3
    for p_ in pools:
        p_.check_errors()
    comp = KVCompressor(group_size=128, bits=4)
    rel, got = {}, {}
    for which, name, x in ((0, "k", K16), (1, "v", V16)):
        c, s_, z = ops.unpack_tokens(pools[0], bt[0], 4096, which)
        got[name] = (c.cpu(), s_.cpu(), z.cpu())
        rel[name] = round(comp.relative_error(x.to(dev), c.view(1, 8, 4096, 128), s_, z), 4)
    gbs = C1_BYTES / (us_q * 1e-6) / 1e9
    blk = {"workload": "quantize+pack K and V [1, 8, 4096, 128] fp16 into 256 INT4 block records of 8 kv heads "
                       "(group 128), then back to fp16 by the Path C route",
           "algorithmic_bytes": C1_BYTES, "value": round(gbs, 2), "unit": "GB/s", "us_per_step": round(us_q, 3),
           "steps": 64, "launch": "hip graph", "roundtrip_us": round(us_rt, 3), "relative_error_pct": rel,
           "roofline": {"bound": "hbm", "achieved": round(gbs, 2), "peak": HBM_PEAK_GBS, "unit": "GB/s",
                        "frac": round(gbs / HBM_PEAK_GBS, 4),
                        "traffic": read_profile("pack_tokens_c1_traffic.txt", "traffic_bytes_per_call")}}
    if args.no_cpu_baseline:
        return blk
    n = cpu_threads(torch)

    def step():
        return tr.compress(K16, 128), tr.compress(V16, 128)

    t, reps, ((kc, kss, kz), (vc, vss, vz)) = time_cpu(step, min(args.cpu_budget, 5.0))
    mism = 0
    for (c, s_, z), name in (((kc, kss, kz), "k"), ((vc, vss, vz), "v")):
        gc, gs, gz = got[name]
        mism += int((c.view(8, 4096, 128) != gc).sum() + (s_.view(torch.int32) != gs.view(torch.int32)).sum() +
                    (z != gz).sum())
    blk["cpu_baseline"] = {"value": round(C1_BYTES / t / 1e9, 4), "unit": "GB/s", "cores": n, "kind": "port",
                           "sample": "%d float32 torch compress passes of K and V (kv_compressor.py ops), median "
                                     "%.1f ms" % (reps, t * 1e3)}
    blk["parity"] = {"code_scale_zp_mismatches_vs_cpu": mism}
    return blk


def bench_scoring(torch, ops, args):
    """Heavy-hitter scoring on the 32K decode workload: the decode launch with score
    outputs against the plain one, the head-averaged weights of the newest token
    (hkv_attn_weights, 32 heads x 32768 items) and the eviction candidates of a 131072-token
    score board (8192 blocks of 16, sink 64, local 4096, 64 candidates)."""
    dev = torch.device("cuda:0")
    torch.cuda.set_device(dev)
    q, K, V = make_inputs(torch)
    R = args.copies
    copies = [build_copy(torch, ops, q, K, V, dev) for _ in range(R)]
    q_dev = q.to(dev)
    out = torch.empty((B, HQ, D), dtype=torch.float16, device=dev)
    ws = ops.DecodeWorkspace(dev)
    n_items = MID + SINK + RECENT
    scores = torch.full((B, HQ, n_items), float("-inf"), dtype=torch.float32, device=dev)
    stats = torch.empty((B, HQ, 2), dtype=torch.float32, device=dev)
    board = torch.zeros(131072, dtype=torch.float32, device=dev)
    board += torch.rand(131072, device=dev, generator=torch.Generator(device=dev).manual_seed(3))
    wts = torch.zeros((1, n_items), dtype=torch.float32, device=dev)

    def dec(i, with_scores):
        c = copies[i % R]
        ops.decode_attention(q_dev, zones=c["zones"], pool=c["pool"], block_table=c["bt"], int4_max_len=MID,
                             workspace=ws, out=out, scores=scores if with_scores else None,
                             score_stats=stats if with_scores else None)

    def timed(fn, n):
        for i in range(max(args.warmup, 2)):
            fn(i)
        torch.cuda.synchronize()
        e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        e0.record()
        for i in range(n):
            fn(i)
        e1.record()
        e1.synchronize()
        return e0.elapsed_time(e1) * 1e3 / n

    n = max(args.steps, 16)
    us_plain = timed(lambda i: dec(i, False), n)
    us_scores = timed(lambda i: dec(i, True), n)
    us_weights = timed(lambda i: ops.attn_weights(scores, stats, out=wts, accumulate=True), n)
    us_cand = timed(lambda i: ops.eviction_candidates(board, 131072, 16, 64, 4096, 64), max(n // 8, 8))
    got = ops.eviction_candidates(board, 131072, 16, 64, 4096, 64).cpu().tolist()
    blk = board.view(8192, 16).double().mean(1).cpu().numpy()
    blk[:4] = float("inf")
    blk[8192 - 256:] = float("inf")
    want = sorted(range(8192), key=lambda i: (blk[i], i))[:64]
    line = {
        "metric": "heavy-hitter scoring cost per decode step at 32K ctx (us)",
        "value": round(us_scores - us_plain + us_weights, 3), "unit": "us", "n_gpus": 1, "steps": n,
        "warmup": args.warmup, "ms_per_step": round((us_scores + us_weights) * 1e-3, 6), "higher_is_better": False,
        "scaling": "weak", "vs_baseline": None, "dtype": "fp32",
        "data": "synthetic (the 32K decode workload's seeded K/V; uniform random score board)",
        "config": {"workload": "decode with score outputs (32 q / 8 kv heads, ctx 32768) + head-averaged weights "
                               "of the newest token + 64 eviction candidates over 131072 scored tokens",
                   "decode_us": round(us_plain, 3), "decode_with_scores_us": round(us_scores, 3),
                   "attn_weights_us": round(us_weights, 3), "eviction_candidates_us": round(us_cand, 3),
                   "score_bytes_written": B * HQ * n_items * 4,
                   "candidates_match_float64_means": got == want},
        "roofline": None,
        "cpu_baseline": None,
    }
    print(json.dumps(line), flush=True)


PROBE_LIB = os.path.join(ROOT, "hetero-kvcache-optimizer_amd", "heterokv", "libhkvprobe.so")
# (pattern, workgroups, waves per workgroup, units in flight per wave): 8 and 16 waves per
# CU at 1x and 2x the decode's 256-workgroup grid, plus the INT4 pool's head-part pattern
PROBE_SHAPES = ("contig:256:8:2,contig:256:8:4,contig:256:8:8,contig:256:16:2,contig:256:16:4,"
                "contig:512:4:4,contig:512:4:8,contig:512:8:2,contig:512:8:4,contig:1024:8:2,"
                "parts:256:8:2,parts:256:8:4,parts:256:16:2,parts:512:8:2")


def bench_probe(torch, args):
    """Streaming-read probes at the 32K decode's size: how fast one launch of a given shape
    reads 48,638,976 bytes (contiguous) or the INT4 pool's 2208-byte head parts of 1788
    records of 8 heads (31,583,232 bytes), with no compute.  Eight rotated copies defeat
    the Infinity Cache; launches are replayed from a HIP graph, HIP events on its stream."""
    import ctypes
    dev = torch.device("cuda:0")
    lib = ctypes.CDLL(PROBE_LIB)
    lib.hkv_probe_stream.restype = ctypes.c_int
    lib.hkv_probe_stream.argtypes = [ctypes.c_void_p, ctypes.c_int64, ctypes.c_int32, ctypes.c_int32, ctypes.c_int32,
                                     ctypes.c_int32, ctypes.c_int32, ctypes.c_int32, ctypes.c_uint32,
                                     ctypes.c_void_p, ctypes.c_void_p]
    R = args.copies
    parts_bytes = HKV * 2208 * ((MID + 15) // 16)
    bufs = [torch.randint(0, 1 << 30, (STEP_BYTES // 4,), dtype=torch.int32, device=dev) for _ in range(R)]
    sink = torch.zeros(1024 * 16 * 64, dtype=torch.int32, device=dev)
    n = max(args.steps, 64)
    n -= n % R
    shapes = [s for s in (args.probe_shapes or PROBE_SHAPES).split(",") if s]
    rows = []
    for sh in shapes:
        pat, grid, waves, depth = sh.split(":")
        grid, waves, depth = int(grid), int(waves), int(depth)
        pattern = {"contig": 0, "parts": 1}[pat]
        nbytes = STEP_BYTES if pattern == 0 else parts_bytes

        def launch(i):
            st = torch.cuda.current_stream(dev).cuda_stream   # the capturing stream under graph capture
            rc = lib.hkv_probe_stream(bufs[i % R].data_ptr(), nbytes, pattern, grid, waves, depth, HKV, 2208,
                                      0x9E3779B9, sink.data_ptr(), ctypes.c_void_p(st))
            if rc != 0:
                raise RuntimeError("hkv_probe_stream(%s) returned %d" % (sh, rc))

        if args.no_graph:
            for i in range(R):
                launch(i)
            ms = event_time_ms(torch, launch, n)
        else:
            ms = graph_time_ms(torch, launch, n, 2, dev)
        rows.append({"shape": sh, "waves_per_cu": waves * grid // 256, "bytes": nbytes, "us": round(ms * 1e3, 3),
                     "gbs": round(nbytes / (ms * 1e-3) / 1e9, 1), "frac": round(nbytes / (ms * 1e-3) / 1e9 / HBM_PEAK_GBS, 4)})
        print("[probe] %-18s %6.2f us  %7.1f GB/s" % (sh, rows[-1]["us"], rows[-1]["gbs"]), file=sys.stderr, flush=True)
    best = max((r for r in rows if r["bytes"] == STEP_BYTES), key=lambda r: r["gbs"], default=None)
    line = {
        "metric": "streaming-read probe GB/s at the 32K decode's byte count",
        "value": best["gbs"] if best else None, "unit": "GB/s", "n_gpus": 1, "steps": n, "warmup": 2,
        "ms_per_step": round(best["us"] * 1e-3, 6) if best else None, "higher_is_better": True, "scaling": "weak",
        "vs_baseline": None, "dtype": "u8", "data": "synthetic (random int32 words, 8 rotated copies)",
        "config": {"workload": "read-only streaming probe (no compute), 48,638,976 bytes contiguous or the "
                               "31,583,232-byte INT4 head-part pattern; %d launches per shape from a HIP graph" % n,
                   "shapes": rows},
        "roofline": {"bound": "hbm", "achieved": best["gbs"] if best else None, "peak": HBM_PEAK_GBS, "unit": "GB/s",
                     "frac": best["frac"] if best else None, "traffic": None},
        "cpu_baseline": None,
    }
    return line


TIMELINE_LIB = os.path.join(ROOT, "hetero-kvcache-optimizer_amd", "heterokv", "libheterokv_timeline.so")


def bench_timeline(torch, args):
    """Phase timeline of the 32K decode kernel, from the library's timeline build
    (HKV_DECODE_TIMELINE: every wave stamps the 100 MHz constant clock at its phase
    boundaries).  The stamps of each sampled launch are read back and reduced to: first data
    consumed (INT4 and fp16 ranges), block ids of the INT4 ranges in LDS, streaming end
    per workgroup (INT4 ranges and fp16 ranges), partial states stored, the last ticket,
    the final merge's loads and the output write of each pair's last workgroup.  A graph of
    the 8 launches is replayed and the stamps of its last launch are read (launches back to
    back, as in the headline bench).  Times are microseconds from that launch's first wave
    start; figures are medians over the samples."""
    import ctypes
    import numpy as np
    from heterokv import _lib
    _lib.LIB_PATH = TIMELINE_LIB
    from heterokv import ops
    lib = _lib.load()
    lib.hkv_decode_timeline_read.restype = ctypes.c_int64
    lib.hkv_decode_timeline_read.argtypes = [ctypes.c_void_p, ctypes.c_int64]
    dev = torch.device("cuda:0")
    q, K, V = make_inputs(torch)
    R = args.copies
    bt = torch.arange((MID + 15) // 16, dtype=torch.int32, device=dev)[None]
    copies = [build_copy(torch, ops, q, K, V, dev, bt) for _ in range(R)]
    q_dev = q.to(dev)
    out = torch.empty((B, HQ, D), dtype=torch.float16, device=dev)
    ws = ops.DecodeWorkspace(dev)
    err = ops.ErrorWord(dev)

    def launch(i):
        c = copies[i % R]
        ops.decode_attention(q_dev, zones=c["zones"], pool=c["pool"], block_table=c["bt"], int4_max_len=MID,
                             workspace=ws, out=out, deterministic=args.deterministic, err=err)

    for i in range(max(args.warmup, R)):
        launch(i)
    torch.cuda.synchronize()
    stream = torch.cuda.Stream(device=dev)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=stream):
        for i in range(R):
            launch(i)
    g.replay()
    torch.cuda.synchronize()
    buf = np.zeros((16384, 16), dtype=np.uint64)
    keys = ("first_data_int4_p50", "first_data_f16_p50", "ids_in_lds_int4_p50", "ids_in_lds_int4_max",
            "stream_end_int4_p50", "stream_end_int4_max", "stream_end_f16_p50", "stream_end_f16_max",
            "stream_end_all_min", "partials_stored_max", "last_ticket_max", "final_loads_done_max",
            "output_written_max")
    samples = {k: [] for k in keys}
    per_xcd = []
    n_s = max(min(args.steps, 256), 8)
    for i in range(n_s):
        g.replay()   # the stamps of the graph's last launch (steady state, launches back to back)
        n = lib.hkv_decode_timeline_read(buf.ctypes.data_as(ctypes.c_void_p), buf.shape[0])
        if n <= 0:
            raise RuntimeError("timeline read failed (%d)" % n)
        t = buf[:n].astype(np.int64)
        t0 = t[:, 0].min()
        us = lambda col: (t[:, col] - t0) / 100.0   # noqa: E731  (100 MHz clock)
        info = t[:, 7]
        n4 = (info >> 24) & 0xFFFFFF
        nfw = info & 0xFFFFFF
        xcd = (info >> 56) & 0xF
        last = ((info >> 48) & 1) == 1
        wg = np.arange(n) // 8
        int4_rng = (n4 > 0) & (nfw == 0)
        f16_rng = (nfw > 0) & (n4 == 0)
        end_wg = np.array([us(2)[wg == w].max() for w in range(n // 8)])
        kind4 = np.array([int4_rng[w * 8] for w in range(n // 8)])
        kindf = np.array([f16_rng[w * 8] for w in range(n // 8)])
        ids = us(1)[int4_rng]
        first = us(8)
        samples["first_data_int4_p50"].append(float(np.median(first[int4_rng])) if int4_rng.any() else None)
        samples["first_data_f16_p50"].append(float(np.median(first[f16_rng])) if f16_rng.any() else None)
        samples["ids_in_lds_int4_p50"].append(float(np.median(ids)) if ids.size else None)
        if os.environ.get("HKV_TIMELINE_WAITS") == "1":
            for key, col, sel in (("prologue_in_f16_p50", 9, f16_rng), ("prologue_in_int4_p50", 10, int4_rng)):
                samples.setdefault(key, []).append(float(np.median(us(col)[sel])) if sel.any() else None)
        samples["ids_in_lds_int4_max"].append(float(ids.max()) if ids.size else None)
        for name, sel in (("int4", kind4), ("f16", kindf)):
            e = end_wg[sel]
            samples["stream_end_%s_p50" % name].append(float(np.median(e)) if e.size else None)
            samples["stream_end_%s_max" % name].append(float(e.max()) if e.size else None)
        samples["stream_end_all_min"].append(float(end_wg.min()))
        samples["partials_stored_max"].append(float(us(3).max()))
        samples["last_ticket_max"].append(float(us(4)[last].max()) if last.any() else None)
        samples["final_loads_done_max"].append(float(us(5)[last].max()) if last.any() else None)
        samples["output_written_max"].append(float(us(6)[last].max()) if last.any() else None)
        per_xcd.append([float(end_wg[np.array([xcd[w * 8] for w in range(n // 8)]) == x].max())
                        for x in range(8) if (xcd == x).any()])
    err.check()
    med = {k: (round(float(np.median([v for v in vals if v is not None])), 3)
               if any(v is not None for v in vals) else None) for k, vals in samples.items()}
    line = {
        "metric": "INT4-KV decode kernel phase timeline at 32K ctx (us from the first wave's start)",
        "value": med["output_written_max"], "unit": "us", "n_gpus": 1, "steps": n_s, "warmup": args.warmup,
        "ms_per_step": None, "higher_is_better": False, "scaling": "weak", "vs_baseline": None, "dtype": "fp16",
        "data": "synthetic (the 32K decode workload's seeded K/V)",
        "config": {"workload": "single-layer INT4-KV decode attention, batch 1, 32 q / 8 kv heads, ctx 32768 = "
                               "64 fp16 sink + 28608 INT4 + 4096 fp16 recent; timeline build of the library, "
                               "last launch of a replayed 8-launch graph",
                   "phases_us_median": med,
                   "stream_end_max_per_xcd_us_median": [round(float(x), 3) for x in np.median(np.array(per_xcd), 0)],
                   "waves_per_launch": int(n)},
        "roofline": None,
        "cpu_baseline": None,
    }
    return line


T_LAYERS, T_HQ, T_HKV, T_HIDDEN, T_INTER, T_VOCAB = 28, 28, 4, 3584, 18944, 152064
T_CTX, T_CHUNK, T_SINK, T_KEEP, T_HOST_FRAC = 131072, 2048, 64, 4160, 0.75
PCIE_GEN5_X16_GBS = 63.0   # 32 GT/s x 16 lanes, 128b/130b encoding, one direction


def _tiered_model(torch, dev):
    """Random-init bf16 Qwen2-style decoder: 28 layers, hidden 3584, 28 q / 4 kv heads,
    head_dim 128, MLP 18944, vocabulary 152064 (Qwen2-VL-7B's text decoder sizes)."""
    from transformers import Qwen2Config, Qwen2ForCausalLM
    from heterokv.engine_wrapper import register_attention
    cfg = Qwen2Config(vocab_size=T_VOCAB, hidden_size=T_HIDDEN, intermediate_size=T_INTER,
                      num_hidden_layers=T_LAYERS, num_attention_heads=T_HQ, num_key_value_heads=T_HKV,
                      max_position_embeddings=T_CTX + 4096, rope_theta=1e6, rms_norm_eps=1e-6,
                      tie_word_embeddings=False, attn_implementation=register_attention())
    torch.manual_seed(0)
    prev = torch.get_default_dtype()
    torch.set_default_dtype(torch.bfloat16)
    try:
        with torch.device(dev):
            model = Qwen2ForCausalLM(cfg)
    finally:
        torch.set_default_dtype(prev)
    return model.eval()


def _decode_tokens(torch, model, cache, tok, pos, n, dev):
    """n greedy decode steps; each ends with a synchronize (the host reads the token id).
    Returns the next token, position, per-token seconds and per-token prefetch stats."""
    times, stats = [], []
    for _ in range(n):
        t0 = time.perf_counter()
        out = model(input_ids=tok, past_key_values=cache, position_ids=torch.tensor([[pos]], device=dev),
                    use_cache=True, logits_to_keep=1)
        tok = out.logits[:, -1:].argmax(-1)
        torch.cuda.synchronize()
        times.append(time.perf_counter() - t0)
        stats.append(cache.prefetch_stats())
        pos += 1
    return tok, pos, times, stats


def _decode_tokens_graph(torch, runner, tok, pos, n, dev):
    """_decode_tokens through a DecodeGraph (one captured decode step replayed per token)."""
    times = []
    for _ in range(n):
        t0 = time.perf_counter()
        logits = runner.step(tok, torch.tensor([[pos]], device=dev))
        tok = logits[:, -1:].argmax(-1)
        torch.cuda.synchronize()
        times.append(time.perf_counter() - t0)
        pos += 1
    return tok, pos, times, []


def _summ(times, stats):
    import statistics
    t = statistics.median(times)
    stall = statistics.median([s["stall_ms"] for s in stats]) if stats else 0.0
    out = {"tok_per_s": round(1.0 / t, 3), "ms_per_token": round(t * 1e3, 3),
           "prefetch_stall_ms_per_token": round(stall, 3),
           "stall_fraction": round(stall / (t * 1e3), 4)}
    if stats and any(s.get("per_layer") for s in stats):
        layers = sorted({l for s in stats for l, _ in s.get("per_layer", [])})
        out["stall_ms_per_layer_median"] = [
            round(statistics.median([ms for s in stats for l2, ms in s.get("per_layer", []) if l2 == l] or [0.0]), 4)
            for l in layers]
    return out


def cpu_baseline_c5(torch, model, budget_s):
    """The reference's decode step restated on the host cores in float32 torch for ONE of the
    28 layers at the 131072-token shape (Path C: dequantize the layer's 126912 INT4 tokens to
    fp16, attention over them plus 64 sink + 4096 recent tokens, 28 q / 4 kv heads; the
    layer's projections and MLP); per token the layer time x 28 plus the final lm_head GEMV."""
    from oracle import torch_ref as tr
    n = cpu_threads(torch)
    mid = T_CTX - T_KEEP
    g = torch.Generator().manual_seed(5)
    kn = torch.randn((T_HKV, mid, D), generator=g).half()
    vn = torch.randn((T_HKV, mid, D), generator=g).half()
    kc, ks, kz = tr.compress(kn, 128)
    vc, vs, vz = tr.compress(vn, 128)
    del kn, vn
    hk = [torch.randn((T_HKV, T_KEEP, D), generator=g).half()]
    hv = [torch.randn((T_HKV, T_KEEP, D), generator=g).half()]
    layer = model.model.layers[0]
    w = {nm: p.detach().float().cpu() for nm, p in layer.named_parameters()}
    lm = model.lm_head.weight.detach().float().cpu()
    x = torch.randn(1, T_HIDDEN)

    def layer_step():
        h = x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + 1e-6) * w["input_layernorm.weight"]
        q = h @ w["self_attn.q_proj.weight"].T + w["self_attn.q_proj.bias"]
        h @ w["self_attn.k_proj.weight"].T
        h @ w["self_attn.v_proj.weight"].T
        a = tr.attend(q.view(T_HQ, 1, D), tr.path_c_keys(kc, ks, kz, hk), tr.path_c_keys(vc, vs, vz, hv))
        o = a.reshape(1, T_HQ * D) @ w["self_attn.o_proj.weight"].T
        h2 = x + o
        h3 = h2 * torch.rsqrt(h2.pow(2).mean(-1, keepdim=True) + 1e-6) * w["post_attention_layernorm.weight"]
        gte = torch.nn.functional.silu(h3 @ w["mlp.gate_proj.weight"].T) * (h3 @ w["mlp.up_proj.weight"].T)
        return h2 + gte @ w["mlp.down_proj.weight"].T

    t_layer, reps, _ = time_cpu(layer_step, budget_s, max_reps=5)
    t_head, _, _ = time_cpu(lambda: x @ lm.T, 1.0, max_reps=3)
    t_tok = T_LAYERS * t_layer + t_head
    return {"value": round(1.0 / t_tok, 5), "unit": "tok/s", "cores": n, "kind": "port",
            "sample": "%d timed pass(es) of one decoder layer at 131072 tokens (float32 torch: Path C dequant "
                      "of 126912 INT4 tokens + attention + projections/MLP, median %.2f s) x 28 + lm_head GEMV"
                      % (reps, t_layer)}


def _tiered_prefill(torch, dev):
    """The C5 model and its 131072-token prompt, prefilled in 2048-token chunks (fused prefill
    kernel) through ChunkedPrefillEngine, four calls of 32768 tokens.  Returns the model, the
    token ids, the cache and the prefill wall seconds."""
    from heterokv.engine_wrapper import ChunkedPrefillEngine, FusedHeteroCache
    t0 = time.perf_counter()
    model = _tiered_model(torch, dev)
    torch.cuda.synchronize()
    print("[c5] model ready in %.1f s" % (time.perf_counter() - t0), file=sys.stderr, flush=True)
    ids = torch.randint(0, T_VOCAB, (1, T_CTX), generator=torch.Generator().manual_seed(1)).to(dev)
    cache = FusedHeteroCache(num_layers=T_LAYERS, sink_tokens=T_SINK, keep_tail=T_KEEP, chunk_size=T_CHUNK,
                             device=str(dev), fused_prefill=True)
    t0 = time.perf_counter()
    with torch.inference_mode():
        eng = ChunkedPrefillEngine(model, cache, chunk_size=T_CHUNK)
        for start in range(0, T_CTX, 16 * T_CHUNK):
            part = ids[:, :start + 16 * T_CHUNK]
            eng.prefill(part[:, start:], position_ids=torch.arange(start, part.shape[1], device=dev)[None])
            torch.cuda.synchronize()
            print("[c5] prefill %d / %d tokens, %.1f s" % (part.shape[1], T_CTX, time.perf_counter() - t0),
                  file=sys.stderr, flush=True)
    return model, ids, cache, time.perf_counter() - t0


def bench_tiered_prefill(torch, args):
    """The C5 model's 128K chunked prefill alone (for a kernel trace of it)."""
    _, _, cache, prefill_s = _tiered_prefill(torch, torch.device("cuda:0"))
    return {"workload": "128K chunked prefill of the C5 model (28 layers, 28 q / 4 kv heads, hidden 3584, random-init "
                        "bf16 weights, 2048-token chunks, sink 64 + recent 4096 fp16, the rest packed to INT4)",
            "prefill_seconds": round(prefill_s, 2), "tokens": T_CTX, "tok_per_s": round(T_CTX / prefill_s, 1),
            "int4_tokens_per_layer": cache._manager.dram_tokens(0)}


def leg_c5(torch, args, timed=8, warm=2):
    """End-to-end tiered decode at 131072 tokens: chunked prefill (2048-token chunks, fused
    prefill kernel), then 75% of every layer's INT4 block records moved to pinned host memory;
    decode with each layer's host records copied on the side stream one layer ahead.  Greedy
    tokens; every variant decodes `timed` tokens after `warm` untimed ones."""
    from heterokv.engine_wrapper import DecodeGraph
    from oracle import torch_ref as tr
    dev = torch.device("cuda:0")
    model, ids, cache, prefill_s = _tiered_prefill(torch, dev)
    mgr = cache._manager
    int4_tokens = mgr.dram_tokens(0)
    out = {}
    with torch.inference_mode():
        tok, pos = ids[:, -1:], T_CTX
        tok, pos, _, _ = _decode_tokens(torch, model, cache, tok, pos, warm, dev)
        tok, pos, tm, st = _decode_tokens(torch, model, cache, tok, pos, timed, dev)
        out["resident"] = _summ(tm, st)
        runner = DecodeGraph(model, cache)
        tok, pos, _, _ = _decode_tokens_graph(torch, runner, tok, pos, max(warm, 3), dev)
        tok, pos, tm, st = _decode_tokens_graph(torch, runner, tok, pos, timed, dev)
        out["resident_graph"] = _summ(tm, st)
        runner.close()
        del runner
        moved = cache.offload_to_host(T_HOST_FRAC, seed=0)
        torch.cuda.synchronize()
        host_bytes = mgr.memory_summary()["host_bytes"]
        # full retrieval (Path C): every host record crosses PCIe every token
        tok, pos, _, _ = _decode_tokens(torch, model, cache, tok, pos, warm, dev)
        b0 = mgr.prefetch_stats()["bytes_h2d"]
        tok, pos, tm, st = _decode_tokens(torch, model, cache, tok, pos, timed, dev)
        full = _summ(tm, st)
        full["h2d_bytes_per_token"] = (st[-1]["bytes_h2d"] - b0) // max(timed, 1)
        out["full"] = full
        # parity: one layer's decode attention over its host-tier records (staged) against the
        # float32 Path C restatement over the same INT4 codes and zones
        layer = 5
        qq = (torch.randn((1, T_HQ, 1, D), generator=torch.Generator().manual_seed(9)) / math.sqrt(D)).half()
        got = mgr.attend_decode(layer, qq.to(dev)).float().cpu()[0, :, 0]
        codes = {nm: [] for nm in ("k_data", "k_scales", "k_zps", "v_data", "v_scales", "v_zps")}
        for key in mgr._layer_chunks(layer):
            e = mgr.chunk_codes(key)
            for nm in codes:
                codes[nm].append(e[nm].cpu())
        zk, zv = mgr.get_hbm_kv(layer)
        kcat = torch.cat([c[0] for c in codes["k_data"]], dim=1)
        vcat = torch.cat([c[0] for c in codes["v_data"]], dim=1)
        nt = kcat.shape[1]
        ksc = torch.cat([s_.view(T_HKV, -1) for s_ in codes["k_scales"]], 1).reshape(-1)
        kzp = torch.cat([z.view(T_HKV, -1) for z in codes["k_zps"]], 1).reshape(-1)
        vsc = torch.cat([s_.view(T_HKV, -1) for s_ in codes["v_scales"]], 1).reshape(-1)
        vzp = torch.cat([z.view(T_HKV, -1) for z in codes["v_zps"]], 1).reshape(-1)
        ref = tr.attend(qq[0].float(), tr.path_c_keys(kcat, ksc, kzp, [zk[0].cpu()]),
                        tr.path_c_keys(vcat, vsc, vzp, [zv[0].cpu()]))[:, 0]
        parity = {"layer": layer, "int4_tokens": nt, "fp16_tokens": int(zk.shape[2]),
                  "max_abs_err_vs_cpu": round(float((got - ref).abs().max()), 6), "tolerance": 2e-3}
        # windowed retrieval (Path A): the top-w_t chunks, w_t from the adaptive controller
        cache.retrieval_window = "adaptive"
        tok, pos, _, _ = _decode_tokens(torch, model, cache, tok, pos, warm, dev)
        b0 = mgr.prefetch_stats()["bytes_h2d"]
        tok, pos, tm, st = _decode_tokens(torch, model, cache, tok, pos, timed, dev)
        win = _summ(tm, st)
        win["h2d_bytes_per_token"] = (st[-1]["bytes_h2d"] - b0) // max(timed, 1)
        win["window_chunks"] = int(mgr._adaptive_controller.stats["current_w"])
        out["windowed"] = win
        # the same two retrievals with each step replayed from a HIP graph (DecodeGraph: each
        # layer's host runs gathered from the pinned arena by a kernel captured before its
        # decode kernel)
        for name, window in (("windowed_graph", "adaptive"), ("full_graph", None)):
            cache.retrieval_window = window
            runner = DecodeGraph(model, cache)
            tok, pos, _, _ = _decode_tokens_graph(torch, runner, tok, pos, max(warm, 3), dev)
            tok, pos, tm, _ = _decode_tokens_graph(torch, runner, tok, pos, timed, dev)
            out[name] = _summ(tm, [])
            runner.close()
            del runner
        cache.retrieval_window = "adaptive"
        # host -> HBM copy rate of one layer's records on the side stream
        pf, st0 = mgr._pf, mgr._layers[0]
        rb = st0.n_host * mgr._staging[0].record_bytes
        ev0, ev1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        torch.cuda.synchronize()
        ev0.record()
        pf.submit([(mgr._staging[0].data.data_ptr(), pf.host_ptr(st0.host_off), rb)], slot=0)
        pf.wait(0)
        ev1.record()
        ev1.synchronize()
        h2d_gbs = rb / (ev0.elapsed_time(ev1) * 1e-3) / 1e9
        cache.check_errors()
    print("[c5] %s" % json.dumps(out), file=sys.stderr, flush=True)
    weights = sum(p.numel() * p.element_size() for p in model.parameters())
    host_per_tok = full["h2d_bytes_per_token"]
    blk = {"workload": "tiered decode: 28-layer Qwen2-style decoder (hidden 3584, 28 q / 4 kv heads, head_dim 128, "
                       "MLP 18944, vocab 152064, random-init bf16), 131072-token prompt prefilled in 2048-token "
                       "chunks, sink 64 + recent 4096 fp16, INT4 middle with 75% of its 16-token blocks in pinned "
                       "host memory, batch 1, greedy",
           "full_tok_per_s": full["tok_per_s"], "windowed_tok_per_s": win["tok_per_s"],
           "full_graph_tok_per_s": out["full_graph"]["tok_per_s"],
           "windowed_graph_tok_per_s": out["windowed_graph"]["tok_per_s"],
           "full_stall_ms_per_token": full["prefetch_stall_ms_per_token"],
           "windowed_stall_ms_per_token": win["prefetch_stall_ms_per_token"],
           "h2d_gbs_one_layer_copy": round(h2d_gbs, 2), "pcie_gen5_x16_gbs": PCIE_GEN5_X16_GBS,
           "h2d_bytes_per_layer_full": host_per_tok // T_LAYERS,
           "stall_bound": "only windowed retrieval (Path A) is not bound by the prefetch stall; full retrieval "
                          "(Path C) moves every host record over PCIe for every token and is bound by the link",
           "unit": "tok/s", "steps": timed, "warmup": warm,
           "int4_tokens_per_layer": int4_tokens, "host_records_moved": moved, "host_bytes": host_bytes,
           "prefill_seconds": round(prefill_s, 1),
           # the reference's end-to-end figure (results_throughput.csv:42, 2.07 tok/s at 131072 tokens
           # on its hardware) counts the 128K prefill plus 64 decode tokens in its wall time
           "wall_tok_per_s_prefill_plus_64_tokens": {
               k: round(64.0 / (prefill_s + 64 * out[k]["ms_per_token"] * 1e-3), 3)
               for k in ("full", "windowed", "full_graph", "windowed_graph", "resident_graph")},
           "variants": out,
           # full retrieval moves every host record over PCIe per token: its bound is the link,
           # priced at the PCIe Gen5 x16 rate (and at this box's measured one-layer copy rate)
           "roofline": {"bound": "pcie", "achieved": round(host_per_tok / (full["ms_per_token"] * 1e-3) / 1e9, 2),
                        "peak": PCIE_GEN5_X16_GBS, "unit": "GB/s",
                        "frac": round(host_per_tok / (full["ms_per_token"] * 1e-3) / 1e9 / PCIE_GEN5_X16_GBS, 4),
                        "frac_of_measured_copy": round(host_per_tok / (full["ms_per_token"] * 1e-3) / 1e9 / h2d_gbs, 4),
                        "traffic": None, "weights_bytes": weights},
           "parity": parity}
    if not args.no_cpu_baseline:
        blk["cpu_baseline"] = cpu_baseline_c5(torch, model, args.cpu_budget * 2)
    del model, cache
    torch.cuda.empty_cache()
    return blk


# ------------------------------------------------------------------------------ C2 headline
def leg_c2(torch, ops, args):
    """The headline: single-layer decode attention at 32K context (one launch per step),
    replayed from HIP graphs over 8 rotated KV copies (the copies play the layers of a
    decode step: each has its own K/V, all share one block table).  The W warm-up
    launches and the K timed launches are each captured in one graph, so the timed
    region is K launches and one graph launch."""
    dev = torch.device("cuda:0")
    q, K, V = make_inputs(torch)
    R = args.copies
    bt = torch.arange((MID + 15) // 16, dtype=torch.int32, device=dev)[None]
    copies = [build_copy(torch, ops, q, K, V, dev, bt) for _ in range(R)]
    q_dev = q.to(dev)
    out = torch.empty((B, HQ, D), dtype=torch.float16, device=dev)
    ws = ops.DecodeWorkspace(dev)
    err = ops.ErrorWord(dev)

    def launch(i):
        c = copies[i % R]
        ops.decode_attention(q_dev, zones=c["zones"], pool=c["pool"], block_table=c["bt"], int4_max_len=MID,
                             workspace=ws, out=out, deterministic=args.deterministic, err=err)

    for i in range(max(R, 8)):
        launch(i)
    torch.cuda.synchronize()
    stream = torch.cuda.Stream(device=dev)
    K_steps, W = args.steps, args.warmup
    graphs = {}
    if not args.no_graph:
        def capture(n):
            g = torch.cuda.CUDAGraph()
            with torch.cuda.graph(g, stream=stream):
                for i in range(n):
                    launch(i)
            return g
        graphs["timed"] = capture(K_steps)
        if W > 0:
            graphs["warm"] = capture(W)

    def run(n, key):
        if args.no_graph:
            with torch.cuda.stream(stream):
                for i in range(n):
                    launch(i)
        elif n > 0:
            graphs[key].replay()

    with torch.cuda.stream(stream):
        run(W, "warm")
    torch.cuda.synchronize()
    ev0 = torch.cuda.Event(enable_timing=True)
    ev1 = torch.cuda.Event(enable_timing=True)
    if not args.no_graph:
        lead_in(torch, stream)
    with torch.cuda.stream(stream):
        ev0.record(stream)
        run(K_steps, "timed")
        ev1.record(stream)
    ev1.synchronize()
    torch.cuda.synchronize()
    ms_total = ev0.elapsed_time(ev1)
    ms_step = ms_total / K_steps
    gbs = STEP_BYTES * K_steps / (ms_total * 1e-3) / 1e9
    err.check()
    cpu = None
    parity = None
    if not args.no_cpu_baseline:
        ref, cpu = cpu_baseline_c2(torch, q, K, V, args.cpu_budget)
        launch(0)
        torch.cuda.synchronize()
        e = float((out[0].float().cpu() - ref).abs().max())
        if not e <= 2e-3:
            raise RuntimeError("GPU decode output differs from the CPU restatement by %.3e" % e)
        parity = {"max_abs_err_vs_cpu": round(e, 6), "tolerance": 2e-3}
    line = {
        "metric": METRIC, "value": round(gbs, 2), "unit": "GB/s", "n_gpus": 1, "steps": K_steps, "warmup": W,
        "ms_per_step": round(ms_step, 6), "higher_is_better": True, "scaling": "weak", "vs_baseline": None,
        "dtype": "fp16",
        "data": "synthetic (seeded N(0,1) K/V with x8 K outlier channels; INT4 middle packed by the build's "
                "quantizer; random-init model weights and seeded token ids for the 128K leg)",
        "config": {"workload": "single-layer INT4-KV decode attention, batch 1, 32 q / 8 kv heads, head_dim 128, "
                               "ctx 32768 = 64 fp16 sink + 28608 INT4 + 4096 fp16 recent",
                   "batch": B, "context": CTX, "q_heads": HQ, "kv_heads": HKV, "head_dim": D,
                   "int4_tokens": MID, "fp16_tokens": SINK + RECENT, "kv_copies_rotated": R,
                   "launch": "eager" if args.no_graph else "hip graph replay",
                   "schedule": "fixed (deterministic)" if args.deterministic else "on demand",
                   "bytes_per_step": STEP_BYTES},
        "roofline": {"bound": "hbm", "achieved": round(gbs, 2), "peak": HBM_PEAK_GBS, "unit": "GB/s",
                     "frac": round(gbs / HBM_PEAK_GBS, 4), "traffic": read_traffic()},
        "cpu_baseline": ({k: (round(v, 4) if isinstance(v, float) else v) for k, v in cpu.items()} if cpu else None),
        "parity": parity,
    }
    return line


LEGS = ("c1", "c3", "c4", "c5")
LEG_KEYS = {"c1": "c1_quant", "c3": "c3_paged", "c4": "c4_prefill", "c5": "offload_128k"}


def main():
    ap = argparse.ArgumentParser(description=__doc__, formatter_class=argparse.RawDescriptionHelpFormatter)
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=4096, help="timed launches of the 32K decode (the headline)")
    ap.add_argument("--warmup", type=int, default=64)
    ap.add_argument("--copies", type=int, default=8)
    ap.add_argument("--no-graph", action="store_true")
    ap.add_argument("--deterministic", action="store_true",
                    help="decode with the fixed block-to-wave schedule (bitwise reproducible)")
    ap.add_argument("--no-cpu-baseline", action="store_true")
    ap.add_argument("--cpu-budget", type=float, default=10.0, help="seconds of CPU work per baseline")
    ap.add_argument("--legs", default=",".join(LEGS),
                    help="nested configuration blocks of the default line: any of c1 (quantize+pack), c3 (batched "
                         "paged decode), c4 (chunked prefill), c5 (128K tiered decode with 75%% host offload); "
                         "'none' for the 32K decode alone")
    ap.add_argument("--workload",
                    choices=["decode", "prefill", "tiered", "tiered-prefill", "paged", "scoring", "quant", "probe",
                             "timeline"],
                    default=None,
                    help="run one configuration alone and print its block as the line (for profiling): decode "
                         "(32K), prefill (C4), tiered (C5), tiered-prefill (the C5 model's 128K chunked prefill alone), paged "
                         "(C3), quant (C1), scoring (heavy hitters), probe "
                         "(streaming-read probes at the decode's byte count), timeline (the 32K decode kernel's "
                         "phase timeline from the library's timeline build)")
    ap.add_argument("--probe-shapes", default=None,
                    help="probe shapes pattern:workgroups:waves:depth, comma-separated (pattern contig or parts)")
    ap.add_argument("--copy-calibration", type=float, default=0.0,
                    help="run only torch's device copy of this many MB (20 launches) so that rocprofv3 "
                         "FETCH_SIZE / WRITE_SIZE can be scaled against a known byte count")
    args = ap.parse_args()
    if args.gpus != 1 or int(os.environ.get("WORLD_SIZE", "1")) != 1:
        print("bench.py: this benchmark measures one GPU only (the decode path would shard by kv head or "
              "sequence, with no exchange between GPUs); run with --gpus 1", file=sys.stderr)
        sys.exit(2)

    import torch

    dev = torch.device("cuda:0")
    torch.cuda.set_device(dev)
    if args.copy_calibration > 0:
        n = int(args.copy_calibration * 1e6) // 4
        src = torch.ones(n, dtype=torch.int32, device=dev)
        dst = torch.empty_like(src)
        for _ in range(20):
            dst.copy_(src)
        torch.cuda.synchronize()
        print(json.dumps({"copy_calibration_bytes_read_per_launch": n * 4,
                          "copy_calibration_bytes_written_per_launch": n * 4, "launches": 20}), flush=True)
        return

    from heterokv import ops

    single = {"prefill": lambda: leg_c4(torch, ops, args), "paged": lambda: leg_c3(torch, ops, args),
              "quant": lambda: leg_c1(torch, ops, args), "tiered": lambda: leg_c5(torch, args),
              "scoring": lambda: bench_scoring(torch, ops, args), "probe": lambda: bench_probe(torch, args),
              "timeline": lambda: bench_timeline(torch, args),
              "tiered-prefill": lambda: bench_tiered_prefill(torch, args)}
    if args.workload in single:
        blk = single[args.workload]()
        if blk is not None:
            print(json.dumps(blk), flush=True)
        return
    line = leg_c2(torch, ops, args)
    legs = [] if args.legs in ("", "none") else [x.strip() for x in args.legs.split(",")]
    for leg in legs:
        if leg not in LEGS:
            raise SystemExit("bench.py: unknown leg %r (choose from %s)" % (leg, ", ".join(LEGS)))
        print("[bench] leg %s" % leg, file=sys.stderr, flush=True)
        t0 = time.perf_counter()
        if leg == "c1":
            blk = leg_c1(torch, ops, args)
        elif leg == "c3":
            blk = leg_c3(torch, ops, args)
        elif leg == "c4":
            blk = leg_c4(torch, ops, args)
        else:
            blk = leg_c5(torch, args)
        blk["leg_seconds"] = round(time.perf_counter() - t0, 1)
        line[LEG_KEYS[leg]] = blk
        torch.cuda.empty_cache()
    print(json.dumps(line), flush=True)


if __name__ == "__main__":
    main()
