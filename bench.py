"""Benchmark of the paged KV hot path on one MI355X.

Headline (the JSON line's value): paged decode attention at Llama-3-8B GQA
shape, batch 64, log-normal contexts up to 8k, as
algorithmic HBM GB/s. A step is one vapi_paged_attention call over that
batch (the split-K decode kernel plus its partial-merge kernel), with every
input already resident in HBM.

Also measured in the same run (under "extras"): KV append GB/s (config 1),
chunked-prefill TFLOP/s (config 3), copy-on-write GB/s (config 4a), swap
GB/s per direction overlapped with a decode launch (config 4b), and the
device-copy / pinned-copy probes. The CPU baseline is the C oracle
(a restatement of vapi's candle CPU path) timed on this box's host cores.

Usage: python bench.py [--gpus 1] [--steps K] [--warmup W] [--only NAME]
"""
from __future__ import annotations

import argparse
import json
import os
import sys
import time
from pathlib import Path

import numpy as np
import torch

ROOT = Path(__file__).resolve().parent
sys.path.insert(0, str(ROOT))

from vapi_amd import workload  # noqa: E402
from vapi_amd.attention import (ForwardBatch, PreparedAttention, paged_attention_append_prepared,  # noqa: E402
                                paged_attention_prepared)
from vapi_amd.backend import KvBlockBackend  # noqa: E402
from vapi_amd.cache import (PagedKvCache, scatter_index, write_kv_to_cache_layers,  # noqa: E402
                             write_rows_indexed)

HBM_PEAK_GBS = 8000.0
BF16_MFMA_PEAK_TFLOPS = 2500.0
DEV = "cuda"


def log(msg):
    print(msg, file=sys.stderr, flush=True)


def timed(fn, steps, warmup):
    """Run fn warmup times, then time `steps` back-to-back runs between one
    pair of HIP events on the current stream (the stream every kernel here
    launches on), synchronized on both sides. Returns (ms per run, wall ms
    for the timed region)."""
    for _ in range(warmup):
        fn()
    torch.cuda.synchronize()
    start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    t0 = time.perf_counter()
    start.record()
    for _ in range(steps):
        fn()
    end.record()
    torch.cuda.synchronize()
    wall = (time.perf_counter() - t0) * 1e3
    return start.elapsed_time(end) / steps, wall


def timed_graph(fn, steps, warmup, replays=7, detail=None):
    """Capture `steps` back-to-back calls of fn into one HIP graph (the way a
    serving loop replays its captured decode step), replay it untimed until
    at least `warmup` calls have run, then time `replays` replays, each
    between its own pair of events. Returns the median replay's ms per call;
    `detail`, if given, receives every replay's us per call."""
    fn()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        with torch.cuda.graph(graph, stream=side):
            for _ in range(steps):
                fn()
    torch.cuda.current_stream().wait_stream(side)
    for _ in range(max(-(-warmup // steps), 1)):
        graph.replay()
    torch.cuda.synchronize()
    evs = [(torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True))
           for _ in range(replays)]
    for a, b in evs:
        a.record()
        graph.replay()
        b.record()
    torch.cuda.synchronize()
    per = sorted(a.elapsed_time(b) / steps for a, b in evs)
    if detail is not None:
        detail.extend(round(x * 1e3, 2) for x in per)
    return per[len(per) // 2]


# ---- config 2: decode (headline) ---------------------------------------------

# Decode calls rotate over this many layers of one pool (each config 2's
# 32k blocks, filled with their own values), as a forward pass's layers
# follow each other. Replaying one layer's call back to back lets the
# 256 MB last-level cache keep some of the previous call's K/V (the adaptive
# work split moves which wave reads a tile, and when), which no forward
# sees: on one box 137 us per call on one layer against 143 us rotating.
DECODE_LAYERS = 4


def setup_decode():
    w = workload.config2_decode()
    cache = PagedKvCache(DECODE_LAYERS, w.num_blocks, w.block_size, w.num_kv_heads, w.head_dim,
                         torch.bfloat16, "HND")
    workload.fill_normal(cache._slab, workload.seed_for(2))
    g = torch.Generator(device=DEV).manual_seed(workload.seed_for(2) + 1)
    q = torch.randn(w.batch, w.num_heads, w.head_dim, generator=g, device=DEV).to(torch.bfloat16)
    batch = ForwardBatch(cu_seqlens_q=w.cu_q().tolist(), cu_seqlens_k=w.cu_k().tolist(),
                         block_tables=[t.tolist() for t in w.tables], max_seqlen_q=1,
                         max_seqlen_k=int(w.lens.max()))
    prep = PreparedAttention.from_batch(batch, DEV)
    out = torch.empty_like(q)
    scale = w.head_dim ** -0.5
    sum_len = int(w.lens.sum())
    n_blocks = sum(len(t) for t in w.tables)
    kv_bytes = sum_len * 2 * w.num_kv_heads * w.head_dim * 2
    alg_bytes = (kv_bytes + 2 * w.batch * w.num_heads * w.head_dim * 2 + n_blocks * 4
                 + 2 * (w.batch + 1) * 4)

    turn = [0]

    def step():
        paged_attention_prepared(q, cache, turn[0] % DECODE_LAYERS, prep, scale, out=out)
        turn[0] += 1

    def step_same_layer():
        paged_attention_prepared(q, cache, 0, prep, scale, out=out)

    return dict(w=w, cache=cache, q=q, batch=batch, prep=prep, step=step,
                step_same_layer=step_same_layer, scale=scale,
                sum_len=sum_len, alg_bytes=alg_bytes, flops=4.0 * w.num_heads * w.head_dim * sum_len)


def bench_decode(steps, warmup):
    d = setup_decode()
    ms, wall = timed(d["step"], steps, warmup)
    gbs = d["alg_bytes"] / (ms * 1e-3) / 1e9
    log(f"decode cfg2: sum_len {d['sum_len']}, {d['alg_bytes'] / 1e6:.1f} MB/step, "
        f"{ms * 1e3:.1f} us/step, {gbs:.0f} GB/s ({gbs / HBM_PEAK_GBS:.1%} of 8 TB/s)")
    # The same call replayed from a HIP graph, as a serving loop that
    # captures its decode step runs it (GraphRunner, backend.rs:893-1216).
    graph_replays = []
    gms = timed_graph(d["step"], steps, warmup, detail=graph_replays)
    log(f"decode cfg2 in a graph: {gms * 1e3:.1f} us/step (median of {len(graph_replays)} "
        f"replays of {steps} calls: {graph_replays}), "
        f"{d['alg_bytes'] / (gms * 1e-3) / 1e9:.0f} GB/s (layers rotating)")
    same = timed_graph(d["step_same_layer"], steps, warmup)
    log(f"decode cfg2 in a graph, one layer replayed: {same * 1e3:.1f} us/step, "
        f"{d['alg_bytes'] / (same * 1e-3) / 1e9:.0f} GB/s (not reported as the value: the "
        "last-level cache keeps part of the previous call's K/V)")
    # Per-call spread: each of `steps` calls between its own pair of events
    # on the stream the kernels run on (median, 10th and 90th percentile).
    evs = [(torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True))
           for _ in range(steps)]
    for a, b in evs:
        a.record()
        d["step"]()
        b.record()
    torch.cuda.synchronize()
    per = np.array([a.elapsed_time(b) * 1e3 for a, b in evs])
    spread = dict(median_us=float(np.median(per)), p10_us=float(np.percentile(per, 10)),
                  p90_us=float(np.percentile(per, 90)), calls=int(steps),
                  graph_us=gms * 1e3, graph_replays_us=graph_replays,
                  layers_rotated=DECODE_LAYERS,
                  one_layer_replayed_graph_us=same * 1e3,
                  one_layer_replayed_graph_gbs=d["alg_bytes"] / (same * 1e-3) / 1e9)
    log(f"decode cfg2 per call: median {spread['median_us']:.1f} us "
        f"(p10 {spread['p10_us']:.1f}, p90 {spread['p90_us']:.1f})")
    d.update(ms=ms, wall=wall, gbs=gbs, graph_ms=gms, spread=spread,
             graph_gbs=d["alg_bytes"] / (gms * 1e-3) / 1e9)
    return d


def bench_gather(d, steps, warmup):
    """gather_kv (a7) on config 2's pool: the longest context's K and V into
    logical order, one launch."""
    w = d["w"]
    i = int(np.argmax(w.lens))
    lk = int(w.lens[i])
    table = torch.from_numpy(w.tables[i].astype(np.int32)).to(DEV)
    k_out = torch.empty(lk, w.num_kv_heads, w.head_dim, dtype=torch.bfloat16, device=DEV)
    v_out = torch.empty_like(k_out)
    from vapi_amd._lib import check, lib
    from vapi_amd.cache import stream_handle
    cache = d["cache"]
    # The timed calls rotate over the layers and over four tables of the
    # same length cut from one permutation of the pool (the first is the
    # sequence's own): 16 sources of 34 MB, so no call reads what the
    # last-level cache kept from the one before.
    nb = table.shape[0]
    perm = np.random.default_rng(7).permutation(w.num_blocks)
    tables = [table] + [torch.from_numpy(perm[j * nb:(j + 1) * nb].astype(np.int32)).to(DEV)
                        for j in range(3)]
    turn = [0]

    def gather():
        t = tables[(turn[0] // DECODE_LAYERS) % len(tables)]
        layer = turn[0] % DECODE_LAYERS
        turn[0] += 1
        check(lib().vapi_kv_gather(cache.pool, layer, t.data_ptr(), nb, lk,
                                   k_out.data_ptr(), v_out.data_ptr(), stream_handle()))

    ms, _ = timed(gather, max(steps, 32), warmup)
    turn[0] = 0
    gather()
    alg = 2 * 2 * k_out.numel() * k_out.element_size() + table.numel() * 4
    gbs = alg / (ms * 1e-3) / 1e9
    ok = torch.equal(k_out[: w.block_size], cache.reference_view(0, "k")[int(w.tables[i][0])])
    log(f"gather cfg2: {lk} keys x K and V, {alg / 1e6:.1f} MB, {ms * 1e3:.1f} us, {gbs:.0f} GB/s")
    return {"keys": lk, "us": round(ms * 1e3, 2), "gbs": round(gbs, 1), "first_block_exact": bool(ok)}


def bench_fused_step(d, steps, warmup):
    """Config 2's decode step with its 64 new tokens appended: the two calls
    (vapi_kv_append, vapi_paged_attention) against the fused
    vapi_paged_attention_append, back to back on one stream."""
    w = d["w"]
    g = torch.Generator(device=DEV).manual_seed(workload.seed_for(2) + 2)
    k_new = torch.randn(w.batch, w.num_kv_heads, w.head_dim, generator=g,
                        device=DEV).to(torch.bfloat16)
    v_new = torch.randn_like(k_new)
    slots = np.array([int(t[(l - 1) // w.block_size]) * w.block_size + (l - 1) % w.block_size
                      for t, l in zip(w.tables, w.lens)], dtype=np.uint32)
    dslots = torch.from_numpy(slots.view(np.int32)).to(DEV)
    cache, q, prep, scale, out = d["cache"], d["q"], d["prep"], d["scale"], torch.empty_like(d["q"])

    turn = [0]

    def two():
        layer = turn[0] % DECODE_LAYERS
        turn[0] += 1
        write_rows_indexed(cache, layer, k_new, v_new, dslots)
        paged_attention_prepared(q, cache, layer, prep, scale, out=out)

    def fused():
        layer = turn[0] % DECODE_LAYERS
        turn[0] += 1
        paged_attention_append_prepared(q, k_new, v_new, dslots, cache, layer, prep, scale,
                                        out=out)

    ms_two, _ = timed(two, steps, warmup)
    ms_fused, _ = timed(fused, steps, warmup)
    # The same two sequences replayed from HIP graphs (no host launch cost).
    g_two = timed_graph(two, steps, warmup)
    g_fused = timed_graph(fused, steps, warmup)
    log(f"decode cfg2 + append of {w.batch} tokens: two calls {ms_two * 1e3:.1f} us, "
        f"fused {ms_fused * 1e3:.1f} us; in graphs {g_two * 1e3:.1f} / {g_fused * 1e3:.1f} us")
    return {"two_calls_us": round(ms_two * 1e3, 2), "fused_us": round(ms_fused * 1e3, 2),
            "two_calls_graph_us": round(g_two * 1e3, 2), "fused_graph_us": round(g_fused * 1e3, 2)}


# ---- f32 pools, other head dims ---------------------------------

def bench_mixed_step(d, steps, warmup):
    """A chunked-prefill serving step on config 2's pool: its first 63
    sequences as decode rows plus one 512-token chunk at positions
    1536..2047, in one call, replayed from a graph: through the prepared
    call that names the step's prefill sequences (what PreparedAttention
    issues) and through vapi_paged_attention_ex without the list (the prefill
    grid then spans every sequence, and the chunk is not split)."""
    from vapi_amd import _lib
    from vapi_amd.cache import stream_handle
    w, cache = d["w"], d["cache"]
    nd = 63
    lens_q = [1] * nd + [512]
    lens_k = [int(x) for x in w.lens[:nd]] + [2048]
    tables = [list(t) for t in w.tables[:nd]]
    # The chunk's 128 blocks: pool blocks no decode row reads.
    used = set(int(x) for t in tables for x in t)
    tables.append([x for x in range(w.num_blocks) if x not in used][:128])
    batch = ForwardBatch(cu_seqlens_q=np.concatenate([[0], np.cumsum(lens_q)]).tolist(),
                         cu_seqlens_k=np.concatenate([[0], np.cumsum(lens_k)]).tolist(),
                         block_tables=tables, max_seqlen_q=512, max_seqlen_k=max(lens_k))
    prep = PreparedAttention.from_batch(batch, DEV)
    q = torch.randn(sum(lens_q), w.num_heads, w.head_dim, device=DEV).to(torch.bfloat16)
    o = torch.empty_like(q)
    scale = w.head_dim ** -0.5
    listed_ms = timed_graph(lambda: paged_attention_prepared(q, cache, 0, prep, scale, out=o),
                            steps, warmup)
    L = _lib.lib()
    b = nd + 1
    need = L.vapi_paged_attention_workspace_size(cache.pool, b, w.num_heads, 512, prep.max_seqlen_k)
    ws = torch.zeros(need, dtype=torch.uint8, device=DEV)

    def unlisted():
        _lib.check(L.vapi_paged_attention_ex(
            cache.pool, 0, q.data_ptr(), o.data_ptr(), prep.seqlens_q.data_ptr(),
            prep.seqlens_k.data_ptr(), prep.block_table.data_ptr(), b, prep.block_table.shape[1],
            512, prep.max_seqlen_k, w.num_heads, scale, -1, 0, 0, ws.data_ptr(), need,
            stream_handle()))

    unlisted_ms = timed_graph(unlisted, steps, warmup)
    res = dict(decode_rows=nd, prefill_chunk=512, prefill_context=2048,
               us=listed_ms * 1e3, us_without_prefill_list=unlisted_ms * 1e3)
    log(f"mixed step (63 decode rows + one 512-token chunk): {res['us']:.1f} us per call, "
        f"{res['us_without_prefill_list']:.1f} us without the prefill list")
    return res


def bench_valu(steps, warmup):
    """f32 pools: config 0 (Qwen3-0.6B-shaped f32 decode, the reference's CPU
    parity case: at most 512 keys, so the short-context kernel), config
    2's batch over an f32 pool (1.5 GB of K/V, the f32-MFMA decode stream),
    the same batch at head_dim 80 (the stream padded to 128), and config 3
    on an f32 pool (the bf16-split prefill) at head_dim 128 and 80."""
    out = {}
    for name, w, heads, kvh, d in (("cfg0_f32", workload.config0_decode_small(), 16, 8, None),
                                   ("cfg2_shape_f32", workload.config2_decode(), 32, 8, None),
                                   ("cfg2_shape_f32_d80", workload.config2_decode(), 32, 8, 80)):
        d = d or w.head_dim
        cache = PagedKvCache(1, w.num_blocks, w.block_size, kvh, d, torch.float32, "HND")
        workload.fill_normal(cache._slab, workload.seed_for(0))
        q = torch.randn(w.batch, heads, d, device=DEV)
        batch = ForwardBatch(cu_seqlens_q=w.cu_q().tolist(), cu_seqlens_k=w.cu_k().tolist(),
                             block_tables=[t.tolist() for t in w.tables], max_seqlen_q=1,
                             max_seqlen_k=int(w.lens.max()))
        prep = PreparedAttention.from_batch(batch, DEV)
        o = torch.empty_like(q)
        call = lambda: paged_attention_prepared(q, cache, 0, prep, d ** -0.5, out=o)  # noqa: E731
        ms, _ = timed(call, max(steps // 2, 5), 3)
        gms = timed_graph(call, max(steps // 2, 5), 3)
        kv = int(w.lens.sum()) * 2 * kvh * d * 4
        out[name] = dict(us=ms * 1e3, graph_us=gms * 1e3, kv_bytes=kv,
                         gbs=kv / (ms * 1e-3) / 1e9, graph_gbs=kv / (gms * 1e-3) / 1e9,
                         path=("short-context decode" if name == "cfg0_f32"
                               else "f32 MFMA decode stream (head_dim 80: padded to 128)"
                               if name.endswith("d80") else "f32 MFMA decode stream"))
        log(f"f32 attention {name}: {ms * 1e3:.1f} us ({gms * 1e3:.1f} us in a graph), "
            f"{kv / 1e6:.1f} MB of K/V, {out[name]['gbs']:.0f} GB/s, {out[name]['path']}")
        del cache
    # Config 3 (32 x 512-token chunks over 4,096 keys) on an f32 pool, at
    # head_dim 128 and 80 (the prefill padded to 128; FLOPs at 80).
    p = workload.config3_prefill()
    for name, d in (("cfg3_f32", 128), ("cfg3_f32_d80", 80)):
        cache = PagedKvCache(1, p.num_blocks, p.block_size, 8, d, torch.float32, "HND")
        workload.fill_normal(cache._slab, workload.seed_for(3))
        q = torch.randn(p.batch * p.len_q, 32, d, device=DEV)
        batch = ForwardBatch(cu_seqlens_q=p.cu_q().tolist(), cu_seqlens_k=p.cu_k().tolist(),
                             block_tables=[t.tolist() for t in p.tables], max_seqlen_q=p.len_q,
                             max_seqlen_k=p.len_k)
        prep = PreparedAttention.from_batch(batch, DEV)
        o = torch.empty_like(q)
        ms, _ = timed(lambda: paged_attention_prepared(q, cache, 0, prep, d ** -0.5, out=o), 3, 2)
        flops = p.flops() * d / 128
        out[name] = dict(ms=ms, flops=flops, tflops=flops / (ms * 1e-3) / 1e12)
        log(f"f32 attention {name}: {ms:.2f} ms, {out[name]['tflops']:.1f} TFLOP/s")
        del cache, q, o
    return out


def bench_small_batches(steps, warmup):
    """Decode latency at small batches (config 2's heads and pool, equal
    contexts): where the call's fixed costs (the first loads, the merge)
    weigh most. Per call, replayed from a HIP graph over rotating tables."""
    cache = PagedKvCache(1, 32768, 16, 8, 128, torch.bfloat16, "HND")
    workload.fill_normal(cache._slab, workload.seed_for(2))
    rng = np.random.default_rng(workload.seed_for(2))
    out = {}
    for b, lk in ((1, 8192), (1, 32768), (4, 4096), (16, 2048)):
        nb = (lk + 15) // 16
        perm = rng.permutation(32768)
        # Consecutive calls read disjoint blocks (up to 16 tables cut from one
        # permutation of the pool), so no call finds the previous one's K/V
        # in the last-level cache: at least 512 MB between reuses.
        n_tab = min(16, 32768 // (b * nb))
        preps = []
        for j in range(n_tab):
            part = perm[j * b * nb:(j + 1) * b * nb]
            batch = ForwardBatch(cu_seqlens_q=list(range(b + 1)),
                                 cu_seqlens_k=[i * lk for i in range(b + 1)],
                                 block_tables=[part[i * nb:(i + 1) * nb].tolist() for i in range(b)],
                                 max_seqlen_q=1, max_seqlen_k=lk)
            preps.append(PreparedAttention.from_batch(batch, DEV))
        q = torch.randn(b, 32, 128, device=DEV).to(torch.bfloat16)
        o = torch.empty_like(q)
        turn = [0]

        def call():
            prep = preps[turn[0] % n_tab]
            turn[0] += 1
            paged_attention_prepared(q, cache, 0, prep, 128 ** -0.5, out=o)

        gms = timed_graph(call, max(steps, 2 * n_tab), warmup)
        kv = b * lk * 8 * 128 * 2 * 2
        out[f"b{b}_k{lk}"] = dict(us=gms * 1e3, gbs=kv / (gms * 1e-3) / 1e9)
    log("decode small batches: " + ", ".join(f"{k} {v['us']:.1f} us" for k, v in out.items()))
    del cache
    return out


def bench_small_prefill(steps, warmup):
    """Prefill latency at small batches (config 3's heads, one causal chunk
    at the end of each context): fewer query tiles than CUs, so the kernel
    splits each tile's keys over several workgroups. Per call, replayed
    from a HIP graph."""
    cache = PagedKvCache(1, 32768, 16, 8, 128, torch.bfloat16, "HND")
    workload.fill_normal(cache._slab, workload.seed_for(3))
    rng = np.random.default_rng(workload.seed_for(3))
    out = {}
    for b, lq, lk in ((1, 512, 4096), (1, 128, 8192), (2, 512, 4096), (4, 512, 4096)):
        nb = (lk + 15) // 16
        perm = rng.permutation(32768)
        batch = ForwardBatch(cu_seqlens_q=[i * lq for i in range(b + 1)],
                             cu_seqlens_k=[i * lk for i in range(b + 1)],
                             block_tables=[perm[i * nb:(i + 1) * nb].tolist() for i in range(b)],
                             max_seqlen_q=lq, max_seqlen_k=lk)
        prep = PreparedAttention.from_batch(batch, DEV)
        q = torch.randn(b * lq, 32, 128, device=DEV).to(torch.bfloat16)
        o = torch.empty_like(q)
        gms = timed_graph(lambda: paged_attention_prepared(q, cache, 0, prep, 128 ** -0.5, out=o),
                          steps, warmup)
        # causal chunk at the end of the context: query i sees lk - lq + i + 1 keys
        flops = 4 * 32 * 128 * b * sum(lk - lq + i + 1 for i in range(lq))
        out[f"b{b}_q{lq}_k{lk}"] = dict(us=gms * 1e3, tflops=flops / (gms * 1e-3) / 1e12)
    log("prefill small batches: " + ", ".join(f"{k} {v['us']:.1f} us ({v['tflops']:.0f} TFLOP/s)"
                                              for k, v in out.items()))
    del cache
    return out


def bench_head_dim_64(steps, warmup):
    """Configs 2 and 3 with head_dim 64 (LFM2's attention layers: 32 q / 8 kv
    heads of 64), on the same MFMA kernels' head_dim-64 builds."""
    w = workload.config2_decode()
    cache = PagedKvCache(DECODE_LAYERS, w.num_blocks, w.block_size, 8, 64, torch.bfloat16,
                         "HND")
    workload.fill_normal(cache._slab, workload.seed_for(2))
    q = torch.randn(w.batch, 32, 64, device=DEV).to(torch.bfloat16)
    batch = ForwardBatch(cu_seqlens_q=w.cu_q().tolist(), cu_seqlens_k=w.cu_k().tolist(),
                         block_tables=[t.tolist() for t in w.tables], max_seqlen_q=1,
                         max_seqlen_k=int(w.lens.max()))
    prep = PreparedAttention.from_batch(batch, DEV)
    out = torch.empty_like(q)
    turn = [0]

    def call():
        paged_attention_prepared(q, cache, turn[0] % DECODE_LAYERS, prep, 0.125, out=out)
        turn[0] += 1

    gms = timed_graph(call, steps, warmup)
    kv = int(w.lens.sum()) * 2 * 8 * 64 * 2
    res = {"decode_cfg2_d64": dict(us=gms * 1e3, kv_bytes=kv, gbs=kv / (gms * 1e-3) / 1e9)}
    del cache, q, out
    p = workload.config3_prefill()
    cache = PagedKvCache(1, p.num_blocks, p.block_size, 8, 64, torch.bfloat16, "HND")
    workload.fill_normal(cache._slab, workload.seed_for(3))
    q = torch.randn(p.batch * p.len_q, 32, 64, device=DEV).to(torch.bfloat16)
    batch = ForwardBatch(cu_seqlens_q=p.cu_q().tolist(), cu_seqlens_k=p.cu_k().tolist(),
                         block_tables=[t.tolist() for t in p.tables], max_seqlen_q=p.len_q,
                         max_seqlen_k=p.len_k)
    prep = PreparedAttention.from_batch(batch, DEV)
    out = torch.empty_like(q)
    ms, _ = timed(lambda: paged_attention_prepared(q, cache, 0, prep, 0.125, out=out),
                  max(steps, 10), 30)
    flops = p.flops() / 2  # head_dim 64
    res["prefill_cfg3_d64"] = dict(ms=ms, flops=flops, tflops=flops / (ms * 1e-3) / 1e12)
    log("head_dim 64: decode cfg2 {:.1f} us ({:.0f} GB/s), prefill cfg3 {:.3f} ms ({:.0f} "
        "TFLOP/s)".format(res["decode_cfg2_d64"]["us"], res["decode_cfg2_d64"]["gbs"], ms,
                          res["prefill_cfg3_d64"]["tflops"]))
    del cache, q, out
    return res


def bench_decode_other_head_dims(steps, warmup):
    """Configs 2 and 3 (32 q / 8 kv heads, bf16) at head_dim 80 and 96
    (Phi-2's and Phi-3's): the decode stream and the prefill kernel at
    D = 128 with zeros past the head dim. Bytes and FLOPs are counted at the
    real head dim (what the padded columns cost shows as a lower rate)."""
    w = workload.config2_decode()
    p = workload.config3_prefill()
    out = {}
    for d in (80, 96):
        cache = PagedKvCache(2, w.num_blocks, w.block_size, 8, d, torch.bfloat16, "HND")
        workload.fill_normal(cache._slab, workload.seed_for(2))
        q = torch.randn(w.batch, 32, d, device=DEV).to(torch.bfloat16)
        o = torch.empty_like(q)
        batch = ForwardBatch(cu_seqlens_q=w.cu_q().tolist(), cu_seqlens_k=w.cu_k().tolist(),
                             block_tables=[t.tolist() for t in w.tables], max_seqlen_q=1,
                             max_seqlen_k=int(w.lens.max()))
        prep = PreparedAttention.from_batch(batch, DEV)
        turn = [0]

        def call():
            paged_attention_prepared(q, cache, turn[0] % 2, prep, d ** -0.5, out=o)
            turn[0] += 1

        us = timed_graph(call, steps, warmup) * 1e3
        kv = int(w.lens.sum()) * 8 * d * 2 * 2
        del cache, q, o
        cache = PagedKvCache(1, p.num_blocks, p.block_size, 8, d, torch.bfloat16, "HND")
        workload.fill_normal(cache._slab, workload.seed_for(3))
        q = torch.randn(p.batch * p.len_q, 32, d, device=DEV).to(torch.bfloat16)
        o = torch.empty_like(q)
        batch = ForwardBatch(cu_seqlens_q=p.cu_q().tolist(), cu_seqlens_k=p.cu_k().tolist(),
                             block_tables=[t.tolist() for t in p.tables], max_seqlen_q=p.len_q,
                             max_seqlen_k=p.len_k)
        prep = PreparedAttention.from_batch(batch, DEV)
        ms, _ = timed(lambda: paged_attention_prepared(q, cache, 0, prep, d ** -0.5, out=o),
                      max(steps, 10), 30)
        flops = p.flops() * d / 128
        out[f"d{d}"] = dict(us=us, gbs=kv / (us * 1e-6) / 1e9, kv_bytes=kv,
                            prefill_ms=ms, prefill_tflops=flops / (ms * 1e-3) / 1e12)
        log(f"head_dim {d}: decode cfg2 {us:.1f} us ({kv / (us * 1e-6) / 1e9:.0f} GB/s), "
            f"prefill cfg3 {ms:.3f} ms ({flops / (ms * 1e-3) / 1e12:.0f} TFLOP/s at d{d})")
        del cache, q, o
    torch.cuda.empty_cache()
    return out


def bench_decode_block_major(steps, warmup):
    """Config 2's decode over a block-major pool of 4 layers (block stride
    8 blocks: each 4 KiB (block, head) tile of a layer sits apart from the
    next block's by every layer's K and V), rotating layers as the headline."""
    w = workload.config2_decode()
    cache = PagedKvCache(DECODE_LAYERS, w.num_blocks, w.block_size, w.num_kv_heads, w.head_dim,
                         torch.bfloat16, "HND", block_major=True)
    workload.fill_normal(cache._slab, workload.seed_for(2))
    q = torch.randn(w.batch, w.num_heads, w.head_dim, device=DEV).to(torch.bfloat16)
    batch = ForwardBatch(cu_seqlens_q=w.cu_q().tolist(), cu_seqlens_k=w.cu_k().tolist(),
                         block_tables=[t.tolist() for t in w.tables], max_seqlen_q=1,
                         max_seqlen_k=int(w.lens.max()))
    prep = PreparedAttention.from_batch(batch, DEV)
    out = torch.empty_like(q)
    turn = [0]

    def call():
        paged_attention_prepared(q, cache, turn[0] % DECODE_LAYERS, prep, 128 ** -0.5, out=out)
        turn[0] += 1

    gms = timed_graph(call, steps, warmup)
    kv = int(w.lens.sum()) * 2 * 8 * 128 * 2
    log(f"decode cfg2 over a block-major pool: {gms * 1e3:.1f} us, "
        f"{kv / (gms * 1e-3) / 1e9:.0f} GB/s of K/V")
    del cache, q, out
    torch.cuda.empty_cache()
    return dict(us=gms * 1e3, gbs=kv / (gms * 1e-3) / 1e9)


def bench_decode_block_size_32(steps, warmup):
    """Config 2's batch (the same contexts and heads) over a pool of 32-key
    blocks, the reference's own block size (vapi_core::config::BLOCK_SIZE),
    16,384 blocks in random order, rotating over 4 layers as the headline."""
    w = workload.config2_decode()
    bs, nb = 32, 16384
    rng = np.random.default_rng(workload.seed_for(2))
    perm = rng.permutation(nb)
    tables, at = [], 0
    for l in w.lens:
        n = (int(l) + bs - 1) // bs
        tables.append(perm[at:at + n].tolist())
        at += n
    cache = PagedKvCache(DECODE_LAYERS, nb, bs, w.num_kv_heads, w.head_dim, torch.bfloat16, "HND")
    workload.fill_normal(cache._slab, workload.seed_for(2))
    q = torch.randn(w.batch, w.num_heads, w.head_dim, device=DEV).to(torch.bfloat16)
    batch = ForwardBatch(cu_seqlens_q=w.cu_q().tolist(), cu_seqlens_k=w.cu_k().tolist(),
                         block_tables=tables, max_seqlen_q=1, max_seqlen_k=int(w.lens.max()))
    prep = PreparedAttention.from_batch(batch, DEV)
    out = torch.empty_like(q)
    turn = [0]

    def call():
        paged_attention_prepared(q, cache, turn[0] % DECODE_LAYERS, prep, 128 ** -0.5, out=out)
        turn[0] += 1

    gms = timed_graph(call, steps, warmup)
    kv = int(w.lens.sum()) * 2 * 8 * 128 * 2
    log(f"decode cfg2 over 32-key blocks: {gms * 1e3:.1f} us, "
        f"{kv / (gms * 1e-3) / 1e9:.0f} GB/s of K/V")
    del cache, q, out
    torch.cuda.empty_cache()
    return dict(us=gms * 1e3, gbs=kv / (gms * 1e-3) / 1e9)


def bench_wide_group(steps, warmup):
    """Config 2's batch with more than 16 query heads per kv head on bf16
    pools: 64 q over 2 kv heads (G = 32: two virtual kv heads of 16 per
    group), 48 q over 1 (G = 48: three of 16) and 71 q over 1 (Falcon-7B's
    G = 71: four of 15 and one of 11). Each virtual kv head reads its
    group's K/V, so K/V are read ceil(G / 16) times; GB/s count them once."""
    w = workload.config2_decode()
    res = {}
    for hq, kvh in ((64, 2), (48, 1), (71, 1)):
        G = hq // kvh
        parts = (G + 15) // 16
        cache = PagedKvCache(DECODE_LAYERS, w.num_blocks, w.block_size, kvh, 128, torch.bfloat16,
                             "HND")
        workload.fill_normal(cache._slab, workload.seed_for(2))
        q = torch.randn(w.batch, hq, 128, device=DEV).to(torch.bfloat16)
        batch = ForwardBatch(cu_seqlens_q=w.cu_q().tolist(), cu_seqlens_k=w.cu_k().tolist(),
                             block_tables=[t.tolist() for t in w.tables], max_seqlen_q=1,
                             max_seqlen_k=int(w.lens.max()))
        prep = PreparedAttention.from_batch(batch, DEV)
        out = torch.empty_like(q)
        turn = [0]

        def call():
            paged_attention_prepared(q, cache, turn[0] % DECODE_LAYERS, prep, 128 ** -0.5,
                                     out=out)
            turn[0] += 1

        gms = timed_graph(call, steps, warmup)
        kv = int(w.lens.sum()) * kvh * 2 * 128 * 2
        log(f"decode cfg2 batch, {hq} q / {kvh} kv heads (G = {G}, {parts} parts): "
            f"{gms * 1e3:.1f} us, {kv / (gms * 1e-3) / 1e9:.0f} GB/s of unique K/V "
            f"({parts * kv / (gms * 1e-3) / 1e9:.0f} GB/s read)")
        res[f"g{G}"] = dict(us=gms * 1e3, kv_bytes=kv, parts=parts,
                            gbs_unique_kv=kv / (gms * 1e-3) / 1e9,
                            gbs_read=parts * kv / (gms * 1e-3) / 1e9)
        del cache, q, out
    torch.cuda.empty_cache()
    return res


def bench_head_dim_256(steps, warmup):
    """Configs 2 and 3 with head_dim 256 (32 q / 8 kv heads of 256) on bf16
    pools: the decode stream at twice config 2's K/V bytes per key, and the
    prefill (one 16-row tile per wave) at twice config 3's FLOPs."""
    w = workload.config2_decode()
    layers = 2
    cache = PagedKvCache(layers, w.num_blocks, w.block_size, 8, 256, torch.bfloat16, "HND")
    workload.fill_normal(cache._slab, workload.seed_for(2))
    q = torch.randn(w.batch, 32, 256, device=DEV).to(torch.bfloat16)
    batch = ForwardBatch(cu_seqlens_q=w.cu_q().tolist(), cu_seqlens_k=w.cu_k().tolist(),
                         block_tables=[t.tolist() for t in w.tables], max_seqlen_q=1,
                         max_seqlen_k=int(w.lens.max()))
    prep = PreparedAttention.from_batch(batch, DEV)
    out = torch.empty_like(q)
    turn = [0]

    def call():
        paged_attention_prepared(q, cache, turn[0] % layers, prep, 256 ** -0.5, out=out)
        turn[0] += 1

    gms = timed_graph(call, steps, warmup)
    kv = int(w.lens.sum()) * 8 * 256 * 2 * 2
    res = {"decode_cfg2_d256": dict(us=gms * 1e3, kv_bytes=kv, gbs=kv / (gms * 1e-3) / 1e9,
                                    frac_of_8tbs=kv / (gms * 1e-3) / 8e12)}
    del cache, q, out
    p = workload.config3_prefill()
    cache = PagedKvCache(1, p.num_blocks, p.block_size, 8, 256, torch.bfloat16, "HND")
    workload.fill_normal(cache._slab, workload.seed_for(3))
    q = torch.randn(p.batch * p.len_q, 32, 256, device=DEV).to(torch.bfloat16)
    batch = ForwardBatch(cu_seqlens_q=p.cu_q().tolist(), cu_seqlens_k=p.cu_k().tolist(),
                         block_tables=[t.tolist() for t in p.tables], max_seqlen_q=p.len_q,
                         max_seqlen_k=p.len_k)
    prep = PreparedAttention.from_batch(batch, DEV)
    out = torch.empty_like(q)
    ms, _ = timed(lambda: paged_attention_prepared(q, cache, 0, prep, 256 ** -0.5, out=out),
                  max(steps, 10), 30)
    flops = p.flops() * 2  # head_dim 256
    res["prefill_cfg3_d256"] = dict(ms=ms, flops=flops, tflops=flops / (ms * 1e-3) / 1e12)
    log("head_dim 256: decode cfg2 {:.1f} us ({:.0f} GB/s), prefill cfg3 {:.3f} ms ({:.0f} "
        "TFLOP/s)".format(res["decode_cfg2_d256"]["us"], res["decode_cfg2_d256"]["gbs"], ms,
                          res["prefill_cfg3_d256"]["tflops"]))
    del cache, q, out
    return res


# ---- config 1: append --------------------------------------------------------------

def bench_append(steps, warmup):
    w = workload.config1_append()
    cache = PagedKvCache(1, w.num_blocks, w.block_size, w.num_kv_heads, w.head_dim,
                         torch.bfloat16, "HND")
    g = torch.Generator(device=DEV).manual_seed(workload.seed_for(1))
    k = torch.randn(w.n_tokens, 8, 128, generator=g, device=DEV).to(torch.bfloat16)
    v = torch.randn(w.n_tokens, 8, 128, generator=g, device=DEV).to(torch.bfloat16)
    idx = scatter_index(w.slots, DEV)

    def append():
        write_rows_indexed(cache, 0, k, v, idx)

    # Host-launched calls: one Python + ctypes call per append through the
    # Python mirror (its argument checks included), and the bare C ABI call
    # with every pointer prepared (what a compiled caller pays per call).
    ms_host, _ = timed(append, steps, warmup)
    from vapi_amd._lib import check as _check, lib as _L
    from vapi_amd.cache import stream_handle as _sh
    fn, pool, sh = _L().vapi_kv_append_ex, cache.pool, _sh()
    kp, vp, ip = k.data_ptr(), v.data_ptr(), idx.data_ptr()

    def append_c():
        fn(pool, 0, kp, vp, ip, w.n_tokens, 0, sh)

    ms_host_c, _ = timed(append_c, max(steps, 50), warmup)
    _check(fn(pool, 0, kp, vp, ip, w.n_tokens, 0, sh))
    # The same appends captured in one HIP graph and replayed, as a serving
    # step would issue its per-layer appends: per-append device time.
    ms = timed_graph(append, steps, warmup)
    alg = w.n_valid * 2 * 8 * 128 * 2 * 2 + w.n_tokens * 4
    gbs = alg / (ms * 1e-3) / 1e9
    log(f"append cfg1: {alg / 1e6:.1f} MB, {ms * 1e3:.2f} us/append in a graph "
        f"({gbs:.0f} GB/s), {ms_host * 1e3:.1f} us/append host-launched")
    # Cold sources: the graph's appends rotate over 24 source sets (384 MB,
    # more than the 256 MB last-level cache), as a fresh layer's K/V rows
    # would arrive, so the reads come from HBM; with VAPI_APPEND_COLD_SOURCE
    # (streaming loads) and without.
    n_sets = 24
    ks = torch.randn(n_sets, w.n_tokens, 8, 128, generator=g, device=DEV).to(torch.bfloat16)
    vs = torch.randn_like(ks)
    it = [0]

    def append_cold(flag):
        i = it[0] % n_sets
        it[0] += 1
        write_rows_indexed(cache, 0, ks[i], vs[i], idx, cold_source=flag)

    ms_cold = timed_graph(lambda: append_cold(True), max(steps, n_sets), warmup)
    ms_cold_plain = timed_graph(lambda: append_cold(False), max(steps, n_sets), warmup)
    gbs_cold = alg / (ms_cold * 1e-3) / 1e9
    log(f"append cfg1, sources rotated over {n_sets} sets: {ms_cold * 1e3:.2f} us/append "
        f"({gbs_cold:.0f} GB/s) with the cold-source flag, {ms_cold_plain * 1e3:.2f} us without; "
        f"host-launched {ms_host_c * 1e3:.2f} us/append through the bare C ABI")
    del ks, vs
    # Ceiling for the cold leg: a trivial sequential copy of the same byte
    # count (the valid rows' K and V), its source rotated over 24 buffers the
    # same way, in ordinary and streaming form.
    from vapi_amd.cache import stream_handle
    plib = probe_lib()
    half = w.n_valid * 2 * 8 * 128 * 2
    half -= half % 16
    srcs = torch.empty(n_sets, half, dtype=torch.uint8, device=DEV)
    dst = torch.empty(half, dtype=torch.uint8, device=DEV)
    cold_probe = {}
    for nt, sfx in ((0, ""), (1, "_nt")):
        def probe_cold(nt=nt):
            i = it[0] % n_sets
            it[0] += 1
            _chk_probe(plib.vapi_probe_copy(dst.data_ptr(), srcs[i].data_ptr(), half, nt,
                                         stream_handle()))
        pms = timed_graph(probe_cold, max(steps, n_sets), warmup)
        cold_probe["copy_seq_cold" + sfx + "_us"] = pms * 1e3
        cold_probe["copy_seq_cold" + sfx + "_gbs"] = 2 * half / (pms * 1e-3) / 1e9
    log("append cold-source ceiling: sequential copy of the same bytes " +
        ", ".join(f"{k} {v:.1f}" for k, v in cold_probe.items()))
    del srcs, dst
    del cache
    # The same step's rows for 4 layers in one launch (vapi_kv_append_layers).
    L = 4
    cache = PagedKvCache(L, w.num_blocks, w.block_size, w.num_kv_heads, w.head_dim,
                         torch.bfloat16, "HND")
    kl = torch.randn(L, w.n_tokens, 8, 128, generator=g, device=DEV).to(torch.bfloat16)
    vl = torch.randn_like(kl)
    ms_l, _ = timed(lambda: write_kv_to_cache_layers(cache, 0, kl, vl, idx), steps, warmup)
    gbs_l = L * alg / (ms_l * 1e-3) / 1e9
    log(f"append cfg1 x {L} layers in one launch: {ms_l * 1e3:.2f} us "
        f"({ms_l * 1e3 / L:.2f} us/layer, {gbs_l:.0f} GB/s)")
    del cache, kl, vl
    return dict(us=ms * 1e3, gbs=gbs, frac=gbs / HBM_PEAK_GBS, bytes=alg,
                cold_us=ms_cold * 1e3, cold_gbs=gbs_cold, cold_frac=gbs_cold / HBM_PEAK_GBS,
                cold_frac_of_cold_copy_probe=gbs_cold / max(cold_probe["copy_seq_cold_gbs"],
                                                            cold_probe["copy_seq_cold_nt_gbs"]),
                cold_flag="VAPI_APPEND_COLD_SOURCE (streaming source loads)",
                cold_us_without_flag=ms_cold_plain * 1e3,
                cold_gbs_without_flag=alg / (ms_cold_plain * 1e-3) / 1e9,
                cold_probe=cold_probe,
                us_host_launched=ms_host * 1e3,
                gbs_host_launched=alg / (ms_host * 1e-3) / 1e9,
                us_host_launched_c_abi=ms_host_c * 1e3,
                gbs_host_launched_c_abi=alg / (ms_host_c * 1e-3) / 1e9,
                layers4_one_launch_us=ms_l * 1e3, layers4_gbs=gbs_l)


# ---- config 3: chunked prefill ----------------------------------------------------

def bench_prefill(steps, warmup):
    w = workload.config3_prefill()
    cache = PagedKvCache(1, w.num_blocks, w.block_size, 8, 128, torch.bfloat16, "HND")
    workload.fill_normal(cache._slab, workload.seed_for(3))
    g = torch.Generator(device=DEV).manual_seed(workload.seed_for(3) + 1)
    q = torch.randn(w.batch * w.len_q, 32, 128, generator=g, device=DEV).to(torch.bfloat16)
    batch = ForwardBatch(cu_seqlens_q=w.cu_q().tolist(), cu_seqlens_k=w.cu_k().tolist(),
                         block_tables=[t.tolist() for t in w.tables], max_seqlen_q=w.len_q,
                         max_seqlen_k=w.len_k)
    prep = PreparedAttention.from_batch(batch, DEV)
    out = torch.empty_like(q)
    ms, _ = timed(lambda: paged_attention_prepared(q, cache, 0, prep, 128 ** -0.5, out=out),
                     steps, warmup)
    tf = w.flops() / (ms * 1e-3) / 1e12
    log(f"prefill cfg3: {w.flops() / 1e12:.3f} TFLOP, {ms:.2f} ms, {tf:.1f} TFLOP/s "
        f"({tf / BF16_MFMA_PEAK_TFLOPS:.1%} of 2.5 PF)")
    del cache, q, out
    gemm = mfma_probe()
    log(f"bf16 GEMM probe (hipBLASLt, 8192^3): {gemm:.0f} TFLOP/s; prefill at "
        f"{tf / gemm:.1%} of it")
    return dict(ms=ms, tflops=tf, frac=tf / BF16_MFMA_PEAK_TFLOPS, flops=w.flops(),
                gemm_probe_tflops=gemm, frac_of_gemm_probe=tf / gemm)


def mfma_probe():
    """Dense bf16 GEMM (torch.matmul -> hipBLASLt), 8192 x 8192 x 8192: what
    a library GEMM reaches of the MFMA peak on this box."""
    n = 8192
    a = torch.randn(n, n, device=DEV).to(torch.bfloat16)
    b = torch.randn(n, n, device=DEV).to(torch.bfloat16)
    c = torch.empty(n, n, device=DEV, dtype=torch.bfloat16)
    ms, _ = timed(lambda: torch.matmul(a, b, out=c), 20, 20)
    return 2.0 * n ** 3 / (ms * 1e-3) / 1e12


# ---- config 4: copy-on-write and swap ---------------------------------------------

def bench_blocks(steps, warmup, decode):
    w = workload.config4_block_ops()
    cache = PagedKvCache(w.num_layers, w.num_blocks, w.block_size, w.num_kv_heads,
                         w.head_dim, torch.bfloat16, "HND")
    workload.fill_normal(cache._slab, workload.seed_for(4))
    be = KvBlockBackend(cache)
    bb = be.block_bytes()
    pairs_dev = torch.from_numpy(w.pairs.astype(np.int32).reshape(-1)).to(DEV)
    from vapi_amd._lib import check, lib
    from vapi_amd.cache import stream_handle

    def copy():
        check(lib().vapi_kv_copy_blocks(cache.pool, pairs_dev.data_ptr(), w.pairs.shape[0],
                                        stream_handle()))

    ms, _ = timed(copy, steps, warmup)
    alg = w.pairs.shape[0] * bb * 2
    copy_gbs = alg / (ms * 1e-3) / 1e9
    log(f"copy cfg4a: {alg / 1e9:.2f} GB moved, {ms:.3f} ms, {copy_gbs:.0f} GB/s")
    # Bit-exactness at full size: every pair's destination equals its source.
    src = torch.from_numpy(w.pairs[:, 0].astype(np.int64)).to(DEV)
    dst = torch.from_numpy(w.pairs[:, 1].astype(np.int64)).to(DEV)
    copy_ok = all(torch.equal(t[src], t[dst]) for t in cache.k + cache.v)
    copy_probes = probes_copy(w, cache)
    bm = bench_copy_block_major(w, pairs_dev, steps, warmup)

    # Swap: 4,096 blocks out to pinned host and back into other blocks.
    n = len(w.swap_ids)
    host = torch.empty(n * bb, dtype=torch.uint8, pin_memory=True)
    staging = torch.empty(256 * bb, dtype=torch.uint8, device=DEV)
    ids_out = torch.from_numpy(w.swap_ids.astype(np.int32)).to(DEV)
    ids_in = torch.from_numpy(w.swap_in_ids.astype(np.int32)).to(DEV)
    side = torch.cuda.Stream()

    def on_side(fn):
        ev0, ev1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        ev0.record(side)
        fn()
        ev1.record(side)
        side.synchronize()
        return ev0.elapsed_time(ev1)

    torch.cuda.synchronize()
    # Three round trips, the median of each direction (a single transfer's
    # rate moves with the host's load).
    outs, ins = [], []
    for _ in range(3):
        outs.append(on_side(lambda: be.swap_out(ids_out, host, staging, stream=side)))
        ins.append(on_side(lambda: be.swap_in(ids_in, host, staging, stream=side)))
    out_ms, in_ms = sorted(outs)[1], sorted(ins)[1]
    swap_ok = True
    for a, b in ((0, 0), (n // 2, n // 2), (n - 1, n - 1)):
        swap_ok &= be.export_block(int(w.swap_ids[a])) == be.export_block(int(w.swap_in_ids[b]))
    # Overlap: swap-out on the side stream while decode steps run on the main stream.
    dec_alone, _ = timed(decode["step"], 10, 2)
    torch.cuda.synchronize()
    ev0, ev1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    ev0.record(side)
    be.swap_out(ids_out, host, staging, stream=side)
    ev1.record(side)
    dec_ms = []
    while not ev1.query():
        e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        e0.record()
        decode["step"]()
        e1.record()
        e1.synchronize()
        dec_ms.append(e0.elapsed_time(e1))
        if len(dec_ms) > 5000:
            break
    side.synchronize()
    overlap_out_ms = ev0.elapsed_time(ev1)
    # Pinned-copy probe (host-link peak).
    probe = torch.empty(1 << 30, dtype=torch.uint8, device=DEV)
    ph = torch.empty(1 << 30, dtype=torch.uint8, pin_memory=True)
    torch.cuda.synchronize()
    d2h = on_side(lambda: _copy_on(side, ph, probe))
    h2d = on_side(lambda: _copy_on(side, probe, ph))
    link = dict(d2h_gbs=(1 << 30) / (d2h * 1e-3) / 1e9, h2d_gbs=(1 << 30) / (h2d * 1e-3) / 1e9)
    gb = n * bb / 1e9
    # Spill tier: 512 evicted blocks into a host-memory store through a
    # 64-block pinned buffer, then promoted into other blocks (batched
    # spill_evicted / promote_from_spill), wall clock.
    from vapi_amd.spill import SpillStore, pinned_buffer, promote, spill_evicted
    ns = 512
    hs = [int(i).to_bytes(32, "little") for i in range(ns)]
    store = SpillStore(None, ns * bb, 0)
    pin = pinned_buffer(cache, 64)
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    exported = spill_evicted(store, cache, zip(hs, w.swap_ids[:ns].tolist()), pin)
    t1 = time.perf_counter()
    restored = promote(store, cache, hs, w.swap_in_ids[:ns].tolist(), pin)
    t2 = time.perf_counter()
    spill_ok = exported == ns and restored == ns and all(
        be.export_block(int(w.swap_ids[i])) == be.export_block(int(w.swap_in_ids[i]))
        for i in (0, ns // 2, ns - 1))
    spill = dict(blocks=ns, export_us_per_block=(t1 - t0) * 1e6 / ns,
                 import_us_per_block=(t2 - t1) * 1e6 / ns,
                 export_gbs=ns * bb / (t1 - t0) / 1e9, import_gbs=ns * bb / (t2 - t1) / 1e9,
                 round_trip_bit_exact=bool(spill_ok))
    log(f"spill tier: {ns} blocks out {spill['export_us_per_block']:.0f} us/block "
        f"({spill['export_gbs']:.1f} GB/s), back {spill['import_us_per_block']:.0f} us/block "
        f"({spill['import_gbs']:.1f} GB/s)")
    store.close()
    # A full store (host memory for 128 blocks, no disk): every put evicts,
    # and the evicted buffers take the next blobs, as in a long-running
    # server whose spill tier has filled.
    store = SpillStore(None, 128 * bb, 0)
    spill_evicted(store, cache, zip(hs[:128], w.swap_ids[:128].tolist()), pin)
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    spill_evicted(store, cache, zip(hs[128:ns], w.swap_ids[128:ns].tolist()), pin)
    t1 = time.perf_counter()
    spill.update(full_store_export_us_per_block=(t1 - t0) * 1e6 / (ns - 128),
                 full_store_export_gbs=(ns - 128) * bb / (t1 - t0) / 1e9)
    log(f"spill tier, full store: {ns - 128} blocks out "
        f"{spill['full_store_export_us_per_block']:.0f} us/block "
        f"({spill['full_store_export_gbs']:.1f} GB/s)")
    store.close()
    # The same spill overlapped with the forward: the pack into device
    # staging is all the model's stream waits for; the copy to host runs on
    # a side stream and the drain puts the blobs into the store. The event
    # span on the model stream also covers the call's host work (the stream
    # is otherwise idle here); the pack kernel alone is shorter.
    from vapi_amd.spill import drain, spill_evicted_async
    store = SpillStore(None, ns * bb, 0)
    pin_all = pinned_buffer(cache, ns)
    staging = torch.empty(ns * bb, dtype=torch.uint8, device=DEV)
    ev0, ev1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    # The model's stream is a stream of its own, as a serving loop's is: on
    # the legacy default stream the span measured 8.6 ms, the default
    # stream waiting for the side stream's copy.
    model = torch.cuda.Stream()
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    with torch.cuda.stream(model):
        ev0.record()
        exported = spill_evicted_async(store, cache, zip(hs, w.swap_ids[:ns].tolist()), staging,
                                       pin_all, side=side)
        ev1.record()
    t1 = time.perf_counter()
    drained = drain(store)
    t2 = time.perf_counter()
    async_ok = exported == drained == ns and all(
        store.get(hs[i], bb) == be.export_block(int(w.swap_ids[i])) for i in (0, ns - 1))
    spill.update(async_call_us=(t1 - t0) * 1e6, async_stream_us=ev0.elapsed_time(ev1) * 1e3,
                 async_drain_ms=(t2 - t1) * 1e3, async_bit_exact=bool(async_ok))
    log(f"spill tier async: {ns} blocks, model stream {spill['async_stream_us']:.0f} us, "
        f"call returns in {spill['async_call_us']:.0f} us, drain {spill['async_drain_ms']:.1f} ms")
    store.close()
    del pin, pin_all, staging
    res = dict(copy_ms=ms, copy_gbs=copy_gbs, copy_frac=copy_gbs / HBM_PEAK_GBS,
               # Against the better of each probe's two forms.
               copy_frac_of_runs_probe=copy_gbs / max(copy_probes["copy_runs16k_gbs"],
                                                      copy_probes["copy_runs16k_nt_gbs"]),
               copy_frac_of_seq_copy_probe=copy_gbs / max(copy_probes["copy_seq_gbs"],
                                                          copy_probes["copy_seq_nt_gbs"]),
               probes=copy_probes, copy_bit_exact=bool(copy_ok),
               copy_block_major=bm,
               swap_out_gbs=gb / (out_ms * 1e-3), swap_in_gbs=gb / (in_ms * 1e-3),
               swap_round_trip_bit_exact=bool(swap_ok),
               swap_out_overlapped_gbs=gb / (overlap_out_ms * 1e-3),
               decode_us_alone=dec_alone * 1e3,
               decode_us_during_swap=float(np.median(dec_ms)) * 1e3 if dec_ms else None,
               pinned_probe=link, swap_bytes_per_direction=n * bb, spill_tier=spill)
    log(f"swap cfg4b: out {res['swap_out_gbs']:.1f} GB/s, in {res['swap_in_gbs']:.1f} GB/s, "
        f"pinned probe d2h {link['d2h_gbs']:.1f} h2d {link['h2d_gbs']:.1f}; decode "
        f"{res['decode_us_alone']:.0f} us alone, {res['decode_us_during_swap']} us during swap")
    del cache, host, ph, probe
    return res


def bench_copy(steps, warmup):
    """Copy-on-write alone (config 4a), for profiling."""
    w = workload.config4_block_ops()
    cache = PagedKvCache(w.num_layers, w.num_blocks, w.block_size, w.num_kv_heads,
                         w.head_dim, torch.bfloat16, "HND")
    workload.fill_normal(cache._slab, workload.seed_for(4))
    be = KvBlockBackend(cache)
    pairs_dev = torch.from_numpy(w.pairs.astype(np.int32).reshape(-1)).to(DEV)
    from vapi_amd._lib import check, lib
    from vapi_amd.cache import stream_handle
    n = w.pairs.shape[0]
    ms, _ = timed(lambda: check(lib().vapi_kv_copy_blocks(cache.pool, pairs_dev.data_ptr(), n,
                                                          stream_handle())), steps, warmup)
    alg = n * be.block_bytes() * 2
    log(f"copy cfg4a: {alg / 1e9:.2f} GB moved, {ms:.3f} ms, {alg / (ms * 1e-3) / 1e9:.0f} GB/s")


def bench_copy_block_major(w, pairs_dev, steps, warmup):
    """Config 4a's pairs on a block-major pool (block_major=True: per block,
    every layer's K and V side by side), where a pair is one 917,504-byte
    run: the same vapi_kv_copy_blocks call."""
    from vapi_amd._lib import check, lib
    from vapi_amd.cache import stream_handle
    cache = PagedKvCache(w.num_layers, w.num_blocks, w.block_size, w.num_kv_heads,
                         w.head_dim, torch.bfloat16, "HND", block_major=True)
    workload.fill_normal(cache._slab, workload.seed_for(4))
    n = w.pairs.shape[0]
    ms, _ = timed(lambda: check(lib().vapi_kv_copy_blocks(cache.pool, pairs_dev.data_ptr(), n,
                                                          stream_handle())), steps, warmup)
    alg = n * KvBlockBackend(cache).block_bytes() * 2
    gbs = alg / (ms * 1e-3) / 1e9
    src = torch.from_numpy(w.pairs[:, 0].astype(np.int64)).to(DEV)
    dst = torch.from_numpy(w.pairs[:, 1].astype(np.int64)).to(DEV)
    ok = all(torch.equal(t[src], t[dst]) for t in cache.k + cache.v)
    log(f"copy cfg4a, block-major pool: {alg / 1e9:.2f} GB moved, {ms:.3f} ms, {gbs:.0f} GB/s"
        f" ({gbs / HBM_PEAK_GBS:.1%} of 8 TB/s), bit-exact {ok}")
    del cache
    torch.cuda.empty_cache()
    return dict(ms=ms, gbs=gbs, frac=gbs / HBM_PEAK_GBS, bit_exact=ok)


def _copy_on(stream, dst, src):
    with torch.cuda.stream(stream):
        dst.copy_(src, non_blocking=True)


# ---- HBM ceiling probes (libvapi_probe.so) ---------------------------------------

_PROBE = None


def probe_lib():
    """The benchmark's probe kernels (vapi_amd/csrc/probes.hip), built by
    vapi_amd.build next to libvapi_kv.so."""
    global _PROBE
    if _PROBE is None:
        import ctypes
        path = ROOT / "vapi_amd" / "libvapi_probe.so"
        if not path.exists():
            raise ImportError(f"{path} is missing: build with `python -m vapi_amd.build`")
        L = ctypes.CDLL(str(path))
        vp, u32, u64 = ctypes.c_void_p, ctypes.c_uint32, ctypes.c_uint64
        # The u32 before the stream: 0 ordinary loads/stores, 1 streaming.
        L.vapi_probe_read.argtypes = [vp, u64, vp, u32, vp]
        L.vapi_probe_read_tiles.argtypes = [vp, vp, u32, u32, vp, u32, vp]
        L.vapi_probe_copy.argtypes = [vp, vp, u64, u32, vp]
        L.vapi_probe_copy_runs.argtypes = [vp, vp, u32, u32, u32, vp]
        _PROBE = L
    return _PROBE


def _probe_time(fn, reps=20, warmup=3):
    ms, _ = timed(lambda: _chk_probe(fn()), reps, warmup)
    return ms


def _chk_probe(rc):
    if rc != 0:
        raise RuntimeError(f"probe launch failed ({rc})")


def decode_tiles(d):
    """The 4 KiB K and V tiles config 2's decode reads, as tile indices of
    its pool slab, in the decode's order (sequence, kv head, block, K/V)."""
    w, cache = d["w"], d["cache"]
    tile = w.block_size * w.head_dim * 2
    k0 = cache.pool.k
    v_off = (cache.pool.v - k0) // tile
    ids = []
    for t, l in zip(w.tables, w.lens):
        blocks = np.asarray(t[: -(-int(l) // w.block_size)], dtype=np.int64)
        for h in range(w.num_kv_heads):
            kt = blocks * w.num_kv_heads + h
            ids.append(np.stack([kt, kt + v_off], 1).reshape(-1))
    return np.concatenate(ids).astype(np.uint32), k0, tile


def probes_decode(dec):
    """Ceilings for the decode, measured on this box on its access pattern
    (same bytes, same granularity; GB/s of bytes read), each with ordinary
    loads and with streaming (non-temporal) loads (`_nt`), the kind the
    decode issues for K/V:
      read_seq:     a sequential read of the decode's K/V byte count;
      read_tiles4k: the decode's own 4 KiB K/V tiles of config 2's pool, in
                    its order (the decode kernel's reads without its math);
      read_runs8k:  the same bytes as random 8 KiB runs of the pool."""
    from vapi_amd.cache import stream_handle
    L, sh = probe_lib(), stream_handle()
    sink = torch.zeros(1024, dtype=torch.int32, device=DEV)
    out = {}
    ids, base, tile = decode_tiles(dec)
    nbytes = int(ids.size) * tile
    buf = torch.empty(nbytes, dtype=torch.uint8, device=DEV)
    dids = torch.from_numpy(ids.view(np.int32)).to(DEV)
    slab_bytes = dec["cache"]._slab.numel() * 2
    n8 = nbytes // 8192
    r8 = np.random.default_rng(8).permutation(slab_bytes // 8192)[:n8].astype(np.uint32)
    d8 = torch.from_numpy(r8.view(np.int32)).to(DEV)
    for nt, sfx in ((0, ""), (1, "_nt")):
        ms = _probe_time(lambda: L.vapi_probe_read(buf.data_ptr(), nbytes, sink.data_ptr(), nt, sh))
        out["read_seq" + sfx + "_gbs"] = nbytes / (ms * 1e-3) / 1e9
        ms = _probe_time(lambda: L.vapi_probe_read_tiles(base, dids.data_ptr(), ids.size, 4096,
                                                          sink.data_ptr(), nt, sh))
        out["read_tiles4k" + sfx + "_gbs"] = nbytes / (ms * 1e-3) / 1e9
        ms = _probe_time(lambda: L.vapi_probe_read_tiles(base, d8.data_ptr(), n8, 8192,
                                                          sink.data_ptr(), nt, sh))
        out["read_runs8k" + sfx + "_gbs"] = n8 * 8192 / (ms * 1e-3) / 1e9
    del buf
    out["decode_kv_bytes"] = nbytes
    log("probes (decode): " + ", ".join(f"{k} {v:.0f}" for k, v in out.items()
                                        if k.endswith("gbs")))
    return out


def probes_copy(w, cache):
    """Ceilings for the block copy (GB/s of bytes read + written):
      copy_runs16k: config 4a's own (src, dst) 16 KiB runs over its pool,
                    every layer, K and V (the block copy's pattern);
      copy_seq:     a sequential device copy of the same byte count;
    each with ordinary and with streaming (`_nt`) loads and stores, the
    kind the block copy issues."""
    from vapi_amd.cache import stream_handle
    L, sh = probe_lib(), stream_handle()
    out = {}
    run = w.block_size * w.num_kv_heads * w.head_dim * 2
    kbase = cache.pool.k
    lstride = cache.pool.layer_stride_bytes // run
    voff = (cache.pool.v - kbase) // run
    pr = []
    for l in range(w.num_layers):
        for off in (0, voff):
            pr.append(np.stack([w.pairs[:, 0].astype(np.int64) + l * lstride + off,
                                w.pairs[:, 1].astype(np.int64) + l * lstride + off], 1))
    pr = np.concatenate(pr).astype(np.uint32)
    dpr = torch.from_numpy(pr.reshape(-1).view(np.int32)).to(DEV)
    cbytes = pr.shape[0] * run
    a = torch.empty(cbytes, dtype=torch.uint8, device=DEV)
    b = torch.empty_like(a)
    for nt, sfx in ((0, ""), (1, "_nt")):
        ms = _probe_time(lambda: L.vapi_probe_copy_runs(kbase, dpr.data_ptr(), pr.shape[0], run,
                                                        nt, sh), reps=10)
        out["copy_runs16k" + sfx + "_gbs"] = 2 * cbytes / (ms * 1e-3) / 1e9
        ms = _probe_time(lambda: L.vapi_probe_copy(b.data_ptr(), a.data_ptr(), cbytes, nt, sh),
                         reps=10)
        out["copy_seq" + sfx + "_gbs"] = 2 * cbytes / (ms * 1e-3) / 1e9
        # The same pairs as whole-block runs (917,504 B: every layer's K and V
        # of a block adjacent, a block-major layout), over the pool's slab.
        blob = run * 2 * w.num_layers
        assert cache._slab.numel() * cache._slab.element_size() >= w.num_blocks * blob
        bpr = torch.from_numpy(w.pairs.astype(np.uint32).reshape(-1).view(np.int32)).to(DEV)
        ms = _probe_time(lambda: L.vapi_probe_copy_runs(cache._slab.data_ptr(), bpr.data_ptr(),
                                                        w.pairs.shape[0], blob, nt, sh), reps=10)
        out["copy_runs_block" + sfx + "_gbs"] = 2 * w.pairs.shape[0] * blob / (ms * 1e-3) / 1e9
    out["copy_bytes_each_way"] = cbytes
    del a, b
    log("probes (copy): " + ", ".join(f"{k} {v:.0f}" for k, v in out.items()
                                      if k.endswith("gbs")))
    return out


# ---- CPU baseline ------------------------------------------------------------------

def cpu_baseline(decode, budget_s=8.0):
    """The candle CPU path on the same config-2 batch, in two restatements,
    each repeated until ~budget_s: the C oracle (OpenMP over sequences,
    scalar f32 loops) and oracle/candle_np.py (candle's own steps: gather,
    cast, repeat_kv, BLAS matmuls, host-built mask, softmax). The faster is
    the reported baseline; both are in the line."""
    import oracle  # checker/baseline only
    from oracle import candle_np  # baseline only
    w = decode["w"]
    cache = decode["cache"]
    # Host copy of just the blocks the batch uses, renumbered densely.
    used = np.concatenate(w.tables).astype(np.int64)
    remap = {int(b): i for i, b in enumerate(used)}
    idx = torch.from_numpy(used).to(DEV)
    kd = cache.reference_view(0, "k")[idx]
    vd = cache.reference_view(0, "v")[idx]
    kc, vc = kd.float().cpu().numpy(), vd.float().cpu().numpy()
    kbits = kd.contiguous().view(torch.int16).cpu().numpy().view(np.uint16)
    vbits = vd.contiguous().view(torch.int16).cpu().numpy().view(np.uint16)
    tables = [[remap[int(b)] for b in t] for t in w.tables]
    q = decode["q"].float().cpu().numpy()
    qbits = decode["q"].contiguous().view(torch.int16).cpu().numpy().view(np.uint16)
    # Every core this process may run on (the box's share of the host).
    threads = len(os.sched_getaffinity(0))
    cu_q, cu_k = w.cu_q(), w.cu_k()

    def rate(fn):
        reps, t0 = 0, time.perf_counter()
        while True:
            fn()
            reps += 1
            if time.perf_counter() - t0 > budget_s or reps >= 50:
                break
        return (time.perf_counter() - t0) / reps, reps

    legs = {}
    sec, reps = rate(lambda: oracle.paged_attention(q, kc, vc, cu_q, cu_k, tables,
                                                    decode["scale"], threads=threads))
    legs["c_oracle"] = dict(
        value=decode["alg_bytes"] / sec / 1e9, ms_per_step=sec * 1e3, reps=reps,
        sample=f"full config-2 decode batch (64 seqs, sum_len {w.lens.sum()}), {reps} passes, "
               f"C oracle with OpenMP over sequences, f32 math on bf16-valued K/V")
    sec, reps = rate(lambda: candle_np.paged_attention(qbits, kbits, vbits, cu_q, cu_k, tables,
                                                       decode["scale"]))
    legs["candle_numpy"] = dict(
        value=decode["alg_bytes"] / sec / 1e9, ms_per_step=sec * 1e3, reps=reps,
        sample=f"full config-2 decode batch (64 seqs, sum_len {w.lens.sum()}), {reps} passes, "
               f"candle's steps in numpy (gather, f32 cast, repeat_kv, BLAS matmuls, mask, "
               f"softmax) on bf16 K/V, BLAS threads as the process allows")
    for k, v in legs.items():
        log(f"cpu baseline ({k}): {v['ms_per_step']:.1f} ms per config-2 step, "
            f"{v['value']:.2f} GB/s")
    best = max(legs, key=lambda k: legs[k]["value"])
    b = legs[best]
    return dict(value=b["value"], unit="GB/s", cores=threads, nproc=os.cpu_count(), kind="port",
                sample=b["sample"], ms_per_step=b["ms_per_step"], legs=legs)


def cpu_baselines_more(decode, budget_s=4.0):
    """The other CPU legs of the benchmark's configs, each on a bounded sample
    with the C oracle, on one core and on every core this process may use: config-2
    decode on one core (the all-core figure is `cpu_baseline`), the config-1
    append scatter (write_rows), the config-3 chunked prefill (the last 64
    query rows of each sequence's chunk) and the config-4a block copy
    (copy_blocks). The multi-core append and copy split the rows or pairs over
    threads (config 1's slots and config 4's pairs never collide)."""
    import oracle  # checker/baseline only
    threads = len(os.sched_getaffinity(0))
    out = {}

    def rate(fn, min_reps, budget):
        fn()  # untimed: first touch of the pages
        reps, t0 = 0, time.perf_counter()
        while reps < min_reps or time.perf_counter() - t0 < budget:
            fn()
            reps += 1
        return (time.perf_counter() - t0) / reps, reps

    # Decode on one core: the same batch as the headline leg.
    w = decode["w"]
    cache = decode["cache"]
    used = np.concatenate(w.tables).astype(np.int64)
    remap = {int(b): i for i, b in enumerate(used)}
    idx = torch.from_numpy(used).to(DEV)
    kc = cache.reference_view(0, "k")[idx].float().cpu().numpy()
    vc = cache.reference_view(0, "v")[idx].float().cpu().numpy()
    tables = [[remap[int(b)] for b in t] for t in w.tables]
    q = decode["q"].float().cpu().numpy()
    reps, t0 = 0, time.perf_counter()
    while reps < 1 or time.perf_counter() - t0 < budget_s:
        oracle.paged_attention(q, kc, vc, w.cu_q(), w.cu_k(), tables, decode["scale"], threads=1)
        reps += 1
    sec = (time.perf_counter() - t0) / reps
    out["decode_cfg2_1core"] = dict(gbs=decode["alg_bytes"] / sec / 1e9, ms=sec * 1e3, reps=reps)
    del kc, vc
    # Append scatter (config 1) into a host pool of the config's size (K only;
    # V is the same work again, counted in the bytes).
    a = workload.config1_append()
    row = a.num_kv_heads * a.head_dim * 2
    pool = np.zeros((a.num_blocks * a.block_size, row), dtype=np.uint8)
    src = np.random.default_rng(1).integers(0, 255, size=(a.n_tokens, row), dtype=np.uint8)
    alg = a.n_valid * 2 * row * 2 + a.n_tokens * 4
    for tag, th in (("1core", 1), ("allcores", threads)):
        sec, reps = rate(lambda: oracle.write_rows(pool, src, a.slots, threads=th), 3, budget_s / 4)
        out[f"append_cfg1_{tag}"] = dict(gbs=alg / (2 * sec) / 1e9, us=2 * sec * 1e6, reps=reps,
                                         threads=th)
    del pool
    # Chunked prefill (config 3): the last 64 query rows of each sequence's
    # 512-row chunk (positions 4032..4095 over 4,096 keys, bottom-right
    # causal as in the full chunk); one sequence on one core, one sequence
    # per thread on every core.
    p = workload.config3_prefill()
    rng = np.random.default_rng(3)
    kp = rng.standard_normal((p.num_blocks, p.block_size, p.num_kv_heads, p.head_dim),
                             dtype=np.float32)
    vp = rng.standard_normal(kp.shape, dtype=np.float32)
    lq = 64
    for tag, nseq, th in (("1core", 1, 1), ("allcores", min(threads, p.batch), threads)):
        qs = rng.standard_normal((nseq * lq, p.num_heads, p.head_dim), dtype=np.float32)
        cu_q = np.arange(nseq + 1, dtype=np.uint32) * lq
        cu_k = np.arange(nseq + 1, dtype=np.uint32) * p.len_k
        tabs = [t.tolist() for t in p.tables[:nseq]]
        flops = 4.0 * p.head_dim * p.num_heads * nseq * sum(
            pos + 1 for pos in range(p.len_k - lq, p.len_k))
        sec, reps = rate(lambda: oracle.paged_attention(qs, kp, vp, cu_q, cu_k, tabs,
                                                        p.head_dim ** -0.5, threads=th),
                         1, budget_s / 2)
        out[f"prefill_cfg3_{tag}"] = dict(tflops=flops / sec / 1e12, ms=sec * 1e3, reps=reps,
                                          threads=th, sample=f"{nseq} seq x {lq} query rows")
    del kp, vp
    # Block copy (config 4a) over per-layer pools holding just the pairs'
    # blocks, renumbered densely.
    c = workload.config4_block_ops()
    blocks = np.unique(c.pairs.reshape(-1))
    ren = {int(b): i for i, b in enumerate(blocks)}
    pairs = np.array([[ren[int(x)], ren[int(y)]] for x, y in c.pairs], dtype=np.uint32)
    blk = c.block_size * c.num_kv_heads * c.head_dim * 2
    ks = [np.zeros((len(blocks), blk), dtype=np.uint8) for _ in range(c.num_layers)]
    vs = [np.zeros((len(blocks), blk), dtype=np.uint8) for _ in range(c.num_layers)]
    alg = len(pairs) * 2 * c.num_layers * blk * 2
    for tag, th in (("1core", 1), ("allcores", threads)):
        sec, reps = rate(lambda: oracle.copy_blocks(ks, vs, pairs, threads=th), 1, budget_s / 2)
        out[f"copy_cfg4a_{tag}"] = dict(gbs=alg / sec / 1e9, ms=sec * 1e3, reps=reps, threads=th)
    del ks, vs
    out["threads_allcores"] = threads
    out["nproc"] = os.cpu_count()
    log("cpu baselines: decode 1 core {:.2f} GB/s; append {:.1f}/{:.1f} GB/s; prefill "
        "{:.4f}/{:.4f} TFLOP/s; copy {:.1f}/{:.1f} GB/s (1 core / {} threads)".format(
            out["decode_cfg2_1core"]["gbs"], out["append_cfg1_1core"]["gbs"],
            out["append_cfg1_allcores"]["gbs"], out["prefill_cfg3_1core"]["tflops"],
            out["prefill_cfg3_allcores"]["tflops"], out["copy_cfg4a_1core"]["gbs"],
            out["copy_cfg4a_allcores"]["gbs"], threads))
    return out


def load_traffic():
    p = ROOT / "profiles" / "paged_decode_config2_traffic.json"
    if p.exists():
        try:
            return json.loads(p.read_text())
        except Exception:
            return None
    return None


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=50)
    ap.add_argument("--warmup", type=int, default=10)
    ap.add_argument("--only", choices=["decode", "append", "prefill", "copy", "blocks", "valu",
                                       "mixed", "shapes", "small", "copy_bm", "gather"],
                    default=None)
    ap.add_argument("--no-cpu", action="store_true")
    ap.add_argument("--calibrate", action="store_true",
                    help="first run one plain 256 MiB device copy, whose FETCH_SIZE/WRITE_SIZE "
                         "counters scale the hot kernels' counters to bytes")
    args = ap.parse_args()
    if args.gpus != 1 or int(os.environ.get("WORLD_SIZE", "1")) > 1:
        print("bench.py measures one GPU only: this build's paged-KV path runs on a single "
              "MI355X (across GPUs it would shard by kv head or by sequence, with no exchange); "
              "run with --gpus 1.",
              file=sys.stderr)
        sys.exit(2)
    torch.cuda.init()
    if args.calibrate:
        # A plain conversion kernel of known traffic: reads 256 MiB of f32,
        # writes 128 MiB of f16 (the only f32->f16 copy in the run).
        src = torch.ones(64 << 20, dtype=torch.float32, device=DEV)
        dst = src.to(torch.float16)
        torch.cuda.synchronize()
        del src, dst
    if args.only == "append":
        bench_append(args.steps, args.warmup)
        return
    if args.only == "copy":
        bench_copy(args.steps, args.warmup)
        return
    if args.only == "gather":
        bench_gather(setup_decode(), args.steps, args.warmup)
        return
    if args.only == "copy_bm":
        w = workload.config4_block_ops()
        pairs_dev = torch.from_numpy(w.pairs.astype(np.int32).reshape(-1)).to(DEV)
        bench_copy_block_major(w, pairs_dev, args.steps, args.warmup)
        return
    if args.only == "prefill":
        bench_prefill(args.steps, args.warmup)
        return
    if args.only == "valu":
        bench_valu(args.steps, args.warmup)
        return
    if args.only == "small":
        bench_small_batches(args.steps, args.warmup)
        bench_small_prefill(args.steps, args.warmup)
        return
    if args.only == "shapes":
        bench_head_dim_64(args.steps, args.warmup)
        bench_wide_group(args.steps, args.warmup)
        bench_head_dim_256(args.steps, args.warmup)
        bench_decode_block_major(args.steps, args.warmup)
        bench_decode_block_size_32(args.steps, args.warmup)
        bench_decode_other_head_dims(args.steps, args.warmup)
        return
    if args.only == "mixed":
        bench_mixed_step(setup_decode(), args.steps, args.warmup)
        return
    dec = bench_decode(args.steps, args.warmup)
    if args.only == "decode":
        return
    extras = {"decode_cfg2_calls": dict(dec["spread"], host_launched_us=dec["ms"] * 1e3,
                                        host_launched_gbs=dec["gbs"])}
    extras["gather_cfg2"] = bench_gather(dec, args.steps, args.warmup)
    extras["fused_step_cfg2"] = bench_fused_step(dec, args.steps, args.warmup)
    extras["mixed_step_cfg2"] = bench_mixed_step(dec, args.steps, args.warmup)
    # Block copy, swap and spill run before the other extras: run after
    # them in one process, the swap's host-to-device rate fell to ~31 GB/s
    # (55.6 alone or first; some full runs still read ~31), while a 1 GiB
    # pinned probe allocated after the swap's 3.76 GB source read at 57
    # GB/s; the cause was not found.
    extras["blocks_cfg4"] = bench_blocks(max(args.steps // 5, 3), 2, dec)
    if args.only in (None,):
        extras["append_cfg1"] = bench_append(args.steps, args.warmup)
        # Prefill runs 1.2 ms per call; its rate climbs over the first ~25
        # calls (849 -> 959 -> 983 TFLOP/s over three runs of 13 calls on one
        # box), so it warms up for 30 calls, as a serving loop's steady state.
        extras["prefill_cfg3"] = bench_prefill(max(args.steps, 10), 30)
        extras["f32_attention"] = bench_valu(args.steps, args.warmup)
        extras["head_dim_64"] = bench_head_dim_64(args.steps, args.warmup)
        extras["wide_groups"] = bench_wide_group(args.steps, args.warmup)
        extras["head_dim_256"] = bench_head_dim_256(args.steps, args.warmup)
        extras["decode_cfg2_block_major"] = bench_decode_block_major(args.steps, args.warmup)
        extras["decode_cfg2_block_size_32"] = bench_decode_block_size_32(args.steps, args.warmup)
        extras["other_head_dims"] = bench_decode_other_head_dims(args.steps, args.warmup)
        extras["decode_small_batches"] = bench_small_batches(args.steps, args.warmup)
        extras["prefill_small_batches"] = bench_small_prefill(args.steps, args.warmup)
    # The gather is a copy of scattered 4 KiB K/V tiles into a contiguous
    # output: its fractions of 8 TB/s and of the random-16 KiB-run copy
    # probe (the nearest measured pattern).
    g, pr = extras["gather_cfg2"], extras["blocks_cfg4"]["probes"]
    g["frac"] = g["gbs"] / HBM_PEAK_GBS
    g["frac_of_runs_copy_probe"] = g["gbs"] / max(pr["copy_runs16k_gbs"], pr["copy_runs16k_nt_gbs"])
    if args.only == "blocks":
        return
    pd = probes_decode(dec)
    extras["probes_decode"] = dict(
        pd,
        decode_call_frac_of_tiles4k=dec["graph_gbs"] / max(pd["read_tiles4k_gbs"],
                                                           pd["read_tiles4k_nt_gbs"]),
        decode_call_frac_of_read_seq=dec["graph_gbs"] / max(pd["read_seq_gbs"],
                                                            pd["read_seq_nt_gbs"]))
    traffic = load_traffic()
    cpu = None if args.no_cpu else cpu_baseline(dec)
    if not args.no_cpu:
        extras["cpu_baselines"] = cpu_baselines_more(dec)
    alg = dec["alg_bytes"]
    line = {
        "metric": "decode paged-attn HBM GB/s & % of peak (B=64, 8B GQA); KV append GB/s",
        "value": round(dec["graph_gbs"], 1),
        "unit": "GB/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": round(dec["graph_ms"], 5),
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "bf16",
        "data": "synthetic (seeded N(0,1) K/V/Q, seeded log-normal context lengths)",
        "config": {"workload": "paged decode attention, BASELINE config 2: 32 q / 8 kv heads, "
                               "head_dim 128, block_size 16, batch 64, log-normal contexts "
                               "median 2k in [256, 8192], 32k-block pool",
                   "sum_context_tokens": dec["sum_len"], "global_batch": 64,
                   "algorithmic_bytes_per_step": alg, "parallelism": "single GPU"},
        "roofline": {"bound": "hbm", "achieved": round(dec["graph_gbs"], 1), "peak": HBM_PEAK_GBS,
                     "unit": "GB/s", "frac": round(dec["graph_gbs"] / HBM_PEAK_GBS, 4),
                     "traffic": traffic.get("bytes_per_call") if traffic else None,
                     "traffic_source": ("profiles/paged_decode_config2_traffic.json: FETCH_SIZE "
                                        "and WRITE_SIZE of a rocprofv3 --pmc run of this call, "
                                        "calibrated on a copy of known size; read from the "
                                        "committed file, not measured in this run"),
                     "kernel": "paged_decode_stream + paged_decode_merge (one vapi_paged_attention call)"},
        "cpu_baseline": cpu,
        # Config 1's append, three ways: replayed from a graph with its source
        # rows warm (as a projection just wrote them), replayed with cold
        # sources (rotated over 384 MB, read with the cold-source flag), and
        # launched call by call from the host through the bare C ABI.
        "kv_append_gbs": round(extras["append_cfg1"]["gbs"], 1) if "append_cfg1" in extras else None,
        "kv_append_cold_gbs": (round(extras["append_cfg1"]["cold_gbs"], 1)
                               if "append_cfg1" in extras else None),
        "kv_append_host_launched_gbs": (round(extras["append_cfg1"]["gbs_host_launched_c_abi"], 1)
                                        if "append_cfg1" in extras else None),
        # Config 4a's copy-on-write: the layer-major pool (each layer's K and
        # V buffers contiguous, as the reference's tensors) and a block-major
        # one (a pair is one contiguous run).
        "kv_copy_gbs": (round(extras["blocks_cfg4"]["copy_gbs"], 1)
                        if "blocks_cfg4" in extras else None),
        "kv_copy_block_major_gbs": (round(extras["blocks_cfg4"]["copy_block_major"]["gbs"], 1)
                                    if "blocks_cfg4" in extras else None),
        # Tokens per second per layer (one GPU): config 2's 64 decode tokens
        # per call, config 1's 3,891 appended tokens per call, config 3's
        # 16,384 prefill query tokens per call.
        "tokens_per_s": {
            "decode_cfg2": round(64 / (dec["graph_ms"] * 1e-3)),
            "append_cfg1": (round(3891 / (extras["append_cfg1"]["us"] * 1e-6))
                            if "append_cfg1" in extras else None),
            "prefill_cfg3": (round(32 * 512 / (extras["prefill_cfg3"]["ms"] * 1e-3))
                             if "prefill_cfg3" in extras else None),
        },
        "extras": extras,
    }
    print(json.dumps(line), flush=True)


if __name__ == "__main__":
    main()
