"""Performance cases of the paged KV-cache path.

Each case is one call (or one layer's pair of calls) that a serving program
makes per layer of a step, through the public entry points of vapi_amd:

  decode    one new token per sequence: cache write + attention, or attention
            alone over a pool that already holds the token
  prefill   a chunk of new tokens per sequence over its earlier context
  mixed     one step of decode rows and prefill chunks together
  append    the cache write alone
  copy      copy-on-write of whole blocks over all layers

A case is a dict of plain values. Sequence lengths follow from the case
alone (`lens_seed` and the ranges beside it); the contents, the block tables
and the slots follow from the seed given to prepare().
"""
from __future__ import annotations

import math

import numpy as np
import torch

from vapi_amd.attention import (ForwardBatch, PreparedAttention,
                                paged_attention_append_prepared, paged_attention_prepared)
from vapi_amd.backend import KvBlockBackend
from vapi_amd.cache import PagedKvCache, scatter_index, write_rows_indexed

DEV = "cuda"
DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}
SIZE = {"bf16": 2, "f16": 2, "f32": 4}
SKIP = 0xFFFFFFFF


def _attn(kind, batch, heads, kv_heads, head_dim, dtype, **kw):
    case = {
        "kind": kind, "batch": batch, "q_heads": heads, "kv_heads": kv_heads,
        "head_dim": head_dim, "dtype": dtype, "block": 16, "layout": "HND",
        # Context before the step: log-normal (median, sigma) clipped to [lo, hi].
        "ctx_median": 2048, "ctx_sigma": 0.75, "ctx_lo": 256, "ctx_hi": 8192,
        # New tokens of a prefill sequence: uniform in [lo, hi].
        "new_lo": 1, "new_hi": 1, "chunks": 0,
        "window": 0, "shared_blocks": 0, "share_group": 1, "append": True, "lens_seed": 1,
    }
    case.update(kw)
    return case


def listed():
    return [
        # One user of an 8B model (32 q / 8 kv heads) generating over a short
        # context: the smallest step, all latency.
        {"name": "decode_b1",
         **_attn("decode", 1, 32, 8, 128, "bf16", ctx_median=1337, ctx_sigma=0.0)},
        # The 0.6B shape in f32 (16 q / 8 kv heads), 8 short sequences.
        {"name": "decode_b8_f32",
         **_attn("decode", 8, 16, 8, 128, "f32", ctx_median=256, ctx_sigma=0.5, ctx_lo=63,
                 ctx_hi=511, lens_seed=8)},
        # A lightly loaded server: 16 sequences of an 8B model, on blocks of
        # 32 in the [block, token, head, d] layout that such a pool may have.
        {"name": "decode_b16",
         **_attn("decode", 16, 32, 8, 128, "bf16", block=32, layout="NHD", lens_seed=16)},
        # The benchmark's decode batch: 64 sequences, contexts 256 to 8,192,
        # attention alone (the token was written by a call of its own).
        {"name": "decode_b64",
         **_attn("decode", 64, 32, 8, 128, "bf16", append=False, lens_seed=0x5EED0002)},
        # A model with as many kv heads as query heads, head_dim 96 and a
        # sliding window of 2,047 keys.
        {"name": "decode_b12_mha_window",
         **_attn("decode", 12, 32, 32, 96, "bf16", window=2047, ctx_median=3000,
                 lens_seed=12)},
        # A step of a busy server with chunked prefill: 63 decode rows and one
        # 512-token chunk in one call, attention alone.
        {"name": "mixed_b64",
         **_attn("mixed", 64, 32, 8, 128, "bf16", chunks=1, new_lo=512, new_hi=512,
                 append=False, lens_seed=0x5EED0002)},
        # One sequence's next chunk: 487 new tokens over 3,412 earlier ones.
        {"name": "prefill_b1",
         **_attn("prefill", 1, 32, 8, 128, "bf16", ctx_median=3412, ctx_sigma=0.0,
                 new_lo=487, new_hi=487, chunks=1)},
        # Chunks of 512 over 3,584 earlier keys for 32 sequences, groups of 8
        # sharing a 2,048-token prefix (the benchmark's prefill batch).
        {"name": "prefill_b32_shared",
         **_attn("prefill", 32, 32, 8, 128, "bf16", ctx_median=3584, ctx_sigma=0.0,
                 new_lo=512, new_hi=512, chunks=32, shared_blocks=128, share_group=8,
                 append=False)},
        # Fresh prompts of very different lengths in one call (28 q / 4 kv
        # heads, f16): nothing before them, causal over themselves.
        {"name": "prefill_fresh_f16",
         **_attn("prefill", 7, 28, 4, 128, "f16", ctx_median=0, ctx_sigma=0.0, ctx_lo=0,
                 new_lo=33, new_hi=3000, chunks=7, lens_seed=27)},
        # f32 prefill of the 0.6B shape: 4 chunks over about 1,500 earlier keys.
        {"name": "prefill_b4_f32",
         **_attn("prefill", 4, 16, 8, 128, "f32", ctx_median=1500, ctx_sigma=0.3,
                 new_lo=300, new_hi=512, chunks=4, lens_seed=4)},
        # The cache write of a 4,096-token step at 8 kv heads, 5% padding.
        {"name": "append_4096",
         "kind": "append", "tokens": 4096, "run": 256, "kv_heads": 8, "head_dim": 128,
         "block": 16, "layout": "HND", "dtype": "bf16", "blocks": 8192, "pad": 0.05},
        # A burst of forks: 256 blocks copied in 28 layers of 4 kv heads.
        {"name": "copy_256",
         "kind": "copy", "pairs": 256, "layers": 28, "kv_heads": 4, "head_dim": 128,
         "block": 16, "dtype": "bf16", "blocks": 640},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "decode", "mixed", "prefill", "prefill", "prefill",
                       "append", "copy"])
    if kind == "append":
        return {"kind": kind, "tokens": _log(rng, 1, 4096), "run": _log(rng, 1, 300),
                "kv_heads": rng.choice([1, 4, 8]), "head_dim": rng.choice([64, 80, 96, 128]),
                "block": rng.choice([16, 32]), "layout": rng.choice(["HND", "NHD"]),
                "dtype": rng.choice(["bf16", "f16", "f32"]), "blocks": 8192,
                "pad": rng.choice([0.0, 0.05])}
    if kind == "copy":
        return {"kind": kind, "pairs": _log(rng, 1, 256), "layers": rng.choice([16, 28, 32]),
                "kv_heads": rng.choice([4, 8]), "head_dim": rng.choice([64, 128]), "block": 16,
                "dtype": "bf16", "blocks": 640}
    dtype = rng.choice(["bf16", "bf16", "bf16", "f16", "f32"])
    heads, kvh = rng.choice([(32, 8), (32, 8), (16, 8), (28, 4), (32, 32), (64, 8)])
    case = _attn(kind, 1, heads, kvh, rng.choice([64, 80, 96, 128, 128, 128]), dtype,
                 block=rng.choice([16, 32]), layout=rng.choice(["HND", "HND", "NHD"]),
                 lens_seed=rng.randrange(1 << 20), append=rng.random() < 0.7)
    if rng.random() < 0.25:
        case["window"] = _log(rng, 128, 4096)
    if kind == "decode":
        case["batch"] = _log(rng, 1, 64)
        case["ctx_median"] = _log(rng, 40, 4000)
        case["ctx_lo"], case["ctx_hi"] = 1, 8192
    else:
        case["chunks"] = _log(rng, 1, 16 if kind == "prefill" else 3)
        case["batch"] = case["chunks"] + (_log(rng, 2, 60) if kind == "mixed" else 0)
        case["new_lo"] = _log(rng, 2, 200)
        case["new_hi"] = case["new_lo"] + _log(rng, 1, 1500)
        case["ctx_lo"], case["ctx_hi"] = 1, 8192
        if kind == "prefill" and rng.random() < 0.4:
            case["ctx_median"], case["ctx_sigma"], case["ctx_lo"] = 0, 0.0, 0
        else:
            case["ctx_median"] = _log(rng, 40, 4000)
    # No dearer than the listed cases of the same kind.
    limit = 3e10 if dtype == "f32" else 4e11
    while True:
        w = work(case)
        if w["bytes"] <= 7e8 and w["flops"] <= limit:
            return case
        if case["new_hi"] > 64:
            case["new_lo"] = max(case["new_lo"] // 2, 2)
            case["new_hi"] = max(case["new_hi"] // 2, case["new_lo"])
        case["ctx_median"] = case["ctx_median"] * 3 // 4
        case["ctx_hi"] = max(case["ctx_hi"] * 3 // 4, 64)


# ---- shapes -----------------------------------------------------------------


def _lens(case):
    """(len_q, len_k) per sequence; the chunks are the last sequences."""
    r = np.random.default_rng(case["lens_seed"])
    b = case["batch"]
    if case["ctx_median"] > 0:
        ctx = np.exp(r.normal(math.log(case["ctx_median"]), case["ctx_sigma"], size=b))
        ctx = np.clip(np.round(ctx), case["ctx_lo"], case["ctx_hi"]).astype(np.int64)
    else:
        ctx = np.zeros(b, np.int64)
    len_q = np.ones(b, np.int64)
    c = case["chunks"]
    if c:
        len_q[b - c:] = r.integers(case["new_lo"], case["new_hi"] + 1, size=c)
    # A decode batch without the cache write holds its token already.
    len_k = ctx + np.where((len_q == 1) & (not case["append"]), 0, len_q)
    return len_q, np.maximum(len_k, len_q)


def _visible(case, len_q, len_k):
    """Visible (query, key) pairs of one sequence, and keys any query sees."""
    p = np.arange(len_k - len_q, len_k, dtype=np.int64)
    lo = np.maximum(0, p - (case["window"] - 1)) if case["window"] else np.zeros_like(p)
    return int((p - lo + 1).sum()), int(len_k - lo.min())


def work(case):
    e = SIZE[case["dtype"]]
    if case["kind"] == "append":
        rows = case["tokens"] - int(round(case["pad"] * case["tokens"]))
        return {"bytes": 4.0 * rows * case["kv_heads"] * case["head_dim"] * e
                + 4.0 * case["tokens"], "flops": 0.0}
    if case["kind"] == "copy":
        return {"bytes": 4.0 * case["pairs"] * case["layers"] * case["kv_heads"] *
                case["head_dim"] * case["block"] * e + 8.0 * case["pairs"], "flops": 0.0}
    len_q, len_k = _lens(case)
    pairs = keys = 0
    for lq, lk in zip(len_q, len_k):
        p, k = _visible(case, int(lq), int(lk))
        pairs, keys = pairs + p, keys + k
    if case["shared_blocks"]:  # a shared prefix is read once per group
        g = case["share_group"]
        keys -= (case["batch"] - -(-case["batch"] // g)) * case["shared_blocks"] * case["block"]
    n = int(len_q.sum())
    kv_row = 2 * case["kv_heads"] * case["head_dim"] * e
    q_row = case["q_heads"] * case["head_dim"] * e
    # K/V once (new rows from the step's own tensors), the new rows' write,
    # Q in and the output out, tables and lengths.
    total = keys * kv_row + (n * kv_row if case["append"] else 0) + 2 * n * q_row
    total += 4 * (int((-(-len_k // case["block"])).sum()) + 2 * (case["batch"] + 1))
    return {"bytes": float(total), "flops": 4.0 * case["head_dim"] * case["q_heads"] * pairs}


# ---- inputs -------------------------------------------------------------------


def _normal(gen, shape, dtype):
    return torch.randn(shape, generator=gen, device=DEV, dtype=torch.float32).to(dtype)


def _slots(table, first, last, block):
    pos = np.arange(first, last, dtype=np.int64)
    return table[pos // block] * block + pos % block


def _attn_inputs(case, seed):
    """Everything of an attention case as plain tensors and arrays: the pool
    contents in the case's layout, Q, the new rows, tables and slots."""
    gen = torch.Generator(device=DEV)
    gen.manual_seed(seed)
    r = np.random.default_rng(seed)
    dt, bs = DTYPES[case["dtype"]], case["block"]
    kvh, d, sh = case["kv_heads"], case["head_dim"], case["shared_blocks"]
    len_q, len_k = _lens(case)
    need = -(-len_k // bs)
    groups = -(-case["batch"] // case["share_group"]) if sh else 0
    nb = int(need.sum()) - sh * (case["batch"] - groups if sh else 0) + 5
    perm = r.permutation(nb).astype(np.int64)
    prefix = [perm[g * sh:(g + 1) * sh] for g in range(groups)]
    at, tables = groups * sh, []
    for s in range(case["batch"]):
        own = int(need[s]) - sh
        tables.append(np.concatenate([prefix[s // case["share_group"]], perm[at:at + own]])
                      if sh else perm[at:at + own])
        at += own
    shape = (nb, kvh, bs, d) if case["layout"] == "HND" else (nb, bs, kvh, d)
    k, v = _normal(gen, shape, dt), _normal(gen, shape, dt)
    n = int(len_q.sum())
    q = _normal(gen, (n, case["q_heads"], d), dt)
    k_new = v_new = slots = None
    if case["append"]:
        k_new, v_new = _normal(gen, (n, kvh, d), dt), _normal(gen, (n, kvh, d), dt)
        slots = np.concatenate([_slots(t, lk - lq, lk, bs)
                                for t, lq, lk in zip(tables, len_q, len_k)])
    return {"k": k, "v": v, "q": q, "k_new": k_new, "v_new": v_new, "slots": slots,
            "tables": tables, "len_q": len_q, "len_k": len_k, "blocks": nb}


def prepare(case, seed):
    if case["kind"] == "append":
        return _prepare_append(case, seed)
    if case["kind"] == "copy":
        return _prepare_copy(case, seed)
    x = _attn_inputs(case, seed)
    cache = PagedKvCache(1, x["blocks"], case["block"], case["kv_heads"], case["head_dim"],
                         DTYPES[case["dtype"]], case["layout"], DEV)
    cache.k[0].copy_(x["k"])
    cache.v[0].copy_(x["v"])
    batch = ForwardBatch(
        cu_seqlens_q=np.concatenate([[0], np.cumsum(x["len_q"])]).tolist(),
        cu_seqlens_k=np.concatenate([[0], np.cumsum(x["len_k"])]).tolist(),
        block_tables=[t.tolist() for t in x["tables"]],
        max_seqlen_q=int(x["len_q"].max()), max_seqlen_k=int(x["len_k"].max()))
    state = {
        "case": case, "cache": cache, "q": x["q"], "scale": case["head_dim"] ** -0.5,
        "left": case["window"] - 1 if case["window"] else None,
        # What a program keeps for the layers of a step.
        "prepared": PreparedAttention.from_batch(batch, DEV, cache, case["q_heads"]),
    }
    if case["append"]:
        state.update(k_new=x["k_new"], v_new=x["v_new"], slots=scatter_index(x["slots"], DEV))
    return state


def _prepare_append(case, seed):
    gen = torch.Generator(device=DEV)
    gen.manual_seed(seed)
    r = np.random.default_rng(seed)
    dt, n, bs = DTYPES[case["dtype"]], case["tokens"], case["block"]
    shape = (n, case["kv_heads"], case["head_dim"])
    k, v = _normal(gen, shape, dt), _normal(gen, shape, dt)
    perm = r.permutation(case["blocks"]).astype(np.int64)
    slots, at, done = [], 0, 0
    while done < n:
        run = min(case["run"], n - done)
        first = int(r.integers(0, bs)) if r.random() < 0.5 else 0
        width = -(-(first + run) // bs)
        slots.append(_slots(perm[at:at + width], first, first + run, bs))
        at, done = at + width, done + run
    slots = np.concatenate(slots)
    slots[r.choice(n, size=int(round(case["pad"] * n)), replace=False)] = SKIP
    cache = PagedKvCache(1, case["blocks"], bs, case["kv_heads"], case["head_dim"], dt,
                         case["layout"], DEV)
    return {"case": case, "cache": cache, "k": k, "v": v, "slots": scatter_index(slots, DEV)}


def _prepare_copy(case, seed):
    gen = torch.Generator(device=DEV)
    gen.manual_seed(seed)
    r = np.random.default_rng(seed)
    dt = DTYPES[case["dtype"]]
    cache = PagedKvCache(case["layers"], case["blocks"], case["block"], case["kv_heads"],
                         case["head_dim"], dt, "HND", DEV)
    for t in cache.k + cache.v:
        t.copy_(_normal(gen, tuple(t.shape), dt))
    perm = r.permutation(case["blocks"])
    p = case["pairs"]
    pairs = [(int(s), int(d)) for s, d in zip(perm[:p], perm[p:2 * p])]
    return {"case": case, "cache": cache, "backend": KvBlockBackend(cache), "pairs": pairs}


# ---- one pass -----------------------------------------------------------------


def run(state):
    case, cache = state["case"], state["cache"]
    if case["kind"] == "append":
        write_rows_indexed(cache, 0, state["k"], state["v"], state["slots"])
        return [cache.k[0], cache.v[0]]
    if case["kind"] == "copy":
        state["backend"].copy_blocks(state["pairs"])
        return cache.k + cache.v
    if case["append"]:
        out = paged_attention_append_prepared(
            state["q"], state["k_new"], state["v_new"], state["slots"], cache, 0,
            state["prepared"], state["scale"], state["left"], 0)
        return [out, cache.k[0], cache.v[0]]
    return [paged_attention_prepared(state["q"], cache, 0, state["prepared"], state["scale"],
                                     state["left"], 0)]


def tolerance(case):
    if case["kind"] in ("append", "copy"):
        return "exact"
    # Two correct results differ by the order of the sums and, in 16 bits, by
    # the rounding of the probabilities and of the output: about four times
    # what the path differs from exact() by (2-norm 2.35e-3, 2.8e-4 and 7e-7;
    # largest over the root mean square 5.4e-2, 1e-2 and 1.6e-5).
    return {"rel": {"bf16": 1e-2, "f16": 1.2e-3, "f32": 3e-6}[case["dtype"]],
            "max": {"bf16": 0.22, "f16": 0.04, "f32": 6.4e-5}[case["dtype"]]}


def exact(case, seed):
    if case["kind"] in ("append", "copy"):
        return None
    x = _attn_inputs(case, seed)
    k, v = x["k"], x["v"]
    if case["layout"] == "HND":
        k, v = k.permute(0, 2, 1, 3), v.permute(0, 2, 1, 3)
    kvh, d, hq = case["kv_heads"], case["head_dim"], case["q_heads"]
    k, v = k.reshape(-1, kvh, d), v.reshape(-1, kvh, d)
    if case["append"]:
        at = torch.from_numpy(x["slots"]).to(DEV)
        k, v = k.clone(), v.clone()
        k[at], v[at] = x["k_new"], x["v_new"]
    out = torch.empty(x["q"].shape, dtype=torch.float64, device=DEV)
    first = 0
    for t, lq, lk in zip(x["tables"], x["len_q"].tolist(), x["len_k"].tolist()):
        at = torch.from_numpy(_slots(t, 0, lk, case["block"])).to(DEV)
        ks, vs = k[at].double(), v[at].double()
        qs = x["q"][first:first + lq].double()
        pos = torch.arange(lk - lq, lk, device=DEV)[:, None]
        key = torch.arange(lk, device=DEV)[None, :]
        hidden = key > pos
        if case["window"]:
            hidden |= key < pos - (case["window"] - 1)
        g = hq // kvh
        for h in range(hq):
            s = (qs[:, h] @ ks[:, h // g].T) * d ** -0.5
            s.masked_fill_(hidden, -math.inf)
            out[first:first + lq, h] = torch.softmax(s, dim=1) @ vs[:, h // g]
        first += lq
    result = [out]
    if case["append"]:
        for t in (k, v):
            t = t.view(x["blocks"], case["block"], kvh, d)
            result.append((t.permute(0, 2, 1, 3) if case["layout"] == "HND" else t).double())
    return result
