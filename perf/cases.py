"""Performance cases of the PagedAttention path: the steps a continuous-batching pipeline has the library do.

A pass of a "step" or "sparse" case is one model step over some decoder layers, exactly as the pipeline drives it: the
step's arrays (`step_begin`), the block table (`set_block_indices`), then one `forward` per layer, each layer with K and V
cache tensors, queries, keys and values of its own.  The layer count of a case is the model's where the step is small
(host work and launches are then shared by as many layers as in real use) and less where one layer is long.  A pass of
an "evict" case is what follows such a step when cache eviction is on: every layer's scores are registered and the
blocks to drop are chosen.

Cache contents are seeded normal values with 1 % outliers at +-8, put into the caches (and quantised) by the library's own
append; block tables are random permutations of a pool larger than the blocks in use.
"""
import importlib.util
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
DTYPES = {"f16": torch.float16, "bf16": torch.bfloat16}
POOL_FACTOR = 1.25


def _package():
    """The package directory's name holds a dot: it is loaded from its path, of the tree the process runs in."""
    name = "openvino_genai_amd"
    if name not in sys.modules:
        root = os.getcwd() if os.path.isdir(os.path.join(os.getcwd(), "openvino.genai_amd")) else ROOT
        path = os.path.join(root, "openvino.genai_amd")
        spec = importlib.util.spec_from_file_location(name, os.path.join(path, "__init__.py"), submodule_search_locations=[path])
        sys.modules[name] = importlib.util.module_from_spec(spec)
        spec.loader.exec_module(sys.modules[name])
    return sys.modules[name]


def _step(name, heads, q, kv, layers, bs=32, scores=False, window=0, decodes=0, past=(0, 0), new=1, chunks=0,
          chunk_past=(0, 0), chunk_new=0, shape_seed=1, kind="step", threshold=0.0):
    """decodes: sequences that schedule `new` tokens each behind past[0] .. past[1] cached ones (drawn by shape_seed);
    chunks: sequences that schedule `chunk_new` prompt tokens each, evenly over chunk_past[0] .. chunk_past[1]."""
    c = dict(kind=kind, Hq=heads[0], Hkv=heads[1], D=heads[2], bs=bs, q=q, kv=kv, layers=layers, scores=scores, window=window,
             decodes=decodes, past_lo=past[0], past_hi=past[1], new=new, chunks=chunks, chunk_past_lo=chunk_past[0],
             chunk_past_hi=chunk_past[1], chunk_new=chunk_new, shape_seed=shape_seed, threshold=threshold)
    return dict(name=name, **c) if name else c


def _evict(name, sequences, layers, mode, cache=1024, bs=32):
    c = dict(kind="evict", sequences=sequences, layers=layers, mode=mode, cache=cache, bs=bs)
    return dict(name=name, **c) if name else c


LLAMA, TINY, QWEN, LONG = (32, 8, 128), (32, 4, 64), (28, 4, 128), (40, 8, 128)


def listed():
    return [
        # one user in a chat: a token per step, all 32 layers; launches and host work decide
        _step("chat_decode_u8", LLAMA, "f16", "u8", 32, decodes=1, past=(1117, 1117)),
        # a small server's batch on a small model with a 16-bit cache, contexts of all lengths, 22 layers
        _step("small_batch_decode_f16", TINY, "f16", "f16", 22, decodes=16, past=(64, 2048)),
        # a full serving batch over the default cache precision, scores on for cache eviction: the headline step
        _step("batch_decode_scores_u8", LLAMA, "f16", "u8", 4, scores=True, decodes=64, past=(4096, 4096)),
        # few users, very long contexts
        _step("long_context_decode_u8", LONG, "f16", "u8", 4, decodes=8, past=(32768, 32768)),
        # the smallest cache precision, a ragged batch
        _step("ragged_decode_u4", LLAMA, "bf16", "u4", 4, decodes=32, past=(256, 4096), shape_seed=5),
        # speculative decoding / prompt lookup: every sequence validates four drafted tokens
        _step("validate_drafts_u8", LLAMA, "f16", "u8", 8, decodes=16, past=(500, 4000), new=5, shape_seed=6),
        # the scheduler's default step: 256 batched tokens, of which one prompt takes what the running sequences leave
        _step("split_fuse_256_u8", LLAMA, "f16", "u8", 8, decodes=15, past=(128, 4000), chunks=1, chunk_past=(1000, 1000),
              chunk_new=241, shape_seed=7),
        # a large step that mixes prompts and running sequences over a 16-bit cache
        _step("mixed_bf16", QWEN, "bf16", "bf16", 2, decodes=60, past=(512, 8192), chunks=4, chunk_past=(0, 8192),
              chunk_new=512, shape_seed=8),
        # a whole prompt in one step over the default cache precision
        _step("prompt_u8", LLAMA, "f16", "u8", 2, chunks=1, chunk_new=6143),
        # one chunk of a very long prompt over a 16-bit cache
        _step("chunk_behind_30000_bf16", QWEN, "bf16", "bf16", 1, chunks=1, chunk_past=(30000, 30000), chunk_new=2048),
        # a chunk of a long prompt with block-sparse prefill
        _step("xattention_chunk_bf16", QWEN, "bf16", "bf16", 2, chunks=1, chunk_past=(14011, 14011), chunk_new=2048,
              kind="sparse", threshold=0.8),
        # the eviction step of a batch: 64 sequences at their cap of 1024 tokens drop a block in each of 32 layers
        _evict("evict_norm_sum", 64, 32, "norm_sum"),
    ]


def _log_int(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def _cost(case):
    """Seconds a pass may take at modest rates (4 TB/s, 0.4 PFLOP/s, 20 us per layer): bounds what `draw` gives."""
    w = work(case)
    return w["bytes"] / 4e12 + w["flops"] / 4e14 + 2e-5 * case["layers"]


def draw(rng):
    """A case of the listed ones' ranges: the head shapes of the library's workloads and tests, every cache type, block
    sizes 16 - 256, batches of 1 - 128 sequences, contexts of 1 - 32768 tokens."""
    limit = max(_cost(c) for c in listed())
    while True:
        kind = rng.choice(["decode"] * 4 + ["validate", "mixed", "mixed", "prompt", "prompt", "sparse", "evict"])
        seed = rng.randrange(1, 1 << 30)
        if kind == "evict":
            c = _evict(None, _log_int(rng, 1, 128), rng.choice([16, 22, 32]), rng.choice(["norm_sum", "sum"]),
                       32 * rng.randrange(16, 65))
        else:
            heads = rng.choice([LLAMA, LLAMA, TINY, QWEN, LONG, (32, 32, 96), (16, 8, 256)])
            q = rng.choice(["f16", "bf16"])
            kv = rng.choice(["u8", "u8", q])
            bs = rng.choice([32, 32, 32, 16, 64, 256])
            scores = rng.random() < 0.3
            window = rng.choice([0, 0, 0, 0, 4096])
            hi = _log_int(rng, 16, 32768)
            lo = hi if rng.random() < 0.3 else _log_int(rng, 1, hi)
            layers = rng.choice([1, 2, 4, 8, 16, 32])
            if kind == "decode":
                if rng.random() < 0.25:  # what only the shape-generic kernels' callers ask for
                    heads, kv = rng.choice([(LLAMA, "u4"), ((32, 8, 80), rng.choice(["u8", q]))])
                c = _step(None, heads, q, kv, layers, bs, scores, window, _log_int(rng, 1, 128), (lo, hi), shape_seed=seed)
            elif kind == "validate":
                c = _step(None, heads, q, kv, layers, bs, scores, window, _log_int(rng, 1, 64), (lo, hi), rng.randrange(2, 9), shape_seed=seed)
            elif kind == "mixed":
                c = _step(None, heads, q, kv, layers, bs, scores, window, _log_int(rng, 1, 64), (lo, hi), 1, rng.randrange(1, 5),
                          (0, _log_int(rng, 1, 8192)), _log_int(rng, 16, 1024), seed)
            elif kind == "prompt":
                p = rng.choice([0, _log_int(rng, 1, 30000)])
                c = _step(None, heads, q, kv, layers, bs, scores, window, chunks=rng.randrange(1, 5), chunk_past=(p, p),
                          chunk_new=_log_int(rng, 16, 8192), shape_seed=seed)
            else:
                p = rng.choice([0, _log_int(rng, 64, 30000)])
                c = _step(None, rng.choice([LLAMA, QWEN, (16, 8, 256)]), q, kv, layers, rng.choice([32, 256]), False, 0,
                          chunks=rng.randrange(1, 3), chunk_past=(p, p), chunk_new=_log_int(rng, 128, 4096), shape_seed=seed,
                          kind="sparse", threshold=rng.choice([0.8, 0.9]))
        while c["layers"] > 1 and _cost(c) > limit:
            c["layers"] //= 2
        if _cost(c) <= limit:
            return c


def _lengths(case):
    """(past, new) per sequence: prompt chunks first, then the running sequences."""
    rng = np.random.Generator(np.random.PCG64(case["shape_seed"]))
    past = np.concatenate([np.linspace(case["chunk_past_lo"], case["chunk_past_hi"], case["chunks"]).round(),
                           rng.integers(case["past_lo"], case["past_hi"] + 1, size=case["decodes"])]).astype(np.int64)
    new = np.concatenate([np.full(case["chunks"], case["chunk_new"]), np.full(case["decodes"], case["new"])]).astype(np.int64)
    return past, new


def _row_bytes(D, kv):
    return D + 8 if kv == "u8" else D // 2 + 8 if kv == "u4" else 2 * D


def work(case):
    """Bytes: every visible cache row of K and V once, queries in and outputs out, the new rows in and into the caches,
    ids and scores; flops: 4 * D per (query row, visible position).  Block-sparse chunks: the positions a threshold of 0.8
    to 0.9 keeps on these inputs are about a tenth of the visible ones."""
    if case["kind"] == "evict":
        tokens = case["sequences"] * case["layers"] * (case["cache"] + case["bs"])
        return {"bytes": 4.0 * tokens + 32.0 * tokens, "flops": 2.0 * tokens}
    past, new = _lengths(case)
    Hq, Hkv, D, w = case["Hq"], case["Hkv"], case["D"], case["window"]
    rows = pairs = 0
    for p, n in zip(past.tolist(), new.tolist()):
        vis = np.arange(p + 1, p + n + 1)
        rows += min(p + n, w + n - 1) if w else p + n
        pairs += int((np.minimum(vis, w) if w else vis).sum())
    share = 0.1 if case["kind"] == "sparse" else 1.0
    rb, T = _row_bytes(D, case["kv"]), int(new.sum())
    nbytes = 2 * Hkv * rb * rows + T * (2 * Hq * D * 2 + 2 * Hkv * D * 2) + 4 * int((past + new).sum()) * (1 if case["scores"] else 0) \
        + 4 * int(((past + new + case["bs"] - 1) // case["bs"]).sum())
    return {"bytes": float(nbytes * case["layers"]), "flops": 4.0 * Hq * D * pairs * share * case["layers"]}


def tolerance(case):
    """Outputs are rounded to the query's type; probabilities enter the products rounded to 11 bits or better and scores
    are staged in f16.  Against the same step evaluated in 64 bits the path was off by up to REL_SEEN (2-norm, outputs and
    scores) and MAX_SEEN; four times that is allowed.  Eviction works in binary64 and selects whole blocks."""
    if case["kind"] == "evict":
        return "exact"
    return {"rel": 4 * REL_SEEN[case["q"]], "max": 4 * MAX_SEEN[case["q"]], "differ": 0.0}


REL_SEEN = {"f16": 2.2e-4, "bf16": 1.7e-3}
MAX_SEEN = {"f16": 8e-4, "bf16": 4e-3}


def _values(n, width, dtype, gen):
    x = torch.randn(n, width, generator=gen, device="cuda", dtype=torch.float32)
    r = torch.rand(n, width, generator=gen, device="cuda", dtype=torch.float32)
    x = torch.where(r < 0.005, 8.0, torch.where(r > 0.995, -8.0, x))
    return x.to(dtype)


def _cached_groups(case, past):
    """The sequences with a cached part, some at a time (the order in which the cached tokens are drawn)."""
    group = max(1, int(2 ** 27 // max(1, int(past.max()) * case["Hkv"] * case["D"])))
    for b0 in range(0, len(past), group):
        idx = np.array([b for b in range(b0, min(len(past), b0 + group)) if past[b] > 0], np.int64)
        if len(idx):
            yield idx


def prepare(case, seed):
    pkg = _package()
    gen = torch.Generator(device="cuda").manual_seed(int(seed))
    if case["kind"] == "evict":
        return _prepare_evict(pkg, case, gen)
    past, new = _lengths(case)
    L, Hq, Hkv, D, bs = case["layers"], case["Hq"], case["Hkv"], case["D"], case["bs"]
    dtype, B, T = DTYPES[case["q"]], len(past), int(new.sum())
    nblk = (past + new + bs - 1) // bs
    bib = np.concatenate([[0], np.cumsum(nblk)]).astype(np.int32)
    pool = int(np.ceil(POOL_FACTOR * bib[-1])) + 1
    table = np.random.Generator(np.random.PCG64(int(seed))).permutation(pool)[:bib[-1]].astype(np.int32)
    rb = pkg.row_bytes(D, case["kv"])
    kc = torch.zeros(L, pool, Hkv, bs, rb, dtype=torch.uint8, device="cuda")
    vc = torch.zeros_like(kc)
    op = pkg.PagedAttention(Hq, Hkv, D, bs, case["q"], case["kv"], num_layers=L, device=0, stream=torch.cuda.current_stream())
    # block-sparse prefill: keys of the first 64 tokens and of a twenty-fifth of the other 64-token blocks lie along a
    # direction that the queries share, as the sink and retrieval blocks of trained models do
    lean = torch.randn(Hkv, D, generator=gen, device="cuda") if case["kind"] == "sparse" else None

    def keys(k, starts, lens):
        if lean is None:
            return k
        heavy = torch.rand(int(lens.max()) // 64 + 1, generator=gen, device="cuda") < 0.04
        heavy[0] = True
        for s, n in zip(starts.tolist(), lens.tolist()):
            m = heavy.repeat_interleave(64)[:n].to(torch.float32)
            k[s:s + n] += (0.85 * m[:, None] * lean.reshape(1, -1)).to(dtype)
        return k

    for idx in _cached_groups(case, past):
        begins = np.concatenate([[0], np.cumsum(past[idx])]).astype(np.int32)
        op.step_begin(np.zeros(len(idx), np.int32), begins, np.concatenate([[0], np.cumsum(nblk[idx])]).astype(np.int32))
        op.set_block_indices(np.concatenate([table[bib[b]:bib[b + 1]] for b in idx]), pool)
        for l in range(L):
            n = int(begins[-1])
            op.kv_append(keys(_values(n, Hkv * D, dtype, gen), begins[:-1], past[idx]), _values(n, Hkv * D, dtype, gen), kc[l], vc[l], layer=l)
    op.synchronize()
    sb = np.concatenate([[0], np.cumsum(new)]).astype(np.int32)
    q = torch.randn(L, T, Hq * D, generator=gen, device="cuda").to(dtype)
    if lean is not None:
        q += (0.85 * lean.repeat_interleave(Hq // Hkv, 0).reshape(1, 1, -1)).to(dtype)
    k = _values(L * T, Hkv * D, dtype, gen).view(L, T, -1)
    v = _values(L * T, Hkv * D, dtype, gen).view(L, T, -1)
    n_scores = int((past + new).sum())
    return dict(case=case, op=op, past=past.astype(np.int32), sb=sb, bib=bib, table=table, pool=pool,
                max_len=int((past + new).max()), thresholds=np.full(B, case["threshold"], np.float32), q=q, k=k, v=v, kc=kc, vc=vc,
                out=torch.zeros_like(q), scores=torch.zeros(L, n_scores, device="cuda") if case["scores"] else None)


def _prepare_evict(pkg, case, gen):
    n, L, bs = case["sequences"], case["layers"], case["bs"]
    agg = pkg.AggregationMode.NORM_SUM if case["mode"] == "norm_sum" else pkg.AggregationMode.SUM
    cfg = pkg.CacheEvictionConfig(32, 128, case["cache"], agg, False)
    tokens = case["cache"] + bs
    ev = pkg.Evictor(cfg, bs, L, 7, max_sequences=n, max_tracked_tokens=tokens + bs, device=0, stream=torch.cuda.current_stream())
    # attention mass per position: a softmax of normal logits, some blocks drawing far more of it than others, times 32 heads
    logits = torch.randn(L, n, tokens, generator=gen, device="cuda")
    logits += 3.0 * torch.randn(L, n, tokens // bs, generator=gen, device="cuda").repeat_interleave(bs, -1)
    scores = 32.0 * torch.softmax(logits, -1)
    slots = np.arange(n, dtype=np.int32)
    # what the prompt's step left: its scores, over as many tokens as the cap (the scores of its last eight query tokens)
    prompt = scores[:, :, :case["cache"]].contiguous()
    ev.register_new_token_scores(slots, [prompt[l].data_ptr() for l in range(L)], np.arange(n + 1, dtype=np.int64) * case["cache"],
                                 np.full(n, 8, np.uint64))
    torch.cuda.synchronize()
    return dict(case=case, ev=ev, scores=scores.contiguous(), slots=slots, offsets=np.arange(n + 1, dtype=np.int64) * tokens,
                aggregated=np.ones(n, np.uint64))


def run(state):
    case = state["case"]
    if case["kind"] == "evict":
        scores = state["scores"]
        state["ev"].register_new_token_scores(state["slots"], [scores[l].data_ptr() for l in range(case["layers"])], state["offsets"],
                                              state["aggregated"])
        dropped = state["ev"].evict_logical_blocks(state["slots"])
        return {"counts": np.array([[len(b) for b in s] for s in dropped], np.int32),
                "blocks": np.array([i for s in dropped for b in s for i in b], np.int32)}
    op = state["op"]
    op.step_begin(state["past"], state["sb"], state["bib"], state["max_len"], None, case["window"], 0.0)
    op.set_block_indices(state["table"], state["pool"])
    if case["kind"] == "sparse":
        op.set_xattention(state["thresholds"], 64, 8)
    q, k, v, kc, vc, out, scores = (state[x] for x in ("q", "k", "v", "kc", "vc", "out", "scores"))
    for l in range(case["layers"]):
        op.forward(q[l], k[l], v[l], kc[l], vc[l], out[l], None if scores is None else scores[l], layer=l)
    return {"out": out, "scores": scores, "key_cache": kc, "value_cache": vc}


def _cached(x, case):
    """What a cache of the case's type holds of rows x [n, Hkv, D], in 64 bits.  Quantised rows: scale = (max - min) / levels
    and zero-point = -min / scale in binary32, codes rounded to nearest."""
    levels = {"u8": 255.0, "u4": 15.0}.get(case["kv"])
    if levels is None:
        return x.double()
    x = x.float()
    mn, mx = x.amin(-1, keepdim=True), x.amax(-1, keepdim=True)
    scale = (mx - mn) / torch.tensor(levels, device=x.device)  # (by a tensor: a Python number would become a reciprocal)
    scale = torch.where(scale == 0, torch.full_like(scale, 1e-4), scale)
    zp, inv = -mn / scale, 1.0 / scale
    codes = (x.double() * inv.double() + zp.double()).float().round().clamp(0, levels)  # one rounding, as a fused multiply-add
    return (codes.double() - zp.double()) * scale.double()


def exact(case, seed):
    """Outputs and scores in 64 bits; cache contents are bytes and have no such value.  None for eviction (block numbers) and for
    block-sparse prefill, where the blocks that are kept hang on comparisons of computed sums."""
    if case["kind"] != "step" or work(case)["flops"] > 4e12:
        return None
    gen = torch.Generator(device="cuda").manual_seed(int(seed))
    past, new = _lengths(case)
    L, Hq, Hkv, D, w = case["layers"], case["Hq"], case["Hkv"], case["D"], case["window"]
    dtype, B, T = DTYPES[case["q"]], len(past), int(new.sum())
    rows = [[[None] * L for _ in range(B)] for _ in range(2)]  # [K | V][sequence][layer]: the cached rows as drawn
    for idx in _cached_groups(case, past):
        begins = np.concatenate([[0], np.cumsum(past[idx])])
        for l in range(L):
            for which in range(2):
                x = _values(int(begins[-1]), Hkv * D, dtype, gen)
                for i, b in enumerate(idx):
                    rows[which][b][l] = x[begins[i]:begins[i + 1]]
    sb = np.concatenate([[0], np.cumsum(new)])
    q = torch.randn(L, T, Hq * D, generator=gen, device="cuda").to(dtype)
    kv_new = [_values(L * T, Hkv * D, dtype, gen).view(L, T, -1) for _ in range(2)]
    out = torch.zeros(L, T, Hq * D, dtype=torch.float64, device="cuda")
    scores = torch.zeros(L, int((past + new).sum()), dtype=torch.float64, device="cuda") if case["scores"] else None
    so = np.concatenate([[0], np.cumsum(past + new)])
    for l in range(L):
        for b in range(B):
            parts = [[rows[j][b][l]] if past[b] else [] for j in range(2)]
            k, v = (_cached(torch.cat(parts[j] + [kv_new[j][l, sb[b]:sb[b + 1]]]).view(-1, Hkv, D), case).transpose(0, 1).contiguous()
                    for j in range(2))
            n_kv, kt = k.shape[1], k.transpose(1, 2).contiguous()
            pos = torch.arange(n_kv, device="cuda")
            step = max(1, int(2 ** 28 // (n_kv * Hq)))  # query tokens at a time
            for t0 in range(0, int(new[b]), step):
                t1 = min(int(new[b]), t0 + step)
                x = q[l, sb[b] + t0:sb[b] + t1].double().view(t1 - t0, Hkv, Hq // Hkv, D).permute(1, 2, 0, 3).reshape(Hkv, -1, D).contiguous()
                p = torch.bmm(x, kt).view(Hkv, Hq // Hkv, t1 - t0, n_kv) / D ** 0.5
                last = int(past[b]) + torch.arange(t0, t1, device="cuda")[:, None]
                p.masked_fill_((pos > last) | ((pos <= last - w) if w else (pos < 0)), float("-inf"))
                p = torch.softmax(p, -1)
                o = torch.bmm(p.view(Hkv, -1, n_kv), v).view(Hkv, Hq // Hkv, t1 - t0, D)
                out[l, sb[b] + t0:sb[b] + t1] = o.permute(2, 0, 1, 3).reshape(t1 - t0, Hq * D)
                if scores is not None and t1 == int(new[b]):  # the default window: the last query token, summed over the heads
                    scores[l, so[b]:so[b + 1]] = p[:, :, -1].sum((0, 1))
    return {"out": out, "scores": scores, "key_cache": None, "value_cache": None}
