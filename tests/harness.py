"""Shared test harness: synthetic tensor contents, the GPU run through the C-ABI, the CPU-checker run, tolerances."""
import numpy as np

from oracle import oracle as O

DT = {"f16": O.DT_F16, "bf16": O.DT_BF16, "u8": O.DT_U8}

# Tolerance of north star: <= 2e-3 relative / 1e-3 absolute on fp16/bf16 outputs and on scores.  The output is
# stored in the query dtype, so half an ulp of that format is unavoidable on top: 2^-11 relative for fp16 (inside
# the 2e-3), 2^-8 for bf16 (added explicitly).
RTOL, ATOL = 2e-3, 1e-3
HALF_ULP = {"f16": 2.0 ** -11, "bf16": 2.0 ** -8}


def assert_close(got, ref, q_dtype, what="out"):
    got = np.asarray(got, np.float64)
    ref = np.asarray(ref, np.float64)
    extra = HALF_ULP[q_dtype] if q_dtype == "bf16" else 0.0
    tol = ATOL + (RTOL + extra) * np.abs(ref)
    assert got.shape == ref.shape, f"{what}: shape {got.shape} != {ref.shape}"
    assert np.isfinite(got).all(), f"{what}: {(~np.isfinite(got)).sum()} of {got.size} values are not finite"
    bad = ~(np.abs(got - ref) <= tol)
    assert not bad.any(), (f"{what}: {bad.sum()} of {bad.size} beyond tolerance; worst |err|={np.abs(got - ref).max():.4g} "
                           f"at ref={ref.flat[np.argmax(np.abs(got - ref))]:.4g}")


def tiny_decode_case():
    return dict(name="tiny_decode_u8", B=3, Hq=8, Hkv=2, D=128, bs=32, q_dtype="f16", kv_dtype="u8",
                past_lens=np.array([37, 130, 64], np.int32), new_lens=np.array([1, 1, 1], np.int32))


def case_from_lens(name, Hq, Hkv, D, bs, q_dtype, kv_dtype, past_lens, new_lens, sliding_window=0,
                   score_aggregation_window=None, scale=None):
    return dict(name=name, B=len(past_lens), Hq=Hq, Hkv=Hkv, D=D, bs=bs, q_dtype=q_dtype, kv_dtype=kv_dtype,
                past_lens=np.asarray(past_lens, np.int32), new_lens=np.asarray(new_lens, np.int32),
                sliding_window=sliding_window, score_aggregation_window=score_aggregation_window, scale=scale)


def build_case(case, seed, outliers=False, pool_factor=2.0):
    """Adds block tables and tensor contents (numpy) to a shape description.

    The past part of the caches is filled with the CPU checker's own append (a prefill of ``past`` tokens per
    sequence), so attention parity does not depend on the GPU append.
    """
    c = dict(case)
    rng = np.random.default_rng(seed)
    B, Hq, Hkv, D, bs = c["B"], c["Hq"], c["Hkv"], c["D"], c["bs"]
    qd, kd = DT[c["q_dtype"]], DT[c["kv_dtype"]]
    past, new = c["past_lens"].astype(np.int64), c["new_lens"].astype(np.int64)
    c["subsequence_begins"] = np.concatenate([[0], np.cumsum(new)]).astype(np.int32)
    nblk = (past + new + bs - 1) // bs
    c["block_indices_begins"] = np.concatenate([[0], np.cumsum(nblk)]).astype(np.int32)
    n_ids = int(c["block_indices_begins"][-1])
    pool = int(np.ceil(pool_factor * n_ids)) + 1
    c["num_blocks"] = pool
    c["block_indices"] = rng.permutation(pool)[:n_ids].astype(np.int32)
    c.setdefault("sliding_window", 0)
    c.setdefault("score_aggregation_window", None)
    if c.get("scale") is None:
        c["scale"] = float(1.0 / np.sqrt(D))
    rb = O.row_bytes(D, kd)

    def synth(n, width):
        x = rng.standard_normal((n, width)).astype(np.float32)
        if outliers:  # 1 % of elements replaced by +-8
            m = rng.random(x.shape) < 0.01
            x[m] = np.where(rng.random(m.sum()) < 0.5, 8.0, -8.0)
        return O.to_bits(x, qd)

    kc = np.zeros((pool, Hkv, bs, rb), np.uint8)
    vc = np.zeros((pool, Hkv, bs, rb), np.uint8)
    if past.sum() > 0:
        psb = np.concatenate([[0], np.cumsum(past)]).astype(np.int32)
        O.kv_append(synth(int(psb[-1]), Hkv * D), synth(int(psb[-1]), Hkv * D), qd, kc, vc, kd,
                    np.zeros(B, np.int32), psb, c["block_indices"], c["block_indices_begins"], Hkv, D, bs)
    T = int(c["subsequence_begins"][-1])
    c["key_cache0"], c["value_cache0"] = kc, vc
    c["query"] = synth(T, Hq * D)
    c["key"] = synth(T, Hkv * D)
    c["value"] = synth(T, Hkv * D)
    return c


def run_case_on_checker(case, num_threads=8, want_scores=True):
    c = case
    qd, kd = DT[c["q_dtype"]], DT[c["kv_dtype"]]
    kc, vc = c["key_cache0"].copy(), c["value_cache0"].copy()
    O.kv_append(c["key"], c["value"], qd, kc, vc, kd, c["past_lens"], c["subsequence_begins"], c["block_indices"],
                c["block_indices_begins"], c["Hkv"], c["D"], c["bs"])
    out, out16, scores = O.paged_attention(c["query"], qd, kc, vc, kd, c["past_lens"], c["subsequence_begins"],
                                           c["block_indices"], c["block_indices_begins"], c["Hq"], c["Hkv"], c["D"],
                                           c["bs"], c["scale"], c["sliding_window"], c["score_aggregation_window"],
                                           want_scores, num_threads)
    return dict(key_cache=kc, value_cache=vc, out=out, out16=out16, scores=scores)


def _torch_dtype(torch, name):
    return {"f16": torch.float16, "bf16": torch.bfloat16}[name]


def to_device_16(torch, bits, name, device):
    return torch.from_numpy(bits.view(np.int16)).to(device).view(_torch_dtype(torch, name))


def run_case_on_gpu(pkg, case, device, want_scores=True, op=None):
    """Runs pa_step_begin / pa_set_block_indices / pa_forward through the C-ABI; returns numpy results."""
    import torch
    c = case
    if op is None:
        op = pkg.PagedAttention(c["Hq"], c["Hkv"], c["D"], c["bs"], c["q_dtype"], c["kv_dtype"], num_layers=1,
                                device=device.index or 0, stream=torch.cuda.current_stream(device))
    q = to_device_16(torch, c["query"], c["q_dtype"], device)
    k = to_device_16(torch, c["key"], c["q_dtype"], device)
    v = to_device_16(torch, c["value"], c["q_dtype"], device)
    kc = torch.from_numpy(c["key_cache0"]).to(device)
    vc = torch.from_numpy(c["value_cache0"]).to(device)
    out = torch.zeros_like(q)
    op.step_begin(c["past_lens"], c["subsequence_begins"], c["block_indices_begins"],
                  int((c["past_lens"] + c["new_lens"]).max()), c["score_aggregation_window"], c["sliding_window"],
                  c["scale"])
    op.set_block_indices(c["block_indices"], c["num_blocks"])
    scores = torch.full((op.total_scores,), float("nan"), dtype=torch.float32, device=device) if want_scores else None
    op.forward(q, k, v, kc, vc, out, scores)
    op.synchronize()
    torch.cuda.synchronize(device)
    return dict(key_cache=kc.cpu().numpy(), value_cache=vc.cpu().numpy(),
                out=out.float().cpu().numpy(), out16=out.view(torch.int16).cpu().numpy().view(np.uint16),
                scores=scores.cpu().numpy() if want_scores else None, op=op)


def spoil_rows_beyond_the_context(c):
    """All-ones bytes -- NaN headers over u8 and u4 rows -- in every cache row behind a sequence's last token, its own blocks'
    included and blocks of no sequence."""
    bs = c["bs"]
    keep = np.zeros((c["num_blocks"], bs), bool)
    for b, (past, new) in enumerate(zip(c["past_lens"], c["new_lens"])):
        pos = np.arange(past + new)
        keep[c["block_indices"][c["block_indices_begins"][b] + pos // bs], pos % bs] = True
    for cache in (c["key_cache0"], c["value_cache0"]):
        cache.transpose(0, 2, 1, 3)[~keep] = 0xFF


def quantised_rows_f64(cache, levels, D):
    """Rows of a u8 (levels 255) or u4 (15) cache as the binary64 values they stand for."""
    hdr = np.ascontiguousarray(cache[..., :8]).view(np.float32).astype(np.float64)
    codes = cache[..., 8:]
    if levels == 15:
        codes = np.stack([codes >> 4, codes & 15], -1).reshape(cache.shape[:-1] + (D,))
    return (codes - hdr[..., 1:]) * hdr[..., :1]


def attention_f64(query, key_cache, value_cache, levels, past, sb, bib, table, Hq, Hkv, D, bs):
    """Causal attention in binary64 over quantised caches that hold the step's rows already; query [T, Hq * D] values."""
    out = np.zeros((int(sb[-1]), Hq, D))
    q = np.asarray(query, np.float64).reshape(-1, Hkv, Hq // Hkv, D)
    for b in range(len(past)):
        n = int(past[b] + sb[b + 1] - sb[b])
        ids = table[bib[b]:bib[b + 1]]
        k, v = (quantised_rows_f64(c[ids], levels, D).transpose(1, 0, 2, 3).reshape(Hkv, -1, D)[:, :n] for c in (key_cache, value_cache))
        for t in range(int(sb[b]), int(sb[b + 1])):
            m = int(past[b]) + t - int(sb[b]) + 1
            x = q[t] @ k[:, :m].transpose(0, 2, 1) / np.sqrt(D)
            p = np.exp(x - x.max(-1, keepdims=True))
            out[t] = (p @ v[:, :m] / p.sum(-1, keepdims=True)).reshape(Hq, D)
    return out.reshape(len(out), Hq * D)


def misrounded(got, exact, q_dtype):
    """How many outputs are not the binary64 result rounded to the query's type.  A result whose error before that last rounding
    is e units in the last place misses with probability e, so the count tells errors apart that the rounding hides."""
    import torch
    want = torch.from_numpy(exact).to(_torch_dtype(torch, q_dtype)).float().numpy()
    return int((np.asarray(got, np.float32) != want).sum())
