"""Mixed steps over 16-bit caches whose matrix and decode kernel run side by side -- a long chunk, or single tokens behind contexts of
very different length -- and ones below that: against the same sequences in steps of their own, and against the CPU checker."""
import numpy as np
import pytest

import harness as H

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("qd,heads,past,new,sw", [
    ("f16", (32, 4, 64), [4000, 700, 33, 1500], [1500, 1, 1, 1], 0),     # 57 GFLOP of chunk work: two streams
    ("bf16", (28, 4, 128), [4000, 700, 33], [800, 1, 1], 0),             # 50 GFLOP
    ("bf16", (28, 4, 128), [4000, 700, 33], [1500, 1, 1], 3000),         # 48 GFLOP within a window
    ("bf16", (28, 4, 128), [4000, 700, 33], [300, 1, 1], 0),             # 18 GFLOP: one stream
])
def test_mixed_step_equals_separate_steps(pkg, qd, heads, past, new, sw):
    import torch
    dev = torch.device("cuda:0")
    (Hq, Hkv, D), bs, B = heads, 32, len(past)
    print(f"case mixed fork {qd} {heads} past {past} new {new}", flush=True)
    gen = torch.Generator(device="cuda").manual_seed(3)
    dt = torch.float16 if qd == "f16" else torch.bfloat16
    past, new = np.array(past, np.int32), np.array(new, np.int32)
    nblk = (past + new + bs - 1) // bs
    table = np.random.default_rng(1).permutation(int(nblk.sum())).astype(np.int32)
    tab = np.split(table, np.cumsum(nblk)[:-1])
    shape = (len(table), Hkv, bs, D)
    kc = torch.randn(shape, generator=gen, device=dev).to(dt).view(torch.uint8)
    vc = torch.randn(shape, generator=gen, device=dev).to(dt).view(torch.uint8)
    T = int(new.sum())
    q = torch.randn(T, Hq * D, generator=gen, device=dev).to(dt)
    k, v = (torch.randn(T, Hkv * D, generator=gen, device=dev).to(dt) for _ in range(2))
    op = pkg.PagedAttention(Hq, Hkv, D, bs, qd, qd, 1, 0, torch.cuda.current_stream(dev))

    def step(which):
        rows = torch.cat([torch.arange(int(new[:b].sum()), int(new[:b + 1].sum())) for b in which]).to(dev)
        sb = np.concatenate([[0], np.cumsum(new[which])]).astype(np.int32)
        bib = np.concatenate([[0], np.cumsum(nblk[which])]).astype(np.int32)
        op.step_begin(past[which], sb, bib, int((past + new)[which].max()), None, sw, 0.0)
        op.set_block_indices(np.concatenate([tab[b] for b in which]), len(table))
        out = torch.zeros(len(rows), Hq * D, dtype=dt, device=dev)
        qi, ki, vi = (x[rows].contiguous() for x in (q, k, v))
        for _ in range(3):  # (later calls of the step next to the tail of earlier ones)
            op.forward(qi, ki, vi, kc, vc, out)
        op.synchronize()
        ran.append(op.kernels_run - {"fold"})
        scored = torch.zeros_like(out)
        scores = torch.full((op.total_scores,), float("nan"), dtype=torch.float32, device=dev)
        op.forward(qi, ki, vi, kc, vc, scored, scores)
        op.synchronize()
        assert op.kernels_run == ({"decode", "matrix", "side_stream"} if "matrix" in ran[-1] and "decode" in ran[-1] else ran[-1])
        H.assert_close(scored.float().cpu().numpy(), out.float().cpu().numpy(), qd, "outputs of the call with scores")
        return out.float().cpu().numpy(), scores.cpu().numpy()

    ran = []
    together, scores = step(list(range(B)))
    assert ran == [{"decode", "matrix", "side_stream"} if new[0] >= 800 else {"decode", "matrix"}]
    n0, s0 = int(new[0]), int(past[0] + new[0])
    # outputs of the same arithmetic cut into other ranges: both sides within the tolerance of the exact result
    for got, got_scores, which in ((together[:n0], scores[:s0], [0]), (together[n0:], scores[s0:], list(range(1, B)))):
        out, sc = step(which)
        H.assert_close(got, out, qd)
        H.assert_close(got_scores, sc, "f16", "scores")


@pytest.mark.parametrize("qd,Hq,Hkv,D,bs,past,new,sw,side", [
    ("f16", 8, 2, 128, 32, [6000, 300, 40, 200], [1, 1, 1, 70], 0, True), ("bf16", 8, 4, 64, 16, [90, 5000, 64, 0], [33, 1, 1, 5], 4500, True),
    ("bf16", 6, 2, 96, 64, [4200, 10], [1, 140], 0, False), ("f16", 4, 4, 128, 32, [4200, 4100, 10], [1, 1, 140], 0, False),
    ("f16", 8, 2, 128, 32, [3998, 30, 9], [1, 1, 64], 0, False), ("f16", 8, 2, 128, 32, [3999, 30, 9], [1, 1, 64], 0, True),
    ("f16", 8, 2, 128, 32, [9000, 30, 9], [1, 1, 64], 3000, False),
])
def test_mixed_step_beside_uneven_contexts(pkg, qd, Hq, Hkv, D, bs, past, new, sw, side):
    import torch
    print(f"case mixed uneven {qd} {Hq}/{Hkv} D{D} past {past} new {new} window {sw}", flush=True)
    case = H.build_case(H.case_from_lens("uneven", Hq, Hkv, D, bs, qd, qd, past, new, sw), seed=D + bs)
    ref = H.run_case_on_checker(case)
    got = H.run_case_on_gpu(pkg, case, torch.device("cuda:0"))
    assert got["op"].kernels_run == {"decode", "matrix", "side_stream"}  # (with scores: always)
    H.assert_close(got["out"], ref["out"], qd)
    H.assert_close(got["scores"], ref["scores"], "f16", "scores")
    plain = H.run_case_on_gpu(pkg, case, torch.device("cuda:0"), want_scores=False, op=got["op"])
    assert plain["op"].kernels_run - {"fold"} == {"decode", "matrix"} | ({"side_stream"} if side else set())
    H.assert_close(plain["out"], ref["out"], qd)
