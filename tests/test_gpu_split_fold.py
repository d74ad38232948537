"""Decode launches whose contexts are cut into splits and that fold the partials themselves (no scores): outputs against the CPU
checker, the same bits on every repeat, and inside a captured graph that is replayed."""
import numpy as np
import pytest

import harness as H

pytestmark = pytest.mark.gpu

CASES = [
    # (query type, cache type, block size, Hq, Hkv, D, past lengths, window)
    ("f16", "u8", 32, 8, 2, 128, [1117], 0), ("bf16", "u8", 16, 4, 4, 64, [900, 33, 0], 0), ("f16", "u8", 64, 12, 4, 96, [2000, 64], 0),
    ("bf16", "u8", 32, 16, 1, 256, [3000], 700), ("f16", "f16", 32, 14, 2, 128, [1500, 5], 0), ("bf16", "bf16", 16, 8, 8, 64, [64, 1030], 0),
    ("f16", "f16", 32, 16, 8, 256, [2500], 0), ("bf16", "bf16", 256, 6, 2, 96, [700, 701, 1], 600),
    ("f16", "u8", 32, 8, 1, 64, [4000], 0), ("bf16", "bf16", 32, 12, 1, 128, [1000, 40], 0),  # the most rows and splits a launch folds
    ("f16", "u8", 32, 16, 1, 128, [40000], 0), ("f16", "f16", 32, 7, 1, 128, [1990], 0),      # too many for that: a merge launch
    ("f16", "f16", 32, 16, 8, 128, [1000] * 37, 0),                                            # ... and of more than a round of workgroups
]


@pytest.mark.parametrize("qd,kd,bs,Hq,Hkv,D,past,sw", CASES)
def test_split_fold(pkg, qd, kd, bs, Hq, Hkv, D, past, sw):
    import torch
    dev = torch.device("cuda:0")
    print(f"case split fold {qd} {kd} bs{bs} {Hq}/{Hkv} D{D} past {past} window {sw}", flush=True)
    case = H.build_case(H.case_from_lens("fold", Hq, Hkv, D, bs, qd, kd, past, [1] * len(past), sw), seed=D + bs)
    ref = H.run_case_on_checker(case, want_scores=False)
    got = H.run_case_on_gpu(pkg, case, dev, want_scores=False)
    ns = got["op"].num_splits
    assert ns > 1
    # one workgroup's trips to the partials: 256 pairs of channels, eight splits each
    passes, trips = -(-(Hq // Hkv) * D // 512), -(-ns // 8)
    one_round = len(past) * Hkv * ns <= (256 if D > 128 else 512)
    assert ("fold" in got["op"].kernels_run) == (one_round and (trips <= 4 if passes == 1 else passes * trips <= 3)), (ns, passes, trips)
    H.assert_close(got["out"], ref["out"], qd)
    again = H.run_case_on_gpu(pkg, case, dev, want_scores=False, op=got["op"])
    assert np.array_equal(got["out16"], again["out16"])
    # with scores (the merge is then part of the score launch) and without, in turn on one context
    scored = H.run_case_on_gpu(pkg, case, dev, want_scores=True, op=got["op"])
    assert "fold" not in scored["op"].kernels_run
    H.assert_close(scored["out"], ref["out"], qd)
    assert np.array_equal(H.run_case_on_gpu(pkg, case, dev, want_scores=False, op=got["op"])["out16"], got["out16"])


def test_split_fold_in_a_graph(pkg):
    import torch
    dev = torch.device("cuda:0")
    case = H.build_case(H.case_from_lens("fold", 32, 8, 128, 32, "f16", "u8", [1117, 300], [1, 1]), seed=4)
    stream = torch.cuda.Stream(dev)
    with torch.cuda.stream(stream):
        op = pkg.PagedAttention(32, 8, 128, 32, "f16", "u8", 1, 0, stream)
        eager = H.run_case_on_gpu(pkg, case, dev, want_scores=False, op=op)
        assert op.num_splits > 1
        q, k, v = (H.to_device_16(torch, case[n], "f16", dev) for n in ("query", "key", "value"))
        kc, vc = (torch.from_numpy(case[n]).to(dev) for n in ("key_cache0", "value_cache0"))
        out = [torch.zeros_like(q) for _ in range(4)]
        torch.cuda.synchronize(dev)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            for o in out:
                op.forward(q, k, v, kc, vc, o)
        for i in range(4):
            for o in out:
                o.zero_()
            graph.replay()
            if i % 2:
                op.forward(q, k, v, kc, vc, out[0])
            torch.cuda.synchronize(dev)
            for o in out:
                assert np.array_equal(o.view(torch.int16).cpu().numpy().view(np.uint16), eager["out16"]), i


def test_split_fold_after_overlapping_launches(pkg):
    """Calls of one context must not overlap; ones that did (here a graph replayed on two streams, every launch the same values in
    the same places) leave the counters of the fold whole: what runs afterwards, alone, is right."""
    import torch
    dev = torch.device("cuda:0")
    case = H.build_case(H.case_from_lens("fold", 32, 8, 128, 32, "f16", "u8", [1117, 300], [1, 1]), seed=4)
    stream, other = torch.cuda.Stream(dev), torch.cuda.Stream(dev)
    with torch.cuda.stream(stream):
        op = pkg.PagedAttention(32, 8, 128, 32, "f16", "u8", 1, 0, stream)
        eager = H.run_case_on_gpu(pkg, case, dev, want_scores=False, op=op)
        assert "fold" in op.kernels_run
        q = H.to_device_16(torch, case["query"], "f16", dev)
        kc, vc = (torch.from_numpy(eager[n]).to(dev) for n in ("key_cache", "value_cache"))  # (the step's rows in place)
        out = torch.zeros_like(q)
        torch.cuda.synchronize(dev)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            for _ in range(20):
                op.attention(q, kc, vc, out)
        second = torch.cuda.CUDAGraph()
        with torch.cuda.graph(second, stream=stream):
            for _ in range(20):
                op.attention(q, kc, vc, out)
        for _ in range(5):
            graph.replay()
            with torch.cuda.stream(other):
                second.replay()
            torch.cuda.synchronize(dev)
        for _ in range(3):
            out.zero_()
            op.attention(q, kc, vc, out)
            torch.cuda.synchronize(dev)
            assert np.array_equal(out.view(torch.int16).cpu().numpy().view(np.uint16), eager["out16"])
