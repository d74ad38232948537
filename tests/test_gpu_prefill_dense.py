"""The straight-to-LDS matrix kernel (dense chunks, head size 128) against the CPU checker: 16-bit caches, and steps over u8 caches
large enough that their rows are widened beforehand."""
import numpy as np
import pytest

import harness as H
from oracle import oracle as O

pytestmark = pytest.mark.gpu

CASES = [
    # (query type, cache type, block size, Hq, Hkv, past lengths, new tokens, window)
    # 16-bit: one row, a wave's rows, a tile's, one more; a last block of 1, 31 and 32 tokens; two and three tiles of one block
    ("f16", "f16", 32, 4, 2, [0], [2], 0), ("bf16", "bf16", 16, 16, 1, [30], [3], 0), ("f16", "f16", 16, 7, 1, [95, 64], [19, 18], 0),
    ("bf16", "bf16", 256, 8, 8, [200, 31], [129, 33], 0), ("f16", "f16", 64, 8, 2, [4097], [40], 100),
    ("bf16", "bf16", 128, 12, 4, [0, 5000, 17], [130, 47, 64], 0), ("bf16", "bf16", 32, 128, 1, [60], [5], 33),
    # u8, too little work to be widened
    ("f16", "u8", 256, 16, 2, [31], [900], 0), ("bf16", "u8", 32, 32, 2, [2100, 1], [560, 50], 777),
]
WIDENED = [
    # u8, widened: one sequence and several beside single tokens, every kind of block; windows that start inside a block, so that the
    # rows widened do not start at a sequence's first
    ("f16", "u8", 32, 16, 1, [300], [1101], 0), ("bf16", "u8", 16, 16, 1, [1000, 0], [517, 800], 0),
    ("f16", "u8", 64, 64, 2, [700, 90, 40], [331, 1, 400], 0), ("f16", "u8", 256, 16, 1, [31], [1400], 0),
    ("bf16", "u8", 32, 32, 2, [2100, 3000, 5], [900, 203, 1], 777), ("f16", "u8", 16, 16, 1, [1500, 0, 4000], [700, 500, 300], 1001),
    ("f16", "u8", 128, 128, 1, [1000, 333], [400, 150], 250),
]


@pytest.mark.parametrize("qd,kd,bs,Hq,Hkv,past,new,sw", CASES + WIDENED)
def test_prefill_dense(pkg, qd, kd, bs, Hq, Hkv, past, new, sw):
    import torch
    dev = torch.device("cuda:0")
    print(f"case dense {qd}/{kd} bs{bs} {Hq}/{Hkv} past {past} new {new} window {sw}", flush=True)
    case = H.build_case(H.case_from_lens("dense", Hq, Hkv, 128, bs, qd, kd, past, new, sw), seed=bs + Hq + len(past), outliers=True)
    ref = H.run_case_on_checker(case)
    H.spoil_rows_beyond_the_context(case)
    got = H.run_case_on_gpu(pkg, case, dev)
    assert ("widen" in got["op"].launches_ahead) == ((qd, kd, bs, Hq, Hkv, past, new, sw) in WIDENED)
    H.assert_close(got["out"], ref["out"], qd)
    H.assert_close(got["scores"], ref["scores"], "f16", "scores")
    again = H.run_case_on_gpu(pkg, case, dev, want_scores=False, op=got["op"])
    assert np.array_equal(again["out16"], got["out16"])


def test_prefill_dense_widened_error_against_64_bits(pkg):
    """No further from the binary64 result than the kernel that widens codes on their way to LDS, which takes the same rows as
    chunks too short to be widened."""
    import torch
    dev = torch.device("cuda:0")
    whole = H.build_case(H.case_from_lens("dense", 16, 1, 128, 32, "f16", "u8", [0], [1400], 0), seed=4, outliers=True)
    got = H.run_case_on_gpu(pkg, whole, dev, want_scores=False)
    assert "widen" in got["op"].launches_ahead
    exact = H.attention_f64(O.from_bits(whole["query"], H.DT["f16"]), got["key_cache"], got["value_cache"], 255, whole["past_lens"],
                            whole["subsequence_begins"], whole["block_indices_begins"], whole["block_indices"], 16, 1, 128, 32)
    op = pkg.PagedAttention(16, 1, 128, 32, "f16", "u8", 1, 0, torch.cuda.current_stream(dev))
    q, k, v = (H.to_device_16(torch, whole[n], "f16", dev) for n in ("query", "key", "value"))
    kc, vc = (torch.zeros(whole[n].shape, dtype=torch.uint8, device=dev) for n in ("key_cache0", "value_cache0"))
    out = torch.zeros_like(q)
    for t in range(0, 1400, 200):
        op.step_begin(np.array([t], np.int32), np.array([0, 200], np.int32), whole["block_indices_begins"], t + 200, None, 0, whole["scale"])
        op.set_block_indices(whole["block_indices"], whole["num_blocks"])
        op.forward(q[t:t + 200], k[t:t + 200], v[t:t + 200], kc, vc, out[t:t + 200])
        assert "widen" not in op.launches_ahead
    op.synchronize()
    ours, theirs = H.misrounded(got["out"], exact, "f16"), H.misrounded(out.float().cpu().numpy(), exact, "f16")
    print(f"misrounded {ours} against {theirs} of {exact.size}", flush=True)
    assert ours <= theirs + 4 * np.sqrt(theirs + 1)  # (counts of rare independent events: four standard deviations)


def test_prefill_dense_infinity_in_the_last_row(pkg):
    """The rows behind a sequence's tokens stand for nothing: an infinite V element of the last token stays infinite for it.  (f16:
    its low halves come only where a token leans on few others; a bf16 weight always is a high half and a low one, which may be
    negative or zero, and then an infinity times both has no value.)"""
    import torch
    case = H.build_case(H.case_from_lens("dense", 4, 2, 128, 32, "f16", "f16", [50], [41], 0), seed=8)
    value = O.from_bits(case["value"], H.DT["f16"]).reshape(41, 2, 128)
    value[-1, :, 5] = np.inf
    got = H.run_case_on_gpu(pkg, dict(case, value=O.to_bits(value.reshape(41, -1), H.DT["f16"])), torch.device("cuda:0"), want_scores=False)
    assert np.all(np.isposinf(got["out"].reshape(41, 4, 128)[-1, :, 5]))
