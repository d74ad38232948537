"""Steps whose sequences schedule a few tokens each over a u8 cache (the decode kernel's few-token variant) against the CPU checker,
with the calls beside them that stay on the matrix kernel: scores wanted, one row too many, block-sparse sequences."""
import numpy as np
import pytest

import harness as H
from oracle import oracle as O

pytestmark = pytest.mark.gpu

CASES = [
    # (query type, block size, Hq, Hkv, D, past lengths, new tokens, window): one and two column groups, tile edges between a
    # sequence's tokens (a wave whose first tile the early tokens do not see), single tokens beside, one split and several
    ("f16", 32, 32, 8, 128, [500, 31, 0, 1290], [5, 5, 5, 5], 0), ("bf16", 16, 8, 2, 128, [30, 31, 63, 15, 2200], [4, 3, 2, 4, 1], 0),
    ("f16", 64, 4, 4, 64, [29, 4000], [32, 17], 0), ("bf16", 256, 16, 1, 64, [255, 700], [2, 1], 40), ("f16", 32, 8, 8, 128, [124], [16], 0),
    ("f16", 32, 6, 2, 64, [95, 300, 64], [5, 5, 1], 33), ("bf16", 32, 40, 8, 128, [64] * 40, [6] * 40, 0), ("f16", 16, 7, 1, 128, [9000], [4], 0),
    # 33 rows and more: the matrix kernel's
    ("f16", 32, 3, 1, 128, [100, 40], [11, 2], 0), ("f16", 32, 4, 2, 96, [70, 40], [3, 2], 0),
]


@pytest.mark.parametrize("qd,bs,Hq,Hkv,D,past,new,sw", CASES)
def test_decode_few(pkg, qd, bs, Hq, Hkv, D, past, new, sw):
    import torch
    dev = torch.device("cuda:0")
    print(f"case decode few {qd} bs{bs} {Hq}/{Hkv} D{D} past {past[:5]} new {new[:5]} window {sw}", flush=True)
    case = H.build_case(H.case_from_lens("few", Hq, Hkv, D, bs, qd, "u8", past, new, sw), seed=D + bs + len(past), outliers=True)
    ref = H.run_case_on_checker(case)
    got = H.run_case_on_gpu(pkg, case, dev, want_scores=False)
    assert np.array_equal(got["key_cache"], ref["key_cache"]) and np.array_equal(got["value_cache"], ref["value_cache"])
    few = D in (64, 128) and max(new) * Hq // Hkv <= 32
    assert got["op"].kernels_run - {"fold"} == ({"decode_few"} if few else {"matrix"} if 1 not in new else {"matrix", "decode", "side_stream"})
    H.assert_close(got["out"], ref["out"], qd)
    scored = H.run_case_on_gpu(pkg, case, dev, op=got["op"])
    assert "matrix" in scored["op"].kernels_run and "decode_few" not in scored["op"].kernels_run
    H.assert_close(scored["out"], ref["out"], qd)
    H.assert_close(scored["scores"], ref["scores"], "f16", "scores")
    again = H.run_case_on_gpu(pkg, case, dev, want_scores=False, op=got["op"])
    assert np.array_equal(again["out16"], got["out16"])


def test_decode_few_beside_xattention(pkg):
    """Thresholds set and taken back between the table's upload and the layer calls: every order gives the step's result."""
    import torch
    dev = torch.device("cuda:0")
    case = H.build_case(H.case_from_lens("few", 8, 2, 128, 32, "f16", "u8", [300, 70], [4, 3]), seed=2)
    ref = H.run_case_on_checker(case, want_scores=False)
    op = pkg.PagedAttention(8, 2, 128, 32, "f16", "u8", 1, 0, torch.cuda.current_stream(dev))
    q, k, v = (H.to_device_16(torch, case[n], "f16", dev) for n in ("query", "key", "value"))
    for order in ("table", "set table", "set table back", "table set", "table set back"):
        kc, vc = (torch.from_numpy(case[n]).to(dev) for n in ("key_cache0", "value_cache0"))
        out = torch.zeros_like(q)
        op.step_begin(case["past_lens"], case["subsequence_begins"], case["block_indices_begins"], 304, None, 0, case["scale"])
        for what in order.split():
            if what == "table":
                op.set_block_indices(case["block_indices"], case["num_blocks"])
            else:  # (a threshold of 1 keeps every block)
                op.set_xattention(np.ones(2, np.float32) if what == "set" else None, 64, 8)
        op.forward(q, k, v, kc, vc, out)
        op.synchronize()
        assert op.kernels_run - {"fold"} == ({"matrix"} if order.endswith("set") or order == "set table" else {"decode_few"})
        H.assert_close(out.float().cpu().numpy(), ref["out"], "f16", order)


def test_decode_few_layer_tables_beside_xattention(pkg):
    """Per-layer tables uploaded in several calls with thresholds set and taken back between them: every layer keeps its own."""
    import torch
    dev = torch.device("cuda:0")
    layers = 6
    case = H.build_case(H.case_from_lens("few", 8, 2, 128, 32, "f16", "u8", [300, 70, 2000], [4, 3, 2]), seed=9)
    ref = H.run_case_on_checker(case, want_scores=False)
    op = pkg.PagedAttention(8, 2, 128, 32, "f16", "u8", layers, 0, torch.cuda.current_stream(dev))
    q, k, v = (H.to_device_16(torch, case[n], "f16", dev) for n in ("query", "key", "value"))
    ids, n_blocks = case["block_indices"], case["num_blocks"]
    rng = np.random.default_rng(0)
    moved = [rng.permutation(n_blocks) for _ in range(layers)]  # layer l holds block i of the case as block moved[l][i]
    for order in ((True, False), (False, True)):
        op.step_begin(case["past_lens"], case["subsequence_begins"], case["block_indices_begins"], 2002, None, 0, case["scale"])
        for half, on in zip((0, 3), order):
            op.set_xattention(np.ones(3, np.float32) if on else None, 64, 8)  # (a threshold of 1 keeps every block)
            op.set_block_indices_per_layer([moved[l][ids] for l in range(half, half + 3)], n_blocks, half)
        for l in range(layers):
            kc, vc = (torch.zeros(case[n].shape, dtype=torch.uint8, device=dev) for n in ("key_cache0", "value_cache0"))
            at = torch.from_numpy(moved[l]).to(dev)
            kc[at], vc[at] = (torch.from_numpy(case[n]).to(dev) for n in ("key_cache0", "value_cache0"))
            out = torch.zeros_like(q)
            op.forward(q, k, v, kc, vc, out, layer=l)
            op.synchronize()
            H.assert_close(out.float().cpu().numpy(), ref["out"], "f16", f"layer {l} {order}")


@pytest.mark.parametrize("qd,Hq,Hkv,D,past,new", [("f16", 16, 4, 128, [3000, 700], [5, 4]), ("f16", 16, 4, 128, [4000], [3]),
                                                  ("f16", 16, 4, 64, [2000, 100], [8, 2]), ("bf16", 32, 8, 128, [3000, 700], [5, 4]),
                                                  ("bf16", 32, 8, 64, [3000, 700], [4, 3])])
def test_decode_few_error_against_64_bits(pkg, qd, Hq, Hkv, D, past, new):
    """No further from the binary64 result than the matrix kernel, which the same step's call with scores runs on."""
    import torch
    dev = torch.device("cuda:0")
    print(f"case decode few error {qd} {Hq}/{Hkv} D{D} past {past} new {new}", flush=True)
    case = H.build_case(H.case_from_lens("few", Hq, Hkv, D, 32, qd, "u8", past, new), seed=D + Hq, outliers=True)
    few = H.run_case_on_gpu(pkg, case, dev, want_scores=False)
    assert few["op"].kernels_run - {"fold"} == {"decode_few"}
    matrix = H.run_case_on_gpu(pkg, case, dev, op=few["op"])
    assert "matrix" in matrix["op"].kernels_run
    exact = H.attention_f64(O.from_bits(case["query"], H.DT[qd]), few["key_cache"], few["value_cache"], 255, case["past_lens"],
                            case["subsequence_begins"], case["block_indices_begins"], case["block_indices"], Hq, Hkv, D, 32)
    ours, theirs = H.misrounded(few["out"], exact, qd), H.misrounded(matrix["out"], exact, qd)
    print(f"misrounded {ours} against {theirs} of {exact.size}", flush=True)
    assert ours <= theirs + 4 * np.sqrt(theirs + 1)  # (counts of rare independent events: four standard deviations)


@pytest.mark.parametrize("qd,D,bs,new", [("f16", 128, 32, [4, 2, 1]), ("bf16", 64, 16, [3, 8, 2])])
def test_decode_few_ignores_garbage_beyond_the_context(pkg, qd, D, bs, new):
    """Rows behind a sequence's last token may hold anything, NaN headers included."""
    import torch
    past = [40, 90, 2001]
    print(f"case decode few garbage {qd} D{D} bs{bs}", flush=True)
    case = H.build_case(H.case_from_lens("few", 8, 2, D, bs, qd, "u8", past, new), seed=6)
    ref = H.run_case_on_checker(case, want_scores=False)
    H.spoil_rows_beyond_the_context(case)
    got = H.run_case_on_gpu(pkg, case, torch.device("cuda:0"), want_scores=False)
    assert got["op"].kernels_run - {"fold"} == {"decode_few"}
    H.assert_close(got["out"], ref["out"], qd)


@pytest.mark.parametrize("vmul", [2.0 ** -60, 2.0 ** 14, 2.0 ** 60])
def test_decode_few_magnitudes(pkg, vmul):
    """bf16 values far outside f16's range: the rows' V scales times a power of two give outputs times it."""
    import torch
    dev = torch.device("cuda:0")
    print(f"case decode few magnitudes V x {vmul}", flush=True)
    case = H.build_case(H.case_from_lens("few", 8, 2, 128, 32, "bf16", "u8", [640, 77], [3, 5]), seed=5)
    plain = H.run_case_on_gpu(pkg, case, dev, want_scores=False)
    vc = case["value_cache0"].copy()
    vc[..., :4] = (np.ascontiguousarray(vc[..., :4]).view(np.float32) * np.float32(vmul)).view(np.uint8)
    value = O.to_bits(O.from_bits(case["value"], H.DT["bf16"]) * np.float32(vmul), H.DT["bf16"])
    got = H.run_case_on_gpu(pkg, dict(case, value_cache0=vc, value=value), dev, want_scores=False)
    # every scaling is exact and each sum goes along with it: only a tile's unit can differ
    assert np.abs(got["out"] / np.float32(vmul) - plain["out"]).max() <= 2.0 ** -8 * np.abs(plain["out"]).max()


@pytest.mark.parametrize("qd,bs,Hq,Hkv,D,past,new,sw", [
    ("f16", 32, 32, 8, 128, [4000, 30, 0, 95], [5, 5, 5, 1], 0), ("bf16", 16, 8, 2, 64, [15, 700], [8, 3], 0),
    ("f16", 64, 4, 4, 64, [31, 4000], [32, 1], 40), ("bf16", 256, 4, 1, 128, [254, 9000], [4, 4], 0)])
@pytest.mark.parametrize("shared", [False, True])
def test_append_in_the_few_token_kernel(pkg, qd, bs, Hq, Hkv, D, past, new, sw, shared):
    """pa_forward against its two halves, bit for bit; `shared`: a sequence more whose past is the first one's context, the rows that
    the same step writes included (its own new rows go behind them or into a block of its own)."""
    import torch
    dev = torch.device("cuda:0")
    case = H.build_case(H.case_from_lens("few", Hq, Hkv, D, bs, qd, "u8", past + [past[0] + new[0]] * shared, new + [2] * shared, sw), seed=bs)
    ids, bib = case["block_indices"].copy(), case["block_indices_begins"]
    if shared:
        n = -(-(past[0] + new[0]) // bs)
        ids[bib[-2]:bib[-2] + n] = ids[:n]
    q, k, v = (H.to_device_16(torch, case[x], qd, dev) for x in ("query", "key", "value"))
    got = []
    for halves in (False, True):
        op = pkg.PagedAttention(Hq, Hkv, D, bs, qd, "u8", 1, 0, torch.cuda.current_stream(dev))
        kc, vc = (torch.from_numpy(case[x]).to(dev) for x in ("key_cache0", "value_cache0"))
        out = torch.zeros_like(q)
        op.step_begin(case["past_lens"], case["subsequence_begins"], bib, int((case["past_lens"] + case["new_lens"]).max()), None, sw, case["scale"])
        op.set_block_indices(ids, case["num_blocks"])
        if halves:
            op.kv_append(k, v, kc, vc)
            op.attention(q, kc, vc, out)
        else:
            op.forward(q, k, v, kc, vc, out)
        op.synchronize()
        assert "decode_few" in op.kernels_run and ("append" in op.launches_ahead) == (shared and not halves)
        got.append((out.view(torch.int16).cpu(), kc.cpu(), vc.cpu()))
    for a, b in zip(*got):
        assert torch.equal(a, b)


def test_append_in_the_few_token_kernel_by_layer(pkg):
    """A table per layer: only the layer in which one sequence reads a block that another one writes has an append launch."""
    import torch
    dev = torch.device("cuda:0")
    print("case few append by layer", flush=True)
    case = H.build_case(H.case_from_lens("few", 16, 4, 128, 32, "f16", "u8", [700, 705, 33], [5, 2, 1]), seed=2)
    ids, bib = case["block_indices"], case["block_indices_begins"]
    shared = ids.copy()
    shared[bib[1]:bib[1] + 22] = ids[:22]  # (positions 0 .. 703; the first sequence's new rows start at 700)
    q, k, v = (H.to_device_16(torch, case[x], "f16", dev) for x in ("query", "key", "value"))
    got = []
    for halves in (False, True):
        op = pkg.PagedAttention(16, 4, 128, 32, "f16", "u8", 3, 0, torch.cuda.current_stream(dev))
        op.step_begin(case["past_lens"], case["subsequence_begins"], bib, 707, None, 0, case["scale"])
        op.set_block_indices_per_layer([ids, shared, ids], case["num_blocks"])
        for layer in range(3):
            kc, vc = (torch.from_numpy(case[x]).to(dev) for x in ("key_cache0", "value_cache0"))
            out = torch.zeros_like(q)
            if halves:
                op.kv_append(k, v, kc, vc, layer)
                op.attention(q, kc, vc, out, layer=layer)
            else:
                op.forward(q, k, v, kc, vc, out, layer=layer)
                assert ("append" in op.launches_ahead) == (layer == 1)
            op.synchronize()
            assert "decode_few" in op.kernels_run
            got.append((out.view(torch.int16).cpu(), kc.cpu(), vc.cpu()))
    for a, b in zip(got[:3], got[3:]):
        assert all(torch.equal(x, y) for x, y in zip(a, b))
