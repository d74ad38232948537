"""Steps prepared while the ones before them still run: nothing of a step may reach the device's copies of an earlier one."""
import numpy as np
import pytest
import torch

import harness as H

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kd,new,blocks", [("u8", 1, 400), ("u8", 5, 400), ("f16", 1, 400), ("f16", 40, 400), ("u8", 1, 60000)])
def test_steps_queued_ahead(pkg, kd, new, blocks):
    """Twelve steps of other lengths and block tables without a wait in between (the last case's tables outgrow the staging area
    again and again) give what each gives by itself."""
    dev = torch.device("cuda:0")
    print(f"case steps ahead {kd} new {new} blocks {blocks}", flush=True)
    rng = np.random.default_rng(new + blocks)
    op = pkg.PagedAttention(8, 2, 128, 32, "f16", kd, 1, 0, torch.cuda.current_stream(dev))
    gen = torch.Generator(device=dev).manual_seed(1)
    kc, vc = (torch.zeros(blocks, 2, 32, pkg.row_bytes(128, kd), dtype=torch.uint8, device=dev) for _ in range(2))
    n = 32 * 40  # rows 0 .. n - 1 of the pool's first forty blocks hold numbers
    op.step_begin(np.zeros(1, np.int32), np.array([0, n], np.int32), np.array([0, 40], np.int32))
    op.set_block_indices(np.arange(40, dtype=np.int32), blocks)
    k0, v0 = (torch.randn(n, 256, generator=gen, device=dev).half() for _ in range(2))
    op.kv_append(k0, v0, kc, vc)
    op.synchronize()
    extra = 20000 if blocks > 1000 else 0  # ids behind a sequence's own: part of its table, never read
    steps = []
    for i in range(12):
        B = int(rng.integers(1, 7))
        past = rng.integers(1, 200, B).astype(np.int32)
        bib = np.concatenate([[0], np.cumsum((past + new + 31) // 32 + extra)]).astype(np.int32)
        ids = np.concatenate([np.concatenate([rng.permutation(40)[:(p + new + 31) // 32], rng.integers(0, blocks, extra)]) for p in past]).astype(np.int32)
        steps.append((past, (np.arange(B + 1) * new).astype(np.int32), bib, ids))
    q, k, v = (torch.randn(6 * new, w, generator=gen, device=dev).half() for w in (1024, 256, 256))

    def run(wait):
        out = torch.zeros(12, 6 * new, 1024, dtype=torch.float16, device=dev)
        ahead = 0
        for i, (past, sb, bib, ids) in enumerate(steps):
            if not wait and i % 4 == 0:
                keep_busy(dev)
            before = torch.cuda.Event()
            before.record()
            op.step_begin(past, sb, bib)
            op.set_block_indices(ids, blocks)
            ahead += not before.query()
            op.attention(q[:sb[-1]], kc, vc, out[i, :sb[-1]])
            if wait:
                op.synchronize()
        op.synchronize()
        # (the large tables wait for the staging area)
        assert wait or blocks > 1000 or ahead >= 3
        return out

    one_by_one = run(True)  # (first: buffers that grow wait for the stream)
    assert torch.equal(run(False), one_by_one)


def keep_busy(dev):
    """Some tens of milliseconds of work on the current stream: what a step queues behind it stays queued while the next one is
    prepared, which has to wait for it, and the one after that, whose arrays take the first one's part of the staging area."""
    x = torch.ones(8192, 8192, dtype=torch.bfloat16, device=dev)
    for _ in range(20):
        x = torch.mm(x, x) * 0.0
    return x


@pytest.mark.parametrize("kd,new,kind", [("u8", [1] * 5, "append"), ("u8", [3, 1, 5, 2], "append"), ("f16", [1] * 4, "append"),
                                         ("u8", [1, 1, 300, 1], "mixed"), ("f16", [400, 700], "thresholds"), ("f16", [1, 500, 1], "tables")])
def test_forwards_queued_ahead(pkg, kd, new, kind):
    """The same through forward, with its appends, scores every other step, both kernels side by side, thresholds and a table per layer:
    outputs, scores and cache rows of steps prepared behind a stream that is still busy are those of steps taken one by one."""
    dev = torch.device("cuda:0")
    print(f"case forwards ahead {kd} new {new} {kind}", flush=True)
    rng = np.random.default_rng(len(new))
    op = pkg.PagedAttention(8, 2, 128, 32, "f16", kd, 2, 0, torch.cuda.current_stream(dev))
    gen = torch.Generator(device=dev).manual_seed(2)
    n, B, blocks = sum(new), len(new), 400
    q, k, v = (torch.randn(n, w, generator=gen, device=dev).half() for w in (1024, 256, 256))
    empty = torch.zeros(2, blocks, 2, 32, pkg.row_bytes(128, kd), dtype=torch.uint8, device=dev)
    steps = []
    for i in range(8):
        past = rng.integers(0, 600, B).astype(np.int32)
        bib = np.concatenate([[0], np.cumsum((past + new + 31) // 32)]).astype(np.int32)
        steps.append((past, bib, [rng.permutation(blocks)[:bib[-1]].astype(np.int32) for _ in range(2)]))
    sb = np.concatenate([[0], np.cumsum(new)]).astype(np.int32)

    def run(wait):
        kc, vc = empty.clone(), empty.clone()
        out = torch.zeros(8, 2, n, 1024, dtype=torch.float16, device=dev)
        scores = torch.zeros(8, 2, n + 600 * B, device=dev)
        ahead = 0
        for i, (past, bib, tables) in enumerate(steps):
            if not wait and i % 4 == 0:
                keep_busy(dev)
            before = torch.cuda.Event()
            before.record()
            op.step_begin(past, sb, bib)
            if kind == "thresholds":
                op.set_xattention([0.8] * B, 64, 8)
            if kind == "tables":
                op.set_block_indices_per_layer(tables, blocks)
            else:
                op.set_block_indices(tables[0], blocks)
            ahead += not before.query()
            for layer in range(2):
                op.forward(q, k, v, kc[layer], vc[layer], out[i, layer], scores[i, layer] if i % 2 else None, layer=layer)
            if wait:
                op.synchronize()
        op.synchronize()
        assert wait or ahead >= 2
        return out, scores, kc, vc

    one_by_one = run(True)
    for ours, theirs in zip(run(False), one_by_one):
        assert torch.equal(ours, theirs)


def test_step_begin_is_refused_under_capture(pkg):
    case = H.build_case(H.tiny_decode_case(), seed=7)
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        op = pkg.PagedAttention(case["Hq"], case["Hkv"], case["D"], case["bs"], case["q_dtype"], case["kv_dtype"], 1, 0, side)
        op.step_begin(case["past_lens"], case["subsequence_begins"], case["block_indices_begins"])
        graph = torch.cuda.CUDAGraph()
        graph.capture_begin()
        try:
            with pytest.raises(Exception):
                op.step_begin(case["past_lens"], case["subsequence_begins"], case["block_indices_begins"])
        finally:
            graph.capture_end()
    op.step_begin(case["past_lens"], case["subsequence_begins"], case["block_indices_begins"])
    op.synchronize()
