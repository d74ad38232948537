"""A mixed step over a 16-bit cache whose chunk is long enough for matrix and decode kernel to run side by side (and one below that)
against the same sequences in steps of their own."""
import numpy as np
import pytest

import harness as H

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("qd,heads,past,new", [
    ("f16", (32, 4, 64), [4000, 700, 33, 1500], [1500, 1, 1, 1]),   # 57 GFLOP of chunk work: two streams
    ("bf16", (28, 4, 128), [4000, 700, 33], [800, 1, 1]),           # 50 GFLOP
    ("bf16", (28, 4, 128), [4000, 700, 33], [300, 1, 1]),           # 18 GFLOP: one stream
])
def test_mixed_step_equals_separate_steps(pkg, qd, heads, past, new):
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
        op.step_begin(past[which], sb, bib, int((past + new)[which].max()), None, 0, 0.0)
        op.set_block_indices(np.concatenate([tab[b] for b in which]), len(table))
        out = torch.zeros(len(rows), Hq * D, dtype=dt, device=dev)
        qi, ki, vi = (x[rows].contiguous() for x in (q, k, v))
        for _ in range(3):  # (later calls of the step next to the tail of earlier ones)
            op.forward(qi, ki, vi, kc, vc, out)
        op.synchronize()
        ran.append(op.kernels_run - {"fold"})
        return out.float().cpu().numpy()

    ran = []
    together = step(list(range(B)))
    assert ran == [{"decode", "matrix", "side_stream"} if new[0] >= 800 else {"decode", "matrix"}]
    n0 = int(new[0])
    # outputs of the same arithmetic cut into other ranges: both sides within the tolerance of the exact result
    H.assert_close(together[:n0], step([0]), qd)
    H.assert_close(together[n0:], step(list(range(1, B))), qd)
