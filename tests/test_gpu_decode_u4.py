"""Steps of single-token sequences over u4 caches (the u4 variant of the decode kernel) against the CPU checker: cache rows
bit-exact, outputs and scores within tolerance; and the steps next to them that stay on the shape-generic kernels."""
import numpy as np
import pytest

import harness as H
from oracle import oracle as O
from test_gpu_generic_shapes import _case

pytestmark = pytest.mark.gpu

CASES = [
    # (query type, D, block size, Hq, Hkv, past lengths, window): tile edges (31 / 32 / 33 positions), one token, several splits,
    # the late append (a sequence's last tile not among the wave's first ones), groups of 1 to 16 heads
    ("f16", 128, 32, 8, 2, [0, 31, 32, 63, 1100], 0), ("bf16", 128, 16, 32, 8, [15, 16, 17, 2500], 0),
    ("bf16", 128, 256, 16, 1, [700, 1], 300), ("f16", 64, 32, 5, 5, [4097, 40], 0), ("bf16", 64, 16, 12, 4, [300, 95, 96], 33),
    ("f16", 256, 32, 16, 8, [500, 1023], 0), ("bf16", 256, 64, 4, 1, [5000], 4096), ("bf16", 128, 32, 4, 4, [127] * 70, 0),
    # left on the shape-generic kernels: 16-token blocks at head size 256, more than 16 heads per kv head, head size 96
    ("f16", 256, 16, 4, 2, [200, 33], 0), ("bf16", 128, 32, 34, 2, [90], 0), ("f16", 96, 32, 4, 2, [161], 0),
]


KERNELS = []  # of the last call


def _run(pkg, torch, c, qd, D, bs, Hq, Hkv, sw, scores_too, forward=True, slopes=None):
    dev = torch.device("cuda:0")
    op = pkg.PagedAttention(Hq, Hkv, D, bs, qd, "u4", 1, 0, torch.cuda.current_stream(dev))
    if slopes is not None:
        op.set_alibi_slopes(slopes)
    q, k, v = (H.to_device_16(torch, c[n], qd, dev) for n in ("q", "k", "v"))
    kc, vc = torch.from_numpy(c["kc"]).to(dev), torch.from_numpy(c["vc"]).to(dev)
    out = torch.zeros_like(q)
    op.step_begin(c["past"], c["sb"], c["bib"], int((c["past"] + c["new"]).max()), None, sw, 0.0)
    op.set_block_indices(c["table"], c["pool"])
    scores = torch.full((op.total_scores,), float("nan"), dtype=torch.float32, device=dev) if scores_too else None
    if forward:
        op.forward(q, k, v, kc, vc, out, scores)
    else:
        op.kv_append(k, v, kc, vc)
        op.attention(q, kc, vc, out, scores)
    op.synchronize()
    KERNELS[:] = [op.kernels_run - {"fold"}]
    return out.float().cpu().numpy(), scores.cpu().numpy() if scores_too else None, kc.cpu().numpy(), vc.cpu().numpy()


def _checked(c, D, bs, Hq, Hkv, sw):
    kc, vc = c["kc"].copy(), c["vc"].copy()
    O.kv_append_kv(c["k"], c["v"], c["qdt"], kc, vc, c["kdt"], c["vdt"], c["past"], c["sb"], c["table"], c["bib"], Hkv, D, D, bs)
    W = np.ones(len(c["past"]), np.int32)
    out, _, sc = O.paged_attention_kv(c["q"], c["qdt"], kc, vc, c["kdt"], c["vdt"], c["past"], c["sb"], c["table"], c["bib"], Hq,
                                      Hkv, D, D, bs, float(1.0 / np.sqrt(D)), sw, W, True, 8)
    return out, sc, kc, vc


@pytest.mark.parametrize("qd,D,bs,Hq,Hkv,past,sw", CASES)
def test_decode_u4(pkg, qd, D, bs, Hq, Hkv, past, sw):
    import torch
    print(f"case decode u4 {qd} D{D} bs{bs} {Hq}/{Hkv} past {past[:5]} window {sw}", flush=True)
    c = _case(np.random.default_rng(D + bs + Hq), qd, D, D, "u4", "u4", bs, Hq, Hkv, past, [1] * len(past))
    ref = _checked(c, D, bs, Hq, Hkv, sw)
    for scores_too, forward in ((True, True), (False, True), (True, False)):
        got = _run(pkg, torch, c, qd, D, bs, Hq, Hkv, sw, scores_too, forward)
        assert KERNELS == [{"generic"} if (D, bs) == (256, 16) or D == 96 or Hq > 16 * Hkv else {"decode"}]
        assert np.array_equal(got[2], ref[2]) and np.array_equal(got[3], ref[3]), "cache bytes differ"
        H.assert_close(got[0], ref[0], qd)
        if scores_too:  # (no rounding to 16 bits on the way: sums of at most Hq probabilities in binary32)
            assert np.abs(got[1] - ref[1]).max() <= 1e-5 * Hq


@pytest.mark.parametrize("qd,D,bs", [("f16", 128, 32), ("bf16", 64, 16), ("bf16", 256, 64)])
def test_decode_u4_ignores_garbage_beyond_the_context(pkg, qd, D, bs):
    """Rows behind a sequence's last token may hold anything, NaN headers included."""
    import torch
    print(f"case decode u4 garbage {qd} D{D} bs{bs}", flush=True)
    c = _case(np.random.default_rng(8), qd, D, D, "u4", "u4", bs, 8, 2, [40, 90, 2001], [1, 1, 1])
    ref = _checked(c, D, bs, 8, 2, 0)
    H.spoil_rows_beyond_the_context(dict(bs=bs, num_blocks=c["pool"], past_lens=c["past"], new_lens=c["new"], block_indices=c["table"],
                                         block_indices_begins=c["bib"], key_cache0=c["kc"], value_cache0=c["vc"]))
    got = _run(pkg, torch, c, qd, D, bs, 8, 2, 0, True)
    assert KERNELS == [{"decode"}]
    H.assert_close(got[0], ref[0], qd)
    assert np.abs(got[1] - ref[1]).max() <= 1e-5 * 8


@pytest.mark.parametrize("vmul,qmul", [(2.0 ** -40, 1.0), (2.0 ** 30, 1.0), (1.0, 2.0 ** 20), (1.0, 2.0 ** -30)])
def test_decode_u4_magnitudes(pkg, vmul, qmul):
    """bf16 values far outside f16's range: V scaled by a power of two gives outputs scaled by it, and queries scaled by one
    (against keys scaled back) give the same outputs."""
    import torch
    D, bs, Hq, Hkv, past = 128, 32, 8, 2, [77, 640]
    print(f"case decode u4 magnitudes V x {vmul} q x {qmul}", flush=True)
    c = _case(np.random.default_rng(3), "bf16", D, D, "u4", "u4", bs, Hq, Hkv, past, [1, 1])

    def scaled(bits, f):
        return O.to_bits((bits.astype(np.uint32) << 16).view(np.float32) * np.float32(f), c["qdt"])

    def scaled_cache(cache, f):  # (the rows' scales; zero-points and codes stay)
        out = cache.copy()
        hdr = out[..., :4].copy().view(np.float32) * np.float32(f)
        out[..., :4] = hdr.view(np.uint8)
        return out

    plain = _run(pkg, torch, c, "bf16", D, bs, Hq, Hkv, 0, True)
    d = dict(c, v=scaled(c["v"], vmul), q=scaled(c["q"], qmul), k=scaled(c["k"], 1.0 / qmul),
             vc=scaled_cache(c["vc"], vmul), kc=scaled_cache(c["kc"], 1.0 / qmul))
    got = _run(pkg, torch, d, "bf16", D, bs, Hq, Hkv, 0, True)
    assert np.isfinite(got[0]).all()
    # every scaling above is exact: the same roundings at every place, so only a subnormal product could tell them apart
    assert np.abs(got[0] / np.float32(vmul) - plain[0]).max() <= 2.0 ** -8 * np.abs(plain[0]).max()
    assert np.abs(got[1] - plain[1]).max() <= 1e-5 * Hq


@pytest.mark.parametrize("qd,D,bs,Hq,Hkv,past,far", [
    ("f16", 128, 32, 8, 2, [4000, 700], False), ("f16", 64, 16, 16, 4, [2000, 31], False), ("f16", 256, 32, 4, 2, [1500], False),
    ("bf16", 128, 32, 16, 2, [4000, 700], False), ("f16", 128, 32, 8, 2, [2500], True), ("bf16", 128, 64, 16, 2, [2500], True),
])
def test_decode_u4_error_against_64_bits(pkg, qd, D, bs, Hq, Hkv, past, far):
    """The matrix instructions are no further from the binary64 result than the shape-generic kernel's binary32 arithmetic, which
    ALiBi slopes too small to move any logit keep the same step on.  far: one V row 2^12 times the others, under a key that no
    query attends to (its weight is far below 2^-12, the others' weights are that far below the largest V scale)."""
    import torch
    print(f"case decode u4 error {qd} D{D} bs{bs} {Hq}/{Hkv} past {past} far {far}", flush=True)
    c = _case(np.random.default_rng(D + Hq), qd, D, D, "u4", "u4", bs, Hq, Hkv, past, [1] * len(past))
    if far:
        at = (c["table"][c["bib"][:-1]], slice(None), 5)  # token 5 of every sequence
        keys = -3.0 * O.from_bits(c["q"], c["qdt"]).reshape(len(past), Hkv, Hq // Hkv, D).sum(2)
        lo, hi = keys.min(-1, keepdims=True), keys.max(-1, keepdims=True)
        codes = np.rint((keys - lo) / (hi - lo) * 15).astype(np.uint8)
        scale = ((hi - lo) / 15).astype(np.float32)
        c["kc"][at] = np.concatenate([scale.view(np.uint8), (-lo / scale).astype(np.float32).view(np.uint8),
                                      codes[..., 0::2] << 4 | codes[..., 1::2]], -1)
        v = c["vc"][at]
        v[..., :4] = (np.ascontiguousarray(v[..., :4]).view(np.float32) * np.float32(4096)).view(np.uint8)
        c["vc"][at] = v
    out, _, kc, vc = _run(pkg, torch, c, qd, D, bs, Hq, Hkv, 0, False)
    assert KERNELS == [{"decode"}]
    generic = _run(pkg, torch, c, qd, D, bs, Hq, Hkv, 0, False, slopes=np.full(Hq, 1e-30, np.float32))[0]
    assert KERNELS == [{"generic"}]
    exact = H.attention_f64(O.from_bits(c["q"], c["qdt"]), kc, vc, 15, c["past"], c["sb"], c["bib"], c["table"], Hq, Hkv, D, bs)
    ours, theirs = H.misrounded(out, exact, qd), H.misrounded(generic, exact, qd)
    print(f"misrounded {ours} against {theirs} of {out.size}", flush=True)
    assert ours <= theirs + 4 * np.sqrt(theirs + 1)  # (counts of rare independent events: four standard deviations)
