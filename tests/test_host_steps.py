"""What the library's host side does between the runtime calls: memory that runs out, copies that are still queued.  The library
runs in a process of its own on a stand-in for the HIP runtime (fake_hip.cpp), which launches nothing and logs what it was asked."""
import os
import subprocess
import sys
import textwrap

import pytest

TESTS = os.path.dirname(os.path.abspath(__file__))

PRELUDE = """
import ctypes, sys
import numpy as np
sys.path.insert(0, {root!r})
rt = ctypes.CDLL({fake!r}, mode=ctypes.RTLD_GLOBAL)
rt.fake_log.restype = ctypes.c_char_p
rt.fake_used.restype = ctypes.c_size_t
rt.fake_late_copies.restype = rt.fake_malloc_failures.restype = rt.fake_pending.restype = ctypes.c_long
rt.fake_set_budget.argtypes = [ctypes.c_size_t]
rt.fake_fail_sizes.argtypes = [ctypes.c_size_t, ctypes.c_size_t]
import __graft_entry__ as entry
pkg = entry.load_package()

class T:  # a tensor as the binding sees one: nothing reads it here
    def __init__(self, *shape):
        self.shape = shape
    def data_ptr(self):
        return 1 << 40

def ran():
    return [l.split()[2] for l in rt.fake_log().decode().splitlines() if l.startswith("run")]

def begin(op, past, new, bs=32, **kw):
    past, new = np.asarray(past, np.int32), np.asarray(new, np.int32)
    bib = np.concatenate([[0], np.cumsum((past + new + bs - 1) // bs)]).astype(np.int32)
    op.step_begin(past, np.concatenate([[0], np.cumsum(new)]), bib, **kw)
    op.set_block_indices(np.arange(bib[-1]) % 1000, 1000)

def forward(op, scores=None):
    rt.fake_clear_log()
    op.forward(T(1), T(1), T(1), T(1000), T(1000), T(1), scores)
    return ran()
def refused(status, fn, *args):
    try:
        fn(*args)
    except pkg.PaError as e:
        assert e.status == status, e
    else:
        assert False
WIDE = 16896  # bytes of a widened (32-token block, kv head)
"""


@pytest.fixture(scope="module")
def on_fake(tmp_path_factory, pkg):
    so = str(tmp_path_factory.mktemp("fake") / "libfake_hip.so")
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-w", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    os.path.join(TESTS, "fake_hip.cpp"), "-o", so], check=True)

    def run(script):
        head = PRELUDE.format(root=os.path.dirname(TESTS), fake=so)
        r = subprocess.run([sys.executable, "-c", head + textwrap.dedent(script)], capture_output=True, text=True, timeout=120)
        assert r.returncode == 0, r.stdout + r.stderr
    return run


def test_mandatory_memory_before_widened_rows(on_fake):
    """A prompt step over u8 whose workspaces do not fit beside its widened rows gives those back and runs without them."""
    on_fake("""
        op = pkg.PagedAttention(16, 1, 128, 32, "f16", "u8")
        begin(op, [300], [1101])
        before = rt.fake_used()
        assert any("widen" in k for k in forward(op))
        workspaces = rt.fake_used() - before
        del op
        wide = 44 * WIDE
        for short in (1, wide // 2, wide):
            op = pkg.PagedAttention(16, 1, 128, 32, "f16", "u8")
            begin(op, [300], [1101])
            held = rt.fake_used()
            rt.fake_set_budget(held + workspaces - short)
            for layer in range(2):
                names = forward(op)
                assert not any("widen" in k or "dense" in k for k in names) and any("pa_prefill16_kernel" in k for k in names), names
            assert rt.fake_used() == held - wide + workspaces
            rt.fake_set_budget(rt.fake_used() + 4096)
            begin(op, [0], [1])  # (a launch behind the failed allocation is not taken for it)
            forward(op)
            del op
            rt.fake_set_budget(1 << 62)
        # what does not fit without them either is still the library's error
        op = pkg.PagedAttention(16, 1, 128, 32, "f16", "u8")
        begin(op, [300], [1101])
        rt.fake_set_budget(rt.fake_used() + workspaces - wide - 1)
        try:
            forward(op)
            assert False
        except pkg.PaError as e:
            assert e.status == -10, e
        rt.fake_set_budget(1 << 62)
        assert any("pa_prefill16_kernel" in k for k in forward(op))
    """)


def test_widened_rows_outlive_a_failed_growth(on_fake):
    """No memory for more widened rows: the step goes without, the rows held serve the steps that fit them, and a long row of such
    steps does not ask the runtime again and again."""
    on_fake("""
        op = pkg.PagedAttention(16, 1, 128, 32, "f16", "u8")
        begin(op, [0], [1400])
        assert any("widen" in k for k in forward(op))
        blocks = (8000 + 3000 + 31) // 32
        rt.fake_fail_sizes(blocks * WIDE, blocks * WIDE)
        for i in range(20):
            begin(op, [8000], [3000])
            assert not any("widen" in k for k in forward(op))
            begin(op, [0], [1400])
            assert any("widen" in k for k in forward(op)), i
        assert rt.fake_malloc_failures() == 1, rt.fake_malloc_failures()
        rt.fake_fail_sizes(1, 0)
        for i in range(300):
            begin(op, [8000], [3000])
        assert any("widen" in k for k in forward(op))  # (after a while it asks again)
    """)


def test_a_call_without_memory_leaves_no_freed_buffer_in_use(on_fake):
    """Larger thresholds' plans or trig tables that find no memory: what they replaced is gone, and calls that need it are refused."""
    on_fake("""
        op = pkg.PagedAttention(8, 2, 128, 32, "f16", "f16")
        begin(op, [3000], [500])
        op.set_xattention([0.9], 64, 16)
        assert any("xatt" in k for k in forward(op))
        for lo, hi in ((1 << 24, 1 << 40), (40000, 1 << 17)):  # (the logits; the block sums)
            rt.fake_fail_sizes(lo, hi)
            refused(-10, op.set_xattention, [0.9], 32, 1)
            rt.fake_fail_sizes(1, 0)
            refused(-4, forward, op)
            begin(op, [3000], [500])
            forward(op)
            op.set_xattention([0.9], 64, 16)
            forward(op)
        op.set_rotation_trig_lut(np.ones((8, 128), np.float32))
        op.rotate_cache(T(1000), [3], [7])
        rt.fake_fail_sizes(64 * 512, 64 * 512)
        refused(-10, op.set_rotation_trig_lut, np.ones((64, 128), np.float32))
        refused(-10, op.rotate_cache, T(1000), [3], [7])
        rt.fake_fail_sizes(1, 0)
        op.set_rotation_trig_lut(np.ones((64, 128), np.float32))
        op.rotate_cache(T(1000), [3], [63])
    """)


def test_a_failed_mixed_step_joins_its_second_stream(on_fake):
    """A mixed step that finds no memory for the chunk's partials has its decode kernel on the second stream already: the context's
    stream waits for it all the same."""
    on_fake("""
        def step():
            op = pkg.PagedAttention(32, 8, 128, 32, "f16", "u8")
            begin(op, [4000, 3000, 2000, 9000], [1, 1, 1, 40])
            return op
        op = step()
        names = forward(op)
        log = rt.fake_log().decode().splitlines()
        forked = [i for i, l in enumerate(log) if l.startswith("run 100") and "decode" in l]
        late = [int(l.split()[1]) for l in log[forked[0]:] if l.startswith("malloc")]
        assert late, log
        op = step()
        rt.fake_fail_sizes(late[0], late[0])
        try:
            forward(op)
            assert False
        except pkg.PaError as e:
            assert e.status == -10
        log = rt.fake_log().decode().splitlines()
        side = [l.split()[1] for l in log if l.startswith("run") and "decode" in l]
        assert side and side[0] != "0", log
        assert log[-1] == "wait 0 " + side[0], log
    """)


def test_copies_of_steps_queued_ahead(on_fake):
    """Steps prepared one behind the other without a wait: no copy finds its part of the staging area written over, also where a step's
    arrays do not fit it, with thresholds, with a table per layer and with rotations in between."""
    on_fake("""
        rng = np.random.default_rng(0)
        op = pkg.PagedAttention(8, 2, 128, 32, "f16", "f16", num_layers=3)
        op.set_rotation_trig_lut(np.ones((64, 128), np.float32))
        ahead = 0
        for i in range(60):
            B = int(rng.integers(1, 6))
            past, new = rng.integers(1, 4000, B).astype(np.int32), rng.integers(1, 900, B).astype(np.int32)
            extra = 30000 if i in (20, 21, 40) else 0
            bib = np.concatenate([[0], np.cumsum((past + new + 31) // 32 + extra)]).astype(np.int32)
            op.step_begin(past, np.concatenate([[0], np.cumsum(new)]), bib)
            ahead += rt.fake_pending(0) > 1  # (its own upload, and some of the step before)
            if i % 3 == 0:
                op.set_xattention(rng.random(B), 64, 8)
            tables = rng.integers(0, 1000, (3, bib[-1]))
            if i // 10 % 2:  # (going over from one table to one per layer waits)
                op.set_block_indices_per_layer(tables, 1000)
            else:
                op.set_block_indices(tables[0], 1000)
            if i % 5 == 0:
                op.rotate_cache(T(1000), np.arange(7), np.arange(7))
            for layer in range(3):
                op.forward(T(1), T(1), T(1), T(1000), T(1000), T(1), layer=layer)
        op.synchronize()
        assert rt.fake_late_copies() == 0
        assert ahead >= 30, ahead
    """)


def test_tables_carry_the_descriptors_their_step_can_use(on_fake):
    """Descriptors of the 16-bit decode kernel go up with a table only in steps that may run it."""
    on_fake("""
        def bytes_up(D, bs, new):
            op = pkg.PagedAttention(8, 4, D, bs, "f16", "f16")
            rt.fake_clear_log()
            begin(op, [500, 900, 100, 300], new, bs)
            return [int(l.split()[1]) for l in rt.fake_log().decode().splitlines() if l.startswith("malloc")][-1]
        for D in (128, 256):
            for bs in (16, 32):
                for new in ([1, 1, 1, 1], [1, 1, 1, 64], [9, 9, 9, 64]):
                    ids = sum(-(-(p + n) // bs) for p, n in zip([500, 900, 100, 300], new))
                    plain = bytes_up(D, bs, new) == -(-4 * ids // 128) * 128
                    assert plain == (1 not in new or (D == 256 and bs == 16 and max(new) > 1)), (D, bs, new)
    """)


def test_a_failed_call_is_not_reported_again(on_fake):
    """The error of a runtime call that failed, pinned or device memory, belongs to the call it failed in, not to the next launch."""
    on_fake("""
        op = pkg.PagedAttention(8, 2, 128, 32, "f16", "f16")
        rt.fake_fail_sizes(1, 1 << 40)
        for _ in range(2):
            refused(-10, begin, op, [30], [4])
            rt.fake_fail_sizes(1, 0)
            begin(op, [30], [4])
            rt.fake_fail_sizes(1, 1 << 40)
            refused(-10, forward, op)
            rt.fake_fail_sizes(1, 0)
            forward(op)
            op = pkg.PagedAttention(8, 2, 128, 32, "f16", "f16")
            rt.fake_fail_sizes(1, 1 << 40)
        rt.fake_fail_sizes(1, 0)
        from openvino_genai_amd.cache_eviction import AggregationMode, CacheEvictionConfig, Evictor
        ev = Evictor(CacheEvictionConfig(32, 64, 192, AggregationMode.SUM, snapkv_window_size=0), 32, 2, 7, 1, 4096)
        ev.register_new_token_scores([0], [1 << 40, 1 << 41], [0, 640])
        rt.fake_fail_sizes(1, 1 << 40)
        refused(-10, ev.block_scores, 0, 0)
        rt.fake_fail_sizes(1, 0)
        assert len(ev.block_scores(0, 0)) > 0
    """)
