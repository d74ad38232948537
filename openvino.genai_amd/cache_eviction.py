"""``AggregationMode`` / ``CacheEvictionConfig`` / ``CacheEvictionAlgorithm`` over the device-resident evictor.

Names follow the reference's Python module (src/python/py_continuous_batching_pipeline.cpp:344-420) and its C++
classes (src/cpp/include/openvino/genai/cache_eviction.hpp:19-226,
src/cpp/src/continuous_batching/cache/cache_eviction.hpp:23-248).
"""
import ctypes as C
import enum

import numpy as np

from . import _lib as L


class AggregationMode(enum.IntEnum):
    SUM = L.PA_AGG_SUM
    NORM_SUM = L.PA_AGG_NORM_SUM
    ADAPTIVE_RKV = L.PA_AGG_ADAPTIVE_RKV


class KVCrushAnchorPointMode(enum.IntEnum):
    RANDOM = L.PA_KVCRUSH_ANCHOR_RANDOM
    ZEROS = L.PA_KVCRUSH_ANCHOR_ZEROS
    ONES = L.PA_KVCRUSH_ANCHOR_ONES
    MEAN = L.PA_KVCRUSH_ANCHOR_MEAN
    ALTERNATING = L.PA_KVCRUSH_ANCHOR_ALTERNATING


class KVCrushConfig:
    """``budget`` blocks per eviction are kept as representatives of the evicted ones; 0 switches KVCrush off."""

    def __init__(self, budget=0, anchor_point_mode=KVCrushAnchorPointMode.RANDOM, rng_seed=0):
        self.budget = int(budget)
        self.anchor_point_mode = KVCrushAnchorPointMode(anchor_point_mode)
        self.rng_seed = int(rng_seed)

    def get_budget(self):
        return self.budget

    def to_string(self):
        return ("KVCrushConfig { \n"
                f"  budget: {self.budget}\n  rng_seed: {self.rng_seed}\n"
                f"  anchor_point_mode: {self.anchor_point_mode.name}\n }}")


class AdaptiveRKVConfig:
    def __init__(self, attention_mass=0.9, window_size=8):
        self.attention_mass = float(attention_mass)
        self.window_size = int(window_size)


class CacheEvictionConfig:
    """Same construction rules as the reference: non-zero sizes and max_cache_size > start_size + recent_size."""

    def __init__(self, start_size=32, recent_size=128, max_cache_size=672, aggregation_mode=AggregationMode.NORM_SUM,
                 apply_rotation=False, snapkv_window_size=8, kvcrush_config=None, adaptive_rkv_config=None):
        if not start_size:
            raise ValueError("CacheEvictionConfig.start_size must be non-zero")
        if not recent_size:
            raise ValueError("CacheEvictionConfig.recent_size must be non-zero")
        if not max_cache_size:
            raise ValueError("CacheEvictionConfig.max_cache_size must be non-zero")
        if max_cache_size <= start_size + recent_size:
            raise ValueError("CacheEvictionConfig.max_cache_size must be larger than CacheEvictionConfig.start_size + "
                             "CacheEvictionConfig.recent_size")
        self.aggregation_mode = AggregationMode(aggregation_mode)
        self.apply_rotation = bool(apply_rotation)
        self.snapkv_window_size = int(snapkv_window_size)
        self.kvcrush_config = kvcrush_config if kvcrush_config is not None else KVCrushConfig()
        self.adaptive_rkv_config = adaptive_rkv_config if adaptive_rkv_config is not None else AdaptiveRKVConfig()
        self._start_size, self._recent_size, self._max_cache_size = int(start_size), int(recent_size), int(max_cache_size)
        self._evictable_size = self._max_cache_size - self._start_size - self._recent_size

    def get_start_size(self):
        return self._start_size

    def get_recent_size(self):
        return self._recent_size

    def get_max_cache_size(self):
        return self._max_cache_size

    def get_evictable_size(self):
        return self._evictable_size

    def to_string(self):
        return ("CacheEvictionConfig { \n"
                f"  start_size: {self._start_size}\n  recent_size: {self._recent_size}\n"
                f"  max_cache_size: {self._max_cache_size}\n  evictable_size: {self._evictable_size}\n"
                f"  aggregation_mode: {self.aggregation_mode.name}\n"
                f"  apply_rotation: {str(self.apply_rotation).lower()}\n"
                f"  snapkv_window_size: {self.snapkv_window_size}\n"
                f"{self.kvcrush_config.to_string()}\n }}")


def _stream_ptr(stream):
    if stream is None:
        return None
    return C.c_void_p(int(getattr(stream, "cuda_stream", stream)))


class Evictor:
    """Pool of per-sequence eviction states in device memory (one slot per tracked sequence)."""

    def __init__(self, config, block_size, num_decoder_layers, max_pool_window_size, max_sequences=1,
                 max_tracked_tokens=4096, device=0, stream=None, ignore_first_n_blocks=None):
        lib = L.lib()
        c = L.pa_evictor_config()
        c.device, c.stream = device, _stream_ptr(stream)
        if isinstance(config, CacheEvictionConfig):
            c.start_size, c.recent_size, c.max_cache_size = (config.get_start_size(), config.get_recent_size(),
                                                             config.get_max_cache_size())
            c.aggregation_mode, c.snapkv_window_size = int(config.aggregation_mode), config.snapkv_window_size
            c.adaptive_rkv_window_size = config.adaptive_rkv_config.window_size
            c.adaptive_rkv_attention_mass = config.adaptive_rkv_config.attention_mass
            c.kvcrush_budget = config.kvcrush_config.budget
            c.kvcrush_anchor_point_mode = int(config.kvcrush_config.anchor_point_mode)
            c.kvcrush_rng_seed = config.kvcrush_config.rng_seed
        else:  # (aggregation_mode, snapkv_window_size[, adaptive_rkv_window_size]) for a bare score manager
            c.aggregation_mode, c.snapkv_window_size = int(config[0]), int(config[1])
            c.adaptive_rkv_window_size = int(config[2]) if len(config) > 2 else 8
            c.adaptive_rkv_attention_mass = 0.9
        c.block_size, c.num_decoder_layers, c.max_pool_window_size = block_size, num_decoder_layers, max_pool_window_size
        c.max_sequences, c.max_tracked_tokens = max_sequences, max_tracked_tokens
        self.layers, self.block_size = num_decoder_layers, block_size
        self.capacity = max_tracked_tokens
        self.norm_sum = c.aggregation_mode == L.PA_AGG_NORM_SUM
        h = C.c_void_p()
        if ignore_first_n_blocks is None:
            L.check(lib.pa_evictor_create(C.byref(c), C.byref(h)), None)
        else:
            L.check(lib.pa_score_manager_create(C.byref(c), ignore_first_n_blocks, C.byref(h)), None)
        self._h = h

    def __del__(self):
        if getattr(self, "_h", None) and L is not None:  # module globals are gone at interpreter exit
            L.lib().pa_evictor_destroy(self._h)
            self._h = None

    def _ck(self, status):
        L.check(status, L.lib().pa_evictor_last_error, self._h)

    def reset_slot(self, slot):
        self._ck(L.lib().pa_evictor_reset_slot(self._h, slot))

    def register_new_token_scores(self, slots, scores_per_layer_ptrs, offsets, num_snapkv_scores=None):
        """``scores_per_layer_ptrs``: device addresses of ``scores.<L>``; sequence i is [offsets[i], offsets[i+1])."""
        slots = np.ascontiguousarray(slots, dtype=np.int32)
        offsets = np.ascontiguousarray(offsets, dtype=np.int64)
        ptrs = (C.c_void_p * self.layers)(*map(int, scores_per_layer_ptrs))
        snap = None
        if num_snapkv_scores is not None:
            snap = np.ascontiguousarray(num_snapkv_scores, dtype=np.uint64)
        self._ck(L.lib().pa_evictor_register_scores(
            self._h, len(slots), slots.ctypes.data_as(C.POINTER(C.c_int32)), ptrs,
            offsets.ctypes.data_as(C.POINTER(C.c_int64)),
            snap.ctypes.data_as(C.POINTER(C.c_uint64)) if snap is not None else None))

    def register_block_diversity(self, slots, diversity_per_layer_ptrs, offsets):
        """``diversity_per_layer_ptrs``: device addresses of ``adaptive_rkv_diversity.<L>``; sequence i's
        [evictable / block_size, evictable] matrix is [offsets[i], offsets[i+1]) in each."""
        slots = np.ascontiguousarray(slots, dtype=np.int32)
        offsets = np.ascontiguousarray(offsets, dtype=np.int64)
        ptrs = (C.c_void_p * self.layers)(*[C.c_void_p(int(p)) for p in diversity_per_layer_ptrs])
        self._ck(L.lib().pa_evictor_register_block_diversity(
            self._h, len(slots), slots.ctypes.data_as(C.POINTER(C.c_int32)), ptrs,
            offsets.ctypes.data_as(C.POINTER(C.c_int64))))

    def evict_logical_blocks(self, slots, max_blocks_per_entry=4096):
        """Returns ``[sequence][layer] -> ascending list of evicted logical block indices``."""
        slots = np.ascontiguousarray(slots, dtype=np.int32)
        n = len(slots) * self.layers
        # no entry gives up more blocks than it tracks: a short row per entry keeps the array within a few pages (64
        # sequences x 32 layers: 0.3 MB instead of 33 MB of untouched ones)
        max_blocks_per_entry = min(max_blocks_per_entry, self.capacity // self.block_size + 1)
        counts = np.zeros(n, np.int32)
        blocks = np.zeros(n * max_blocks_per_entry, np.int32)
        self._ck(L.lib().pa_evictor_evict(self._h, len(slots), slots.ctypes.data_as(C.POINTER(C.c_int32)),
                                          counts.ctypes.data_as(C.POINTER(C.c_int32)),
                                          blocks.ctypes.data_as(C.POINTER(C.c_int32)), max_blocks_per_entry))
        # all entries' blocks in one list, then one slice per entry
        ends = np.cumsum(counts, dtype=np.int64)
        shift = np.arange(n, dtype=np.int64) * max_blocks_per_entry - (ends - counts)
        flat = blocks[np.arange(ends[-1] if n else 0) + np.repeat(shift, counts)].tolist()
        ends = ends.tolist()
        entries = [flat[a:b] for a, b in zip([0] + ends, ends)]
        return [entries[i:i + self.layers] for i in range(0, n, self.layers)]

    def remove_scores(self, slot, layer, blocks):
        b = np.ascontiguousarray(sorted(blocks), dtype=np.int32)
        self._ck(L.lib().pa_evictor_remove_scores(self._h, slot, layer, b.ctypes.data_as(C.POINTER(C.c_int32)), len(b)))

    def get_evictable_block_range(self, slot, layer=0):
        b, e = C.c_uint64(0), C.c_uint64(0)
        self._ck(L.lib().pa_evictor_get_range(self._h, slot, layer, C.byref(b), C.byref(e)))
        return b.value, e.value

    def get_max_cache_size_after_eviction(self):
        return int(L.lib().pa_evictor_max_cache_size_after_eviction(self._h))

    def get_state(self, slot, layer):
        n = C.c_uint64(0)
        self._ck(L.lib().pa_evictor_get_state(self._h, slot, layer, C.byref(n), None, None, 0))
        scores = np.zeros(n.value, np.float64)
        counters = np.zeros(n.value if self.norm_sum else 0, np.uint64)
        if n.value:
            self._ck(L.lib().pa_evictor_get_state(
                self._h, slot, layer, C.byref(n), scores.ctypes.data_as(C.POINTER(C.c_double)),
                counters.ctypes.data_as(C.POINTER(C.c_uint64)) if self.norm_sum else None, n.value))
        return scores, counters

    def block_scores(self, slot, layer):
        cap = self.capacity // self.block_size + 1
        out = np.zeros(cap, np.float64)
        n = C.c_uint64(0)
        self._ck(L.lib().pa_evictor_block_scores(self._h, slot, layer, out.ctypes.data_as(C.POINTER(C.c_double)), cap,
                                                 C.byref(n)))
        return out[:n.value].copy()


class _HostScoresMixin:
    """Accepts host score vectors (as the reference's unit tests do) by staging them in device memory."""

    def _stage(self, layer_scores):
        import torch
        self._staged = [torch.from_numpy(np.ascontiguousarray(s, dtype=np.float32)).to(f"cuda:{self._device}")
                        if len(s) else torch.zeros(1, device=f"cuda:{self._device}") for s in layer_scores]
        torch.cuda.synchronize()
        lens = {len(s) for s in layer_scores}
        if len(lens) != 1:
            raise ValueError("every layer must carry the same number of scores")
        return [t.data_ptr() for t in self._staged], lens.pop()


class CacheEvictionAlgorithm(_HostScoresMixin):
    """One sequence's eviction state; mirrors the reference class of the same name (one evictor slot)."""

    def __init__(self, eviction_config, block_size, num_decoder_layers, max_pool_window_size, device=0,
                 max_tracked_tokens=4096):
        self._device = device
        self._ev = Evictor(eviction_config, block_size, num_decoder_layers, max_pool_window_size, 1,
                           max_tracked_tokens, device)
        self._layers = num_decoder_layers

    def get_max_cache_size_after_eviction(self):
        return self._ev.get_max_cache_size_after_eviction()

    def get_evictable_block_range(self, layer=0):
        return self._ev.get_evictable_block_range(0, layer)

    def register_new_token_scores(self, attention_scores_for_all_decoder_layers, skipped_logical_block_ids=(),
                                  num_snapkv_scores=0):
        if len(skipped_logical_block_ids):
            raise NotImplementedError("scores of steps with skipped blocks are not registered "
                                      "(pipeline_impl.cpp:909-912 of the reference does the same)")
        ptrs, n = self._stage(attention_scores_for_all_decoder_layers)
        self._ev.register_new_token_scores([0], ptrs, [0, n], [num_snapkv_scores])

    def register_block_diversity(self, block_diversity_for_all_decoder_layers):
        ptrs, n = self._stage(block_diversity_for_all_decoder_layers)
        self._ev.register_block_diversity([0], ptrs, [0, n])

    def evict_logical_blocks(self):
        return self._ev.evict_logical_blocks([0])[0]

    def get_scores(self):
        return [self._ev.get_state(0, l)[0] for l in range(self._layers)]

    def get_counters(self):
        return [self._ev.get_state(0, l)[1] for l in range(self._layers)]

    def block_scores(self, layer):
        return self._ev.block_scores(0, layer)


class EvictionScoreManager(_HostScoresMixin):
    """Bare score tracker (no areas); mirrors the reference class of the same name."""

    def __init__(self, block_size, num_decoder_layers, max_pool_window_size, aggregation_mode,
                 ignore_first_n_blocks=0, snapkv_window_size=0, adaptive_rkv_window_size=8, device=0,
                 max_tracked_tokens=4096):
        self._device = device
        self._ev = Evictor((aggregation_mode, snapkv_window_size, adaptive_rkv_window_size), block_size,
                           num_decoder_layers,
                           max_pool_window_size, 1, max_tracked_tokens, device, None, ignore_first_n_blocks)
        self._layers = num_decoder_layers

    def register_new_token_scores(self, attention_scores_for_all_decoder_layers, skipped_logical_block_ids=(),
                                  num_snapkv_scores=0):
        if len(skipped_logical_block_ids):
            raise NotImplementedError("skip sets are not supported on the device path")
        ptrs, n = self._stage(attention_scores_for_all_decoder_layers)
        self._ev.register_new_token_scores([0], ptrs, [0, n], [num_snapkv_scores])

    def remove_scores(self, evicted_block_indices, decoder_layer_idx):
        self._ev.remove_scores(0, decoder_layer_idx, evicted_block_indices)

    def get_scores(self):
        return [self._ev.get_state(0, l)[0] for l in range(self._layers)]

    def get_counters(self):
        return [self._ev.get_state(0, l)[1] for l in range(self._layers)]


def _u64(values):
    return np.ascontiguousarray(sorted(int(v) for v in values) if isinstance(values, (set, frozenset)) else
                                [int(v) for v in values], dtype=np.uint64)


def _p(a, t):
    return a.ctypes.data_as(C.POINTER(t))


def _select_check(status):
    L.check(status, lambda _h: L.lib().pa_select_last_error(), True)


class AdaptiveRKVBlockCalculator:
    """Mirror of the reference's ``AdaptiveRKVBlockCalculator`` (host arithmetic on block scores)."""

    def __init__(self, attention_mass, block_size):
        self.attention_mass, self.block_size = float(attention_mass), int(block_size)

    def get_diversity_block_set(self, max_num_blocks_kept, evictable_area_block_scores):
        """(blocks left for the diversity filter, number of blocks kept for their attention mass)"""
        sc = np.ascontiguousarray(evictable_area_block_scores, dtype=np.float64)
        out = np.zeros(max(1, sc.size), np.uint64)
        n, kept = C.c_uint64(0), C.c_uint64(0)
        _select_check(L.lib().pa_adaptive_rkv_diversity_block_set(
            self.attention_mass, int(max_num_blocks_kept), _p(sc, C.c_double), sc.size, _p(out, C.c_uint64),
            C.byref(n), C.byref(kept)))
        return set(int(v) for v in out[:n.value]), int(kept.value)

    def get_filtered_block_diversity(self, unfiltered_diversity, eviction_size, diversity_blocks):
        u = np.ascontiguousarray(unfiltered_diversity, dtype=np.float64)
        st = _u64(set(diversity_blocks))
        out = np.zeros(max(1, int(eviction_size) // self.block_size), np.float64)
        _select_check(L.lib().pa_adaptive_rkv_filtered_block_diversity(
            self.block_size, _p(u, C.c_double), u.size, int(eviction_size), _p(st, C.c_uint64), st.size,
            _p(out, C.c_double)))
        return out[:int(eviction_size) // self.block_size]

    def get_most_diverse_blocks(self, num_blocks_left_to_fill, diversity_blocks, filtered_block_diversity):
        st = _u64(set(diversity_blocks))
        f = np.ascontiguousarray(filtered_block_diversity, dtype=np.float64)
        out = np.zeros(max(1, st.size), np.uint64)
        n = C.c_uint64(0)
        _select_check(L.lib().pa_adaptive_rkv_most_diverse_blocks(
            int(num_blocks_left_to_fill), _p(st, C.c_uint64), st.size, _p(f, C.c_double), f.size,
            _p(out, C.c_uint64), C.byref(n)))
        return set(int(v) for v in out[:n.value])


class KVCrushAlgorithm:
    """Mirror of the reference's ``KVCrushAlgorithm`` (host arithmetic on token scores)."""

    def __init__(self, kvcrush_config, block_size):
        self.block_size = int(block_size)
        h = C.c_void_p()
        _select_check(L.lib().pa_kvcrush_create(kvcrush_config.budget, int(kvcrush_config.anchor_point_mode),
                                                kvcrush_config.rng_seed, self.block_size, C.byref(h)))
        self._h = h

    def __del__(self):
        if getattr(self, "_h", None) and L is not None:
            L.lib().pa_kvcrush_destroy(self._h)
            self._h = None

    def _ck(self, status):
        L.check(status, L.lib().pa_kvcrush_last_error, self._h)

    def create_indicators_kvcrush(self, num_tokens_in_evictable_blocks, layer_scores):
        sc = np.ascontiguousarray(layer_scores, dtype=np.float64)
        out = np.zeros(max(1, num_tokens_in_evictable_blocks), np.uint8)
        self._ck(L.lib().pa_kvcrush_create_indicators(self._h, num_tokens_in_evictable_blocks, _p(sc, C.c_double),
                                                      sc.size, _p(out, C.c_uint8)))
        return [int(v) for v in out[:num_tokens_in_evictable_blocks]]

    def create_anchor_point_kvcrush(self, num_tokens_in_evictable_blocks, indicators):
        ind = np.ascontiguousarray(indicators, dtype=np.uint8)
        out = np.zeros(self.block_size, np.uint8)
        self._ck(L.lib().pa_kvcrush_create_anchor_point(self._h, num_tokens_in_evictable_blocks, _p(ind, C.c_uint8),
                                                        _p(out, C.c_uint8)))
        return [int(v) for v in out]

    def calculate_hamming_distance_kvcrush(self, num_tokens_in_evictable_blocks, indicators, anchor_point):
        ind = np.ascontiguousarray(indicators, dtype=np.uint8)
        an = np.ascontiguousarray(anchor_point, dtype=np.uint8)
        nb = num_tokens_in_evictable_blocks // self.block_size
        out = np.zeros(max(1, nb), np.uint64)
        self._ck(L.lib().pa_kvcrush_hamming_distances(self._h, num_tokens_in_evictable_blocks, _p(ind, C.c_uint8),
                                                      _p(an, C.c_uint8), _p(out, C.c_uint64)))
        return [int(v) for v in out[:nb]]

    def get_representative_blocks_kvcrush(self, block_distances, blocks_eligible_for_kvcrush):
        d = _u64(list(block_distances))
        el = _u64(list(blocks_eligible_for_kvcrush))
        out = np.zeros(max(1, el.size), np.uint64)
        n = C.c_uint64(0)
        self._ck(L.lib().pa_kvcrush_representative_blocks(self._h, _p(d, C.c_uint64), d.size, _p(el, C.c_uint64),
                                                          el.size, _p(out, C.c_uint64), C.byref(n)))
        return [int(v) for v in out[:n.value]]

    def get_indices_of_blocks_to_retain_using_kvcrush(self, num_tokens_in_evictable_blocks, evicted_block_indices,
                                                      layer_scores):
        ev = _u64(list(evicted_block_indices))
        sc = np.ascontiguousarray(layer_scores, dtype=np.float64)
        out = np.zeros(max(1, ev.size), np.uint64)
        n = C.c_uint64(0)
        self._ck(L.lib().pa_kvcrush_blocks_to_retain(self._h, num_tokens_in_evictable_blocks, _p(ev, C.c_uint64),
                                                     ev.size, _p(sc, C.c_double), sc.size, _p(out, C.c_uint64),
                                                     C.byref(n)))
        return [int(v) for v in out[:n.value]]


def snapkv_num_token_scores_to_aggregate(snapkv_window_size, prompt_len, num_scheduled_tokens, num_processed_tokens):
    """SnapKVScoreAggregationCalculator::get_num_token_scores_to_aggregate."""
    return int(L.lib().pa_snapkv_num_scores(snapkv_window_size, prompt_len, num_scheduled_tokens, num_processed_tokens))


def rotation_trig_lut(block_size, max_blocks, head_size, rope_theta=10000.0):
    """The [max_blocks, head_size] table of cosines | negated sines the pipeline hands to the model
    (``_prepare_rotation_data_storage``)."""
    lut = np.zeros((max_blocks, head_size), np.float32)
    L.check(L.lib().pa_rotation_trig_lut(block_size, max_blocks, head_size, float(rope_theta),
                                         lut.ctypes.data_as(C.POINTER(C.c_float))), None)
    return lut


class CacheRotationCalculator:
    """Mirror of the reference's ``CacheRotationCalculator``: which kept blocks move after an eviction, and by how
    much.  ``get_rotation_data`` returns dicts with ``logical_block_idx`` (after eviction), ``rotation_delta``
    (tokens) and, unless ``deltas_only``, the per-token ``sines`` / ``cosines`` rows."""

    def __init__(self, block_size, max_context_length_in_blocks, kv_head_size, rope_theta=10000.0):
        self.block_size, self.max_blocks, self.head_size = block_size, max_context_length_in_blocks, kv_head_size
        lut = rotation_trig_lut(block_size, max_context_length_in_blocks, kv_head_size, rope_theta)
        self._cos, self._sin = lut[:, :kv_head_size // 2], lut[:, kv_head_size // 2:]

    def get_head_size(self):
        return self.head_size

    def get_sin_lut(self):
        return self._sin

    def get_cos_lut(self):
        return self._cos

    def get_rotation_data(self, evicted_block_logical_indices, num_logical_blocks_before_eviction, deltas_only=True):
        ev = np.ascontiguousarray(sorted(int(v) for v in evicted_block_logical_indices), np.int64)
        cap = max(1, int(num_logical_blocks_before_eviction))
        idx, delta, n = np.zeros(cap, np.int32), np.zeros(cap, np.int32), C.c_int32(0)
        p32 = lambda a: a.ctypes.data_as(C.POINTER(C.c_int32))
        L.check(L.lib().pa_rotation_data(ev.ctypes.data_as(C.POINTER(C.c_int64)), len(ev),
                                         int(num_logical_blocks_before_eviction), self.block_size, self.max_blocks,
                                         p32(idx), p32(delta), cap, C.byref(n)), None)
        out = []
        for i in range(n.value):
            d = dict(logical_block_idx=int(idx[i]), rotation_delta=int(delta[i]))
            if not deltas_only:
                row = int(delta[i]) // self.block_size
                d["sines"] = [self._sin[row].copy() for _ in range(self.block_size)]
                d["cosines"] = [self._cos[row].copy() for _ in range(self.block_size)]
            out.append(d)
        return out
