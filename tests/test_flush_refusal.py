"""CPU checks that a flush which is refused, or whose launch fails, leaves the cache's counts and page indexes
as they were: a pool never names tokens that were not packed, and a later flush takes the same places; and that
rows which are not the ring's are refused."""
import pytest
import torch

from r2omni_amd import _lib
from r2omni_amd import cache as rc
from r2omni_amd.policy import PageClass, plan_from_pages

HEADS, TOKENS, RING = 2, 96, 128


def _state(cache):
    fields = [(f, getattr(p.page_index, f).tolist()) for p in cache.pools
              for f in ("original_page_ids", "physical_offsets", "lengths", "global_token_indices", "logical_positions")]
    arenas = [(a.active_length, a.capacity) for a in
              (cache.compact_key, cache.compact_value, cache.compact_int4_value, cache.bf16_key) if a is not None]
    counts = [p.token_count for p in cache.pools]
    if cache.metadata_arena is not None:
        counts += [getattr(cache.metadata_arena, f"{t}_{n}_count") for t in ("int4", "int2") for n in ("page", "token")]
    rows = [None if p.fp_v is None else tuple(p.fp_v.shape) for p in cache.pools]
    return fields, arenas, counts, rows


def _cache(generated, arena=True, matched=False):
    """A cache of host tensors with a full ring (one FP, one INT4 and one INT2 page of 32 tokens)."""
    plan = plan_from_pages([0, 32, 64], [32] * 3, [int(PageClass.FP_PAGE), int(PageClass.INT4_PAGE), int(PageClass.INT2_PAGE)],
                           recent_fp_capacity=RING)
    tab = rc._tier_page_table(plan)
    meta, index, evicted, (ring_g, ring_l, length) = rc._build_metadata_arena(
        tab, rc._expand_tier_tokens(tab, "cpu"), plan.global_token_indices, plan.logical_positions, page_size=32,
        recent_capacity=RING, int2_reserve=128, int4_reserve=128 if generated == "int4" else 0)
    row = lambda n: torch.zeros(HEADS, n, 128, dtype=torch.bfloat16)  # noqa: E731
    u8, f16 = dict(dtype=torch.uint8), dict(dtype=torch.float16)
    i4 = rc.CompactInt4ValueArena(torch.zeros(HEADS, 160, 64, **u8), torch.zeros(HEADS, 160, 1), 32, 160, torch.bfloat16)
    i2 = rc.CompactInt2ValueArena(torch.zeros(HEADS, 256, 32, **u8), torch.zeros(HEADS, 256, 4, 1, **f16),
                                  torch.zeros(HEADS, 256, 4, 1, **u8), 32, 256, torch.bfloat16)
    key = rc.CompactInt4KeyArena(torch.zeros(HEADS, 256, 64, **u8), torch.zeros(HEADS, 8, 128, **f16),
                                 torch.zeros(HEADS, 8, 128, **u8), TOKENS, 256, (0, 32, 64), torch.bfloat16, superblock_size=32)
    rows = rc.BF16KeyArena(row(128), TOKENS, 128, (0, TOKENS, TOKENS))
    int4 = generated == "int4"
    pools = [rc.PrecisionPool("fp", index[0], fp_v=row(32)), rc.PrecisionPool("int4", index[1], packed_v=i4 if int4 else None),
             rc.PrecisionPool("int2", index[2], packed_v=i2),
             rc.PrecisionPool("recent_fp", index[3], fp_k=row(RING), fp_v=row(RING), active_length=RING, capacity=RING,
                              length_device=length, global_index_buffer=ring_g, logical_position_buffer=ring_l)]
    kw = dict(bf16_key=rows) if matched else dict(compact_key=key, compact_value=i2, compact_int4_value=i4 if int4 else None)
    return rc.ThreePrecisionCache(*pools, evicted, 32, 128, matched, "v_fourq_k_int4_compact",
                                  metadata_arena=meta if arena and not matched else None, generated_value_precision=generated, **kw)


@pytest.fixture
def host_only(monkeypatch):
    """Every launch is refused, as the library refuses its arguments; host tensors pass for device ones."""
    calls = []

    def call(name, *args):
        calls.append(name)
        raise ValueError(f"{name}: refused")

    monkeypatch.setattr(_lib, "call", call)
    monkeypatch.setattr(_lib, "require_device", lambda t, what: None)
    monkeypatch.setattr(_lib, "stream_of", lambda device: 0)
    return calls


@pytest.mark.parametrize("append", [False, True])
@pytest.mark.parametrize("arena", [True, False])
@pytest.mark.parametrize("generated", ["int2", "int4"])
def test_a_refused_flush_leaves_the_cache_as_it_was(host_only, generated, arena, append):
    cache, stats = _cache(generated, arena), rc.DynamicCacheStats()
    before, length = _state(cache), cache.recent_fp_pool.active_length
    for _ in range(2):
        with pytest.raises(ValueError, match="r2o_ring_flush: refused"):
            if append:
                row = torch.zeros(HEADS, 1, 128, dtype=torch.bfloat16)
                rc.append_generated_token(cache, row, row, global_token_index=1, logical_position=1, stats=stats)
            else:
                rc.flush_full_recent_pool(cache, stats)
    assert host_only == ["r2o_ring_flush"] * 2
    assert _state(cache) == before and cache.recent_fp_pool.active_length == length and stats == rc.DynamicCacheStats()


def test_a_matched_flush_that_cannot_grow_leaves_the_cache_as_it_was(host_only, monkeypatch):
    def full(self, key_block):
        raise torch.OutOfMemoryError("no room to grow")

    monkeypatch.setattr(rc.BF16KeyArena, "append_block", full)
    cache, stats = _cache("int2", matched=True), rc.DynamicCacheStats()
    before = _state(cache)
    with pytest.raises(torch.OutOfMemoryError):
        rc.flush_full_recent_pool(cache, stats)
    assert not host_only and _state(cache) == before and stats == rc.DynamicCacheStats()


BAD_ROWS = {
    "fewer heads": lambda k: (k[:1], k[:1]),
    "more heads": lambda k: (torch.cat([k, k]), torch.cat([k, k])),
    "narrow rows": lambda k: (k[..., :64], k[..., :64]),
    "other type": lambda k: (k.half(), k.half()),
    "host value": lambda k: (k, k.clone()),
    "host key": lambda k: (k.clone(), k),
}


@pytest.mark.parametrize("form", BAD_ROWS)
@pytest.mark.parametrize("length", [0, RING])
def test_rows_that_are_not_the_rings_are_refused(monkeypatch, form, length):
    """The append kernels read [Hkv, 128] rows of the ring's type on its GPU, with and without a flush before."""
    from r2omni_amd.splitk import append_recent_fp_triton

    def launched(name, *args):
        raise AssertionError(f"{name} was launched")

    def require(t, what):
        if what.startswith("new_") and not hasattr(t, "on_device"):
            raise RuntimeError(f"{what} must live on the GPU")

    monkeypatch.setattr(_lib, "call", launched)
    monkeypatch.setattr(_lib, "require_device", require)
    monkeypatch.setattr(_lib, "stream_of", lambda device: 0)
    key = torch.zeros(HEADS, 1, 128, dtype=torch.bfloat16)
    key.on_device = True
    rows = BAD_ROWS[form](key)
    if not form.startswith("host"):
        for t in rows:
            t.on_device = True
    cache, stats = _cache("int2"), rc.DynamicCacheStats()
    cache.recent_fp_pool.active_length = length
    before = _state(cache)
    kw = dict(global_token_index=1, logical_position=1)
    with pytest.raises((ValueError, RuntimeError), match="ring|GPU"):
        rc.append_generated_token(cache, *rows, stats=stats, **kw)
    if length < RING:
        with pytest.raises((ValueError, RuntimeError), match="ring|GPU"):
            append_recent_fp_triton(cache, *rows, **kw)
    assert _state(cache) == before and stats == rc.DynamicCacheStats()
