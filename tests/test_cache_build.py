"""CPU checks of the cache build's native page table against the torch restatement of the same arena."""
import ctypes

import numpy as np
import pytest
import torch

from r2omni_amd import _lib
from r2omni_amd.cache import _build_metadata_arena, _expand_tier_tokens, _metadata_words, _tier_page_table
from test_abi import _c_layout
from test_layouts import _random_plan


def _native(plan, tokens, page_size, reserve4, reserve2, ring):
    table = plan.host_page_table.contiguous()
    n = int(table.shape[1])
    counts = np.empty(8, np.int64)
    rc = _lib.load().r2o_cache_pages(table.data_ptr(), n, tokens, counts.ctypes.data, counts.ctypes.data + 32)
    if rc:
        return rc, None, None
    sizes = dict(page_size=page_size, recent_capacity=ring, int2_reserve=reserve2, int4_reserve=reserve4)
    page_words, total = _metadata_words(counts[:4], counts[4:], **sizes)
    words = np.full(page_words + 3 * n, 77, np.int64)
    call = lambda room: _lib.load().r2o_cache_page_words(table.data_ptr(), n, page_size, reserve4, reserve2, ring,  # noqa: E731
                                                         words.ctypes.data, room)
    assert call(words.size - 1) == 1
    assert call(words.size) == 0
    return counts, words, (page_words, total)


@pytest.mark.parametrize("seed", range(12))
@pytest.mark.parametrize("reserve4,reserve2,ring", [(0, 0, 128), (96, 128, 256)])
def test_native_page_words_match_the_torch_arena(seed, reserve4, reserve2, ring):
    plan, offs, lens, _ = _random_plan(seed, page_sizes=(1, 17, 32))
    tab = _tier_page_table(plan)
    tokens = _expand_tier_tokens(tab, "cpu")
    gi = torch.arange(sum(lens))
    storage = _build_metadata_arena(tab, tokens, gi, gi, page_size=32, recent_capacity=ring, int2_reserve=reserve2,
                                    int4_reserve=reserve4)[0].storage.numpy()
    counts, words, (page_words, total) = _native(plan, sum(lens), 32, reserve4, reserve2, ring)
    assert counts[:4].tolist() == np.diff(tab.first_page).tolist() and counts[4:].tolist() == tab.tier_tokens.tolist()
    assert storage.size == total
    np.testing.assert_array_equal(words[:page_words], storage[:page_words])
    start, length, position = words[page_words:].reshape(3, -1)
    got = np.full(sum(lens), -1)
    for s, n, p in zip(start, length, position):
        got[p:p + n] = np.arange(s, s + n)
    np.testing.assert_array_equal(got, tokens.numpy())


def test_native_page_table_refuses_what_does_not_fit():
    plan, _, lens, _ = _random_plan(3)
    assert _native(plan, sum(lens) - 1, 32, 0, 0, 128)[0] == 1      # a page past the sequence
    table = plan.host_page_table.clone()
    for row, value in ((0, 9), (0, -1), (1, -32), (2, -1)):         # unknown classes, negative pages
        bad = table.clone()
        bad[row, 0] = value
        counts = np.empty(8, np.int64)
        assert _lib.load().r2o_cache_pages(bad.data_ptr(), int(bad.shape[1]), sum(lens), counts.ctypes.data,
                                           counts.ctypes.data + 32) == 1
    words = np.empty(10000, np.int64)
    assert _lib.load().r2o_cache_page_words(table.data_ptr(), int(table.shape[1]), 32, 16, 0, 128, words.ctypes.data, 10000) == 1


def test_build_and_flush_struct_layouts_match_header(tmp_path):
    for struct, cls in (("r2o_cache_build_params", _lib.CacheBuild), ("r2o_ring_flush_params", _lib.RingFlush)):
        names = [f[0] for f in cls._fields_]
        offsets, size = _c_layout(struct, names, tmp_path)
        assert [getattr(cls, n).offset for n in names] == offsets, struct
        assert ctypes.sizeof(cls) == size, struct


def test_build_and_flush_refuse_before_any_launch():
    lib = _lib.load()
    assert lib.r2o_cache_build(None, None) == 1 and lib.r2o_ring_flush(None, None) == 1
    assert lib.r2o_cache_build(_lib.CacheBuild(), None) == 1 and lib.r2o_ring_flush(_lib.RingFlush(), None) == 1
