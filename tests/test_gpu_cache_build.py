"""The two-launch cache build against the arenas' own builders and a torch-filled metadata arena: ragged
pages, evicted and empty tiers, spare capacity, both generated-value modes and rows off 16 bytes."""
import dataclasses

import pytest
import torch

pytestmark = pytest.mark.gpu

FP, I4, I2, EV = 1, 2, 5, 0
CASES = [
    # variant, generated values, superblock, group, page size, ring, append capacity, tiers drawn, page lengths, dtype, offset
    ("v_fourq_k_int4_compact", "int2", 32, 32, 32, 128, None, (FP, I4, I2, EV), (1, 7, 32), torch.bfloat16, 0),
    ("v_fourq_k_int4_compact", "int4", 64, 64, 16, 256, 300, (FP, I4, I2), (16, 5), torch.float16, 3),
    ("v_fourq_k_int2_compact", "int2", 128, 128, 64, 128, 5000, (I2,), (64,), torch.bfloat16, 0),
    ("v_fourq_k_int2_compact", "int4", 128, 32, 32, 128, 130, (FP, EV), (32, 31), torch.bfloat16, 0),
    ("v_fourq_k_bf16", "int2", 32, 64, 32, 384, 260, (FP, I4, EV), (32, 9), torch.bfloat16, 8),
    ("v_fourq_k_bf16", "int2", 32, 32, 32, 128, 0, (I4,), (32,), torch.float16, 0),
]


def _fill_free_memory(dev):
    """Makes memory that a build may take hold 0x77: requests up to 1 MiB come from a pool of their own, so blocks of
    many sizes are filled in both, small ones for the gaps between live tensors, and freed together."""
    torch.cuda.empty_cache()
    held = [torch.full((size,), 0x77, dtype=torch.uint8, device=dev)
            for size, count in ((512, 1024), (1 << 12, 256), (1 << 16, 128), (1 << 20, 24), (1 << 22, 8)) for _ in range(count)]
    del held
    for t in [torch.empty(size, dtype=torch.uint8, device=dev) for size in (512, 1 << 12, 100_000, 900_000, 2_000_000)]:
        assert (t == 0x77).all(), t.numel()


@pytest.mark.parametrize("case", range(len(CASES)))
@pytest.mark.parametrize("host_table", [True, False])
def test_build_is_its_parts(case, host_table):
    import r2omni_amd as ro
    from r2omni_amd.cache import _build_metadata_arena, _expand_tier_tokens, _tier_page_table
    from r2omni_amd.policy import plan_from_pages

    if not torch.cuda.is_available():
        pytest.skip("needs an MI355X")
    dev = torch.device("cuda:0")
    variant, gen, sb, group, ps, ring, append, tiers, page_lens, dtype, offset = CASES[case]
    g = torch.Generator().manual_seed(case)
    pick = lambda seq: [seq[int(i)] for i in torch.randint(len(seq), (70,), generator=g)]  # noqa: E731
    lens, cls = pick(page_lens), pick(tiers)
    offs = [sum(lens[:i]) for i in range(70)]
    s = sum(lens)
    plan = plan_from_pages(offs, lens, cls, recent_fp_capacity=ring, device=dev)
    if not host_table:
        plan = dataclasses.replace(plan, host_page_table=None)
    plan = dataclasses.replace(plan, global_token_indices=plan.global_token_indices * 3 + 1,
                               logical_positions=plan.logical_positions + 11)
    k, v = (torch.empty(3 * s * 128 + offset, dtype=dtype, device=dev)[offset:].view(3, s, 128) for _ in range(2))
    k.copy_(torch.randn(3, s, 128, generator=g)), v.copy_(torch.randn(3, s, 128, generator=g))
    _fill_free_memory(dev)
    c = ro.build_three_precision_cache(k, v, plan, page_size=ps, key_quantization_superblock=sb, int2_group_size=group,
                                       generated_value_precision=gen, cache_variant=variant,
                                       compact_key_append_capacity=append)
    room = ring if append is None else append
    tab = _tier_page_table(plan)
    tokens = _expand_tier_tokens(tab, "cpu")
    a, b, d = (int(x) for x in tab.tier_tokens[:3])
    fp, i4, i2 = tokens[:a].to(dev), tokens[a:a + b].to(dev), tokens[a + b:a + b + d].to(dev)
    reserve2, reserve4 = (0 if x is None else x.numel() - n for x, n in
                          ((c.metadata_arena.int2_global_index_buffer, d), (c.metadata_arena.int4_global_index_buffer, b)))
    want = _build_metadata_arena(tab, tokens, plan.global_token_indices.cpu(), plan.logical_positions.cpu(), page_size=ps,
                                 recent_capacity=ring, int2_reserve=reserve2, int4_reserve=reserve4)[0]
    assert torch.equal(c.metadata_arena.storage.cpu(), want.storage)
    if variant == "v_fourq_k_bf16":
        assert reserve2 == reserve4 == 0
        n = a + b + d
        assert torch.equal(c.bf16_key.rows[:, :n], k[:, tokens[:n].to(dev)]) and not c.bf16_key.rows[:, n:].any()
    else:
        build = ro.build_compact_int4_key_arena if "int4" in variant else ro.build_compact_int2_key_arena
        key = build(k, (fp, i4, i2), append_capacity=room, superblock_size=sb)
        assert (c.compact_key.active_length, c.compact_key.capacity, c.compact_key.segment_offsets) == \
            (key.active_length, key.capacity, key.segment_offsets)
        for x, y in zip(c.compact_key.allocation_tensors(), key.allocation_tensors()):
            assert x.shape == y.shape and torch.equal(x, y)
        free = key.capacity - key.active_length
        assert reserve2 == min(c.compact_value.capacity - d, free) // ps * ps
        assert reserve4 == (min(c.compact_int4_value.capacity - b, free) // ps * ps if gen == "int4" else 0)
    two = ro.build_compact_int2_value_arena(v, i2, append_capacity=0 if gen == "int4" else room, group_size=group)
    for x, y in zip(c.compact_value.allocation_tensors(), two.allocation_tensors()):
        assert x.shape == y.shape and torch.equal(x, y)
    if gen == "int4":
        from r2omni_amd.cache import build_compact_int4_value_arena
        four = build_compact_int4_value_arena(v, i4, append_capacity=room)
        assert torch.equal(c.compact_int4_value.packed, four.packed) and torch.equal(c.compact_int4_value.scale, four.scale)
    elif b:
        four = ro.fused_gather_pack_int4_value(v, i4)
        assert torch.equal(c.int4_pool.packed_v.packed, four.packed) and torch.equal(c.int4_pool.packed_v.scale, four.scale)
    else:
        assert c.int4_pool.packed_v is None
    assert (c.fp_pool.fp_v is None) == (a == 0) and (a == 0 or torch.equal(c.fp_pool.fp_v, v[:, fp]))
    pool = c.recent_fp_pool
    assert not pool.fp_k.any() and not pool.fp_v.any() and int(pool.length_device) == 0
    assert (pool.global_index_buffer == -1).all() and (pool.logical_position_buffer == -1).all()


def test_build_refuses_plans_outside_the_sequence():
    import r2omni_amd as ro
    from r2omni_amd.policy import plan_from_pages

    if not torch.cuda.is_available():
        pytest.skip("needs an MI355X")
    dev = torch.device("cuda:0")
    k = torch.zeros(2, 64, 128, dtype=torch.bfloat16, device=dev)
    with pytest.raises(ValueError, match="inside the K/V sequence"):
        ro.build_three_precision_cache(k, k, plan_from_pages([0, 40], [32, 32], [FP, I4], device=dev))
    plan = dataclasses.replace(plan_from_pages([0, 32], [32, 32], [FP, I4], device=dev),
                               global_token_indices=torch.arange(63, device=dev))
    with pytest.raises(ValueError, match="cover the K/V sequence"):
        ro.build_three_precision_cache(k, k, plan)


@pytest.mark.parametrize("n", [1, 63, 64, 130])
@pytest.mark.parametrize("src_off,dst_off", [(0, 0), (1, 0), (0, 3), (4, 8)])
def test_gather_moves_rows_that_start_anywhere(n, src_off, dst_off):
    from r2omni_amd import _lib

    if not torch.cuda.is_available():
        pytest.skip("needs an MI355X")
    g = torch.Generator().manual_seed(n)
    at = lambda rows, off: torch.zeros(2 * rows * 128 + off, dtype=torch.int16, device="cuda:0")[off:].view(2, rows, 128)  # noqa: E731
    src, dst = at(n + 3, src_off), at(n + 2, dst_off)
    src.copy_(torch.randint(-2 ** 15, 2 ** 15, src.shape, generator=g, dtype=torch.int32).to(torch.int16))
    for index in (torch.randperm(n + 3, generator=g)[:n].to(src.device), None):
        dst.fill_(5)
        _lib.call("r2o_gather_rows", _lib.ptr(src), 2, n + 3, _lib.ptr(index), n, _lib.ptr(dst), n + 2,
                  _lib.stream_of(src.device))
        assert torch.equal(dst[:, :n], src[:, :n] if index is None else src[:, index]) and (dst[:, n:] == 5).all()


@pytest.mark.parametrize("variant", ["v_fourq_k_int4_compact", "v_fourq_k_int2_compact"])
@pytest.mark.parametrize("types", [(torch.bfloat16, torch.float16), (torch.float16, torch.bfloat16)])
def test_keys_and_values_of_different_types(variant, types):
    """Two packing launches in place of one: the same arenas as the builders of each."""
    import r2omni_amd as ro
    from r2omni_amd.policy import plan_from_pages

    if not torch.cuda.is_available():
        pytest.skip("needs an MI355X")
    dev = torch.device("cuda:0")
    g = torch.Generator().manual_seed(2)
    k, v = (torch.randn(3, 32 * 11, 128, generator=g).to(t).to(dev) for t in types)
    cls = [(FP, I4, I2, EV)[i % 4] for i in range(11)]
    plan = plan_from_pages([32 * i for i in range(11)], [32] * 11, cls, device=dev)
    _fill_free_memory(dev)
    c = ro.build_three_precision_cache(k, v, plan, cache_variant=variant)
    fp, i4, i2 = (torch.cat([torch.arange(32 * i, 32 * i + 32) for i in range(11) if cls[i] == t]).to(dev) for t in (FP, I4, I2))
    build = ro.build_compact_int4_key_arena if "int4" in variant else ro.build_compact_int2_key_arena
    for x, y in zip(c.compact_key.allocation_tensors(),
                    build(k, (fp, i4, i2), append_capacity=128, superblock_size=32).allocation_tensors()):
        assert torch.equal(x, y)
    for x, y in zip(c.compact_value.allocation_tensors(),
                    ro.build_compact_int2_value_arena(v, i2, append_capacity=128, group_size=32).allocation_tensors()):
        assert torch.equal(x, y)
    four = ro.fused_gather_pack_int4_value(v, i4)
    assert torch.equal(c.int4_pool.packed_v.packed, four.packed) and torch.equal(c.int4_pool.packed_v.scale, four.scale)
    assert torch.equal(c.fp_pool.fp_v, v[:, fp])


@pytest.mark.parametrize("offset", [0, 1, 4])
def test_matched_build_of_rows_that_start_anywhere(offset):
    import r2omni_amd as ro
    from r2omni_amd.policy import plan_from_pages

    if not torch.cuda.is_available():
        pytest.skip("needs an MI355X")
    dev = torch.device("cuda:0")
    lens, cls = [32, 7, 32, 20, 32], [FP, I2, EV, I4, FP]
    offs, s = [sum(lens[:i]) for i in range(5)], sum(lens)
    g = torch.Generator().manual_seed(offset)
    k, v = (torch.empty(3 * s * 128 + offset, dtype=torch.bfloat16, device=dev)[offset:].view(3, s, 128) for _ in range(2))
    k.copy_(torch.randn(3, s, 128, generator=g)), v.copy_(torch.randn(3, s, 128, generator=g))
    c = ro.build_three_precision_cache(k, v, plan_from_pages(offs, lens, cls, device=dev), matched_fp=True)
    kept = torch.cat([torch.arange(o, o + n) for o, n, t in zip(offs, lens, cls) if t != EV]).to(dev)
    assert torch.equal(c.fp_pool.fp_k, k[:, kept]) and torch.equal(c.fp_pool.fp_v, v[:, kept])
    assert c.fp_pool.page_index.global_token_indices.tolist() == kept.tolist()
