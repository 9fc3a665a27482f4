"""Bit-exactness of the packers where their kernels' lane and tile layouts end: row counts around a wave's
and a block's rows, every group and dtype, sources that start off a 16-byte boundary, quotients on and
next to a rounding tie, and ranges at both ends of fp32."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

DTYPES = {"bfloat16": torch.bfloat16, "float16": torch.float16}


def _dev():
    if not torch.cuda.is_available():
        pytest.skip("needs an MI355X")
    return torch.device("cuda:0")


def _rows(n, seed, dtype, heads=2):
    """Rows whose quotients x / step meet ties: multiples of powers of two beside random rows."""
    gen = torch.Generator().manual_seed(seed)
    x = torch.randn(heads, n, 128, generator=gen)
    kind = torch.randint(0, 6, (heads, n, 1), generator=gen)
    steps = torch.randint(-14, 15, (heads, n, 128), generator=gen).float() * 0.25
    x = torch.where(kind == 1, steps, x)                       # few distinct values: exact ties
    x = torch.where(kind == 2, torch.full_like(x, 0.75), x)    # constant rows
    x = torch.where(kind == 3, torch.zeros_like(x), x)         # the 1e-6 step clamp
    x = torch.where(kind == 4, x * 2.0 ** -20, x)
    return x.to(DTYPES[dtype])


def _offset(t, elements):
    """A contiguous copy of ``t`` that starts ``elements`` elements into its storage."""
    buf = torch.empty(t.numel() + elements, dtype=t.dtype, device=t.device)
    out = buf[elements:].view(t.shape)
    out.copy_(t)
    return out


@pytest.mark.parametrize("dtype", sorted(DTYPES))
@pytest.mark.parametrize("n,offset", [(1, 0), (3, 0), (16, 0), (17, 1), (63, 0), (64, 4), (65, 0), (129, 8), (1000, 0)])
def test_value_packers_match_the_oracle(n, offset, dtype):
    import r2omni_amd as ro
    from oracle.quant import quantize_int2_value, quantize_int4_value

    dev = _dev()
    cpu = _rows(n + 5, n, dtype)
    v = _offset(cpu.to(dev), offset)
    idx = torch.randperm(n + 5, generator=torch.Generator().manual_seed(n))[:n]
    want = cpu[:, idx].float().numpy()
    p, s = quantize_int4_value(want)
    got = ro.fused_gather_pack_int4_value(v, idx.to(dev))
    np.testing.assert_array_equal(got.packed.view(2, n, 64).cpu().numpy(), p)
    np.testing.assert_array_equal(got.scale.cpu().numpy(), s)
    for group in (32, 64, 128):
        p, s, z = quantize_int2_value(want, group)
        a = ro.build_compact_int2_value_arena(v, idx.to(dev), group_size=group, append_capacity=7)
        np.testing.assert_array_equal(a.packed[:, :n].cpu().numpy(), p)
        np.testing.assert_array_equal(a.scale[:, :n].cpu().numpy(), s)
        np.testing.assert_array_equal(a.zero_point[:, :n].cpu().numpy(), z)
        assert not a.packed[:, n:].any() and not a.scale[:, n:].any() and not a.zero_point[:, n:].any()


def test_value_packers_at_the_ends_of_the_range():
    """bf16 rows near fp32's largest value (the range overflows), infinities and NaN: a quotient that is not
    a number takes the lowest code, and the rows beside them in the wave keep theirs."""
    import r2omni_amd as ro
    from oracle.quant import quantize_int2_value, quantize_int4_value

    dev = _dev()
    x = _rows(64, 3, "bfloat16", heads=1)
    x[0, 5] = x[0, 5] * 2.0 ** 126                  # past the fast quotient's range
    x[0, 6, ::2], x[0, 6, 1::2] = 3.0e38, -3.0e38   # a range of infinity over finite values
    x[0, 9, 40] = float("inf")
    x[0, 10, 41] = float("nan")
    x[0, 11] = float("nan")
    x[0, 14] = x[0, 14] * 2.0 ** -130               # subnormal
    v = x.to(dev)
    nan, inf = torch.isnan(x).numpy(), torch.isinf(x).numpy()
    clean = torch.where(torch.isnan(x), torch.zeros_like(x), x).float().numpy()  # 0 is in every range
    with np.errstate(invalid="ignore", over="ignore"):
        p4, s4 = quantize_int4_value(clean)
        p2, s2, z2 = quantize_int2_value(clean, 64)

    def codes(packed, bits):
        return np.stack([(packed >> (bits * i)) & (2 ** bits - 1) for i in range(8 // bits)], -1).reshape(1, 64, 128)

    w4, w2 = codes(p4, 4), codes(p2, 2)
    w4[nan | inf] = 9       # -7
    w2[nan | inf] = 0
    got = ro.fused_gather_pack_int4_value(v, torch.arange(64, device=dev))
    np.testing.assert_array_equal(codes(got.packed.view(1, 64, 64).cpu().numpy(), 4), w4)
    np.testing.assert_array_equal(got.scale.cpu().numpy(), s4)
    a = ro.build_compact_int2_value_arena(v, torch.arange(64, device=dev), group_size=64)
    np.testing.assert_array_equal(codes(a.packed[:, :64].cpu().numpy(), 2), w2)
    np.testing.assert_array_equal(a.scale[:, :64].cpu().numpy(), s2)
    np.testing.assert_array_equal(a.zero_point[:, :64].cpu().numpy(), z2)


KEYS = {4: ("build_compact_int4_key_arena", "quantize_int4_key_per_channel", "dequantize_int4_key"),
        2: ("build_compact_int2_key_arena", "quantize_int2_key_per_channel", "dequantize_int2_key")}


@pytest.mark.parametrize("dtype", sorted(DTYPES))
@pytest.mark.parametrize("bits,superblock", [(b, sb) for b in (4, 2) for sb in (32, 64, 128)])
@pytest.mark.parametrize("n,offset", [(1, 0), (31, 2), (33, 0), (127, 0), (128, 0), (161, 8), (700, 0)])
def test_key_packers_match_the_oracle_through_a_flush(n, offset, bits, superblock, dtype):
    """A gathered build of n tokens, then a flush of 128 that requantises the partial tail superblock."""
    import r2omni_amd as ro
    from oracle import quant

    dev = _dev()
    build, quantise, dequantise = KEYS[bits]
    quantise, dequantise = getattr(quant, quantise), getattr(quant, dequantise)
    cpu = torch.cat([_rows(128, n + 17 * b, dtype).transpose(1, 2) for b in range(n // 128 + 1)] + [_rows(3, n, dtype)], 1)
    cpu = cpu[:, -(n + 3):].contiguous()  # the row kinds as channel kinds
    idx = torch.randperm(n + 3, generator=torch.Generator().manual_seed(n))[:n]
    segments = [idx[: n // 2].to(dev), idx[n // 2: n // 2].to(dev), idx[n // 2:].to(dev)]
    arena = getattr(ro, build)(_offset(cpu.to(dev), offset), segments, append_capacity=256, superblock_size=superblock)
    src = cpu[:, idx].float().numpy()

    def check(total, packed, scale, zero, first=0):
        blocks = -(-total // superblock)
        np.testing.assert_array_equal(arena.packed[:, first:total].cpu().numpy(), packed)
        np.testing.assert_array_equal(arena.scale[:, first // superblock:blocks].cpu().numpy(), scale)
        np.testing.assert_array_equal(arena.zero_point[:, first // superblock:blocks].cpu().numpy(), zero)
        assert not arena.packed[:, total:].any() and not arena.scale[:, blocks:].any()
        assert not arena.zero_point[:, blocks:].any() and not arena.kernel_operands[:, blocks:].any()

    packed, scale, zero = quantise(src, superblock)
    check(n, packed, scale, zero)
    ring = _rows(130, n + 1, dtype)
    first = n // superblock * superblock
    old = quant.round_to_dtype(dequantise(packed, scale, zero, first, n - first, superblock), dtype)
    arena.append_superblock(ring.to(dev)[:, :128], source_tokens=130)
    want = quantise(np.concatenate((old, ring[:, :128].float().numpy()), axis=1), superblock)
    check(n + 128, *want, first=first)


def test_int4_key_packer_at_the_ends_of_the_range():
    """Channels whose range overflows fp32, holds infinities or NaN or is subnormal; the channels beside them
    in a lane keep theirs."""
    import r2omni_amd as ro
    from oracle.quant import quantize_int4_key_per_channel

    dev = _dev()
    x = _rows(64, 5, "bfloat16", heads=1)
    x[0, :, 3] *= 2.0 ** 126
    x[0, ::2, 8], x[0, 1::2, 8] = 3.0e38, -3.0e38
    x[0, 7, 17] = float("inf")
    x[0, 40, 26] = float("nan")
    x[0, :, 35] = float("nan")
    x[0, :, 44] *= 2.0 ** -130
    nan, inf = torch.isnan(x).numpy(), torch.isinf(x).numpy()
    with np.errstate(invalid="ignore", over="ignore"):
        packed, scale, zero = quantize_int4_key_per_channel(torch.where(torch.isnan(x), torch.zeros_like(x), x).float().numpy(), 32)
    codes = np.stack((packed & 15, packed >> 4), -1).reshape(1, 64, 128)
    codes[nan | inf] = 0
    arena = ro.build_compact_int4_key_arena(x.to(dev), [torch.arange(64, device=dev)] + [torch.arange(0, device=dev)] * 2,
                                            superblock_size=32)
    got = arena.packed[:, :64].cpu().numpy()
    np.testing.assert_array_equal(np.stack((got & 15, got >> 4), -1).reshape(1, 64, 128), codes)
    np.testing.assert_array_equal(arena.scale[:, :2].cpu().numpy(), scale)
    np.testing.assert_array_equal(arena.zero_point[:, :2].cpu().numpy(), zero)


@pytest.mark.parametrize("append", [False, True])
@pytest.mark.parametrize("ring,superblock,variant,gen", [
    (128, 32, "v_fourq_k_int4_compact", "int2"), (256, 128, "v_fourq_k_int2_compact", "int2"),
    (384, 64, "v_fourq_k_int4_compact", "int4"), (160, 32, "v_fourq_k_int4_compact", "int2")])
def test_ring_flush_is_its_parts(ring, superblock, variant, gen, append):
    """Two flushes in one call each, against the arenas' own appends and a ring moved by torch (rings that
    move nothing, less than a flush, one flush and two)."""
    import r2omni_amd as ro
    from r2omni_amd.policy import PageClass, plan_from_pages

    dev = _dev()
    pages = 9
    plan = plan_from_pages([32 * i for i in range(pages)], [32] * pages,
                           [int((PageClass.FP_PAGE, PageClass.INT4_PAGE, PageClass.INT2_PAGE)[i % 3]) for i in range(pages)],
                           recent_fp_capacity=ring, device=dev)
    gen_k = torch.Generator().manual_seed(ring)
    k, v = (torch.randn(3, 32 * pages, 128, generator=gen_k).to(torch.bfloat16).to(dev) for _ in range(2))
    kw = dict(page_size=32, key_quantization_superblock=superblock, cache_variant=variant, generated_value_precision=gen,
              compact_key_append_capacity=512)
    cache, parts = (ro.build_three_precision_cache(k, v, plan, **kw) for _ in range(2))
    stats, at = ro.DynamicCacheStats(), 32 * pages
    rows = torch.randn(2, 700, 3, 1, 128, generator=gen_k).to(torch.bfloat16).to(dev)
    want_ring = []  # (k row, v row, global, logical)
    for step in range(2):
        while cache.recent_fp_pool.active_length < ring:
            i = at - 32 * pages
            ro.append_generated_token(cache, rows[0, i], rows[1, i], global_token_index=at, logical_position=3 * at, stats=stats)
            want_ring.append((rows[0, i, :, 0], rows[1, i, :, 0], at, 3 * at))
            at += 1
        oldest = want_ring[:128]
        kb, vb = (torch.stack([r[e] for r in oldest], 1).contiguous() for e in (0, 1))
        parts.compact_key.append_superblock(kb)
        if gen == "int4":
            parts.compact_int4_value.append_block(vb)
            parts.metadata_arena.append_int4_pages(parts.int4_pool, *(torch.tensor([r[e] for r in oldest], device=dev) for e in (2, 3)), 32)
        else:
            parts.compact_value.append_superblock(vb)
            parts.metadata_arena.append_int2_pages(parts.int2_pool, *(torch.tensor([r[e] for r in oldest], device=dev) for e in (2, 3)), 32)
        want_ring = want_ring[128:]
        if append:
            i = at - 32 * pages
            assert ro.append_generated_token(cache, rows[0, i], rows[1, i], global_token_index=at, logical_position=3 * at, stats=stats)
            want_ring.append((rows[0, i, :, 0], rows[1, i, :, 0], at, 3 * at))
            at += 1
        else:
            assert ro.flush_full_recent_pool(cache, stats)
        n, pool = len(want_ring), cache.recent_fp_pool
        assert pool.active_length == n == int(pool.length_device)
        assert pool.page_index.lengths.tolist() == [min(max(n - 32 * p, 0), 32) for p in range(ring // 32)]
        for e, t in ((0, pool.fp_k), (1, pool.fp_v)):
            if n:
                assert torch.equal(t[:, :n], torch.stack([r[e] for r in want_ring], 1))
        assert pool.global_index_buffer[:n].tolist() == [r[2] for r in want_ring]
        assert pool.logical_position_buffer[:n].tolist() == [r[3] for r in want_ring]
        a, b = cache.compact_key, parts.compact_key
        for x, y in ((a.packed, b.packed), (a.scale, b.scale), (a.zero_point, b.zero_point), (a.kernel_operands, b.kernel_operands)):
            assert torch.equal(x, y)
        a, b = (c.compact_int4_value if gen == "int4" else c.compact_value for c in (cache, parts))
        assert a.active_length == b.active_length and torch.equal(a.packed, b.packed) and torch.equal(a.scale, b.scale)
        for x, y in zip(cache.pools[:3], parts.pools[:3]):
            for f in ("original_page_ids", "physical_offsets", "lengths", "global_token_indices", "logical_positions"):
                assert torch.equal(getattr(x.page_index, f), getattr(y.page_index, f))
    assert stats.flushed_tokens == 256


@pytest.mark.parametrize("variant,gen,superblock", [("v_fourq_k_int4_compact", "int2", 32), ("v_fourq_k_int2_compact", "int4", 128)])
@pytest.mark.parametrize("row,ring,arena", [(1, 0, 0), (4, 0, 0), (0, 1, 0), (0, 0, 1), (0, 0, 4), (3, 4, 1)])
def test_a_flush_of_buffers_off_16_bytes(row, ring, arena, variant, gen, superblock):
    """The appended row, the ring's rows or the arenas start ``row``, ``ring``, ``arena`` elements into their memory:
    the flush that ends with an append moves and packs them in smaller pieces, to the same bytes."""
    import r2omni_amd as ro
    from r2omni_amd.policy import PageClass, plan_from_pages

    dev = _dev()
    cls = [int((PageClass.FP_PAGE, PageClass.INT4_PAGE, PageClass.INT2_PAGE)[i % 3]) for i in range(5)]
    plan = plan_from_pages([32 * i for i in range(5)], [32] * 5, cls, recent_fp_capacity=256, device=dev)
    g = torch.Generator().manual_seed(row + 10 * ring + 100 * arena)
    k, v = (torch.randn(3, 160, 128, generator=g).to(torch.bfloat16).to(dev) for _ in range(2))
    kw = dict(page_size=32, key_quantization_superblock=superblock, cache_variant=variant, generated_value_precision=gen,
              compact_key_append_capacity=512)
    want, cache = (ro.build_three_precision_cache(k, v, plan, **kw) for _ in range(2))
    pool, key = cache.recent_fp_pool, cache.compact_key
    value = cache.compact_int4_value if gen == "int4" else cache.compact_value
    if ring:
        pool.fp_k, pool.fp_v = _offset(pool.fp_k, ring), _offset(pool.fp_v, ring)
    if arena:
        for a, names in ((key, ("packed", "scale", "zero_point")), (value, ("packed", "scale") + ("zero_point",) * (gen == "int2"))):
            for name in names:
                setattr(a, name, _offset(getattr(a, name), arena))
    rows = torch.randn(2, 257, 3, 1, 128, generator=g).to(torch.bfloat16).to(dev)
    for c, off in ((want, 0), (cache, row)):
        stats = ro.DynamicCacheStats()
        for i in range(257):
            flushed = ro.append_generated_token(c, _offset(rows[0, i], off), _offset(rows[1, i], off), global_token_index=160 + i,
                                                logical_position=7 * i, stats=stats)
        assert flushed and stats.flushed_tokens == 128

    def tensors(c):
        p, a = c.recent_fp_pool, c.compact_int4_value if gen == "int4" else c.compact_value
        return [*c.compact_key.allocation_tensors(), *a.allocation_tensors(), p.fp_k[:, :129], p.fp_v[:, :129],
                p.global_index_buffer[:129], p.logical_position_buffer[:129], p.length_device, p.page_index.lengths,
                c.metadata_arena.storage]

    for x, y in zip(tensors(cache), tensors(want)):
        assert torch.equal(x, y)
