"""INT2-K decode around the group size where a tile's logits are split over the MFMA's two column halves
(at most 8 query heads per KV head) or not, with segments that end inside a tile, every value tier,
both row dtypes, a fused append and the folded rotation, against the CPU oracle to the decode bar."""
import pytest
import torch

from test_gpu_parity import _bf16_np, _compare, _cuda, _oracle_for

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("gqa", [1, 4, 7, 8, 9, 16])
@pytest.mark.parametrize("probs,superblock,group", [((0.3, 0.3, 0.4), 32, 32), ((0.2, 0.3, 0.5), 64, 64),
                                                    ((0.1, 0.4, 0.5), 128, 128), ((0.0, 0.0, 1.0), 128, 128)])
def test_int2_keys_match_oracle_at_every_group_size(gqa, probs, superblock, group):
    import r2omni_amd as ro
    from r2omni_amd.workloads import DecodeConfig, build_request_cache, make_request
    from oracle.attention import mixed_reference, output_transform
    from oracle.quant import bf16_bits_to_f32

    dev = _cuda()
    cfg = DecodeConfig("t", 2 * gqa, 2, (16 * 83 + 37,), probs, recent=37, superblock=superblock, group=group, page=16,
                       variant="int2k")
    data = make_request(cfg, 16 * 83 + 37, seed=500 + gqa, device=dev)
    cache = build_request_cache(cfg, data)
    ex = ro.prepare_splitk_executor(cache, ro.allocate_splitk_workspace(cache, num_query_heads=2 * gqa), output_hadamard=True)
    out = ex(data.query.contiguous())
    torch.cuda.synchronize()
    q = bf16_bits_to_f32(_bf16_np(data.query))
    _compare(out, output_transform(mixed_reference(q, _oracle_for(data, cfg)), True), f"gqa {gqa} {probs} {group}")


@pytest.mark.parametrize("gqa", [7, 9])
@pytest.mark.parametrize("dtype", ["bfloat16", "float16"])
def test_split_heads_with_append_and_rotation_equal_the_separate_launch(gqa, dtype):
    """The folded rotation reads its query rows by the same head mapping: bit-identical to the call on rows
    that a separate launch rotated, with the appended row and the ring."""
    import r2omni_amd as ro
    from r2omni_amd.workloads import DecodeConfig, build_request_cache, make_request

    dev = _cuda()
    cfg = DecodeConfig("t", 2 * gqa, 2, (16 * 60 + 20,), (0.3, 0.3, 0.4), recent=20, superblock=64, group=32, page=16,
                       variant="int2k", dtype=dtype)
    data = make_request(cfg, 16 * 60 + 20, seed=700 + gqa, device=dev)
    dt = getattr(torch, dtype)
    gen = torch.Generator().manual_seed(gqa)
    k, v = (torch.randn(1, 2, 128, generator=gen).to(dt).to(dev) for _ in range(2))
    ang = torch.rand(3, 1, 1, 128, generator=gen) * 6.3
    cos, sin = ang.cos().to(dt).to(dev), ang.sin().to(dt).to(dev)
    at = 16 * 60 + 20
    got = []
    for fold in (True, False):
        cache = build_request_cache(cfg, data)
        ex = ro.prepare_splitk_executor(cache, ro.allocate_splitk_workspace(cache, num_query_heads=2 * gqa), output_hadamard=True)
        if fold:
            out = ex(data.query, append=(k, v, at, at), rotary=ro.FusedRotary(cos, sin, (16, 24, 24), True, True))
        else:
            q2, k2, v2 = ro.qwen_qk_mrope(data.query[:, :, None], k[:, :, None], cos, sin, (16, 24, 24),
                                          apply_hadamard=True, value=v[:, :, None])
            out = ex(q2[:, :, 0].contiguous(), append=(k2[:, :, 0].contiguous(), v2[:, :, 0].contiguous(), at, at))
        got.append((out.clone(), cache.recent_fp_pool.fp_k, cache.recent_fp_pool.fp_v))
    for a, b in zip(*got):
        assert torch.equal(a, b)
