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
