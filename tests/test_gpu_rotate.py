"""The rotation kernels over a prompt: token counts around a wave's and a block's, head runs split over waves
or not, tables read as aligned runs or element by element, and rows that start off a 16-byte boundary."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

CASES = [
    # batch, hq, hkv, tokens, sections, table form, element offset of q
    (1, 28, 4, 5, (16, 24, 24), "rows", 0),
    (3, 7, 1, 16, (16, 24, 24), "rows", 0),
    (1, 16, 2, 1031, (16, 24, 24), "rows", 0),       # several heads a wave
    (1, 6, 3, 4099, (16, 24, 24), "rows", 1),
    (2, 4, 2, 17, (13, 25, 26), "rows", 0),          # a section ends inside a lane's channels
    (1, 5, 5, 33, (16, 24, 24), "strided", 0),       # channel stride 2
    (1, 5, 5, 33, (64, 0, 0), "offset", 8),
]


def _np32(t):
    return t.detach().float().cpu().numpy()


def _moved(t, elements):
    buf = torch.empty(t.numel() + elements, dtype=t.dtype, device=t.device)
    out = buf[elements:].view(t.shape)
    return out.copy_(t)


def _tables(gen, axes, b, t, form, dtype):
    ang = torch.rand(axes, b, t, 128, generator=gen) * 6.3
    out = []
    for x in (ang.cos().to(dtype).cuda(), ang.sin().to(dtype).cuda()):
        if form == "strided":
            buf = torch.empty(axes, b, t, 256, dtype=dtype, device="cuda")
            buf[..., ::2] = x
            x = buf[..., ::2]
        elif form == "offset":
            x = _moved(x, 3)
        out.append(x)
    return out


@pytest.mark.parametrize("hadamard", [False, True])
@pytest.mark.parametrize("dtype,table", [(torch.bfloat16, torch.bfloat16), (torch.float16, torch.float32)])
@pytest.mark.parametrize("case", range(len(CASES)))
def test_mrope_of_a_prompt_is_bit_exact(case, dtype, table, hadamard):
    import r2omni_amd as ro
    from oracle.quant import normalized_fwht, round_to_dtype
    from oracle.rope import qwen_mrope

    if not torch.cuda.is_available():
        pytest.skip("needs an MI355X")
    b, hq, hkv, t, sections, form, offset = CASES[case]
    gen = torch.Generator().manual_seed(case)
    q, k, v = (_moved(torch.randn(b, h, t, 128, generator=gen).to(dtype).cuda(), offset) for h in (hq, hkv, hkv))
    cos, sin = _tables(gen, 3, b, t, form, table)
    got = ro.qwen_qk_mrope(q, k, cos, sin, sections, apply_hadamard=hadamard, value=v)
    name = str(dtype).split(".")[1]
    for x, y in ((q, got[0]), (k, got[1])):
        np.testing.assert_array_equal(_np32(y), qwen_mrope(_np32(x), _np32(cos), _np32(sin), sections,
                                                           hadamard=hadamard, dtype=name))
    want = round_to_dtype(normalized_fwht(_np32(v)), name) if hadamard else _np32(v)
    np.testing.assert_array_equal(_np32(got[2]), want)
    np.testing.assert_array_equal(_np32(ro.triton_fwht_128(v)), round_to_dtype(normalized_fwht(_np32(v)), name))


def _norm_rope(x, weight, cos, sin, dtype):
    """oracle.rope.qwen3_norm_rope with the squares summed in the kernel's order: x[t]^2 + x[t + 64]^2, then
    halves of t (a sum in another order moves a rounding of the norm, and a difference of two products near
    zero by any number of its own steps)."""
    from oracle.quant import round_to_dtype

    r = lambda v: round_to_dtype(np.asarray(v, dtype=np.float32), dtype)  # noqa: E731
    s = x[..., :64] * x[..., :64] + x[..., 64:] * x[..., 64:]
    while s.shape[-1] > 1:
        half = s.shape[-1] // 2
        s = s[..., :half] + s[..., half:]
    inv = np.float32(1) / np.sqrt(s / np.float32(128) + np.float32(1e-6))
    w = r(weight * r(x * inv))
    rot = np.concatenate((-w[..., 64:], w[..., :64]), axis=-1)
    a, b = r(w * cos[:, None]), r(rot * sin[:, None])
    # the GPU's root may differ in its last bit, which can move x * inv and so the weighted value by a step
    # (spacing at most 2^-7 of a bf16 value, 2^-10 of an fp16 one), each product by another and the sum by one
    unit = 2.0 ** -7 if dtype == "bfloat16" else 2.0 ** -10
    return r(a + b), unit * (3 * np.abs(a) + 3 * np.abs(b) + np.abs(a + b)) + 2.0 ** -24


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("case", range(len(CASES)))
def test_qwen3_norm_rope_of_a_prompt_matches_the_oracle(case, dtype):
    import r2omni_amd as ro

    if not torch.cuda.is_available():
        pytest.skip("needs an MI355X")
    b, hq, hkv, t, _, form, offset = CASES[case]
    gen = torch.Generator().manual_seed(100 + case)
    q, k = (_moved((torch.randn(b, h, t, 128, generator=gen) * 3).to(dtype).cuda(), offset) for h in (hq, hkv))
    wq, wk = ((torch.rand(128, generator=gen) * 2).to(dtype).cuda() for _ in range(2))
    cos, sin = (x[0] for x in _tables(gen, 1, b, t, form, dtype))
    got = ro.qwen3_qk_norm_rope(q, k, wq, wk, cos, sin, eps=1e-6)
    name = str(dtype).split(".")[1]
    for x, w, y in ((q, wq, got[0]), (k, wk, got[1])):
        want, step = _norm_rope(_np32(x), _np32(w), _np32(cos), _np32(sin), name)
        assert (np.abs(_np32(y) - want) <= step).all() and (_np32(y) == want).mean() > 0.999
