"""The decode call's two host routes: the forms that the host module takes and those that it leaves to the
Python path give the same bytes, the same ring and the same errors, on any stream and under graph capture."""
import pytest
import torch

from test_gpu_parity import _cuda

pytestmark = pytest.mark.gpu

TOKENS = 16 * 40 + 20


def _executor(dtype="bfloat16", recent=20, batch=1, stacked=False, native=True, length=None):
    import r2omni_amd as ro
    from r2omni_amd.workloads import DecodeConfig, build_request_cache, make_request

    dev = _cuda()
    cfg = DecodeConfig("t", 8, 2, (TOKENS,) * batch, (0.3, 0.3, 0.4), recent=recent, superblock=32, group=32, page=16, dtype=dtype)
    requests = [make_request(cfg, TOKENS, seed=40 + i, device=dev) for i in range(batch)]
    caches = [build_request_cache(cfg, r) for r in requests]
    parts = [ro.prepare_splitk_executor(c, ro.allocate_splitk_workspace(c, num_query_heads=8)) for c in caches]
    ex = ro.stack_homogeneous_splitk_executors(parts) if stacked else parts[0]
    if not native:
        ex._template = ex._prepare_static()[:3] + (None,)
    return ex, torch.cat([r.query for r in requests]).contiguous()


def _rows(batch, dtype, four=False):
    gen = torch.Generator().manual_seed(5)
    shape = (batch, 2, 1, 128) if four else (batch, 2, 128)
    return [torch.randn(shape, generator=gen).to(getattr(torch, dtype)).cuda() for _ in range(2)]


def _unaligned(t):
    flat = torch.empty(t.numel() + 1, dtype=t.dtype, device=t.device)
    flat[1:] = t.flatten()
    return flat[1:].view(t.shape)


def _ring(ex):
    pools = ex.batched_recent or [c.recent_fp_pool for c in ex.caches]
    return [t.clone() for p in pools for t in (p.fp_k, p.fp_v, p.length_device, p.global_index_buffer, p.logical_position_buffer)]


FORMS = {
    "plain": lambda q, k, v: (q, None),
    "token axis": lambda q, k, v: (q[:, :, None], (k[:, :, None], v[:, :, None], TOKENS, TOKENS)),
    "ints": lambda q, k, v: (q, (k, v, TOKENS, TOKENS + 3)),
    "lists": lambda q, k, v: (q, (k, v, [TOKENS] * len(q), tuple(TOKENS + i for i in range(len(q))))),
    "tensor positions": lambda q, k, v: (q, (k, v, torch.tensor([TOKENS] * len(q)), torch.tensor([7] * len(q)))),
    "unaligned rows": lambda q, k, v: (_unaligned(q), (_unaligned(k), _unaligned(v), TOKENS, TOKENS)),
    "strided token axis": lambda q, k, v: (q, (torch.stack([k, k], 2)[:, :, :1], torch.stack([v, v], 2)[:, :, :1], 1, 2)),
    "other query type": lambda q, k, v: (q.to(torch.float16 if q.dtype == torch.bfloat16 else torch.bfloat16), None),
    "list for a tuple": lambda q, k, v: (q, [k, v, TOKENS, TOKENS]),
    "wrong heads": lambda q, k, v: (q[:, :7].contiguous(), None),
    "strided query": lambda q, k, v: (torch.cat([q, q], 2)[:, :, :128], None),
    "float32 rows": lambda q, k, v: (q, (k.float(), v.float(), 1, 2)),
    "float32 query": lambda q, k, v: (q.float(), None),
    "short rows": lambda q, k, v: (q, (k[:, :1].contiguous(), v[:, :1].contiguous(), 1, 2)),
    "host rows": lambda q, k, v: (q, (k.cpu(), v.cpu(), 1, 2)),
    "too many positions": lambda q, k, v: (q, (k, v, [1] * (len(q) + 1), 2)),
    "fractional position": lambda q, k, v: (q, (k, v, 1.5, 2)),
}


@pytest.mark.parametrize("dtype,batch,stacked", [("bfloat16", 1, False), ("float16", 1, False), ("bfloat16", 3, True)])
@pytest.mark.parametrize("form", FORMS)
def test_both_routes_agree(form, dtype, batch, stacked):
    got = []
    for native in (True, False):
        ex, q = _executor(dtype, batch=batch, stacked=stacked, native=native)
        query, append = FORMS[form](q, *_rows(batch, dtype))
        ex.workspace.output.zero_()
        try:
            result = [ex(query, append).clone(), ex(query, append).clone()], None
        except Exception as e:
            result = None, (type(e), str(e))
        torch.cuda.synchronize()
        got.append((result, _ring(ex), ex.batched_recent_lengths))
    (a, ring_a, own_a), (b, ring_b, own_b) = got
    assert a[1] == b[1] and own_a == own_b
    for x, y in zip([*(a[0] or ()), *ring_a], [*(b[0] or ()), *ring_b]):
        assert torch.equal(x, y)


@pytest.mark.parametrize("stacked", [False, True])
def test_a_full_ring_is_refused_before_the_launch(stacked):
    ex, q = _executor(batch=2 if stacked else 1, stacked=stacked)
    k, v = _rows(len(q), "bfloat16")
    own = ex.batched_recent_lengths
    full = ex.caches[0].recent_fp_pool.capacity
    if stacked:
        own[:] = [3, full]
    else:
        ex.caches[0].recent_fp_pool.active_length = full
    before = _ring(ex)
    with pytest.raises(RuntimeError, match="full Recent-FP pool"):
        ex(q, (k, v, 1, 1))
    torch.cuda.synchronize()
    assert all(torch.equal(x, y) for x, y in zip(before, _ring(ex)))
    assert not stacked or own == [3, full]


def test_replaced_workspace_other_streams_and_capture():
    import r2omni_amd as ro

    ex, q = _executor()
    want = ex(q).clone()
    ex.workspace = ro.allocate_splitk_workspace(ex.caches[0], num_query_heads=8)  # the old one's arguments do not serve
    assert torch.equal(ex(q), want) and ex._template[0] is ex.workspace
    ex.workspace.output = torch.zeros_like(want)  # a caller's own output tensor
    assert ex(q) is ex.workspace.output and torch.equal(ex.workspace.output, want)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    late = torch.zeros_like(q)
    torch.cuda.synchronize()
    with torch.cuda.stream(side):
        late.copy_(q)  # ordered before the call only if the call is on this stream
        got = ex(late).clone()
    side.synchronize()
    assert torch.equal(got, want)
    graph = torch.cuda.CUDAGraph()
    query = q.clone()
    with torch.cuda.graph(graph):
        ex(query)
    for scale in (1.0, 0.5, 1.0):
        query.copy_(q * scale)
        graph.replay()
        torch.cuda.synchronize()
        got = ex.workspace.output.clone()
        assert torch.equal(got, ex(query))


NATIVE = {"plain", "token axis", "ints", "lists", "other query type"}


@pytest.mark.parametrize("dtype,batch,stacked", [("bfloat16", 1, False), ("float16", 1, False), ("bfloat16", 3, True)])
@pytest.mark.parametrize("form", FORMS)
def test_each_form_takes_its_route(form, dtype, batch, stacked, monkeypatch):
    """The forms of a model's step are launched by the host module without reaching the Python path; it leaves
    every other form to that path."""
    from r2omni_amd import _lib

    ex, q = _executor(dtype, batch=batch, stacked=stacked)
    query, append = FORMS[form](q, *_rows(batch, dtype))
    ex(q)  # prepares the handle
    ex.workspace.output.zero_()
    own = None if ex.batched_recent_lengths is None else list(ex.batched_recent_lengths)
    rc = _lib.host().decode(ex._template[3], query, append, ex.workspace.output, ex.caches, own)
    torch.cuda.synchronize()
    assert rc == (0 if form in NATIVE else None)
    assert bool(ex.workspace.output.any()) == (form in NATIVE)

    def python_path(*args):
        raise NotImplementedError("the Python path")

    monkeypatch.setattr(ex, "_prepare_call", python_path)
    if form in NATIVE:
        ex(query, append)
    else:
        with pytest.raises(NotImplementedError):
            ex(query, append)
    torch.cuda.synchronize()
