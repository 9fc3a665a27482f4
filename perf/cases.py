"""Performance cases of the SSPA packed-KV path, each through the package's public entry points.

Four kinds of work, as the model integration issues them for every decoder layer:
  decode  one split-K attention call with the fused Recent-FP append (every layer of every decode step)
  build   the packed cache of a prompt (once per layer after prefill)
  rotate  a prompt's Q/K rotation and the Hadamard transform of the K and V rows that are cached
  flush   the append of a token to a full Recent-FP ring (once per layer every 128 decode steps)
The head geometries are the Qwen2.5-Omni 3B and 7B language models' and MiniCPM-o-4.5's; lengths, tiers,
superblocks and groups those of ``r2omni_amd.workloads.CONFIGS`` and of the benchmark, and odd ones.
Inputs: N(0, 1) rows with 4 key outlier channels x 8, a precision tier per page drawn from the case's
shares (what is left of 1 is evicted), pages that end where the modality changes when ``ragged``.  Each
query head looks for one token of the history, as a trained model's heads do: without that every output
is an average of thousands of independent rows, next to zero.
"""
import math
import os
import random
import sys

import torch

sys.path.insert(0, os.path.abspath("r2-omni_amd"))

import r2omni_amd as ro  # noqa: E402

D = 128
RING = 128  # the manager's Recent-FP capacity for the released profiles
SECTIONS = (16, 24, 24)
GEOMETRY = {"3b": (16, 2), "7b": (28, 4), "minicpm": (32, 8)}
TIERS = ("fp", "int4", "int2")
VARIANT = {"int4": "v_fourq_k_int4_compact", "int2": "v_fourq_k_int2_compact", "bf16": "v_fourq_k_bf16",
           "matched": "v_fourq_k_int4_compact"}


def _cache(model, shares, keys="int4", superblock=32, group=32, dtype="bfloat16", page=64, ragged=False, gen="int2"):
    hq, hkv = GEOMETRY[model]
    return {"hq": hq, "hkv": hkv, "fp": shares[0], "int4": shares[1], "int2": shares[2], "keys": keys,
            "superblock": superblock, "group": group, "dtype": dtype, "page": page, "ragged": ragged, "gen": gen}


def _decode(name, lengths, recent, cache, rotary="", hadamard=True):
    return {"name": name, "op": "decode", "lengths": ",".join(map(str, lengths)), "recent": recent, "rotary": rotary,
            "hadamard": hadamard, **cache}


def listed():
    return [
        # the smallest call: a short chat, one request, every value INT4, an empty ring (launches and latency)
        _decode("decode_3b_4k", (4096,), 0, _cache("3b", (0.0, 1.0, 0.0))),
        # one long-context request of the small model, mixed value tiers
        _decode("decode_3b_32k", (32641,), 127, _cache("3b", (0.2, 0.5, 0.3))),
        # the headline: a served batch of uneven requests
        _decode("decode_7b_ragged_8k_64k", (8065, 16257, 32641, 65409), 127, _cache("7b", (0.15, 0.45, 0.4))),
        # a layer of the end-to-end decode: eight 32k requests, the step's mRoPE and Hadamard folded in
        _decode("decode_7b_8x32k_rotary", (32641,) * 8, 127, _cache("7b", (0.15, 0.45, 0.4)), rotary="mrope"),
        # one very long request of the all-lowbit profile
        _decode("decode_minicpm_128k", (130945,), 127, _cache("minicpm", (0.0, 0.0, 1.0), superblock=128, group=128)),
        # the same with INT2 keys
        _decode("decode_minicpm_128k_int2k", (130945,), 127,
                _cache("minicpm", (0.0, 0.0, 1.0), keys="int2", superblock=128, group=128)),
        # a float16 model with unquantised (matched) rows, two requests of odd lengths
        _decode("decode_7b_matched_fp16", (5003, 12289), 40,
                _cache("7b", (0.3, 0.3, 0.3), keys="matched", dtype="float16", page=32, ragged=True), hadamard=False),
        # the cache of a short prompt
        {"name": "build_3b_4k", "op": "build", "tokens": 4096, **_cache("3b", (0.2, 0.5, 0.3), page=32)},
        # the cache of a long prompt, pages cut at modality changes, a part of them evicted
        {"name": "build_7b_64k", "op": "build", "tokens": 65409,
         **_cache("7b", (0.15, 0.4, 0.35), page=32, ragged=True)},
        # the largest prompt, INT2 keys and values
        {"name": "build_minicpm_128k_int2k", "op": "build", "tokens": 130945,
         **_cache("minicpm", (0.0, 0.0, 1.0), keys="int2", superblock=128, group=128)},
        # a long prompt's rotation
        {"name": "rotate_7b_32k", "op": "rotate", "kind": "mrope", "batch": 1, "tokens": 32768, "hq": 28, "hkv": 4,
         "dtype": "bfloat16"},
        # one token into a full ring of 256: the oldest 128 are packed, the rest move down
        {"name": "flush_7b", "op": "flush", "tokens": 16300, "ring": 256, **_cache("7b", (0.15, 0.45, 0.4))},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _draw_cache(rng, keys):
    model = rng.choice(sorted(GEOMETRY))
    a, b, c = (rng.random() for _ in range(3))
    keep = rng.choice((1.0, 1.0, 0.9)) / (a + b + c)
    shares = rng.choice(((a * keep, b * keep, c * keep), (0.15, 0.45, 0.4), (0.0, 1.0, 0.0), (0.0, 0.0, 1.0)))
    return _cache(model, tuple(round(s, 3) for s in shares), keys=rng.choice(keys), superblock=rng.choice((32, 64, 128)),
                  group=rng.choice((32, 64, 128)), dtype=rng.choice(("bfloat16", "bfloat16", "float16")),
                  page=rng.choice((16, 32, 64)), ragged=rng.random() < 0.5)


def draw(rng):
    op = rng.choice(("decode", "decode", "decode", "build", "build", "rotate", "rotate", "flush"))
    if op == "rotate":
        hq, hkv = GEOMETRY[rng.choice(sorted(GEOMETRY))]
        batch = rng.choice((1, 1, 2, 8))
        return {"op": op, "kind": rng.choice(("mrope", "qwen3")), "batch": batch, "hq": hq, "hkv": hkv,
                "tokens": _log_int(rng, 1, 900000 // (batch * (hq + hkv))),
                "dtype": rng.choice(("bfloat16", "bfloat16", "float16"))}
    if op == "build":
        c = _draw_cache(rng, ("int4", "int4", "int2", "bf16", "matched"))
        most = (600000 if c["keys"] in ("bf16", "matched") else 900000) // c["hkv"]
        return {"op": op, "tokens": _log_int(rng, 512, min(131072, most)), **c}
    if op == "flush":
        c = dict(_draw_cache(rng, ("int4", "int4", "int2")), gen=rng.choice(("int2", "int2", "int4")))
        return {"op": op, "tokens": _log_int(rng, 1024, 32768), "ring": rng.choice((128, 256)), **c}
    c = _draw_cache(rng, ("int4", "int4", "int2", "bf16", "matched"))
    wide = 4 if c["keys"] in ("bf16", "matched") else 1  # rows four times as large
    batch = rng.choice((1, 1, 2, 3, 4, 8))
    most = min(131072, 1000000 // (c["hkv"] * batch * wide))
    rotary = rng.choice(("", "", "mrope", "qwen3"))
    case = _decode("", [_log_int(rng, 700, most) for _ in range(batch)], rng.randrange(RING), c, rotary=rotary,
                   hadamard=rng.random() < 0.7)
    del case["name"]
    return case


# ------------------------------------------------------------------------------------------- inputs
def _gen(seed, part):
    return torch.Generator(device="cuda").manual_seed((int(seed) * 1009 + part) & 0x7FFFFFFF)


def _randn(gen, *shape):
    return torch.randn(*shape, generator=gen, device="cuda")


def _dtype(case):
    return getattr(torch, case["dtype"])


def _pages(case, tokens, seed):
    """(offsets, lengths, tier of each page: 0, 1, 2 or 3 = evicted) on the host.  The page lengths and each
    tier's token count are the case's; which of the full pages a tier gets is the seed's."""
    rng = random.Random(tokens)
    page, lengths, left = case["page"], [], tokens
    while left:
        run = min(left, rng.randrange(1, 12 * page) if case["ragged"] else left)
        left -= run
        lengths += [page] * (run // page) + ([run % page] if run % page else [])
    marks = [case["fp"], case["fp"] + case["int4"], case["fp"] + case["int4"] + case["int2"]]
    marks[2] = 1.0 if marks[2] > 0.999 else marks[2]
    tiers = [sum(u >= m for m in marks) for u in (rng.random() for _ in lengths)]
    tiers[0] = min(tiers[0], 2)  # a cache of evicted pages alone is not built
    full = [i for i, n in enumerate(lengths) if n == page]
    for i, t in zip(full, random.Random(seed).sample([tiers[i] for i in full], len(full))):
        tiers[i] = t
    lengths = torch.tensor(lengths)
    return lengths.cumsum(0) - lengths, lengths, torch.tensor(tiers)


def _rows(case, tokens, seed, part):
    """K and V [Hkv, tokens, 128] of one request."""
    gen = _gen(seed, part)
    outliers = torch.randperm(D, generator=torch.Generator().manual_seed(seed * 31 + part))[:4].cuda()
    k = _randn(gen, case["hkv"], tokens, D)
    k[:, :, outliers] *= 8.0
    return k.to(_dtype(case)), _randn(gen, case["hkv"], tokens, D).to(_dtype(case))


def _tables(case, batch, tokens, axes, start=0):
    """cos / sin of three slowly different position streams (text, height, width), as the model forms them."""
    inv = 1.0 / (1.0e6 ** (torch.arange(64, device="cuda", dtype=torch.float64) / 64.0))
    pos = start + torch.arange(tokens, device="cuda", dtype=torch.float64) + 17 * torch.arange(batch, device="cuda")[:, None]
    pos = torch.stack([torch.floor(pos / (a + 1)) for a in range(axes)])
    ang = (pos[..., None] * inv).repeat(1, 1, 1, 2)
    cos, sin = ang.cos().to(_dtype(case)), ang.sin().to(_dtype(case))
    return (cos, sin) if axes == 3 else (cos[0], sin[0])


def _plan(case, tokens, seed, ring):
    offsets, lengths, tiers = _pages(case, tokens, seed)
    cls = torch.tensor([int(ro.PageClass.FP_PAGE), int(ro.PageClass.INT4_PAGE), int(ro.PageClass.INT2_PAGE),
                        int(ro.PageClass.EVICTED_PAGE)])[tiers]
    return ro.plan_from_pages(offsets, lengths, cls, recent_fp_capacity=ring, device="cuda")


def _build(case, k, v, plan):
    return ro.build_three_precision_cache(
        k, v, plan, page_size=case["page"], key_quantization_superblock=case["superblock"],
        int2_group_size=case["group"], generated_value_precision=case["gen"], matched_fp=case["keys"] == "matched",
        cache_variant=VARIANT[case["keys"]], compact_key_append_capacity=260)


def _lengths(case):
    return [int(n) for n in case["lengths"].split(",")]


def _decode_inputs(case, seed):
    """Per request: K, V of the history, K, V of the ring tokens; then the step's query and K / V rows."""
    reqs = []
    for r, n in enumerate(_lengths(case)):
        k, v = _rows(case, n + case["recent"], seed, 2 * r)
        reqs.append((k[:, :n].contiguous(), v[:, :n].contiguous(), k[:, n:].contiguous(), v[:, n:].contiguous()))
    gen, b = _gen(seed, 999), len(reqs)
    q, nk, nv = (_randn(gen, b, h, D) for h in (case["hq"], case["hkv"], case["hkv"]))
    for r, (k, _, _, _) in enumerate(reqs):  # about half of a head's weight on its token
        at = torch.randint(int(k.shape[1]), (case["hq"],), generator=torch.Generator().manual_seed(seed + r)).cuda()
        want = k[torch.arange(case["hq"], device="cuda") // (case["hq"] // case["hkv"]), at].float()
        q[r] += torch.where(want.abs() < 4, want, 0.0) * (0.1 * math.log(int(k.shape[1])) + 0.05)
    if case["rotary"]:  # the projection before its rotation
        cos, sin = _step_tables(case, b)
        q = _hadamard(q) if case["hadamard"] else q
        q = _rotated(case, "mrope" if case["rotary"] == "mrope" else "plain", q[:, :, None], cos, -sin)[:, :, 0]
    return reqs, q.to(_dtype(case)), nk.to(_dtype(case)), nv.to(_dtype(case))


def _step_tables(case, batch):
    return _tables(case, batch, 1, 3 if case["rotary"] == "mrope" else 1, max(_lengths(case)) + case["recent"])


def _norm_weights(case, seed):
    gen = _gen(seed, 998)
    return [(1.4 + 0.1 * _randn(gen, D)).to(_dtype(case)) for _ in range(2)]


# ------------------------------------------------------------------------------------------ prepare
def prepare(case, seed):
    return {"decode": _prepare_decode, "build": _prepare_build, "rotate": _prepare_rotate, "flush": _prepare_flush}[
        case["op"]](case, seed)


def _prepare_decode(case, seed):
    reqs, q, nk, nv = _decode_inputs(case, seed)
    caches, execs = [], []
    for r, (k, v, rk, rv) in enumerate(reqs):
        n = int(k.shape[1])
        cache = _build(case, k, v, _plan(case, n, seed + r, RING))
        for i in range(case["recent"]):
            ro.append_recent_fp_triton(cache, rk[:, i:i + 1], rv[:, i:i + 1], global_token_index=n + i, logical_position=n + i)
        ws = ro.allocate_splitk_workspace(cache, num_query_heads=case["hq"])
        caches.append(cache)
        execs.append(ro.prepare_splitk_executor(cache, ws, output_hadamard=case["hadamard"]))
    ex = execs[0] if len(execs) == 1 else ro.stack_homogeneous_splitk_executors(execs)
    rings = [c.recent_fp_pool for c in caches] if len(execs) == 1 else ex.batched_recent
    rotary = None
    if case["rotary"]:
        cos, sin = _step_tables(case, len(reqs))
        rotary = ro.FusedRotary(cos, sin, SECTIONS, case["hadamard"], case["hadamard"]) if case["rotary"] == "mrope" \
            else ro.FusedQwen3Rotary(cos, sin, *_norm_weights(case, seed), 1e-6, case["hadamard"], case["hadamard"])
    at = [n + case["recent"] for n in _lengths(case)]
    return {"op": "decode", "ex": ex, "q": q, "append": (nk, nv, at, at), "rotary": rotary, "rings": rings,
            "lengths": [case["recent"]] * len(reqs), "caches": caches}


def _prepare_build(case, seed):
    k, v = _rows(case, case["tokens"], seed, 0)
    return {"op": "build", "case": case, "k": k, "v": v, "plan": _plan(case, case["tokens"], seed, RING)}


def _rotate_inputs(case, seed):
    gen, b, t = _gen(seed, 0), case["batch"], case["tokens"]
    return [_randn(gen, b, h, t, D).to(_dtype(case)) for h in (case["hq"], case["hkv"], case["hkv"])]


def _prepare_rotate(case, seed):
    q, k, v = _rotate_inputs(case, seed)
    cos, sin = _tables(case, case["batch"], case["tokens"], 3 if case["kind"] == "mrope" else 1)
    return {"op": "rotate", "kind": case["kind"], "q": q, "k": k, "v": v, "cos": cos, "sin": sin,
            "w": _norm_weights(case, seed)}


def _prepare_flush(case, seed):
    n, ring = case["tokens"], case["ring"]
    k, v = _rows(case, n + ring + 1, seed, 0)
    cache = _build(case, k[:, :n].contiguous(), v[:, :n].contiguous(), _plan(case, n, seed, ring))
    for i in range(n, n + ring):
        ro.append_recent_fp_triton(cache, k[:, i:i + 1], v[:, i:i + 1], global_token_index=i, logical_position=i)
    meta, pool = cache.metadata_arena, cache.int4_pool if case["gen"] == "int4" else cache.int2_pool
    values = cache.compact_int4_value if case["gen"] == "int4" else cache.compact_value
    mark = (cache.compact_key.active_length, values.active_length, meta.int4_page_count, meta.int4_token_count,
            meta.int2_page_count, meta.int2_token_count, pool.page_index)
    return {"op": "flush", "cache": cache, "pool": pool, "values": values, "mark": mark, "ring": ring, "at": n + ring,
            "k": k[:, n + ring:].contiguous(), "v": v[:, n + ring:].contiguous()}


# ---------------------------------------------------------------------------------------------- run
def run(state):
    return {"decode": _run_decode, "build": _run_build, "rotate": _run_rotate, "flush": _run_flush}[state["op"]](state)


def _ring(pool):
    return [pool.fp_k, pool.fp_v, pool.global_index_buffer, pool.logical_position_buffer, pool.length_device]


def _run_decode(s):
    # the step is made again at the same place: a stacked executor counts its rings' tokens itself, a
    # single one leaves that to the caller
    ex = s["ex"]
    if ex.batched_recent_lengths is not None:
        ex.batched_recent_lengths[:] = s["lengths"]
    out = ex(s["q"], append=s["append"], rotary=s["rotary"])
    return [out] + [_ring(r) for r in s["rings"]]


def _arenas(cache):
    ck, kb, cv, i4 = cache.compact_key, cache.bf16_key, cache.compact_value, cache.int4_pool.packed_v
    out = {"fp_v": cache.fp_pool.fp_v}
    if ck is not None:
        out["k"], out["k_scale"], out["k_zero"] = ck.packed, ck.scale, ck.zero_point
    if kb is not None:
        out["k_rows"] = kb.rows
    if cv is not None:
        out["v2"], out["v2_scale"], out["v2_zero"] = cv.packed, cv.scale, cv.zero_point
    if i4 is not None:
        out["v4"], out["v4_scale"] = i4.packed, i4.scale
    return out


def _indexes(cache):
    return [[p.page_index.original_page_ids, p.page_index.physical_offsets, p.page_index.lengths,
             p.page_index.global_token_indices, p.page_index.logical_positions] for p in cache.pools]


def _run_build(s):
    cache = _build(s["case"], s["k"], s["v"], s["plan"])
    return {"arenas": _arenas(cache), "indexes": _indexes(cache), "evicted": cache.evicted_global_indices,
            "ring": _ring(cache.recent_fp_pool)}


def _run_rotate(s):
    """A prompt: the attention takes the rotated Q and K, the cache the Hadamard transform of K and V."""
    if s["kind"] == "mrope":
        q, k = ro.qwen_qk_mrope(s["q"], s["k"], s["cos"], s["sin"], SECTIONS)
    else:
        q, k = ro.qwen3_qk_norm_rope(s["q"], s["k"], *s["w"], s["cos"], s["sin"])
    return [q, k, ro.triton_fwht_128(k), ro.triton_fwht_128(s["v"])]


def _run_flush(s):
    # the flush is made again at the same place: the host's counts go back to the full ring first
    c, m = s["cache"], s["cache"].metadata_arena
    (c.compact_key.active_length, s["values"].active_length, m.int4_page_count, m.int4_token_count, m.int2_page_count,
     m.int2_token_count, s["pool"].page_index) = s["mark"]
    c.recent_fp_pool.active_length = s["ring"]
    ro.append_generated_token(c, s["k"], s["v"], global_token_index=s["at"], logical_position=s["at"],
                              stats=ro.DynamicCacheStats())
    return {"arenas": _arenas(c), "indexes": _indexes(c), "ring": _ring(c.recent_fp_pool)}


# --------------------------------------------------------------------------------------------- work
def _token_bytes(case):
    """Stored bytes of one history token and KV head, (K, V); evicted tokens store nothing."""
    matched = case["keys"] == "matched"
    kept = case["fp"] + case["int4"] + case["int2"]
    k = {"int4": 64 + 384 / case["superblock"], "int2": 32 + 512 / case["superblock"]}.get(case["keys"], 256)
    v = 256 * kept if matched else 256 * case["fp"] + 68 * case["int4"] + (32 + 384 / case["group"]) * case["int2"]
    return k * kept, v


def work(case):
    if case["op"] == "rotate":
        rows, kv = case["batch"] * case["tokens"], case["hkv"]
        return {"bytes": rows * (256 * (2 * case["hq"] + 5 * kv) + 512),
                "flops": rows * D * (3 * (case["hq"] + kv) + 16 * kv)}
    k, v = _token_bytes(case)
    if case["op"] == "build":
        rows = case["tokens"] * case["hkv"]
        kept = case["fp"] + case["int4"] + case["int2"]
        return {"bytes": rows * (512 * kept + k + v) + 32 * case["tokens"], "flops": rows * D * 2 * 6 * kept}
    if case["op"] == "flush":
        move = case["ring"] - 128
        kb = {"int4": 64 + 384 / case["superblock"], "int2": 32 + 512 / case["superblock"]}[case["keys"]]
        vb = 68 if case["gen"] == "int4" else 32 + 384 / case["group"]
        return {"bytes": case["hkv"] * (128 * (512 + kb + vb) + move * 1024 + 1024) + 4096 + 32 * move,
                "flops": case["hkv"] * 128 * D * 2 * 6}
    total, b = sum(_lengths(case)), len(_lengths(case))
    ring = b * (case["recent"] + 1)
    return {"bytes": case["hkv"] * (total * (k + v) + ring * 512) + b * (case["hq"] * 512 + case["hkv"] * 1024),
            "flops": 4 * D * case["hq"] * (total * (case["fp"] + case["int4"] + case["int2"]) + ring)}


def tolerance(case):
    # packed codes, scales, indices and ring rows are defined to the bit
    if case["op"] in ("build", "flush"):
        return "exact"
    if case["op"] == "rotate":
        return {"rel": 2e-3, "max": 1e-2} if case["dtype"] == "bfloat16" else {"rel": 4e-4, "max": 2e-3}
    # bf16 outputs: 0.16 to 0.27 per cent from 64 bits over every key format, measured at 4k to 128k tokens
    return {"rel": 1e-2, "max": 6e-2}


# -------------------------------------------------------------------------------------------- exact
def _hadamard(x):
    h = torch.ones(1, 1, dtype=torch.float64, device=x.device)
    for _ in range(7):
        h = torch.cat((torch.cat((h, h), 1), torch.cat((h, -h), 1)), 0)
    return x.double() @ h / math.sqrt(D)


def _tier_tokens(case, tokens, seed):
    """Token indices of the FP, INT4 and INT2 pools in storage order."""
    offsets, lengths, tiers = _pages(case, tokens, seed)
    if case["keys"] == "matched":
        tiers = torch.where(tiers < 3, 0, 3)
    index = torch.repeat_interleave(torch.arange(len(lengths)), lengths)
    return [torch.nonzero(tiers[index] == t).flatten().cuda() for t in range(3)]


def _blocks(x, sb):
    """[H, S, D] as [H, blocks, sb, D], the last row repeated to the end of its block."""
    pad = -x.shape[1] % sb
    if pad:
        x = torch.cat((x, x[:, -1:].expand(-1, pad, -1)), 1)
    return x.view(x.shape[0], -1, sb, D)


def _divided(x, by):
    return x / torch.full_like(x, by)  # a true quotient: by a number, torch multiplies by its reciprocal on the GPU


def _key_quant(x, case):
    """(scale, dequantised rows in 64 bits) of compact keys [H, S, D] in storage order."""
    n, b = x.shape[1], _blocks(x.float(), case["superblock"])
    if case["keys"] == "int4":
        mn, mx = b.amin(2, keepdim=True).clamp(max=0), b.amax(2, keepdim=True).clamp(min=0)
        step = _divided(mx - mn, 15.0).clamp(min=1e-6)
        zero = torch.round(-mn / step).clamp(0, 15)
        code = torch.round(b / step + zero).clamp(0, 15)
        deq = (code.double() - zero) * step.half().double()
    else:
        mn, mx = b.amin(2, keepdim=True), b.amax(2, keepdim=True)
        span = mx - mn
        step = _divided(span, 3.0)
        inv = torch.where(span > 0, span.clamp(min=1e-30).reciprocal() * 3.0, 0.0)
        zero = torch.where(span > 0, torch.round(-mn * inv), 0.0)
        off = torch.where(span > 0, -zero * step, mn)
        code = torch.round(b * inv + zero).clamp(0, 3)
        deq = code.double() * step.half().double() + off.half().double()
    return step[:, :, 0].double(), deq.reshape(x.shape[0], -1, D)[:, :n]


def _value_quant(x, bits, group):
    x = x.float()
    if bits == 4:
        step = _divided(x.abs().amax(2, keepdim=True), 7.0).clamp(min=1e-6)
        return step.double(), torch.round(x / step).clamp(-7, 7).double() * step.double()
    g = x.view(*x.shape[:2], D // group, group)
    mn, mx = g.amin(3, keepdim=True).clamp(max=0), g.amax(3, keepdim=True).clamp(min=0)
    step = _divided(mx - mn, 3.0).clamp(min=1e-6)
    zero = torch.round(-mn / step).clamp(0, 3)
    code = torch.round(g / step + zero).clamp(0, 3)
    return step.double(), ((code.double() - zero) * step.half().double()).reshape(x.shape)


def _rotate_half(x):
    return torch.cat((-x[..., 64:], x[..., :64]), -1)


def _rotated(case, kind, x, cos, sin, weight=None):
    """The rotation in 64 bits; x [B, H, T, D]."""
    x, cos, sin = x.double(), cos.double(), sin.double()
    if kind == "mrope":
        axis = torch.tensor([0] * SECTIONS[0] + [1] * SECTIONS[1] + [2] * SECTIONS[2], device=x.device).repeat(2)
        cos, sin = (torch.stack([t[a, ..., d] for d, a in enumerate(axis.tolist())], -1) for t in (cos, sin))
    if weight is not None and kind == "qwen3":
        x = x * torch.rsqrt(x.square().mean(-1, keepdim=True) + 1e-6) * weight.double()
    return x * cos[:, None] + _rotate_half(x) * sin[:, None]


def _exact_decode(case, seed):
    reqs, q, nk, nv = _decode_inputs(case, seed)
    dt, kind = _dtype(case), case["rotary"]
    if kind:
        cos, sin = _step_tables(case, len(reqs))
        wq, wk = _norm_weights(case, seed)
        q, nk = _rotated(case, kind, q[:, :, None], cos, sin, wq)[:, :, 0], _rotated(case, kind, nk[:, :, None], cos, sin, wk)[:, :, 0]
        if case["hadamard"]:
            q, nk, nv = _hadamard(q), _hadamard(nk), _hadamard(nv)
        q, nk, nv = q.to(dt), nk.to(dt), nv.to(dt)
    gqa, outs, rings = case["hq"] // case["hkv"], [], []
    for r, (k, v, rk, rv) in enumerate(reqs):
        tiers = _tier_tokens(case, int(k.shape[1]), seed + r)
        order = torch.cat(tiers)
        heads = []
        for h in range(case["hkv"]):
            kk, vv = k[h:h + 1, order], v[h:h + 1]
            kd = _key_quant(kk, case)[1] if case["keys"] in ("int4", "int2") else kk.double()
            if case["keys"] == "matched":
                vd = vv[:, order].double()
            else:
                vd = torch.cat((vv[:, tiers[0]].double(), _value_quant(vv[:, tiers[1]], 4, 0)[1],
                                _value_quant(vv[:, tiers[2]], 2, case["group"])[1]), 1)
            kd = torch.cat((kd[0], rk[h].double(), nk[r, h][None].double()))
            vd = torch.cat((vd[0], rv[h].double(), nv[r, h][None].double()))
            p = torch.softmax(q[r, h * gqa:(h + 1) * gqa].double() @ kd.T / math.sqrt(D), -1)
            heads.append(p @ vd)
        outs.append(torch.cat(heads))
        ring = [torch.zeros(case["hkv"], RING, D, dtype=torch.float64, device="cuda") for _ in range(2)]
        for t, old, new in ((ring[0], rk, nk[r]), (ring[1], rv, nv[r])):
            t[:, :case["recent"]], t[:, case["recent"]] = old.double(), new.double()
        rings.append(ring + [None, None, None])
    out = torch.stack(outs)
    return [_hadamard(out) if case["hadamard"] else out] + rings


def _exact_build(case, seed):
    """The quantisation steps; every other output is whole numbers or rows as they were."""
    k, v = _rows(case, case["tokens"], seed, 0)
    tiers = _tier_tokens(case, case["tokens"], seed)
    out = {}
    if case["keys"] in ("int4", "int2"):
        step = _key_quant(k[:, torch.cat(tiers)], case)[0]
        capacity = max(128, -(-(sum(len(t) for t in tiers) + 260) // 128) * 128)
        out["k_scale"] = torch.zeros(case["hkv"], capacity // case["superblock"], D, dtype=torch.float64, device="cuda")
        out["k_scale"][:, :step.shape[1]] = step
    if case["keys"] != "matched":
        n2, g = len(tiers[2]), D // case["group"]
        out["v2_scale"] = torch.zeros(case["hkv"], max(128, -(-(n2 + 260) // 128) * 128), g, 1, dtype=torch.float64, device="cuda")
        out["v2_scale"][:, :n2] = _value_quant(v[:, tiers[2]], 2, case["group"])[0]
        if len(tiers[1]):
            out["v4_scale"] = _value_quant(v[:, tiers[1]], 4, 0)[0]
    return {"arenas": out} if out else None


def _exact_rotate(case, seed):
    q, k, v = _rotate_inputs(case, seed)
    cos, sin = _tables(case, case["batch"], case["tokens"], 3 if case["kind"] == "mrope" else 1)
    wq, wk = _norm_weights(case, seed)
    q, k = _rotated(case, case["kind"], q, cos, sin, wq), _rotated(case, case["kind"], k, cos, sin, wk)
    return [q, k, _hadamard(k.to(_dtype(case))), _hadamard(v)]


def _exact_flush(case, seed):
    """The ring after the flush; the packed bytes are defined by the stored 32-bit steps alone."""
    n, ring = case["tokens"], case["ring"]
    rows = []
    for x in _rows(case, n + ring + 1, seed, 0):
        r = x[:, n:n + ring].double()
        r[:, :ring - 128] = r[:, 128:].clone()
        r[:, ring - 128] = x[:, n + ring].double()
        rows.append(r)
    return {"ring": rows}


def exact(case, seed):
    return {"decode": _exact_decode, "build": _exact_build, "rotate": _exact_rotate, "flush": _exact_flush}[case["op"]](
        case, seed)
