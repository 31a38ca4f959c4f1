"""The calls a user of this framework makes, as measured cases.

Four public entry points: ``ops.ragged_paged_attention`` (decode, prefill and mixed batches over a
paged K/V pool), ``ops.CapturedCalls`` (a model step's calls as one graph), ``fused.invoke`` (the
fused Inkling decode step) and ``inkling.inkling_rpa`` (the v1 Inkling contract).  Lengths, heads,
page sizes and pools are the benchmark configurations of ``tpu_cake_amd.workloads``, the sizes its
tests sweep, and the shard of a GQA model's heads on one GPU of several (Hq 8 / Hkv 2).

A case fixes every size (lengths come from ``len_seed``); tensor values and the page permutation
come from the seed given to ``prepare``.
"""

import math
import pathlib
import sys

import numpy as np
import torch

_PACKAGE = str(pathlib.Path(__file__).resolve().parent.parent / "tpu-cake_amd")
if _PACKAGE not in sys.path:
    sys.path.insert(0, _PACKAGE)

from tpu_cake_amd import fused, inkling, ops  # noqa: E402

POOL_FACTOR = 1.25  # pages in the pool per page in use (the benchmark's choice)
FP8_MAX = 448.0
SIGMA = 0.5         # of the log-normal lengths (the benchmark's choice)

# the most one pass of a listed case reads and computes: drawn cases stay below
MAX_BYTES = 640e6
MAX_FLOPS = 360e9


def _operator(name, **sizes):
    """One ``ragged_paged_attention`` call: ``decode`` sequences of one query token, then ``chunks``
    sequences of chunk_lo..chunk_hi query tokens over 0..prior_hi earlier keys."""
    case = dict(kind="operator", decode=0, lens="uniform", len_lo=1, len_hi=1, median=2048, chunks=0, chunk_lo=0,
                chunk_hi=0, prior_hi=0, hq=32, hkv=8, dim=128, page=64, max_len=8192, dtype="bf16", window=0,
                soft_cap=0.0, layers=0, spare=0, len_seed=98)
    case.update(sizes)
    return dict(case, name=name) if name else case


def listed():
    return [
        # the smallest call: four short sequences on a model shard, page 16; launches and latency count
        _operator("tiny_decode", decode=4, len_lo=1, len_hi=512, hq=8, hkv=2, page=16, max_len=512, len_seed=97),
        # the same kind of step as a serving loop runs it: 16 layers' calls captured into one graph, the
        # batch padded to its bucket (6 live sequences of 8)
        _operator("graph_decode_step", decode=6, spare=2, len_lo=1, len_hi=512, hq=8, hkv=2, page=16, max_len=512,
                  layers=16, len_seed=96),
        # the benchmark's headline: GQA decode over ragged lengths
        _operator("gqa_decode", decode=64, lens="lognormal", len_lo=128, len_hi=8192),
        # the same batch over an fp8 cache with per-(page, head) scales
        _operator("fp8_decode", decode=64, lens="lognormal", len_lo=128, len_hi=8192, dtype="fp8"),
        # many users, most with short contexts, one or two very long ones
        _operator("heavy_tail_decode", decode=256, lens="pareto", len_lo=16, len_hi=131072, hq=64, max_len=131072,
                  len_seed=101),
        # decode in a sliding-window layer
        _operator("window_decode", decode=64, lens="lognormal", len_lo=128, len_hi=8192, window=512),
        # continuous batching: decode rows beside prefill chunks
        _operator("mixed_batch", decode=24, len_lo=512, len_hi=8192, chunks=4, chunk_lo=512, chunk_hi=512,
                  prior_hi=3584, len_seed=99),
        # new prompts only, whole and causal, ragged lengths: the largest compute
        _operator("prompt_prefill", chunks=4, chunk_lo=2048, chunk_hi=6144, len_seed=103),
        # a model shard's chunked prefill with a few decode rows, page 16, odd lengths
        _operator("shard_prefill", decode=9, len_lo=1, len_hi=2048, chunks=5, chunk_lo=33, chunk_hi=1023,
                  prior_hi=1500, hq=8, hkv=2, page=16, max_len=4096, len_seed=104),
        # continuous batching of a model with 64-dim heads
        _operator("mixed_batch_d64", decode=24, len_lo=512, len_hi=8192, chunks=4, chunk_lo=512, chunk_hi=512,
                  prior_hi=3584, dim=64, len_seed=99),
        # the fused Inkling decode step: cache write, relative bias and attention
        dict(name="inkling_fused_step", kind="fused", seqs=64, median=2048, hq=32, hkv=8, dim=128, page=64, rel_dim=16,
             rel_extent=512, len_seed=102),
        # the v1 Inkling contract at its own shapes
        dict(name="inkling_v1_contract", kind="v1", seqs=4, len_lo=1, len_hi=128, hq=4, hkv=4, dim=32, page=16,
             len_seed=0),
    ]


def _log(rng, lo, hi):
    """An integer in [lo, hi], spread evenly over its logarithm."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    while True:
        case = _draw(rng)
        w = work(case)
        if w["bytes"] <= MAX_BYTES and w["flops"] <= MAX_FLOPS:
            return case


def _draw(rng):
    family = rng.choice(["small", "small", "decode", "decode", "decode", "mixed", "mixed", "prefill", "prefill", "graph",
                         "fused", "v1"])
    seed = rng.randrange(1 << 30)
    hkv = rng.choice([1, 2, 4, 8])
    hq = hkv * rng.choice([1, 4, 4, 8])
    page = rng.choice([16, 16, 32, 64, 64, 128])
    if family == "fused":
        return dict(kind="fused", seqs=_log(rng, 1, 96), median=_log(rng, 128, 4096), hq=hq, hkv=hkv,
                    dim=rng.choice([64, 128, 128]), page=page, rel_dim=16, rel_extent=rng.choice([128, 512]),
                    len_seed=seed)
    if family == "v1":
        return dict(kind="v1", seqs=_log(rng, 1, 16), len_lo=1, len_hi=_log(rng, 64, 1500), hq=hq, hkv=hkv,
                    dim=rng.choice([32, 64, 128]), page=rng.choice([16, 32, 64]), len_seed=seed)
    base = dict(hq=hq, hkv=hkv, dim=rng.choice([64, 128, 128, 128, 256]), page=page, len_seed=seed,
                dtype=rng.choice(["bf16", "bf16", "bf16", "fp8"]))
    if rng.random() < 0.2:
        base["window"] = _log(rng, 128, 4096)
    if rng.random() < 0.1:
        base["soft_cap"] = 50.0
    if family in ("small", "graph"):  # short contexts, few sequences
        hi = _log(rng, 64, 1024)
        base.update(decode=_log(rng, 1, 32), len_lo=1, len_hi=hi, max_len=max(512, 1 << (hi - 1).bit_length()))
        if family == "graph":
            base.update(layers=rng.randint(8, 32), spare=rng.randint(0, 3), decode=_log(rng, 1, 16))
    elif family == "decode":
        lens = rng.choice(["lognormal", "uniform", "pareto"])
        hi = _log(rng, 1024, 131072) if lens == "pareto" else _log(rng, 1024, 16384)
        base.update(decode=_log(rng, 2, 320), lens=lens, len_lo=16, len_hi=hi, median=_log(rng, 256, 4096),
                    max_len=max(2048, 1 << (hi - 1).bit_length()))
    elif family == "mixed":
        base.update(decode=_log(rng, 1, 64), len_lo=64, len_hi=_log(rng, 512, 8192), chunks=rng.randint(1, 6),
                    chunk_lo=_log(rng, 16, 128), chunk_hi=_log(rng, 128, 1024), prior_hi=_log(rng, 64, 4096),
                    max_len=16384)
    else:
        base.update(chunks=_log(rng, 1, 8), chunk_lo=_log(rng, 64, 512), chunk_hi=_log(rng, 512, 6144),
                    prior_hi=rng.choice([0, 0, 1024]), max_len=8192)
    return _operator(None, **base)


def _lengths(case):
    """(kv lengths, query lengths) of the case's sequences."""
    rng = np.random.default_rng(case["len_seed"])
    if case["kind"] == "fused":
        z = rng.standard_normal(case["seqs"])
        lens = np.clip(np.rint(np.exp(math.log(case["median"]) + SIGMA * z)), 1, 8192).astype(np.int64)
        return lens, np.ones_like(lens)
    if case["kind"] == "v1":
        lens = rng.integers(case["len_lo"], case["len_hi"], size=case["seqs"], endpoint=True)
        return lens, np.ones_like(lens)
    n, lo, hi = case["decode"], case["len_lo"], case["len_hi"]
    if case["lens"] == "lognormal":
        lens = np.rint(np.exp(math.log(case["median"]) + SIGMA * rng.standard_normal(n)))
    elif case["lens"] == "pareto":
        lens = np.floor(16.0 * (1.0 + rng.pareto(1.2, size=n)))
    else:
        lens = rng.integers(lo, hi, size=n, endpoint=True)
    lens = np.clip(lens, lo, hi).astype(np.int64)
    prior = rng.integers(0, case["prior_hi"], size=case["chunks"], endpoint=True)
    chunk = rng.integers(case["chunk_lo"], max(case["chunk_lo"], case["chunk_hi"]), size=case["chunks"], endpoint=True)
    return np.concatenate([lens, prior + chunk]), np.concatenate([np.ones(n, np.int64), chunk])


def _normal(shape, seed, stream, scale=1.0):
    g = torch.Generator(device="cuda").manual_seed(int(seed) * 64 + stream)
    return (torch.randn(shape, generator=g, device="cuda", dtype=torch.float32) * scale).to(torch.bfloat16)


def _int32(values):
    return torch.as_tensor(np.ascontiguousarray(values, dtype=np.int32)).cuda()


def _page_lists(lens, page, seed):
    """Each sequence's pages out of a shuffled pool: (lists, pages in the pool)."""
    need = -(-lens // page)
    pool = max(1, math.ceil(POOL_FACTOR * int(need.sum())))
    perm = np.random.default_rng(seed).permutation(pool).astype(np.int32)
    return np.split(perm[: int(need.sum())], np.cumsum(need)[:-1]), pool


def _quantize(kv):
    """fp8-e4m3 codes and fp32 scales max|x| / 448 per (page, kv head, K or V)."""
    pages, page, comb, dim = kv.shape
    scales = torch.empty(pages, comb // 2, 2, dtype=torch.float32, device="cuda")
    codes = torch.empty(kv.shape, dtype=torch.float8_e4m3fn, device="cuda")
    for p0 in range(0, pages, 256):
        x = kv[p0:p0 + 256].float().view(-1, page, comb // 2, 2, dim)
        amax = x.abs().amax(dim=(1, 4))
        s = torch.where(amax > 0, amax / FP8_MAX, torch.ones_like(amax))
        codes[p0:p0 + 256] = (x / s[:, None, :, :, None]).clamp_(-FP8_MAX, FP8_MAX).view(-1, page, comb, dim).to(codes.dtype)
        scales[p0:p0 + 256] = s
    return codes, scales


def _operator_inputs(case, seed):
    """(args, keywords) of each layer's call; the metadata is shared, as in a model step."""
    lens, qlens = _lengths(case)
    n, rows = len(lens), len(lens) + case["spare"]
    lists, pool = _page_lists(lens, case["page"], seed)
    table = np.zeros((rows, -(-case["max_len"] // case["page"])), np.int32)  # unused slots hold page 0
    for i, pages in enumerate(lists):
        table[i, :len(pages)] = pages
    cu = np.zeros(rows + 1, np.int32)
    cu[1:n + 1] = np.cumsum(qlens)
    cu[n + 1:] = cu[n]
    meta = (_int32(np.concatenate([lens, np.zeros(case["spare"])])), _int32(table), _int32(cu), _int32([n]))
    keywords = dict(sm_scale=1.0 / math.sqrt(case["dim"]), sliding_window=case["window"] or None,
                    soft_cap=case["soft_cap"] or None)
    calls = []
    for layer in range(max(1, case["layers"])):
        q = _normal((int(cu[-1]) + case["spare"], case["hq"], case["dim"]), seed, 2 * layer)
        kv = _normal((pool, case["page"], 2 * case["hkv"], case["dim"]), seed, 2 * layer + 1)
        more = {}
        if case["dtype"] == "fp8":
            kv, more["kv_scales"] = _quantize(kv)
        calls.append(((q, kv, *meta), dict(keywords, **more)))
    return calls


def _fused_inputs(case, seed):
    lens, _ = _lengths(case)
    lists, pool = _page_lists(lens, case["page"], seed)
    n, hq, hkv, dim = case["seqs"], case["hq"], case["hkv"], case["dim"]
    cache = _normal((pool, case["page"], 2 * hkv, 128), seed, 3, 0.25)
    cache[..., dim:] = 0  # rows are padded to 128 with zeros
    cu_kv = np.concatenate([[0], np.cumsum(-(-lens // case["page"]) * case["page"])])
    return (_normal((n, hq, dim), seed, 0), _normal((n, hkv, dim), seed, 1), _normal((n, hkv, dim), seed, 2), cache,
            _int32(lens), _int32(np.concatenate(lists)), _int32(np.arange(n + 1)), _int32(cu_kv), _int32([n] * 3),
            _normal((n, hq, case["rel_dim"]), seed, 4, 0.4), _normal((case["rel_dim"], case["rel_extent"]), seed, 5, 0.4))


def _v1_inputs(case, seed):
    lens, _ = _lengths(case)
    per_seq = -(-case["len_hi"] // case["page"])
    n, hkv, dim = case["seqs"], case["hkv"], case["dim"]
    table = np.random.default_rng(seed).permutation(n * per_seq).reshape(n, per_seq)
    pool = (n * per_seq, case["page"], hkv, dim)
    return (_normal((n, case["hq"], dim), seed, 0), _normal(pool, seed, 1), _normal(pool, seed, 2), _int32(table),
            _int32(lens), _normal((case["hq"], case["len_hi"]), seed, 3, 0.5))


def prepare(case, seed):
    if case["kind"] == "fused":
        lens, _ = _lengths(case)  # an engine knows its lengths on the host
        return {"kind": "fused", "args": _fused_inputs(case, seed), "pages_per_seq": int((-(-lens // case["page"])).max())}
    if case["kind"] == "v1":
        return {"kind": "v1", "args": _v1_inputs(case, seed)}
    calls = _operator_inputs(case, seed)
    if case["layers"]:
        return {"kind": "graph", "step": ops.CapturedCalls(calls)}
    return {"kind": "operator", "call": calls[0]}


def run(state):
    if state["kind"] == "operator":
        args, keywords = state["call"]
        return ops.ragged_paged_attention(*args, **keywords)
    if state["kind"] == "graph":
        return state["step"].replay()
    if state["kind"] == "fused":
        return fused.invoke(*state["args"], pages_per_seq=state["pages_per_seq"])
    return inkling.inkling_rpa(*state["args"])


def _visible(lens, qlens, window):
    """Per sequence: (keys read, sum over query tokens of the keys each sees)."""
    for length, ql in zip(lens.tolist(), qlens.tolist()):
        hi = length - ql + 1 + np.arange(ql, dtype=np.int64)
        lo = np.maximum(hi - window, 0) if window else np.zeros_like(hi)
        yield int(hi[-1] - lo[0]), int((hi - lo).sum())


def work(case):
    lens, qlens = _lengths(case)
    layers = max(1, case.get("layers", 0))
    seen = list(_visible(lens, qlens, case.get("window", 0)))
    keys, visible = sum(s[0] for s in seen), sum(s[1] for s in seen)
    tokens = int(qlens.sum())
    elem = 1 if case.get("dtype") == "fp8" else 2
    pages = sum(-(-s[0] // case["page"]) for s in seen)
    size = 2 * keys * case["hkv"] * case["dim"] * elem + 4 * tokens * case["hq"] * case["dim"]
    size += 4 * (pages + 2 * len(lens))
    if elem == 1:
        size += 8 * pages * case["hkv"]
    flops = 4 * visible * case["hq"] * case["dim"]
    if case["kind"] == "fused":
        # the cache's rows are 128 wide whatever the head dim; the new rows are read and written once
        biased = int(np.minimum(lens, case["rel_extent"]).sum())
        size += 2 * keys * case["hkv"] * (128 - case["dim"]) * 2 + 8 * len(lens) * case["hkv"] * case["dim"]
        size += 2 * case["rel_dim"] * (case["rel_extent"] + len(lens) * case["hq"])
        flops += 2 * biased * case["hq"] * case["rel_dim"]
    if case["kind"] == "v1":
        size += 2 * case["hq"] * int(lens.max())
    return {"bytes": layers * size, "flops": layers * flops}


def tolerance(case):
    # bf16 outputs from fp32 sums, probabilities rounded to bf16 against a moving maximum, fp8 pools'
    # V dequantised to bf16: every path measures 0.0019 to 0.0028 from the float64 results
    return {"rel": 1e-2}


def _softmax_rows(scores):
    scores -= scores.amax(dim=-1, keepdim=True)
    scores.exp_()
    return scores.div_(scores.sum(dim=-1, keepdim=True))


def _attend(q, k, v, first, scale, window=0, soft_cap=0.0, bias=None):
    """q [tokens, heads, D] of one kv head over k, v [keys, D] in float64; token t sits at key
    position first + t.  bias [heads, keys]."""
    out = torch.empty_like(q)
    pos = torch.arange(k.shape[0], device="cuda")
    step = max(1, int(2 ** 27 // (k.shape[0] * q.shape[1])))
    for t0 in range(0, q.shape[0], step):
        qt = q[t0:t0 + step]
        s = (qt.reshape(-1, q.shape[2]) @ k.t()).view(qt.shape[0], qt.shape[1], -1).mul_(scale)
        if soft_cap:
            s = soft_cap * torch.tanh(s / soft_cap)
        if bias is not None:
            s += bias
        at = first + t0 + torch.arange(qt.shape[0], device="cuda")
        hidden = pos[None, :] > at[:, None]
        if window:
            hidden |= pos[None, :] <= at[:, None] - window
        s.masked_fill_(hidden[:, None, :], -math.inf)
        out[t0:t0 + step] = (_softmax_rows(s).view(-1, k.shape[0]) @ v).view(qt.shape)
    return out


def _exact_operator(case, args, keywords):
    q, kv, lens, table, cu, _ = args
    group, page = case["hq"] // case["hkv"], case["page"]
    out = torch.zeros(q.shape, dtype=torch.float64, device="cuda")
    scales = keywords.get("kv_scales")
    lens, cu = lens.tolist(), cu.tolist()
    for i in range(len(lens) - case["spare"]):
        pages = table[i, : -(-lens[i] // page)].long()
        rows = slice(cu[i], cu[i + 1])
        for h in range(case["hkv"]):
            if scales is None:
                k, v = (kv[pages, :, 2 * h + c].double() for c in (0, 1))
            else:
                k, v = (kv.view(torch.uint8)[pages, :, 2 * h + c].view(kv.dtype).float().double()
                        * scales[pages, h, c].double()[:, None, None] for c in (0, 1))
            k, v = (x.reshape(-1, case["dim"])[: lens[i]] for x in (k, v))
            heads = slice(h * group, (h + 1) * group)
            out[rows, heads] = _attend(q[rows, heads].double(), k, v, lens[i] - (cu[i + 1] - cu[i]),
                                       keywords["sm_scale"], case["window"], case["soft_cap"])
    return out


def _exact_fused(case, args):
    q, new_k, new_v, cache, lens, pages, _, cu_kv, _, states, proj = args
    cache, page, dim = cache.clone(), case["page"], case["dim"]
    group = case["hq"] // case["hkv"]
    out = torch.zeros(q.shape, dtype=torch.float64, device="cuda")
    for i, length in enumerate(lens.tolist()):
        first = int(cu_kv[i]) // page
        own = pages[first: first + -(-length // page)].long()
        last, slot = int(own[-1]), (length - 1) % page
        cache[last, slot, 0::2, :dim] = new_k[i]
        cache[last, slot, 1::2, :dim] = new_v[i]
        cache[last, slot, :, dim:] = 0
        rel = states[i].double() @ proj.double()  # [hq, extent] by distance from the new token
        near = min(length, case["rel_extent"])
        bias = torch.zeros(case["hq"], length, dtype=torch.float64, device="cuda")
        bias[:, length - near:] = rel[:, :near].flip(1)
        for h in range(case["hkv"]):
            k, v = (cache[own, :, 2 * h + c, :dim].reshape(-1, dim)[:length].double() for c in (0, 1))
            heads = slice(h * group, (h + 1) * group)
            out[i:i + 1, heads] = _attend(q[i:i + 1, heads].double(), k, v, length - 1, 1.0 / dim, bias=bias[heads])
    return out, cache


def _exact_v1(case, args):
    q, key_cache, value_cache, table, lens, bias = args
    group, dim = case["hq"] // case["hkv"], case["dim"]
    out = torch.zeros(q.shape, dtype=torch.float64, device="cuda")
    for i, length in enumerate(lens.tolist()):
        own = table[i].long()
        for h in range(case["hkv"]):
            k, v = (c[own, :, h].reshape(-1, dim)[:length].double() for c in (key_cache, value_cache))
            heads = slice(h * group, (h + 1) * group)
            out[i:i + 1, heads] = _attend(q[i:i + 1, heads].double(), k, v, length - 1, 1.0 / dim,
                                          bias=bias[heads, :length].double())
    return out


def exact(case, seed):
    """The same results in float64, without this package."""
    if case["kind"] == "fused":
        return _exact_fused(case, _fused_inputs(case, seed))
    if case["kind"] == "v1":
        return _exact_v1(case, _v1_inputs(case, seed))
    results = [_exact_operator(case, *call) for call in _operator_inputs(case, seed)]
    return results if case["layers"] else results[0]
