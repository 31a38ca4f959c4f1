"""Batches whose prefill sequences the attention kernel weighs between tiles and row blocks (64-dim heads, other
pages than whole chunks, kv heads not in fours): the tiles themselves (prefill_tiles=2) where they can go wrong,
the weighed choice on both sides of its line, and that a small chunk beside decode rows is not slower for it.

Bar: max-abs <= 2e-2 against the oracle where |out| < 4, as in the random sweeps (one bf16 ulp above)."""

import numpy as np
import pytest
import torch

from oracle import rpa_oracle as orc
from tpu_cake_amd import ops
from tpu_cake_amd.workloads import make_custom

pytestmark = pytest.mark.gpu

# (query tokens, keys): chunk edges, the unrolled loop's remainders, rows that see one key only
EDGES = [(16, 16), (17, 31), (32, 32), (33, 33), (31, 127), (64, 128), (65, 129), (96, 160), (129, 161), (16, 1025),
         (40, 1056), (1, 700), (1, 33), (130, 255)]


def _check(case, knobs, **kw):
    got = ops.run_case(case, **knobs, **kw).float().cpu().numpy()
    ref = orc.bf16_round(orc.ref_ragged_paged_attention(
        case.q, case.kv_pages, case.kv_lens, case.page_indices, case.cu_q_lens, case.num_seqs, sm_scale=case.sm_scale,
        kv_scales=case.kv_scales, kv_dtype=case.kv_dtype, probs_bf16=True, **kw))
    tv = ref.shape[0]
    assert np.all(np.isfinite(got))
    assert np.allclose(got[:tv], ref, atol=0.02, rtol=0.02)
    assert np.max(np.abs(got[:tv] - ref)[np.abs(ref) < 4], initial=0.0) <= 2e-2
    assert np.all(got[tv:] == 0.0)


@pytest.mark.parametrize("kw", [{}, dict(sliding_window=45), dict(mask_value=-2.5)])
@pytest.mark.parametrize("dtype", ["bf16", "fp8"])
@pytest.mark.parametrize("dim,page,hkv,g", [(128, 16, 2, 4), (128, 24, 1, 8), (128, 1, 3, 1), (128, 64, 6, 2),
                                            (128, 32, 5, 3), (64, 64, 8, 4), (64, 16, 2, 4), (64, 32, 1, 1),
                                            (64, 20, 3, 16)])
def test_tiles(cuda, dtype, dim, page, hkv, g, kw):
    print(f"[case] {dtype} D {dim} page {page} Hkv {hkv} G {g} {kw}", flush=True)
    q_lens, kv_lens = zip(*EDGES)
    _check(make_custom(kv_lens=kv_lens, q_lens=q_lens, num_q_heads=hkv * g, num_kv_heads=hkv, head_dim=dim,
                       page_size=page, kv_dtype=dtype, seed=dim + page + hkv), dict(prefill_tiles=2), **kw)


@pytest.mark.parametrize("dim,page,dtype", [(128, 16, "bf16"), (64, 16, "bf16"), (128, 64, "fp8"), (64, 32, "fp8")])
def test_tiles_over_several_table_segments(cuda, dim, page, dtype):
    print(f"[case] long prior, {dtype} D {dim} page {page}", flush=True)
    _check(make_custom(kv_lens=[9001, 2500], q_lens=[40, 16], num_q_heads=4, num_kv_heads=1, head_dim=dim,
                       page_size=page, kv_dtype=dtype, seed=77 + page), dict(prefill_tiles=2))


@pytest.mark.parametrize("dim,page,hkv,dtype", [(128, 16, 2, "bf16"), (128, 64, 2, "fp8"), (64, 64, 4, "bf16")])
@pytest.mark.parametrize("chunk,prior", [(16, 0), (64, 900), (200, 100), (640, 300)])
def test_weighed(cuda, dim, page, hkv, dtype, chunk, prior):
    print(f"[case] {dtype} D {dim} page {page} Hkv {hkv}, {chunk} tokens over {prior}", flush=True)
    _check(make_custom(kv_lens=[50, 333, 1000, chunk + prior, 7, chunk], q_lens=[1, 1, 1, chunk, 1, chunk],
                       num_q_heads=4 * hkv, num_kv_heads=hkv, head_dim=dim, page_size=page, kv_dtype=dtype,
                       seed=chunk + prior, num_tokens=2 * chunk + 30), {})


def _us(case, **kw):
    d = ops.case_to_device(case, "cuda")
    scales = d.pop("kv_scales", None)
    call = ((d["q"], d["kv_pages"], d["kv_lens"], d["page_indices"], d["cu_q_lens"], d["num_seqs"]),
            dict(sm_scale=case.sm_scale, kv_scales=scales, **kw))
    step = ops.CapturedCalls([call] * 10)
    times = []
    for _ in range(9):
        a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        a.record()
        step.replay()
        b.record()
        torch.cuda.synchronize()
        times.append(a.elapsed_time(b) * 100)
    return sorted(times)[4]


@pytest.mark.parametrize("page,dtype", [(64, "fp8"), (16, "bf16")])
def test_a_small_chunk_beside_decode_rows(cuda, page, dtype):
    # 35 us against 32 and 43 against 41; as tiles the one chunk took 55 and 62
    lens = np.random.default_rng(5).integers(64, 4096, size=64).tolist()
    case = make_custom(kv_lens=lens + [1064], q_lens=[1] * 64 + [64], num_q_heads=8, num_kv_heads=2, page_size=page,
                       kv_dtype=dtype, seed=1)
    weighed, rows = _us(case), _us(case, prefill_tiles=-1)
    print(f"[case] {dtype} page {page}: {weighed:.1f} us, row blocks {rows:.1f} us", flush=True)
    assert weighed < 1.3 * rows


def _exact(case):
    """The call's rows in float64."""
    pages, page, hkv = case.page_indices, case.page_size, case.num_kv_heads
    g = case.num_q_heads // hkv
    kv = torch.from_numpy(orc.bf16_to_f32(case.kv_pages)).cuda().double()
    q = torch.from_numpy(orc.bf16_to_f32(case.q)).cuda().double()
    out = torch.zeros_like(q)
    for i, n in enumerate(case.kv_lens):
        rows = kv[torch.from_numpy(pages[i, : -(-n // page)].astype(np.int64)).cuda()].flatten(0, 1)[:n]
        at = slice(int(case.cu_q_lens[i]), int(case.cu_q_lens[i + 1]))
        ql = at.stop - at.start
        hidden = torch.arange(n, device="cuda") > torch.arange(n - ql, n, device="cuda")[:, None]
        for h in range(hkv):
            k, v = rows[:, 2 * h], rows[:, 2 * h + 1]
            for head in range(h * g, (h + 1) * g):
                s = (q[at, head] @ k.t()) * case.sm_scale
                out[at, head] = torch.softmax(s.masked_fill(hidden, -torch.inf), 1) @ v
    return out


def test_small_batches_are_as_precise_as_the_prefill_kernel(cuda):
    # it cuts a small batch into short chains over all CUs (0.00223); tiles against one lazily moved maximum 0.00233,
    # moved with every chunk 0.00202; a million values tell errors 0.3 percent apart
    err = np.zeros(2)
    norm = 0.0
    for seed in range(2):
        case = make_custom(kv_lens=[1317, 1032], q_lens=[943, 475], num_q_heads=4, num_kv_heads=1, page_size=64, seed=seed)
        ref = _exact(case)
        norm += float((ref ** 2).sum())
        for i, kw in enumerate((dict(), dict(prefill_tiles=1))):
            err[i] += float(((ops.run_case(case, **kw).double() - ref) ** 2).sum())
    err = np.sqrt(err / norm)
    print(f"[case] weighed {err[0]:.6f}, prefill kernel {err[1]:.6f}", flush=True)
    assert err[0] <= 1.01 * err[1]


def test_long_batches(cuda):
    # past the size up to which the maximum moves with every chunk: 0.0023 relative, as the other tiles
    print("[case] prompts of 1500 tokens, Hq 24 / Hkv 6", flush=True)
    case = make_custom(kv_lens=[1500, 1601, 1700], q_lens=[1500, 1400, 1500], num_q_heads=24, num_kv_heads=6,
                       page_size=64, seed=2)
    ref = _exact(case)
    got = ops.run_case(case).double()
    assert float((got - ref).norm() / ref.norm()) <= 3e-3
    assert float((got - ref).abs()[ref.abs() < 4].max()) <= 2e-2
