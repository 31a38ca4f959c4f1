"""GPU parity of the prefill tiles where they can go wrong: key counts at and around 32-key chunks and
the ring's four slots, one-row remainders of a 128-row tile, page sizes that split a chunk, one to six
kv heads (workgroups of several stream-K workers), 64- and 128-dim heads, fp8 scales of either sign,
segments of the chunk table, tiles split over workgroups, windows, soft caps and finite mask values.

Bar: max-abs <= 2e-2 against the oracle where |out| < 4, as in the random sweeps (one bf16 ulp above)."""

import numpy as np
import pytest
import torch

from oracle import rpa_oracle as orc
from tpu_cake_amd import ops
from tpu_cake_amd.workloads import make_custom

pytestmark = pytest.mark.gpu


def _check(case, **kw):
    out = ops.run_case(case, **kw)
    torch.cuda.synchronize()
    got = out.float().cpu().numpy()
    ref = orc.bf16_round(orc.ref_ragged_paged_attention(
        case.q, case.kv_pages, case.kv_lens, case.page_indices, case.cu_q_lens, case.num_seqs, sm_scale=case.sm_scale,
        kv_scales=case.kv_scales, kv_dtype=case.kv_dtype, probs_bf16=True, **kw))
    tv = ref.shape[0]
    assert np.all(np.isfinite(got))
    assert np.allclose(got[:tv], ref, atol=0.02, rtol=0.02)
    small = np.abs(ref) < 4
    assert np.max(np.abs(got[:tv] - ref)[small], initial=0.0) <= 2e-2
    assert np.all(got[tv:] == 0.0)


# (query tokens, keys): chunk edges, the unrolled loop's remainders, rows that see one key only
EDGES = [(16, 16), (17, 31), (32, 32), (33, 33), (31, 127), (64, 128), (65, 129), (96, 160), (129, 161), (16, 1025),
         (40, 1056), (1, 700), (1, 33), (130, 255)]


@pytest.mark.parametrize("dtype", ["bf16", "fp8"])
@pytest.mark.parametrize("dim,page,hkv,g", [(128, 16, 2, 4), (128, 24, 1, 8), (128, 1, 3, 1), (128, 64, 6, 2),
                                            (128, 32, 5, 3), (128, 64, 4, 4), (64, 64, 8, 4), (64, 16, 2, 4),
                                            (64, 32, 1, 1), (64, 20, 3, 16)])
def test_chunk_and_tile_edges(cuda, dtype, dim, page, hkv, g):
    print(f"[case] {dtype} D {dim} page {page} Hkv {hkv} G {g}", flush=True)
    q_lens, kv_lens = zip(*EDGES)
    _check(make_custom(kv_lens=kv_lens, q_lens=q_lens, num_q_heads=hkv * g, num_kv_heads=hkv, head_dim=dim,
                       page_size=page, kv_dtype=dtype, seed=dim + page + hkv))


@pytest.mark.parametrize("dim,page,hkv", [(128, 16, 2), (64, 64, 4), (64, 8, 1), (128, 64, 1)])
@pytest.mark.parametrize("kw", [dict(sliding_window=45), dict(soft_cap=20.0), dict(mask_value=-2.5),
                                dict(sliding_window=300, soft_cap=9.0)])
def test_masks(cuda, dim, page, hkv, kw):
    print(f"[case] D {dim} page {page} Hkv {hkv} {kw}", flush=True)
    _check(make_custom(kv_lens=[700, 90, 1500, 33, 64], q_lens=[200, 90, 65, 17, 1], num_q_heads=4 * hkv,
                       num_kv_heads=hkv, head_dim=dim, page_size=page, seed=31 + dim + page), **kw)


@pytest.mark.parametrize("dim,page", [(128, 64), (128, 16), (64, 32)])
def test_fp8_scales_of_either_sign(cuda, dim, page):
    # the plain path folds a page's K scale into the exponent and must notice one that is not positive
    print(f"[case] negative K scales, D {dim} page {page}", flush=True)
    case = make_custom(kv_lens=[900, 333, 64], q_lens=[140, 100, 64], num_q_heads=8, num_kv_heads=2, head_dim=dim,
                       page_size=page, kv_dtype="fp8", seed=5 + page)
    case.kv_scales = case.kv_scales.copy()
    case.kv_scales[::3, :, 0] *= -1.0
    case.kv_scales[1::5, :, 0] = 0.0
    _check(case)


@pytest.mark.parametrize("dim,page", [(128, 16), (64, 16), (128, 64)])
def test_long_prior_spans_table_segments(cuda, dim, page):
    # more chunks than one table segment holds, few enough tiles that they are split over workgroups
    print(f"[case] long prior, D {dim} page {page}", flush=True)
    _check(make_custom(kv_lens=[9001, 2500], q_lens=[40, 16], num_q_heads=4, num_kv_heads=1, head_dim=dim,
                       page_size=page, seed=77 + page))
    _check(make_custom(kv_lens=[3333, 1200], q_lens=[64, 30], num_q_heads=8, num_kv_heads=2, head_dim=dim,
                       page_size=page, kv_dtype="fp8", seed=78 + page))
