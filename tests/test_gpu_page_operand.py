"""Decode with pages that split a 32-key unit and more than 16 query heads per kv head, which keeps the operand
layout for 128-dim heads and for one or two wider than 64: both sides of that rule, bf16 pools plain and scaled.

Bar: max-abs <= 2e-2 against the oracle where |out| < 4, as in the random sweeps (one bf16 ulp above)."""

import numpy as np
import pytest
import torch

from oracle import rpa_oracle as orc
from tpu_cake_amd import ops
from tpu_cake_amd.workloads import make_custom

pytestmark = pytest.mark.gpu

LENS = [1, 15, 16, 17, 31, 32, 33, 47, 48, 49, 64, 65, 1000, 1031]


@pytest.mark.parametrize("kw", [{}, dict(k_scale=0.8, v_scale=1.3), dict(sliding_window=40), dict(soft_cap=15.0)])
@pytest.mark.parametrize("dim,page,hkv,g", [(128, 16, 1, 32), (128, 24, 4, 17), (128, 16, 8, 20), (112, 7, 2, 32),
                                            (96, 16, 1, 24), (96, 16, 3, 20), (256, 48, 2, 20), (256, 16, 3, 17),
                                            (64, 16, 1, 32), (128, 16, 2, 16)])
def test_groups_past_16(cuda, dim, page, hkv, g, kw):
    print(f"[case] D {dim} page {page} Hkv {hkv} G {g} {kw}", flush=True)
    # (a page table too long for the one-launch form; one sequence holds several tokens)
    case = make_custom(kv_lens=LENS + [300], q_lens=[1] * len(LENS) + [3], num_q_heads=hkv * g, num_kv_heads=hkv,
                       head_dim=dim, page_size=page, pages_per_seq=-(-4200 // page), seed=dim + page + hkv + g)
    got = ops.run_case(case, **kw).float().cpu().numpy()
    ref = orc.bf16_round(orc.ref_ragged_paged_attention(
        case.q, case.kv_pages, case.kv_lens, case.page_indices, case.cu_q_lens, case.num_seqs, sm_scale=case.sm_scale,
        probs_bf16=True, **kw))
    assert np.all(np.isfinite(got))
    assert np.allclose(got, ref, atol=0.02, rtol=0.02)
    assert np.max(np.abs(got - ref)[np.abs(ref) < 4], initial=0.0) <= 2e-2


@pytest.mark.parametrize("hkv,g,tiles", [(8, 20, 3), (8, 17, 0), (2, 32, -1)])
def test_groups_past_16_beside_a_prompt(cuda, hkv, g, tiles):
    print(f"[case] Hkv {hkv} G {g} prefill_tiles {tiles}", flush=True)
    case = make_custom(kv_lens=[700, 33, 150], q_lens=[1, 1, 70], num_q_heads=hkv * g, num_kv_heads=hkv, page_size=16,
                       seed=hkv + g)
    got = ops.run_case(case, prefill_tiles=tiles).float().cpu().numpy()
    ref = orc.bf16_round(orc.ref_ragged_paged_attention(
        case.q, case.kv_pages, case.kv_lens, case.page_indices, case.cu_q_lens, case.num_seqs, sm_scale=case.sm_scale,
        probs_bf16=True))
    assert np.all(np.isfinite(got))
    assert np.allclose(got, ref, atol=0.02, rtol=0.02)
    assert np.max(np.abs(got - ref)[np.abs(ref) < 4], initial=0.0) <= 2e-2
