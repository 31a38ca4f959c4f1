"""GPU parity of decode through whole cache rows where a 32-key unit lies in several pages: page sizes that are
not a multiple of 32, every head-dim width, key counts around units and pages, scaled caches and masks."""

import numpy as np
import pytest
import torch

from oracle import rpa_oracle as orc
from tpu_cake_amd import ops
from tpu_cake_amd.workloads import make_custom

pytestmark = pytest.mark.gpu

LENS = [1, 15, 16, 17, 31, 32, 33, 47, 48, 49, 64, 65, 1000, 1024, 1031]


@pytest.mark.parametrize("dim,page,hkv,g,kw", [
    (128, 16, 2, 4, {}), (128, 1, 4, 4, {}), (128, 48, 8, 1, dict(sliding_window=40)),
    (128, 24, 3, 5, dict(k_scale=0.8, v_scale=1.3)), (128, 16, 8, 8, dict(mask_value=-3.0)),
    (64, 16, 4, 4, {}), (64, 20, 8, 2, dict(k_scale=0.8, v_scale=1.3)), (64, 5, 1, 16, dict(soft_cap=15.0)),
    (32, 16, 8, 1, {}), (96, 16, 2, 3, dict(k_scale=0.8, v_scale=1.3)), (40, 7, 2, 2, {}), (112, 1000, 1, 4, {}),
    (256, 16, 2, 4, {}), (256, 80, 3, 2, dict(sliding_window=500, k_scale=0.8, v_scale=1.3))])
def test_pages_across_units(cuda, dim, page, hkv, g, kw):
    print(f"[case] D {dim} page {page} Hkv {hkv} G {g} {kw}", flush=True)
    # (a page table too long for the one-launch form; two sequences hold several tokens)
    lens, q_lens = LENS + [300, 77], [1] * len(LENS) + [5, 2]
    case = make_custom(kv_lens=lens, q_lens=q_lens, num_q_heads=hkv * g, num_kv_heads=hkv, head_dim=dim,
                       page_size=page, pages_per_seq=-(-4200 // page), seed=dim + page + hkv + g)
    out = ops.run_case(case, **kw)
    torch.cuda.synchronize()
    got = out.float().cpu().numpy()
    ref = orc.bf16_round(orc.ref_ragged_paged_attention(
        case.q, case.kv_pages, case.kv_lens, case.page_indices, case.cu_q_lens, case.num_seqs, sm_scale=case.sm_scale,
        probs_bf16=True, **kw))
    tv = ref.shape[0]
    assert np.all(np.isfinite(got))
    # bf16 probabilities and outputs: the tolerance of every operator test (2e-2, one bf16 ulp above 4)
    assert np.allclose(got[:tv], ref, atol=0.02, rtol=0.02)
    small = np.abs(ref) < 4
    assert np.max(np.abs(got[:tv] - ref)[small], initial=0.0) <= 2e-2
    assert np.all(got[tv:] == 0.0)
