"""Soft caps far above the scores, where soft_cap * tanh(s / soft_cap) is s to fp32 rounding: in the one-launch
kernel, the co-resident prefill tiles (64- and 128-dim heads, bf16 and fp8) and the stream-K rows.

Bar: max-abs <= 2e-2 against the oracle where |out| < 4, as in the random sweeps (one bf16 ulp above).  tanhf is
good to a few ulp, so a score is off by at most its own 1e-6; a form that cancels is off by cap * 2e-8."""

import numpy as np
import pytest
import torch

from oracle import rpa_oracle as orc
from tpu_cake_amd import ops
from tpu_cake_amd.workloads import make_custom

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cap", [1e3, 1e6, 1e8, -1e9])
@pytest.mark.parametrize("path,dim,page,dtype", [("direct", 128, 16, "bf16"), ("direct", 64, 32, "fp8"),
                                                 ("tiles", 128, 64, "bf16"), ("tiles", 64, 16, "bf16"),
                                                 ("tiles", 128, 32, "fp8"), ("rows", 128, 64, "bf16")])
def test_soft_cap_far_above_the_scores(cuda, path, dim, page, dtype, cap):
    print(f"[case] {path} {dtype} D {dim} page {page} cap {cap}", flush=True)
    lens, q_lens = ([1, 33, 300, 500], [1] * 4) if path == "direct" else ([333, 65, 1200], [70, 65, 16])
    case = make_custom(kv_lens=lens, q_lens=q_lens, num_q_heads=8, num_kv_heads=2, head_dim=dim, page_size=page,
                       pages_per_seq=(512 if path == "direct" else 2048) // page, kv_dtype=dtype, seed=dim + page)
    knobs = dict(rows=dict(prefill_tiles=-1), tiles=dict(prefill_tiles=2), direct={})[path]
    got = ops.run_case(case, soft_cap=cap, **knobs).float().cpu().numpy()
    ref = orc.bf16_round(orc.ref_ragged_paged_attention(
        case.q, case.kv_pages, case.kv_lens, case.page_indices, case.cu_q_lens, case.num_seqs, sm_scale=case.sm_scale,
        kv_scales=case.kv_scales, kv_dtype=case.kv_dtype, probs_bf16=True, soft_cap=cap))
    assert np.all(np.isfinite(got))
    assert np.allclose(got, ref, atol=0.02, rtol=0.02)
    assert np.max(np.abs(got - ref)[np.abs(ref) < 4], initial=0.0) <= 2e-2
