"""Finite scores far below -1e30, in every kernel that keeps a running maximum: a third of the keys at -2^107 times
sm_scale and the rest at twice that, so that a row's output is the mean of V over the visible ones of the first kind.

Products and sums of powers of two are exact, so only the probabilities' sum and the output round (one bf16 ulp)."""

import numpy as np
import pytest
import torch

from oracle import rpa_oracle as orc
from tpu_cake_amd import ops
from tpu_cake_amd.workloads import make_custom

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("path,dim,page", [("tiles", 128, 64), ("tiles", 128, 16), ("tiles", 64, 32),
                                           ("direct", 128, 16), ("rows", 128, 64)])
def test_scores_below_1e30(cuda, path, dim, page):
    print(f"[case] {path} D {dim} page {page}", flush=True)
    lens, q_lens = ([1, 33, 300], [1, 1, 1]) if path == "direct" else ([333, 65, 2100], [70, 65, 16])
    case = make_custom(kv_lens=lens, q_lens=q_lens, num_q_heads=8, num_kv_heads=2, head_dim=dim, page_size=page,
                       pages_per_seq=(512 if path == "direct" else 2112) // page, seed=dim + page, sm_scale=1.0,
                       values="host")
    big = np.float32(2.0 ** 50)
    case.q = orc.bf16_from_f32(np.full(case.q.shape, big))
    kv, want = case.kv_pages.copy(), []
    for i, n in enumerate(lens):
        at = np.arange(n)
        pages, slots = case.page_indices[i, at // page], at % page
        k = np.where(at % 3 == 0, -big, -2 * big).astype(np.float32)
        kv[pages, slots, 0::2] = orc.bf16_from_f32(np.broadcast_to(k[:, None, None], (n, 2, dim)).copy())
        v = orc.bf16_to_f32(kv[pages, slots, 1::2])  # [n, hkv, dim]
        for t in range(n - q_lens[i], n):
            want.append(np.repeat(v[: t + 1][at[: t + 1] % 3 == 0].mean(0), 4, axis=0))
    case.kv_pages = kv
    knobs = dict(rows=dict(prefill_tiles=-1), tiles=dict(prefill_tiles=2), direct={})[path]
    got = ops.run_case(case, **knobs).float().cpu().numpy()
    want = np.stack(want)
    assert np.all(np.isfinite(got))
    assert np.allclose(got, want, atol=1e-2, rtol=2.0 ** -7)
