"""The one-launch form's error against float64 beside that of the scheduled launches (prefill_tiles=-1), which cut
each sequence into short ranges of chunks: no larger.

Both round a chunk's probabilities and the output to bf16 (relative error about 0.002 in all); over 16 x 8 sequences
of 64 rows x 128 dims the two errors are each known to about 0.2 percent, so 2 percent tells them apart."""

import numpy as np
import pytest
import torch

from oracle import rpa_oracle as orc
from tpu_cake_amd import ops
from tpu_cake_amd.workloads import make_custom

pytestmark = pytest.mark.gpu


def _exact(case, dim, g):
    pages, page = case.page_indices, case.page_size
    kv = torch.from_numpy(orc.bf16_to_f32(case.kv_pages)).cuda().double()
    q = torch.from_numpy(orc.bf16_to_f32(case.q)).cuda().double()
    out = []
    for i, n in enumerate(case.kv_lens):
        rows = kv[torch.from_numpy(pages[i, : -(-n // page)].astype(np.int64)).cuda()].flatten(0, 1)[:n]
        k, v = (rows[:, c::2].repeat_interleave(g, 1).transpose(0, 1).contiguous() for c in (0, 1))  # [hq, n, dim]
        s = (k @ q[i][:, :, None]).squeeze(2) * case.sm_scale
        out.append((torch.softmax(s, 1)[:, None] @ v).squeeze(1))
    return torch.stack(out)


@pytest.mark.parametrize("dim,keys", [(128, 512), (128, 1024), (64, 1024), (256, 512)])
def test_error_is_no_larger_than_split(cuda, dim, keys):
    print(f"[case] D {dim} keys {keys}", flush=True)
    err = np.zeros(2)
    norm = 0.0
    for seed in range(16):
        case = make_custom(kv_lens=[keys - 3 * i for i in range(8)], q_lens=[1] * 8, num_q_heads=8, num_kv_heads=2,
                           head_dim=dim, page_size=16, pages_per_seq=keys // 16, seed=seed)
        ref = _exact(case, dim, 4)
        norm += float((ref ** 2).sum())
        for i, kw in enumerate((dict(), dict(prefill_tiles=-1))):
            err[i] += float(((ops.run_case(case, **kw).double() - ref) ** 2).sum())
    err = np.sqrt(err / norm)
    print(f"  one launch {err[0]:.6f}, split {err[1]:.6f}", flush=True)
    assert err[0] <= 1.02 * err[1]
