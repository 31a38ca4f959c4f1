"""The fused step's error word where the host preflight was skipped: a sequence with no new token is flagged as a
token with no place in the cache (bit 0) and as q_len > kv_len (bit 3), in one launch and in two."""

import numpy as np
import pytest
import torch

from oracle import rpa_fused_oracle as fo
from tpu_cake_amd import fused

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("pages_per_seq", [8, 512])  # of 16 keys: the one-launch form, the scheduled launches
def test_a_sequence_without_a_token_is_flagged(cuda, pages_per_seq):
    print(f"[case] pages per sequence {pages_per_seq}", flush=True)
    inp = fo.fused_inputs_like(3, nseq=3, hq=8, hkv=2, d=128, page_size=16, pool_pages=24, lengths=[40, 100, 17],
                               rel_dim=16, extent=64)
    args = [torch.from_numpy(np.ascontiguousarray(inp[n]).view(np.int16).copy()).view(torch.bfloat16).cuda()
            if inp[n].dtype == np.uint16 else torch.from_numpy(np.ascontiguousarray(inp[n])).cuda()
            for n in fused.INPUT_NAMES]
    with torch.cuda.stream(torch.cuda.Stream()):
        good, _ = fused.invoke(*args, pages_per_seq=pages_per_seq)
        assert fused.read_error_word() == 0
        args[fused.INPUT_NAMES.index("kv_lengths")][1] = 0
        out, _ = fused.invoke(*args, pages_per_seq=pages_per_seq)
        assert fused.read_error_word() == 9
        assert torch.equal(out[[0, 2]], good[[0, 2]])
