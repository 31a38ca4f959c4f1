"""GPU parity of small calls (one workgroup per sequence and kv head, one launch): key counts around
32-key chunks and the eight waves' turns, several tokens per sequence, padded and empty sequences, every
head-dim width, short pages, masks, and the bounds of the rule that picks this form."""

import numpy as np
import pytest
import torch

from oracle import rpa_oracle as orc
from tpu_cake_amd import ops
from tpu_cake_amd.workloads import make_custom

pytestmark = pytest.mark.gpu

LENS = [1, 2, 31, 32, 33, 63, 65, 127, 255, 256, 257, 300, 511, 512]


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
    small = np.abs(ref) < 4  # one bf16 ulp is more than 2e-2 above
    assert np.max(np.abs(got[:tv] - ref)[small], initial=0.0) <= 2e-2
    assert np.all(got[tv:] == 0.0)


def _case(dim=128, page=16, hkv=2, g=4, lens=LENS, cap=None, **kw):
    cap = cap or (512 if dim == 256 else 768 if page in (20, 24) else 1024)
    return make_custom(kv_lens=lens, q_lens=kw.pop("q_lens", [1] * len(lens)), num_q_heads=hkv * g, num_kv_heads=hkv,
                       head_dim=dim, page_size=page, pages_per_seq=-(-cap // page), seed=dim + page + hkv + g, **kw)


def _is_direct(case):
    return ops.attention_grid(case, cus=256) == (case.page_indices.shape[0] * case.num_kv_heads, 8)


@pytest.mark.parametrize("dim,page,hkv,g,dtype", [
    (128, 16, 2, 4, "bf16"), (128, 64, 8, 4, "bf16"), (128, 1, 1, 32, "bf16"), (64, 16, 4, 1, "bf16"),
    (32, 24, 3, 5, "bf16"), (96, 32, 1, 8, "bf16"), (256, 16, 2, 4, "bf16"), (128, 16, 2, 4, "fp8"),
    (128, 64, 4, 8, "fp8"), (64, 32, 2, 2, "fp8"), (256, 64, 1, 4, "fp8"), (256, 20, 3, 1, "fp8"), (96, 16, 2, 3, "fp8")])
def test_lengths(cuda, dim, page, hkv, g, dtype):
    print(f"[case] {dtype} D {dim} page {page} Hkv {hkv} G {g}", flush=True)
    case = _case(dim, page, hkv, g, kv_dtype=dtype)
    assert _is_direct(case) == (case.page_indices.shape[1] * page * max(dim, 64) <= 1024 * 128)
    _check(case)


@pytest.mark.parametrize("kw", [dict(sliding_window=40), dict(soft_cap=15.0), dict(mask_value=-3.0),
                                dict(k_scale=0.8, v_scale=1.3), dict(sliding_window=200, soft_cap=8.0)])
def test_options(cuda, kw):
    print(f"[case] {kw}", flush=True)
    _check(_case(lens=[1, 45, 300, 700, 1024], page=32), **kw)


def test_tokens_padding_and_empty_sequences(cuda):
    # at most one token per sequence SLOT: a sequence may still hold several (rows in blocks of 16)
    print("[case] q_lens 5, 1, 9, 2 of 24 slots", flush=True)
    case = _case(lens=[5, 200, 400, 900], q_lens=[5, 1, 9, 2], g=8, max_num_seqs=24, num_tokens=20)
    assert _is_direct(case)
    _check(case)
    _check(case, sliding_window=50)


def test_rule_bounds(cuda):
    # a longer page table, more tokens than slots or a schedule knob keep the split form; same results
    print("[case] rule bounds", flush=True)
    small, wide = _case(cap=1024), _case(cap=1040)
    assert _is_direct(small) and not _is_direct(wide)
    assert _is_direct(_case(dim=64, cap=2048)) and not _is_direct(_case(dim=256, cap=1024))
    assert not _is_direct(_case(lens=[40] * 300, q_lens=[1] * 300))  # 600 (sequence, kv head) pairs
    _check(wide)
    knob = ops.run_case(small, waves_per_cu=4).float()
    direct = ops.run_case(small).float()
    assert torch.max((knob - direct).abs()).item() <= 2e-2


def test_bad_page_ids_are_flagged_not_read(cuda):
    print("[case] page ids out of range", flush=True)
    case = _case(lens=[100, 64, 300], page=16)
    case.page_indices = case.page_indices.copy()
    case.page_indices[1, 2] = 1 << 20
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        out = ops.run_case(case)
        assert ops.read_error_word() & 1
    good = ops.run_case(_case(lens=[100, 64, 300], page=16))
    torch.cuda.synchronize()
    assert torch.equal(out[[0, 2]], good[[0, 2]])


@pytest.mark.parametrize("dim,page,extent", [(128, 16, 128), (64, 64, 512), (120, 1, 16), (32, 24, 64)])
def test_fused_step(cuda, dim, page, extent):
    from oracle import rpa_fused_oracle as fo
    from tpu_cake_amd import fused

    print(f"[case] fused D {dim} page {page} E {extent}", flush=True)
    lens = [1, 2, 16, 32, 33, 64, 257, 500, 1000]
    pool = int(sum(-(-x // page) for x in lens) * 1.25) + 2
    inp = fo.fused_inputs_like(dim + page, nseq=len(lens), hq=8, hkv=2, d=dim, page_size=page, pool_pages=pool,
                               lengths=lens, rel_dim=16, extent=extent)
    args = [torch.from_numpy(np.ascontiguousarray(inp[n]).view(np.int16).copy()).view(torch.bfloat16).cuda()
            if inp[n].dtype == np.uint16 else torch.from_numpy(np.ascontiguousarray(inp[n])).cuda()
            for n in fused.INPUT_NAMES]
    out, cache = fused.run_preflighted(*args)
    torch.cuda.synchronize()
    want, want_cache = fo.inkling_fused_rpa_reference(inp)
    bits = cache.view(torch.int16).cpu().numpy().view(np.uint16).reshape(inp["cache"].shape)
    assert np.array_equal(bits, want_cache)
    assert np.max(np.abs(out.float().cpu().numpy() - orc.bf16_to_f32(want))) <= 2e-2
    assert fused.read_error_word() == 0
