"""The two forms of the v1 Inkling decode: one launch over the caller's caches, and the packed form (the caches
copied into the operator's layout in the workspace, then its launches).  Which form a call takes is read from the
workspace: only the packed form writes past the operator's own part of it.

Bar: max-abs <= 2e-2 against the oracle on the same bf16 inputs (bf16 probabilities and outputs)."""

import ctypes

import numpy as np
import pytest
import torch

from oracle import rpa_oracle as orc
from tpu_cake_amd import _lib, inkling

pytestmark = pytest.mark.gpu
TOL = 2e-2
MARK = 0xA5


def _bf16(x):
    return torch.from_numpy(orc.bf16_from_f32(np.asarray(x, np.float32)).view(np.int16)).view(torch.bfloat16).cuda()


def _inputs(lengths, hq, hkv, d, page, keys, seed):
    rng = np.random.default_rng(seed)
    b, mp = len(lengths), keys // page
    used = -(-max(lengths) // page)
    pool = b * used + 2
    table = np.zeros((b, mp), np.int32)
    table[:, :used] = rng.permutation(pool)[: b * used].reshape(b, used)
    arrays = [rng.normal(size=(b, hq, d)), rng.normal(size=(pool, page, hkv, d)), rng.normal(size=(pool, page, hkv, d))]
    arrays = [orc.bf16_to_f32(orc.bf16_from_f32(a.astype(np.float32))) for a in arrays]
    bias = orc.bf16_to_f32(orc.bf16_from_f32(rng.normal(scale=0.5, size=(hq, keys)).astype(np.float32)))
    return (*arrays, table, np.asarray(lengths, np.int32), bias)


def _shape(args):
    q, k, table, bias = args[0], args[1], args[3], args[5]
    return _lib.RpaInklingShape(num_seqs=q.shape[0], num_q_heads=q.shape[1], num_kv_heads=k.shape[2],
                                head_dim=q.shape[2], total_pages=k.shape[0], page_size=k.shape[1],
                                pages_per_seq=table.shape[1], bias_len=bias.shape[1])


def _call(args, out=None):
    """rpa_inkling_decode on device tensors with a workspace of its own; (rc, out, whether caches were packed)."""
    lib, shape, stream = _lib.load(), _shape(args), torch.cuda.current_stream().cuda_stream
    op = _lib.RpaShape(args[0].shape[0], args[0].shape[1], args[1].shape[2], 128, args[1].shape[0], args[1].shape[1],
                       args[3].shape[0], args[3].shape[1], _lib.RPA_KV_BF16)
    packed_at = -(-lib.rpa_workspace_size(ctypes.byref(op)) // 256) * 256
    ws = torch.full((lib.rpa_inkling_workspace_size(ctypes.byref(shape)),), MARK, dtype=torch.uint8, device="cuda")
    _lib.check(lib.rpa_workspace_init(ws.data_ptr(), ws.numel(), stream))
    out = torch.empty_like(args[0]) if out is None else out
    rc = lib.rpa_inkling_decode(ctypes.byref(shape), 1.0 / args[0].shape[2], *[t.data_ptr() for t in args],
                                out.data_ptr(), ws.data_ptr(), ws.numel(), stream)
    torch.cuda.synchronize()
    return rc, out, bool((ws[packed_at:packed_at + 4096] != MARK).any())


def _device(host):
    return [*map(_bf16, host[:3]), torch.from_numpy(host[3]).cuda(), torch.from_numpy(host[4]).cuda(), _bf16(host[5])]


def _max_abs(out, host):
    ref = orc.bf16_round(orc.inkling_rpa_reference(*host))
    got = out.float().cpu().numpy()
    assert np.all(np.isfinite(got))
    return float(np.max(np.abs(got - ref)))


# lengths, hq, hkv, d, page, keys of the page table, packed
FORMS = [
    ([1, 31, 33, 500, 4096], 16, 8, 64, 64, 4096, False),   # the longest table of the one-launch form
    ([1, 31, 33, 500, 4128], 16, 8, 64, 32, 4128, True),    # one chunk past it, chunks in one page
    ([1, 31, 33, 500, 4104], 8, 4, 128, 24, 4104, True),    # and in several
    ([7, 64, 200], 4, 4, 20, 16, 256, True),                # a head dim that is no multiple of 8
    ([7, 64, 200], 4, 4, 32, 16, 256, False),
    ([4096], 32, 1, 128, 16, 4096, True),                   # one CU per kv head would read it all, twice
    ([900, 1000], 64, 1, 64, 16, 1024, True),               # four turns over the same keys, a small pool
    ([100, 512], 32, 1, 128, 16, 512, False),
]


@pytest.mark.parametrize("lengths,hq,hkv,d,page,keys,packed", FORMS)
def test_forms(cuda, lengths, hq, hkv, d, page, keys, packed):
    print(f"[case] H {hq} Hkv {hkv} D {d} page {page} keys {keys} packed {packed}", flush=True)
    host = _inputs(lengths, hq, hkv, d, page, keys, keys + d)
    rc, out, did_pack = _call(_device(host))
    assert rc == 0
    assert _max_abs(out, host) <= TOL
    assert did_pack == packed


@pytest.mark.parametrize("d,which", [(64, 0), (64, 1), (64, 2), (64, 6), (128, 0), (128, 6), (32, 6)])
def test_tensors_off_their_alignment(cuda, d, which):
    # 0 the query, 1 and 2 the caches, 6 the output, one element past a 16-byte boundary: the packed form
    print(f"[case] D {d} tensor {which} at an odd address", flush=True)
    host = _inputs([7, 64, 200], 8, 4, d, 16, 256, 3)
    args = _device(host)
    args.append(torch.empty_like(args[0]))
    flat = torch.empty(args[which].numel() + 1, dtype=torch.bfloat16, device="cuda")
    flat[1:] = args[which].flatten()
    args[which] = flat[1:].view(args[which].shape)
    rc, out, did_pack = _call(args[:6], out=args[6])
    assert rc == 0 and did_pack
    assert _max_abs(out, host) <= TOL
    assert _max_abs(inkling.inkling_rpa(*args[:6], out=args[6]), host) <= TOL


def test_out_may_alias_the_query_below_128_dims_only(cuda):
    print("[case] out is the query", flush=True)
    for keys, packed in ((256, False), (4112, True)):
        host = _inputs([7, 64, 200], 8, 4, 64, 16, keys, 4)
        args = _device(host)
        rc, out, did_pack = _call(args, out=args[0])
        assert rc == 0 and did_pack == packed
        assert _max_abs(out, host) <= TOL
        wide = _device(_inputs([7, 64, 200], 8, 4, 128, 16, keys, 5))
        assert _call(wide, out=wide[0])[0] == -1  # RPA_E_INVALID
