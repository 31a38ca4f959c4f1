"""Which calls run as one launch (rpa_attention_grid on a nominal device; no GPU): the rule's bounds, and the
schedule knobs, each of which keeps the launches it describes."""

import types

import numpy as np
import pytest

from tpu_cake_amd import build, contracts, ops


@pytest.fixture(scope="module", autouse=True)
def library():
    if not build.OUTPUT.exists():
        build.build()


def _case(tokens=60, slots=60, g=4, hkv=4, dim=128, page=64, keys=1024, dtype="bf16"):
    shape = lambda *s: np.empty(s, np.uint8)  # noqa: E731
    return types.SimpleNamespace(q=shape(tokens, hkv * g, dim), kv_pages=shape(2, page, 2 * hkv, dim),
                                 page_indices=shape(slots, -(-keys // page)), kv_dtype=dtype, sm_scale=1.0)


def _direct(case, knobs=None):
    slots, hkv = case.page_indices.shape[0], case.kv_pages.shape[2] // 2
    return ops.attention_grid(case, knobs, cus=256) == (slots * hkv, 8)


@pytest.mark.parametrize("dtype", ["bf16", "fp8"])
@pytest.mark.parametrize("knobs,direct", [
    (None, True), (dict(waves_per_cu=8), True), (dict(waves_per_cu=4), False), (dict(prefill_tiles=-1), False),
    (dict(prefill_tiles=1), False), (dict(prefill_tiles=2), False), (dict(prefill_tiles=3), False),
    (dict(prefill_cost=0.3), False)])
def test_schedule_knobs_keep_their_launches(dtype, knobs, direct):
    assert _direct(_case(dtype=dtype), knobs) == direct


@pytest.mark.parametrize("kw,direct", [
    ({}, True), (dict(tokens=61), False), (dict(keys=1025), False), (dict(dim=64, keys=2048), True),
    (dict(dim=32, keys=2049), False), (dict(dim=256, keys=512), True), (dict(dim=256, keys=513), False),
    (dict(page=20, keys=1020), True),
    # more pairs than CUs: a second round of workgroups
    (dict(slots=65), False), (dict(slots=65, keys=512), True), (dict(slots=128, keys=513), False),
    (dict(slots=129, keys=64), False), (dict(slots=65, keys=512, dtype="fp8"), False),
    (dict(slots=65, keys=256, dtype="fp8"), True), (dict(slots=128, dim=64, keys=2048, dtype="fp8"), True),
    (dict(slots=65, dim=256, keys=128), False), (dict(slots=65, dim=256, keys=64), True),
    (dict(slots=65, dim=256, keys=512, dtype="fp8"), True), (dict(slots=65, dim=32, keys=2048), True),
    (dict(slots=65, dim=64, keys=1088), False),
    # more than 16 query heads per kv head: several turns over the same keys
    (dict(slots=4, tokens=4, hkv=1, g=32), False), (dict(slots=4, tokens=4, hkv=1, g=32, keys=512), True),
    (dict(slots=14, tokens=14, hkv=1, g=32), True), (dict(slots=4, tokens=4, hkv=1, g=64, keys=256), False),
    (dict(slots=4, tokens=4, hkv=1, g=64, keys=128), True), (dict(hkv=1, g=64, keys=512), True),
    (dict(hkv=1, g=65, keys=64), False), (dict(slots=128, g=32, keys=576), False),
    (dict(slots=128, g=32, keys=512), True), (dict(slots=65, g=64, keys=256), True)])
def test_bounds(kw, direct):
    case = _case(**kw)
    assert _direct(case) == direct
    hkv, table = case.kv_pages.shape[2] // 2, case.page_indices.shape[1] * case.kv_pages.shape[1]
    assert contracts.direct_call(case.q.shape[0], case.page_indices.shape[0], hkv, case.q.shape[2], table,
                                 case.q.shape[1] // hkv, case.kv_dtype) == direct
