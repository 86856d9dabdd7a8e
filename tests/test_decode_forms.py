"""Which form of the decode attention a plan gets, and how its workgroups spread over the chip: host
rules only (256 compute units are assumed where there is no GPU)."""
import ctypes

import numpy as np
import pytest

from deserve_amd import _lib

CUS, XCDS = 256, 8


def _plan(lens, n_kv, group=4, d=128, page=16, target=0, dtype=_lib.BF16):
    """(shares, items, most tiles of an item)."""
    lib = _lib.lib()
    n = -(-np.asarray(lens, np.int64) // page)
    indptr = np.concatenate([[0], np.cumsum(n)]).astype(np.int32)
    last = np.array([(x - 1) % page + 1 if x else 0 for x in lens], np.int32)
    cap = lib.dskv_decode_plan_bound(len(lens), int(n.sum()) * page)
    plan = np.zeros(cap, np.int32)
    items, wgs, words, ws = ctypes.c_int32(), ctypes.c_int32(), ctypes.c_int64(), ctypes.c_int64()
    out = [ctypes.byref(x) for x in (items, wgs, words, ws)]
    head = (indptr.ctypes.data, last.ctypes.data, len(lens), page, n_kv * group, n_kv, d)
    rc = lib.dskv_decode_plan_typed(*head, dtype, target, plan.ctypes.data, cap, *out)
    assert rc == 0, _lib.last_error()
    table = plan[4 + wgs.value + 1 + 2 * len(lens): words.value].reshape(-1, 8)
    return wgs.value, items.value, int((-(-(table[:, 2] - table[:, 1]) // 16)).max())


def _launch(items, shares, n_kv, group=4, d=128, dtype=_lib.BF16):
    splits = ctypes.c_int32(-1)
    n = _lib.lib().dskv_decode_launch(items, shares, n_kv * group, n_kv, d, dtype, ctypes.byref(splits))
    return int(n), bool(splits.value)


@pytest.mark.parametrize("n_kv", range(1, 65))
def test_no_xcd_gets_more_workgroups_than_it_has_units(n_kv):
    """The split form's workgroups fill a compute unit's LDS: a 33rd on an XCD waits for another to end."""
    for lens in ([1777], [300, 512, 700, 900], [64] * 32):
        shares, items, _ = _plan(lens, n_kv)
        workgroups, splits = _launch(items, shares, n_kv)
        if splits:
            assert workgroups == shares * n_kv          # every id has work
            assert -(-workgroups // XCDS) <= CUS // XCDS
    assert _launch(3, CUS // n_kv, n_kv) == (CUS // n_kv * n_kv, True)


@pytest.mark.parametrize("n_kv,group,lens,splits", [
    (8, 4, [16 * 240] * 8, True), (8, 4, [16 * 245] * 8, False),            # 1920 tiles: 60 a share
    (8, 4, [16 * 40] * 48, True), (8, 4, [16 * 41] * 48, False),
    (8, 8, [16 * 20] * 64, True), (8, 8, [16 * 21] * 64, False),            # many requests: 40 a share
    (8, 4, [16 * 160] * 16, True), (8, 4, [16 * 161] * 16, False),          # requests in many parts: 80 a share
    (8, 1, [16 * 180] * 8, True), (8, 1, [16 * 185] * 8, False),            # small groups: three quarters
    (24, 1, [16 * 93] * 8, True), (24, 1, [16 * 95] * 8, False),            # 240 of 256 units busy: 750 tiles
    (40, 1, [16 * 56] * 8, True), (40, 1, [16 * 57] * 8, False),
    (16, 1, [16 * 320] * 8, True), (64, 1, [16 * 320] * 8, True),           # every unit busy: 2560 tiles
    (12, 4, [16 * 320] * 8, True), (12, 4, [16 * 321] * 8, False), (12, 1, [16 * 241] * 8, False),
    (4, 4, [16 * 64] * 8, True), (4, 4, [16 * 65] * 8, False), (4, 4, [16 * 192], True), (4, 4, [16 * 193], False), (8, 4, [16 * 2240], True), (8, 4, [16 * 2241], False),
    (2, 4, [16 * 20] * 8, False), (2, 4, [16 * 1200] + [100] * 23, True),   # lopsided
    (1, 8, [16 * 200] * 8, False), (1, 8, [16 * 630] * 8, True),
])
def test_which_batches_split_a_head_over_the_waves_of_a_workgroup(n_kv, group, lens, splits):
    shares, items, _ = _plan(lens, n_kv, group=group)
    assert _launch(items, shares, n_kv, group)[1] == splits
    total = sum(-(-x // 16) for x in lens)
    if not splits and total >= 1024:      # a share per compute unit, as large plans have
        assert shares == max(CUS, CUS // n_kv + 1)


def _mixed(qo_lens, kv_lens, n_kv=8, route=_lib.ROUTE_AUTO, page=16):
    """(shares, items) of the decode rows of a batch planned as prefill."""
    lib = _lib.lib()
    n = -(-np.asarray(kv_lens, np.int64) // page)
    indptr = np.concatenate([[0], np.cumsum(n)]).astype(np.int32)
    last = np.array([(x - 1) % page + 1 for x in kv_lens], np.int32)
    qo = np.concatenate([[0], np.cumsum(qo_lens)]).astype(np.int32)
    cap = lib.dskv_mixed_plan_bound(len(qo_lens), int(qo[-1]), int(n.sum()) * page)
    plan, info = np.zeros(cap, np.int32), _lib.MixedPlanInfo()
    rc = lib.dskv_mixed_plan(qo.ctypes.data, indptr.ctypes.data, last.ctypes.data, len(qo_lens), page, 4 * n_kv,
                             n_kv, 128, 0, route, plan.ctypes.data, cap, ctypes.byref(info))
    assert rc == 0 and info.layout == _lib.LAYOUT_SEPARATE, _lib.last_error()
    return info.n_decode_workgroups, info.n_decode_items


@pytest.mark.parametrize("tiles,splits", [(80, True), (81, False)])
def test_rows_of_a_prefill_batch_have_one_rule_with_and_without_chunks(tiles, splits):
    """No counters there: parts are merged by a launch of their own, and the line lies lower."""
    rows = [16 * tiles] * 8
    alone = _mixed([1] * 8, rows)
    beside = _mixed([1] * 8 + [100], rows + [100], route=_lib.ROUTE_TWO_LAUNCHES)
    assert alone == beside and _launch(alone[1], alone[0], 8)[1] == splits


@pytest.mark.parametrize("d", [128, 64])
@pytest.mark.parametrize("n_kv,lens", [
    (8, [20000] + [64] * 128), (8, [16000] + [100] * 140), (8, [300] * 130), (8, [50, 150] * 12),
    (8, [300, 900] * 32), (8, [20000]), (8, [512] * 8), (16, [400] * 40), (4, [64] * 128), (2, [2000] * 3)])
def test_no_wave_of_an_fp32_batch_walks_longer_than_in_shares_of_a_unit_each(n_kv, lens, d):
    """Planner and launcher agree: where the plan has few, large shares, four waves have an item each."""
    shares, items, longest = _plan(lens, n_kv, d=d, dtype=_lib.F32)
    splits = _launch(items, shares, n_kv, d=d, dtype=_lib.F32)[1]
    _, _, longest_of_256 = _plan(lens, n_kv, d=d, target=CUS, dtype=_lib.F32)
    assert -(-longest // (4 if splits else 1)) <= longest_of_256


@pytest.mark.parametrize("n_kv,lens,d,splits", [
    (8, [512] * 8, 128, True), (8, [512] * 17, 128, False), (8, [530] * 8, 128, False),
    (8, [100] * 24, 128, False), (8, [20] * 64, 128, False), (4, [1000], 128, True), (8, [11000], 128, False),
    (8, [16 * 1250] + [60] * 23, 128, True), (2, [5000] * 3, 128, True), (1, [100] * 24, 128, True),
    (1, [1000] * 24, 128, False), (1, [900] * 24, 128, True), (12, [60] * 16, 128, True), (8, [25] * 24, 128, True), (8, [4096], 128, True), (8, [4097], 128, False), (1, [20000], 128, True), (8, [40] * 24, 64, True), (8, [20] * 64, 64, False)])
def test_which_fp32_batches_split_an_item_over_four_waves(n_kv, lens, d, splits):
    shares, items, _ = _plan(lens, n_kv, d=d, dtype=_lib.F32)
    assert _launch(items, shares, n_kv, d=d, dtype=_lib.F32)[1] == splits


def test_untyped_plans_are_those_of_16_bit_pages():
    lib, lens = _lib.lib(), [700, 40, 3]
    n = -(-np.asarray(lens) // 16)
    indptr, last = np.concatenate([[0], np.cumsum(n)]).astype(np.int32), np.array([12, 8, 3], np.int32)
    out = [ctypes.byref(t()) for t in (ctypes.c_int32, ctypes.c_int32, ctypes.c_int64, ctypes.c_int64)]
    head = (indptr.ctypes.data, last.ctypes.data, 3, 16, 32, 8, 128)
    cap = lib.dskv_decode_plan_bound(3, 743)
    a, b = np.zeros(cap, np.int32), np.zeros(cap, np.int32)
    assert lib.dskv_decode_plan(*head, 0, a.ctypes.data, cap, *out) == 0
    assert lib.dskv_decode_plan_typed(*head, _lib.F16, 0, b.ctypes.data, cap, *out) == 0
    assert np.array_equal(a, b)
    assert lib.dskv_decode_plan_typed(*head, 7, 0, b.ctypes.data, cap, *out) == -1 and "dtype" in _lib.last_error()
