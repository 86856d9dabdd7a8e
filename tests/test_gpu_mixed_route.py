"""Which form a mixed batch takes when the planner chooses: a launch of tiles only, with or without its walks shared by
several workgroups, or one launch of decode workgroups and tiles.  Both sides of every line of the rule, the batches it
leaves alone, and what the chosen form computes, against the oracle and against all rows as tiles."""
import ctypes

import numpy as np
import pytest
import torch

from deserve_amd import _lib
from kvutil import assert_bound_bites, attention_bound, make_scenario, to_torch
from oracle import c_oracle

SEPARATE, SHARED = _lib.LAYOUT_SEPARATE, _lib.LAYOUT_SHARED
CASES = [
    # (name, kv_lens, qo_lens, P, Hq, Hkv, dtype, layout, workgroups a tile)
    ("one_long_row", [3001, 40], [1, 40], 16, 32, 8, "bf16", SHARED, 0),
    ("long_rows_page8_group8", [5300, 3700, 67, 67], [1, 1, 67, 67], 8, 64, 8, "f16", SHARED, 0),
    ("chunk_between_long_rows", [5900, 150, 6500], [1, 33, 1], 16, 32, 8, "bf16", SHARED, 0),
    ("long_rows_page4", [1900, 1000, 20], [1, 1, 5], 4, 32, 8, "bf16", SHARED, 0),
    ("two_kv_heads", [1500, 90], [1, 70], 16, 8, 2, "bf16", SHARED, 0),
    ("walk_before_the_line", [17 * 32, 8], [1, 8], 16, 32, 8, "bf16", SEPARATE, 0),
    ("walk_at_the_line", [18 * 32, 8], [1, 8], 16, 32, 8, "bf16", SHARED, 0),
    ("walks_of_the_chunk_as_long", [1100, 1200], [1, 200], 16, 64, 8, "bf16", SEPARATE, 0),
    ("short_rows_short_prompts", [50] * 12 + [30] * 3, [1] * 12 + [30] * 3, 8, 32, 8, "bf16", SEPARATE, 4),
    ("short_rows_halves", [55] * 24 + [34, 34], [1] * 24 + [34, 34], 8, 64, 8, "bf16", SEPARATE, 2),
    ("rows_too_many_for_short", [55] * 40 + [34], [1] * 40 + [34], 8, 32, 8, "bf16", SHARED, 0),
    ("dozen_beside_as_long_a_chunk", [282] * 14 + [371], [1] * 14 + [5], 8, 32, 8, "bf16", SHARED, 0),
    ("dozen_of_longer_rows", [372] * 12 + [18], [1] * 12 + [18], 16, 32, 8, "bf16", SHARED, 0),
    ("page2", [3001, 40], [1, 40], 2, 32, 8, "bf16", SEPARATE, 0),
    ("row_without_tokens", [3001, 0, 40], [1, 1, 40], 16, 32, 8, "bf16", SHARED, 0),
    ("no_rows_of_one", [3001, 40, 7], [1, 40, 0], 16, 32, 8, "bf16", SHARED, 0),
]


def _plan(kv, qo, P, Hq, Hkv, dtype=_lib.BF16, target=0, route=_lib.ROUTE_AUTO):
    lib, at = _lib.lib(), lambda a: np.concatenate([[0], np.cumsum(a)]).astype(np.int32)
    pages, qo_indptr = at(-(-np.asarray(kv) // P)), at(qo)
    last = np.array([(n - 1) % P + 1 if n else 0 for n in kv], np.int32)
    cap = lib.dskv_mixed_plan_bound(len(kv), int(qo_indptr[-1]), int(pages[-1]) * P)
    plan, info = np.zeros(cap, np.int32), _lib.MixedPlanInfo()
    assert lib.dskv_mixed_plan_typed(qo_indptr.ctypes.data, pages.ctypes.data, last.ctypes.data, len(kv), P, Hq, Hkv, 128,
                                     dtype, target, route, plan.ctypes.data, cap, ctypes.byref(info)) == 0
    return info, plan[: info.plan_words].copy()


@pytest.mark.parametrize("case", CASES, ids=[c[0] for c in CASES])
def test_which_form_a_mixed_batch_takes(case):
    """(256 compute units, also assumed where there is no GPU)"""
    name, kv, qo, P, Hq, Hkv, dtype, layout, workgroups = case
    info, plan = _plan(kv, qo, P, Hq, Hkv)
    assert (info.layout, info.tile_workgroups) == (layout, workgroups)
    rows = sum(1 for n, m in zip(kv, qo) if m == 1 and n > 0)
    assert info.n_decode_rows == (rows if layout == SHARED else 0)
    assert info.n_decode_rows + info.n_tile_rows == sum(qo)
    # the plan is the one that asking for the form gives, word for word
    same, words = _plan(kv, qo, P, Hq, Hkv, route=_lib.ROUTE_SHARED_LAUNCH if layout == SHARED else _lib.ROUTE_OFF)
    assert bytes(same) == bytes(info) and np.array_equal(words, plan)
    # a caller's own number of workgroups and 32 bits: a few rows stay tiles
    if rows < 12:
        for other in ({"target": 512}, {"target": -1}, {"dtype": _lib.F32}):
            assert _plan(kv, qo, P, Hq, Hkv, **other)[0].layout == SEPARATE


@pytest.mark.parametrize("case", CASES, ids=[c[0] for c in CASES])
def test_the_bound_lets_no_row_miss_a_key(case):
    name, kv, qo, P, Hq, Hkv, dtype, layout, workgroups = case
    sc = make_scenario(83, kv_lens=kv, qo_lens=qo, P=P, Hq=Hq, Hkv=Hkv, D=128, dtype=dtype)
    want = c_oracle.prefill_attn(sc.q, sc.qo_indptr, sc.pages, sc.kv_page_indices, sc.kv_page_indptr, sc.kv_last_page_lens, dtype)
    assert_bound_bites(sc, want, attention_bound(sc, want))


@pytest.mark.gpu
@pytest.mark.parametrize("case", CASES, ids=[c[0] for c in CASES])
def test_mixed_batches_match_oracle_and_tiles(case):
    from deserve_amd.paged_ops import BatchPrefillWithPagedKVCacheWrapper

    name, kv, qo, P, Hq, Hkv, dtype, layout, workgroups = case
    print("[case] mixed route", *case, flush=True)
    sc = make_scenario(83, kv_lens=kv, qo_lens=qo, P=P, Hq=Hq, Hkv=Hkv, D=128, dtype=dtype)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a, np.int32)).cuda()
    indptr, tab, tabptr, last = (dev(a) for a in (sc.qo_indptr, sc.kv_page_indices, sc.kv_page_indptr,
                                                  sc.kv_last_page_lens))
    w = BatchPrefillWithPagedKVCacheWrapper(torch.empty(64 << 20, dtype=torch.uint8, device="cuda"))
    q, pages = to_torch(sc.q, dtype), to_torch(sc.pages, dtype)
    results = []
    for route in (True, False):
        w.begin_forward(indptr, tabptr, tab, last, Hq, Hkv, 128, P, route_one_row_requests=route)
        assert w._info.layout == (layout if route else SEPARATE)
        results.append(w.forward(q, pages, out=torch.full_like(q, float("nan"))))
    got, tiles = (r.float().cpu().numpy() for r in results)
    assert np.isfinite(got).all()
    want = c_oracle.prefill_attn(sc.q, sc.qo_indptr, sc.pages, sc.kv_page_indices, sc.kv_page_indptr,
                                 sc.kv_last_page_lens, dtype, True)
    bound = attention_bound(sc, want)
    for form in (got, tiles):
        off = np.abs(form - want) / bound
        assert off.max() <= 1, (np.unravel_index(off.argmax(), off.shape), off.max())



def test_a_caller_with_little_room_keeps_the_tiles():
    lib = _lib.lib()
    qo, pages, last = (np.array(a, np.int32) for a in ([0, 1, 41], [0, 188, 191], [9, 8]))
    bound = lib.dskv_mixed_plan_bound(2, 41, 3001 + 40)
    for cap, layout in ((bound, SHARED), (bound - 1, SEPARATE), (400, SEPARATE)):
        plan, info = np.zeros(bound, np.int32), _lib.MixedPlanInfo()
        assert lib.dskv_mixed_plan_typed(qo.ctypes.data, pages.ctypes.data, last.ctypes.data, 2, 16, 32, 8, 128, _lib.BF16, 0,
                                         _lib.ROUTE_AUTO, plan.ctypes.data, cap, ctypes.byref(info)) == 0
        assert info.layout == layout and not plan[cap:].any()


@pytest.mark.parametrize("group", [4, 8])
def test_a_dozen_rows_are_tiles_only_where_the_kernel_of_short_walks_takes_them(group):
    """(the kernel of long walks is further off for them than the shared launch, which they had before there was a choice)"""
    rng, seen = np.random.default_rng(group), {}
    for _ in range(400):
        rows, chunks = int(rng.integers(12, 41)), int(rng.integers(1, 4))
        kv, qo = rng.integers(2, int(rng.choice([60, 250, 600, 1000])), rows).tolist(), [1] * rows
        for _ in range(chunks):
            qo.append(int(rng.integers(2, 300)))
            kv.append(qo[-1] + int(rng.choice([0, rng.integers(0, 900)])))
        had = _plan(kv, qo, 16, 8 * group, 8, target=-1)[0].layout      # no choice with a number of workgroups
        now = _plan(kv, qo, 16, 8 * group, 8)[0]
        if had == SHARED:
            assert now.layout == SHARED or now.tile_workgroups, (kv, qo)
        seen[had, now.layout, bool(now.tile_workgroups)] = True
    assert (SHARED, SHARED, False) in seen and (SHARED, SEPARATE, True) in seen
