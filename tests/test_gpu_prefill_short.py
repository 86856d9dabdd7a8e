"""The prefill attention of few short walks: a tile's columns shared by four workgroups or by two, 256 keys in LDS at a
time, key groups of a workgroup merged there.  Edges of the quarters, the blocks, the rounds and the rule that takes a plan
to them; against the oracle, and against the same plan walked by one workgroup a tile."""
import ctypes

import numpy as np
import pytest
import torch

from deserve_amd import _lib
from kvutil import assert_bound_bites, attention_bound, make_scenario, to_torch
from oracle import c_oracle

CASES = [
    # (name, kv_lens, qo_lens, P, Hq, Hkv, dtype, workgroups a tile)
    ("two_tokens", [2], [2], 16, 32, 8, "bf16", 4),
    ("quarter_edges", [15, 16, 17, 33], [15, 16, 17, 33], 16, 32, 8, "f16", 4),
    ("block_edges", [31, 32, 33, 64, 65], [7, 16, 17, 2, 33], 8, 32, 8, "bf16", 4),
    ("key_group_without_blocks", [96, 40, 97], [5, 40, 70], 16, 32, 8, "bf16", 4),
    ("one_round", [256, 255], [64, 256], 16, 32, 8, "bf16", 4),
    ("two_rounds", [257, 512, 289], [33, 64, 40], 16, 32, 8, "f16", 4),
    ("long_walk_of_few_columns", [257], [32], 16, 32, 8, "bf16", 0),
    ("three_rounds", [513], [200], 16, 32, 8, "bf16", 4),
    ("four_rounds_behind_tokens", [1024, 769, 60], [40, 64, 60], 8, 32, 8, "bf16", 4),
    ("four_rounds_group8", [1000], [129], 16, 64, 8, "f16", 4),
    ("as_many_as_units", [128] * 4, [128] * 4, 16, 32, 8, "bf16", 4),
    ("one_more_than_units", [128] * 4 + [2], [128] * 4 + [2], 16, 32, 8, "bf16", 2),
    ("halves", [250] * 3 + [203, 17], [250] * 3 + [203, 17], 8, 32, 8, "f16", 2),
    ("halves_behind_tokens", [214, 90, 256] * 5, [64, 33, 40] * 5, 16, 32, 8, "bf16", 2),
    ("halves_of_two_rounds", [257] + [250] * 4, [257] + [250] * 4, 16, 32, 8, "bf16", 0),
    ("more_halves_than_units", [250] * 5, [250] * 5, 16, 32, 8, "bf16", 0),
    ("no_rows_between", [40, 60, 1, 9], [40, 0, 1, 9], 16, 32, 8, "bf16", 4),
    ("fewer_keys_than_rows", [20, 0, 3], [40, 5, 3], 16, 32, 8, "bf16", 4),
    ("group1_page8", [129, 40], [129, 7], 8, 8, 8, "bf16", 4),
    ("group3_page32", [200, 90], [70, 90], 32, 12, 4, "bf16", 4),
    ("group7", [130, 260], [130, 50], 16, 28, 4, "f16", 4),
    ("group8_halves", [203, 17, 120], [203, 17, 120], 8, 64, 8, "f16", 2),
    ("group20", [150, 9], [33, 2], 16, 40, 2, "f16", 4),
    ("kv17", [50, 20], [50, 3], 64, 17, 17, "bf16", 4),
    ("page4", [40, 9], [40, 9], 4, 32, 8, "bf16", 0),
]


def test_which_plans_share_their_tiles():
    """(256 compute units, also assumed where there is no GPU)"""
    lib, at = _lib.lib(), lambda a: np.concatenate([[0], np.cumsum(a)]).astype(np.int32)
    for name, kv, qo, P, Hq, Hkv, dtype, workgroups in CASES:
        pages, qo_indptr = at(-(-np.asarray(kv) // P)), at(qo)
        last = np.array([(n - 1) % P + 1 if n else 0 for n in kv], np.int32)
        cap = lib.dskv_mixed_plan_bound(len(kv), int(qo_indptr[-1]), int(pages[-1]) * P)
        plan, info = np.zeros(cap, np.int32), _lib.MixedPlanInfo()
        rc = lib.dskv_mixed_plan_typed(qo_indptr.ctypes.data, pages.ctypes.data, last.ctypes.data, len(kv), P, Hq, Hkv, 128,
                                       _lib.BF16, 0, _lib.ROUTE_OFF, plan.ctypes.data, cap, ctypes.byref(info))
        assert rc == 0 and info.n_splits == 1, name
        assert info.tile_workgroups == workgroups and info.layout == _lib.LAYOUT_SEPARATE, name
        # a caller's own number of workgroups, 32 bits: never
        for target, route, typed in ((512, _lib.ROUTE_OFF, _lib.BF16), (0, _lib.ROUTE_OFF, _lib.F32)):
            assert lib.dskv_mixed_plan_typed(qo_indptr.ctypes.data, pages.ctypes.data, last.ctypes.data, len(kv), P, Hq, Hkv,
                                             128, typed, target, route, plan.ctypes.data, cap, ctypes.byref(info)) == 0
            assert info.tile_workgroups == 0, name


def test_a_walk_past_four_rounds_is_cut():
    lib = _lib.lib()
    for keys, shared in ((1024, True), (1025, False)):
        pages = -(-keys // 16)
        qo, indptr, last = (np.array(a, np.int32) for a in ([0, 200], [0, pages], [keys - 16 * (pages - 1)]))
        cap = lib.dskv_mixed_plan_bound(1, 200, keys)
        plan, info = np.zeros(cap, np.int32), _lib.MixedPlanInfo()
        assert lib.dskv_mixed_plan_typed(qo.ctypes.data, indptr.ctypes.data, last.ctypes.data, 1, 16, 32, 8, 128, _lib.BF16, 0,
                                         _lib.ROUTE_AUTO, plan.ctypes.data, cap, ctypes.byref(info)) == 0
        assert info.tile_workgroups == (4 if shared else 0) and info.n_splits == (1 if shared else 2)
        assert info.tile_workspace_bytes == 0 or not shared


@pytest.mark.parametrize("case", CASES, ids=[c[0] for c in CASES])
def test_the_bound_lets_no_row_miss_a_key(case):
    name, kv, qo, P, Hq, Hkv, dtype, workgroups = case
    sc = make_scenario(71, kv_lens=kv, qo_lens=qo, P=P, Hq=Hq, Hkv=Hkv, D=128, dtype=dtype)
    want = c_oracle.prefill_attn(sc.q, sc.qo_indptr, sc.pages, sc.kv_page_indices, sc.kv_page_indptr, sc.kv_last_page_lens, dtype)
    assert_bound_bites(sc, want, attention_bound(sc, want))


@pytest.mark.gpu
@pytest.mark.parametrize("case", CASES, ids=[c[0] for c in CASES])
def test_short_walks_match_oracle_and_whole_tiles(case):
    from deserve_amd.paged_ops import (BatchPrefillWithPagedKVCacheWrapper, append_paged_kv_cache, apply_rope,
                                       rope_table)

    name, kv, qo, P, Hq, Hkv, dtype, workgroups = case
    print("[case] short walks", *case, flush=True)
    sc = make_scenario(71, kv_lens=kv, qo_lens=qo, P=P, Hq=Hq, Hkv=Hkv, D=128, dtype=dtype)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a, np.int32)).cuda()
    indptr, tab, tabptr, last = (dev(a) for a in (sc.qo_indptr, sc.kv_page_indices, sc.kv_page_indptr,
                                                  sc.kv_last_page_lens))
    w = BatchPrefillWithPagedKVCacheWrapper(torch.empty(64 << 20, dtype=torch.uint8, device="cuda"))
    w.begin_forward(indptr, tabptr, tab, last, Hq, Hkv, 128, P, route_one_row_requests=False)
    assert w._info.tile_workgroups == workgroups
    workgroups = w._info.tile_workgroups = workgroups or 4   # longer walks and more of them: slower, and as right
    q, pages = to_torch(sc.q, dtype), to_torch(sc.pages, dtype)
    offsets = dev(np.maximum(sc.kv_lens - sc.qo_lens, 0))
    run = lambda q, **k: w.forward(q, pages, out=torch.full_like(q, float("nan")), **k)
    for causal in (True, False):
        got = run(q, causal=causal)
        assert bool(torch.isfinite(got.float()).all())
        want = c_oracle.prefill_attn(sc.q, sc.qo_indptr, sc.pages, sc.kv_page_indices, sc.kv_page_indptr,
                                     sc.kv_last_page_lens, dtype, causal)
        bound = attention_bound(sc, want, causal)
        w._info.tile_workgroups = 0
        whole = run(q, causal=causal)
        w._info.tile_workgroups = workgroups
        for form in (got, whole):
            off = np.abs(form.float().cpu().numpy() - want) / bound
            assert off.max() <= 1, (causal, np.unravel_index(off.argmax(), off.shape), off.max())
    if min(np.asarray(kv) - np.asarray(qo)) < 0:
        return
    k, v = to_torch(sc.k, dtype), to_torch(sc.v, dtype)
    q_rot, k_rot = apply_rope(q, k, indptr, offsets, interleave=True, rope_theta=5e5)
    new = pages.clone()
    append_paged_kv_cache(k_rot, v, indptr, pages, tab, tabptr, last)
    want = run(q_rot)
    got = w.forward(q, new, out=torch.full_like(q, float("nan")), k_append=k, v_append=v,
                    rope_table=rope_table(indptr, offsets, q.shape[0], 128, 5e5))
    assert torch.equal(got.view(torch.int16), want.view(torch.int16)) and torch.equal(new.view(torch.int16), pages.view(torch.int16))
