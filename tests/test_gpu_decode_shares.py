"""The small-batch decode attention on the shares that its planner lays out: requests that lie whole in a share with one
to three tiles for each of its waves, several of them in a share, requests cut into shares of a round; q heads per kv
head from 1 to 8 (heads are dealt to waves in pairs); pages of 32 to 4 tokens.  Against the oracle, and the
launch that rotates and appends against the calls one by one."""
import ctypes

import numpy as np
import pytest
import torch

from kvutil import make_scenario, max_rel_err_per_request, to_torch
from oracle import c_oracle

pytestmark = pytest.mark.gpu

CASES = [
    # (name, kv_lens, P, Hq, Hkv, dtype, shares, whether requests are cut)
    ("one_round", [128], 16, 32, 8, "bf16", 1, False),
    ("a_token_past_a_round", [129], 16, 32, 8, "bf16", 1, False),
    ("two_rounds", [256, 241], 16, 32, 8, "f16", 2, False),
    ("three_rounds_cut", [272], 16, 32, 8, "bf16", 3, True),
    ("several_to_a_share", [40, 17, 16, 1, 33, 100, 90, 5], 16, 32, 8, "bf16", 4, False),
    ("empty_ones_among_them", [0, 40, 0, 90, 0], 16, 32, 8, "bf16", 2, False),
    ("short_beside_cut", [20, 700, 9, 400], 16, 32, 8, "f16", 12, True),
    ("group1_page8", [250, 129], 8, 16, 16, "bf16", 2, False),
    ("group2_page32", [250, 400], 32, 16, 8, "f16", 6, True),
    ("group3_page4", [250, 60, 200], 4, 24, 8, "bf16", 3, False),
    ("group5_page8", [250, 400], 8, 40, 8, "f16", 6, True),
    ("group6", [250, 400, 3], 16, 48, 8, "bf16", 7, True),
    ("group7_page8", [129, 700], 8, 56, 8, "bf16", 8, True),
    ("group8_page8", [250, 400], 8, 64, 8, "f16", 6, True),
]


def _dev(a):
    return torch.from_numpy(np.ascontiguousarray(a, np.int32)).cuda()


@pytest.mark.parametrize("case", CASES, ids=[c[0] for c in CASES])
def test_shares_match_oracle_and_separate_calls(case):
    from deserve_amd import _lib
    from deserve_amd.paged_ops import BatchDecodeWithPagedKVCacheWrapper, rope_append_paged_kv_cache

    name, lens, P, Hq, Hkv, dtype, shares, cut = case
    print("[case] decode shares", *case, flush=True)
    sc = make_scenario(97, kv_lens=lens, qo_lens=[1] * len(lens), P=P, Hq=Hq, Hkv=Hkv, D=128, dtype=dtype)
    w = BatchDecodeWithPagedKVCacheWrapper(torch.empty(64 << 20, dtype=torch.uint8, device="cuda"))
    tables = (_dev(sc.kv_page_indices), _dev(sc.kv_page_indptr), _dev(sc.kv_last_page_lens))
    w.begin_forward(tables[1], tables[0], tables[2], Hq, Hkv, 128, P)
    flag = ctypes.c_int32()
    _lib.lib().dskv_decode_launch(w._n_items, w._n_workgroups, Hq, Hkv, 128, _lib.BF16, ctypes.byref(flag))
    assert flag.value and w._n_workgroups == shares and (w._n_items > len(lens)) == cut
    q, k, v, pages = (to_torch(x, dtype) for x in (sc.q, sc.k, sc.v, sc.pages))
    outs = [w.forward(q, pages, out=torch.full_like(q, float("nan"))) for _ in range(4)]
    want = c_oracle.decode_attn(sc.q, sc.pages, sc.kv_page_indices, sc.kv_page_indptr, sc.kv_last_page_lens, dtype)
    live = np.asarray(lens) > 0
    got = outs[0].float().cpu().numpy()
    assert np.isfinite(got).all() and not got[~live].any()
    if live.any():
        assert max_rel_err_per_request(got[live], want[live]) <= 2e-2
    assert all(torch.equal(o.view(torch.int16), outs[0].view(torch.int16)) for o in outs[1:])
    assert int(w._counters.abs().max()) == 0
    if not live.all():
        return
    indptr, offsets = _dev(np.arange(len(lens) + 1)), _dev(np.asarray(lens) - 1)
    one, sep = pages.clone(), pages.clone()
    q_rot = rope_append_paged_kv_cache(q, k, v, indptr, offsets, sep, *tables, rope_theta=5e5)
    a = w.forward(q, one, k_append=k, v_append=v, rope_offsets=offsets, rope_theta=5e5)
    b = w.forward(q_rot, sep)
    assert torch.equal(one.view(torch.int16), sep.view(torch.int16)) and torch.equal(a.view(torch.int16), b.view(torch.int16))
