"""The two forms of the 16-bit decode attention, plain, with the step's token appended inside the launch
and with RoPE inside.  As the planner's own rule picks them: plans filled up with workgroups without
work, one head in 256 split shares, requests in so many parts that a merge launch follows the split
form, the deployed batch of 75 on 8-token pages.  And the form whose waves are kv heads on every kind
of page and with more than one workgroup per share, in explicit shares: small batches of these shapes
have the split form by themselves."""
import ctypes

import numpy as np
import pytest
import torch

from kvutil import make_scenario, max_rel_err_per_request, to_torch
from oracle import c_oracle

pytestmark = pytest.mark.gpu

CASES = [
    # (name, kv_lens, P, Hq, Hkv, dtype, target, splits a head over waves)
    ("two_heads_filled_up", [700, 1, 33, 16], 16, 8, 2, "bf16", 0, False),
    ("one_head_filled_up", [40, 300, 17], 8, 8, 1, "f16", 0, False),
    ("four_heads_one_request", [4000], 16, 16, 4, "bf16", 0, False),
    ("two_heads_lopsided", [16 * 700 + 3] + [40 + i for i in range(9)], 16, 8, 2, "bf16", 0, True),
    ("one_head_256_shares", [16 * 1700, 16 * 3310 + 5], 16, 4, 1, "f16", 0, True),
    ("parts_in_the_dozens", [16 * 500 + 1], 16, 10, 5, "bf16", 0, True),
    ("75_on_page8", [200 + 7 * i for i in range(75)], 8, 16, 8, "f16", 0, False),
    ("page8_bf16", [3000, 700, 9, 8, 1, 600], 8, 32, 8, "bf16", 64, False),
    ("page8_f16_group8", [2100, 1999, 16, 7], 8, 64, 8, "f16", 64, False),
    ("page4", [3001, 1200, 5, 4], 4, 32, 8, "bf16", 64, False),
    ("page2", [2500, 1700, 2, 1], 2, 16, 8, "f16", 64, False),
    ("page32", [2500, 1700, 31, 33], 32, 16, 8, "bf16", 64, False),
    ("kv12_page8", [1500, 700, 33], 8, 24, 12, "bf16", 32, False),
    ("kv16", [1500, 700, 33], 16, 32, 16, "f16", 32, False),
    ("kv17_one_wave_in_the_last_workgroup", [1500, 700, 33], 16, 17, 17, "bf16", 32, False),
    ("eight_wave_merge", [33000], 16, 8, 8, "bf16", 256, False),
]


def _dev(a):
    return torch.from_numpy(np.ascontiguousarray(a, np.int32)).cuda()


@pytest.mark.parametrize("case", CASES, ids=[c[0] for c in CASES])
def test_form_matches_oracle_and_separate_calls(case):
    from deserve_amd import _lib
    from deserve_amd.paged_ops import (BatchDecodeWithPagedKVCacheWrapper, append_paged_kv_cache,
                                       rope_append_paged_kv_cache)

    name, lens, P, Hq, Hkv, dtype, target, splits = case
    print("[case] decode form", *case, flush=True)
    sc = make_scenario(83, kv_lens=lens, qo_lens=[1] * len(lens), P=P, Hq=Hq, Hkv=Hkv, D=128, dtype=dtype)
    w = BatchDecodeWithPagedKVCacheWrapper(torch.empty(64 << 20, dtype=torch.uint8, device="cuda"))
    tables = (_dev(sc.kv_page_indices), _dev(sc.kv_page_indptr), _dev(sc.kv_last_page_lens))
    w.begin_forward(tables[1], tables[0], tables[2], Hq, Hkv, 128, P, target_workgroups=target)
    flag = ctypes.c_int32()
    _lib.lib().dskv_decode_launch(w._n_items, w._n_workgroups, Hq, Hkv, 128, _lib.BF16, ctypes.byref(flag))
    assert bool(flag.value) == splits
    q, k, v, pages = (to_torch(x, dtype) for x in (sc.q, sc.k, sc.v, sc.pages))
    got = w.forward(q, pages, out=torch.full_like(q, float("nan")))
    want = c_oracle.decode_attn(sc.q, sc.pages, sc.kv_page_indices, sc.kv_page_indptr, sc.kv_last_page_lens, dtype)
    out = got.float().cpu().numpy()
    assert np.isfinite(out).all() and max_rel_err_per_request(out, want) <= 2e-2
    # the appended token, without and with rotation, against the calls one by one
    indptr, offsets = _dev(np.arange(len(lens) + 1)), _dev(np.asarray(lens) - 1)
    one, sep = pages.clone(), pages.clone()
    append_paged_kv_cache(k, v, indptr, sep, *tables)
    a, b = w.forward(q, one, k_append=k, v_append=v), w.forward(q, sep)
    assert torch.equal(one.view(torch.int16), sep.view(torch.int16)) and torch.equal(a.view(torch.int16), b.view(torch.int16))
    one, sep = pages.clone(), pages.clone()
    q_rot = rope_append_paged_kv_cache(q, k, v, indptr, offsets, sep, *tables, rope_theta=5e5)
    a = w.forward(q, one, k_append=k, v_append=v, rope_offsets=offsets, rope_theta=5e5)
    b = w.forward(q_rot, sep)
    assert torch.equal(one.view(torch.int16), sep.view(torch.int16)) and torch.equal(a.view(torch.int16), b.view(torch.int16))
