"""The decode attention of fp32 rows and of head sizes other than 128 in the plans of small batches:
four waves split an item's tokens and meet in LDS.  Edges: items with fewer tokens than waves, one
more than a turn of all waves (4 x 16), requests without tokens, cut requests, groups of 1 to 8 q
heads (3 padded to 4), head sizes of 8 and 40, pages of 3 tokens; and as many items as take a
wave each again."""
import numpy as np
import pytest
import torch

from kvutil import make_scenario, max_rel_err_per_request, to_torch
from oracle import c_oracle

pytestmark = pytest.mark.gpu

CASES = [
    # (name, kv_lens, P, Hq, Hkv, D, dtype, target shares)
    ("eight_of_512", [512] * 8, 16, 32, 8, 128, "f32", 0),
    ("a_turn_and_a_token", [65, 1, 16, 17, 64], 16, 32, 8, 128, "f32", 1),
    ("empty_and_cut", [0, 300, 0, 77, 1000], 8, 16, 2, 128, "f32", 20),
    ("group1_d8_page3", [5, 260], 3, 2, 2, 8, "f32", 3),
    ("group3_d40", [333, 64], 16, 12, 4, 40, "f16", 4),
    ("group8_d64", [700, 31], 16, 32, 4, 64, "bf16", 16),
    ("group2_d128_odd_page", [400, 50], 5, 8, 4, 128, "f32", 9),
    ("a_wave_per_item", [9 + i % 5 for i in range(150)], 16, 32, 8, 128, "f32", 0),
]


@pytest.mark.parametrize("case", CASES, ids=[c[0] for c in CASES])
def test_gqa_decode_in_few_shares_matches_oracle(case):
    from deserve_amd.paged_ops import BatchDecodeWithPagedKVCacheWrapper

    name, lens, P, Hq, Hkv, D, dtype, target = case
    print("[case] gqa decode", name, P, Hq, Hkv, D, dtype, target, flush=True)
    sc = make_scenario(67, kv_lens=lens, qo_lens=[1] * len(lens), P=P, Hq=Hq, Hkv=Hkv, D=D, dtype=dtype)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a, np.int32)).cuda()
    w = BatchDecodeWithPagedKVCacheWrapper(torch.empty(16 << 20, dtype=torch.uint8, device="cuda"))
    w.begin_forward(dev(sc.kv_page_indptr), dev(sc.kv_page_indices), dev(sc.kv_last_page_lens), Hq, Hkv, D, P,
                    target_workgroups=target)
    assert w._n_workgroups * Hkv <= torch.cuda.get_device_properties(0).multi_processor_count
    assert (w._n_items * Hkv > 1024) == (name == "a_wave_per_item")
    q, pages = to_torch(sc.q, dtype), to_torch(sc.pages, dtype)
    out = w.forward(q, pages, out=torch.full_like(q, float("nan")))
    torch.cuda.synchronize()
    want = c_oracle.decode_attn(sc.q, sc.pages, sc.kv_page_indices, sc.kv_page_indptr, sc.kv_last_page_lens, dtype)
    got, live = out.float().cpu().numpy(), np.asarray(lens) > 0
    assert np.isfinite(got).all() and not got[~live].any()
    # 32-bit sums of up to 1000 terms: sqrt(1000) roundings of 2^-24 with a margin of ten; 16 bits: the storage type
    assert max_rel_err_per_request(got[live], want[live]) <= (2e-5 if dtype == "f32" else 2e-2)
