"""The decode attention of small batches: a workgroup per (share, kv head) whose waves split the
share's tiles, and the merge of cut requests inside the launch.  Sizes at its edges: slices that
hold no tile, one, several requests or a part of one; one share and as many as there may be;
groups of 1 to 8 q heads; pages of 16, 8 and 4 tokens; requests without tokens."""
import numpy as np
import pytest
import torch

from kvutil import make_scenario, max_rel_err_per_request, to_torch
from oracle import c_oracle

pytestmark = pytest.mark.gpu

CASES = [
    # (name, kv_lens, P, Hq, Hkv, dtype, target shares)
    ("one_token", [1], 16, 32, 8, "bf16", 0),
    ("one_tile_and_a_token", [17], 16, 32, 8, "f16", 0),
    ("nine_tiles_in_eight_waves", [16 * 9], 16, 32, 8, "bf16", 1),
    ("a_request_per_wave_and_more", [3, 16, 1, 40, 16, 5, 17, 2, 90, 1, 33], 16, 32, 8, "bf16", 2),
    ("empty_requests_between", [0, 30, 0, 0, 200, 0], 16, 32, 8, "bf16", 3),
    ("most_parts", [16 * 40 + 5], 16, 32, 8, "bf16", 32),
    ("two_sets_end_in_a_share", [200, 130, 310, 170], 16, 64, 8, "bf16", 7),
    ("group1_kv16", [300, 77], 16, 16, 16, "f16", 16),
    ("group3_page8", [250, 9, 64], 8, 12, 4, "bf16", 5),
    ("group8_page4", [100, 33, 700], 4, 16, 2, "f16", 40),
    ("default_plan", [1777, 300, 12], 8, 64, 8, "bf16", 0),
]


@pytest.mark.parametrize("case", CASES, ids=[c[0] for c in CASES])
def test_split_decode_matches_oracle_and_the_merge_launch(case):
    from deserve_amd.paged_ops import BatchDecodeWithPagedKVCacheWrapper

    name, lens, P, Hq, Hkv, dtype, target = case
    print("[case] split decode", *case, flush=True)
    sc = make_scenario(61, kv_lens=lens, qo_lens=[1] * len(lens), P=P, Hq=Hq, Hkv=Hkv, D=128, dtype=dtype)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a, np.int32)).cuda()
    w = BatchDecodeWithPagedKVCacheWrapper(torch.empty(16 << 20, dtype=torch.uint8, device="cuda"))
    w.begin_forward(dev(sc.kv_page_indptr), dev(sc.kv_page_indices), dev(sc.kv_last_page_lens), Hq, Hkv, 128, P,
                    target_workgroups=target)
    assert w._n_workgroups * Hkv <= torch.cuda.get_device_properties(0).multi_processor_count
    q, pages = to_torch(sc.q, dtype), to_torch(sc.pages, dtype)
    outs = [w.forward(q, pages, out=torch.full_like(q, float("nan"))) for _ in range(20)]
    two = torch.full_like(q, float("nan"))
    w.forward(q, pages, out=two, phases=1)
    w.forward(q, pages, out=two, phases=2)
    torch.cuda.synchronize()
    want = c_oracle.decode_attn(sc.q, sc.pages, sc.kv_page_indices, sc.kv_page_indptr, sc.kv_last_page_lens, dtype)
    live = np.asarray(lens) > 0
    got = outs[0].float().cpu().numpy()
    assert np.isfinite(got).all() and not got[~live].any()
    assert max_rel_err_per_request(got[live], want[live]) <= 2e-2
    for o in outs[1:]:      # whichever part finishes last, the sums are taken in the same order
        assert torch.equal(o.view(torch.int16), outs[0].view(torch.int16))
    # the two merges add the same fp32 numbers in another order: one unit of the 16-bit result's last
    # place (2^-7 of it in bf16, 2^-10 in f16), or fp32 noise of the row's scale beside a zero
    ulp = 2.0 ** (-7 if dtype == "bf16" else -10)
    diff = (two.float() - outs[0].float()).abs()
    assert bool((diff <= ulp * outs[0].float().abs() + 1e-6).all()), float(diff.max())
    assert int(w._counters.abs().max()) == 0      # every launch leaves the counters as it found them
