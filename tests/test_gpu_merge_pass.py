"""The merge pass of rows in parts: a workgroup per (row, eight heads), a thread per four dims.  Sizes
at its edges: rows in two to eight parts (each requested in one go), in 9, 16, 17 and 33 (a workgroup for every two
heads, whose four groups of threads take a quarter each: quarters of unequal length, more than eight in one),
rows without parts beside them, head counts that do not fill a workgroup or need several, both element types."""
import numpy as np
import pytest
import torch

from kvutil import make_scenario, max_rel_err_per_request, to_torch
from oracle import c_oracle

pytestmark = pytest.mark.gpu

CASES = [
    # (name, tiles of each request (shares of four tiles), Hq, Hkv, dtype)
    ("two_to_five", [8, 2, 12, 0, 16, 20], 32, 8, "bf16"),
    ("six_to_nine", [24, 28, 32, 36, 1], 64, 8, "f16"),
    ("16_17_33", [64, 68, 132, 3], 12, 4, "bf16"),
    ("one_head", [40, 9], 1, 1, "bf16"),
    ("17_heads", [40, 21, 50], 17, 17, "f16"),
]


@pytest.mark.parametrize("case", CASES, ids=[c[0] for c in CASES])
def test_merge_pass_matches_oracle(case):
    from deserve_amd.paged_ops import BatchDecodeWithPagedKVCacheWrapper

    name, tiles, Hq, Hkv, dtype = case
    print("[case] merge pass", *case, flush=True)
    lens = [max(16 * t - 3, 0) for t in tiles]
    sc = make_scenario(64, kv_lens=lens, qo_lens=[1] * len(lens), P=16, Hq=Hq, Hkv=Hkv, D=128, dtype=dtype)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a, np.int32)).cuda()
    w = BatchDecodeWithPagedKVCacheWrapper(torch.empty(64 << 20, dtype=torch.uint8, device="cuda"))
    w.begin_forward(dev(sc.kv_page_indptr), dev(sc.kv_page_indices), dev(sc.kv_last_page_lens), Hq, Hkv, 128, 16,
                    target_workgroups=sum(tiles) // 4)
    assert len(lens) < w._n_items <= 32 * len(lens)             # cut, and merged by the pass under test
    q, pages = to_torch(sc.q, dtype), to_torch(sc.pages, dtype)
    out = torch.full_like(q, float("nan"))
    w.forward(q, pages, out=out, phases=1)
    w.forward(q, pages, out=out, phases=2)
    want = c_oracle.decode_attn(sc.q, sc.pages, sc.kv_page_indices, sc.kv_page_indptr, sc.kv_last_page_lens, dtype)
    live = np.asarray(lens) > 0
    got = out.float().cpu().numpy()
    assert np.isfinite(got).all() and not got[~live].any()
    assert max_rel_err_per_request(got[live], want[live]) <= 2e-2
