"""Query tiles leave their rows through LDS, 16 lanes to a column: groups that do not divide a wave's
32 columns, tiles with one live row and one missing row, whole tiles, tiles in parts and the shared
launch - every row of the request, in a tensor whose other rows stay untouched."""
import numpy as np
import pytest
import torch

from deserve_amd import _lib
from kvutil import make_scenario, max_rel_err_per_request, to_torch
from oracle import c_oracle

pytestmark = pytest.mark.gpu

# (Hq, Hkv, dtype); rows per eight-wave tile: 8 * (32 // group)
GROUPS = [(3, 1, "bf16"), (10, 2, "f16"), (7, 1, "bf16"), (24, 2, "bf16"), (17, 1, "f16"), (32, 1, "bf16")]


@pytest.mark.parametrize("case", GROUPS, ids=[f"group{q // k}_{d}" for q, k, d in GROUPS])
def test_rows_out_of_tiles(case):
    from deserve_amd.paged_ops import BatchPrefillWithPagedKVCacheWrapper

    Hq, Hkv, dtype = case
    rows = 8 * (32 // (Hq // Hkv))
    print("[case] rows out of tiles", *case, flush=True)
    qo = [1, rows - 1, rows + 1, 3]
    kv = [40, rows + 1200, rows + 1, 3]
    sc = make_scenario(65, kv_lens=kv, qo_lens=qo, P=16, Hq=Hq, Hkv=Hkv, D=128, dtype=dtype)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a, np.int32)).cuda()
    w = BatchPrefillWithPagedKVCacheWrapper(torch.empty(64 << 20, dtype=torch.uint8, device="cuda"))
    q, pages = to_torch(sc.q, dtype), to_torch(sc.pages, dtype)
    want = c_oracle.prefill_attn(sc.q, sc.qo_indptr, sc.pages, sc.kv_page_indices, sc.kv_page_indptr,
                                 sc.kv_last_page_lens, dtype)
    parts = set()
    # groups over 16 have no decode form: their one-row request stays a tile
    for route, target in ((False, -1), (False, 1024), (_lib.ROUTE_SHARED_LAUNCH, 0), (_lib.ROUTE_SHARED_LAUNCH, -1)):
        w.begin_forward(dev(sc.qo_indptr), dev(sc.kv_page_indptr), dev(sc.kv_page_indices), dev(sc.kv_last_page_lens),
                        Hq, Hkv, 128, 16, target_workgroups=target, route_one_row_requests=route)
        parts.add(w._n_splits)
        held = torch.full((q.shape[0] + 2 * rows,) + tuple(q.shape[1:]), 7.0, dtype=q.dtype, device="cuda")
        out = held[rows: rows + q.shape[0]]
        w.forward(q, pages, out=out)
        torch.cuda.synchronize()
        got = held.float().cpu().numpy()
        assert max_rel_err_per_request(got[rows:-rows], want) <= 2e-2, (route, target)
        assert (got[:rows] == 7.0).all() and (got[-rows:] == 7.0).all(), (route, target)
    assert {1, 2} <= parts
