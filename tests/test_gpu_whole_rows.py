"""K read by whole rows and through LDS (the decode form for small batches, and the decode rows of a
shared mixed launch), with NaN in every page slot that holds no token: lengths around a tile and
a page, a tile across two pages and more, the newest token in the pages or still on its way."""
import numpy as np
import pytest
import torch

from deserve_amd import _lib
from kvutil import make_scenario, max_rel_err_per_request, to_torch
from oracle import c_oracle

pytestmark = pytest.mark.gpu

TOL = {"bf16": 2e-2, "f16": 2e-2}   # of a row's own scale: 16-bit probabilities and results
LENS = [1, 15, 16, 17, 31, 33, 8, 255, 1, 700, 64, 9, 129]


def _with_nan(sc, dtype):
    """The pool with NaN in the slots past every request's end and in the pages nobody owns."""
    pages = to_torch(sc.pages, dtype)
    held = torch.zeros(pages.shape[0], sc.P, dtype=torch.bool)
    for b, n in enumerate(sc.kv_lens):
        for t in range(int(n)):
            held[sc.kv_page_indices[sc.kv_page_indptr[b] + t // sc.P], t % sc.P] = True
    return torch.where(held.cuda()[:, None, :, None, None], pages, torch.full_like(pages, float("nan")))


@pytest.mark.parametrize("dtype,P", [("bf16", 16), ("bf16", 32), ("f16", 8), ("bf16", 4), ("f16", 1)])
@pytest.mark.parametrize("shared", [False, True], ids=["small_batch", "shared_launch"])
def test_slots_without_a_token_do_not_matter(dtype, P, shared):
    from deserve_amd.paged_ops import BatchDecodeWithPagedKVCacheWrapper, BatchPrefillWithPagedKVCacheWrapper

    print("[case] whole rows", dtype, P, shared, flush=True)
    if shared and P < 4:
        pytest.skip("the shared launch takes pages of four tokens and more")
    qo = [1] * len(LENS) + ([40] if shared else [])
    sc = make_scenario(91, kv_lens=LENS + ([90] if shared else []), qo_lens=qo, P=P, Hq=32, Hkv=8, D=128, dtype=dtype)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a, np.int32)).cuda()
    qo_ptr, tab, tabptr, last = (dev(a) for a in (sc.qo_indptr, sc.kv_page_indices, sc.kv_page_indptr,
                                                  sc.kv_last_page_lens))
    q, pages = to_torch(sc.q, dtype), _with_nan(sc, dtype)
    ws = torch.empty(64 << 20, dtype=torch.uint8, device="cuda")
    want = c_oracle.prefill_attn(sc.q, sc.qo_indptr, sc.pages, sc.kv_page_indices, sc.kv_page_indptr,
                                 sc.kv_last_page_lens, dtype, causal=True)
    if shared:
        w = BatchPrefillWithPagedKVCacheWrapper(ws)
        w.begin_forward(qo_ptr, tabptr, tab, last, 32, 8, 128, P, route_one_row_requests=_lib.ROUTE_SHARED_LAUNCH)
        assert w._info.layout == _lib.LAYOUT_SHARED
        got = w.forward(q, pages)
        torch.cuda.synchronize()
        assert max_rel_err_per_request(got.float().cpu().numpy(), want) <= TOL[dtype]
        return
    w = BatchDecodeWithPagedKVCacheWrapper(ws)
    w.begin_forward(tabptr, tab, last, 32, 8, 128, P)
    assert w._n_workgroups * 8 <= 256       # the form for small batches
    got = w.forward(q, pages)
    torch.cuda.synchronize()
    assert max_rel_err_per_request(got.float().cpu().numpy(), want) <= TOL[dtype]
    if w.fused_append_supported(q.dtype):   # the newest token taken from k and v, its slot NaN until then
        tails = [(sc.kv_page_indices[sc.kv_page_indptr[b + 1] - 1], (n - 1) % P) for b, n in enumerate(LENS)]
        k, v = (torch.stack([pages[p, half, s] for p, s in tails]) for half in (0, 1))
        holed = pages.clone()
        for p, s in tails:
            holed[p, :, s] = float("nan")
        again = w.forward(q, holed, k_append=k, v_append=v)
        torch.cuda.synchronize()
        assert torch.equal(again.view(torch.int16), got.view(torch.int16))
        assert torch.equal(holed.view(torch.int16), pages.view(torch.int16))
