"""Appends to pages from number 2^30 on, where twice the number no longer fits 32 bits: one-token pages of 32 bytes."""
import pytest
import torch


@pytest.mark.gpu
@pytest.mark.parametrize("requests", [3, 70])    # owners by ballot, by search
def test_append_beyond_two_to_the_30_pages(requests):
    from deserve_amd.paged_ops import append_paged_kv_cache

    n = (1 << 30) + 4096
    if torch.cuda.mem_get_info()[0] < 40 << 30:
        pytest.skip("a pool of 34 GB does not fit")
    print("[case] append far", requests, flush=True)
    pages = torch.empty((n, 2, 1, 1, 8), dtype=torch.bfloat16, device="cuda")
    ids = torch.tensor([n - 2, (1 << 30) - 1, 1 << 30] + [(1 << 30) + 9 + 3 * i for i in range(requests - 3)],
                       dtype=torch.int64, device="cuda")
    near = torch.cat([ids - 1, ids, ids + 1, torch.arange(64, device="cuda")]).unique()
    pages[near] = 0
    want = pages[near]
    k, v = (torch.randn((requests, 1, 8), device="cuda").bfloat16() for _ in range(2))
    at = torch.searchsorted(near, ids)
    want[at] = torch.stack([k, v], 1)[:, :, None]
    ptr = torch.arange(requests + 1, dtype=torch.int32, device="cuda")
    append_paged_kv_cache(k, v, ptr, pages, ids.int(), ptr, torch.ones(requests, dtype=torch.int32, device="cuda"))
    assert torch.equal(pages[near].view(torch.int16), want.view(torch.int16))
    del pages
    torch.cuda.empty_cache()
