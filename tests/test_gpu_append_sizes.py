"""The append kernel's forms: row sets of 1, 2 and 4 KiB (as many registers as they fill), the sizes around them and one
that no lane holds whole; pages of any size; 63 and 64 requests.  Bit for bit, untouched bytes included."""
import numpy as np
import pytest
import torch

from kvutil import from_torch, make_scenario, to_torch
from oracle import kv_oracle as orc

HEADS = {512: 2, 1024: 4, 1280: 5, 2048: 8, 4096: 16, 4352: 17}   # bytes of a row set: kv heads of 16 bits


@pytest.mark.gpu
@pytest.mark.parametrize("P", [16, 12])
@pytest.mark.parametrize("row_bytes", list(HEADS))
def test_append_of_every_row_set(row_bytes, P):
    from deserve_amd.paged_ops import append_paged_kv_cache

    print("[case] append sizes", row_bytes, P, flush=True)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a, np.int32)).cuda()
    for kv, qo in (([1, 40, 2 * P, 300], [1, 33, 0, 9]), ([20 + 3 * i for i in range(64)], [i % 5 for i in range(64)])):
        sc = make_scenario(23, kv_lens=kv, qo_lens=qo, P=P, Hq=HEADS[row_bytes], Hkv=HEADS[row_bytes], D=128, dtype="bf16")
        want, pages = sc.pages.copy(), to_torch(sc.pages, "bf16")
        orc.append_paged_kv(want, sc.k, sc.v, sc.qo_indptr, sc.kv_page_indices, sc.kv_page_indptr, sc.kv_last_page_lens)
        append_paged_kv_cache(to_torch(sc.k, "bf16"), to_torch(sc.v, "bf16"), dev(sc.qo_indptr), pages,
                              dev(sc.kv_page_indices), dev(sc.kv_page_indptr), dev(sc.kv_last_page_lens))
        assert np.array_equal(from_torch(pages, "bf16").view(np.uint16), want.view(np.uint16))
