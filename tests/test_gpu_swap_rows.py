"""Scattered pages over the link as rows of a rectangle: page sizes on both sides of the row sizes, what is
left over behind whole rows, and the host memory that keeps the linear copy (pageable, odd addresses)."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("memory", ["pinned", "pageable", "odd"])
@pytest.mark.parametrize("page,heads,dim,n", [(8, 1, 64, 3),       # 2 KiB pages, less than a row in all
                                              (8, 1, 64, 35),      # 2 KiB pages, a row and a rest
                                              (8, 8, 64, 7),       # 16 KiB: a row each
                                              (5, 3, 40, 61),      # 2400 bytes: rows that no page ends with
                                              (16, 8, 128, 9)])    # 64 KiB
def test_rows_of_every_page_size_and_memory(page, heads, dim, n, memory):
    from deserve_amd.kvcache import _native
    from deserve_amd.kvcache.paged.page_pool import GpuPagePool

    print("[case]", page, heads, dim, n, memory, flush=True)
    layers, dev = 3, torch.device("cuda")
    pool = GpuPagePool(layers, 70, page, dev, torch.bfloat16, heads, dim)
    rng = np.random.default_rng(page * n)
    before = torch.from_numpy(rng.integers(0, 1 << 15, tuple(pool.pages.shape), dtype=np.int16))
    pool.pages.view(torch.int16).copy_(before)
    ids = torch.from_numpy(rng.permutation(70)[:n].astype(np.int32))
    words = layers * n * pool.page_bytes // 2
    shift = 1 if memory == "odd" else 0

    def host():
        return torch.zeros(words + shift, dtype=torch.int16, pin_memory=memory != "pageable")[shift:]

    engine = _native.SwapEngine(1 << 20)
    out, back = host(), host()
    engine.swap_out(out, pool, ids)
    engine.wait()
    want = before[:, ids.long()].reshape(-1)
    assert torch.equal(out, want)
    new = torch.from_numpy(rng.integers(0, 1 << 15, words, dtype=np.int16))
    back.copy_(new)
    engine.swap_in(pool, back, ids)
    engine.wait()
    after = before.clone()
    after[:, ids.long()] = new.reshape(layers, n, *before.shape[2:])
    assert torch.equal(pool.pages.view(torch.int16).cpu(), after)
    back.copy_(want)
    engine.exchange(out, back, pool, ids)
    engine.wait()
    assert torch.equal(out, new) and torch.equal(pool.pages.view(torch.int16).cpu(), before)
    engine.close()
