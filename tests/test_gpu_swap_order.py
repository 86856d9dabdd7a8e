"""Swap-outs and swap-ins travel beside each other but act on the pool, and on host memory they
share, in the order of the calls: seeded sequences of calls and of kernels that overwrite pages
behind fence_pages(), against the same sequence on numpy arrays.  Staging of 1 MiB (a ring of 4)
under transfers of up to 3 MiB: chunks, wraps and stretches that wait for their copy."""
import numpy as np
import pytest
import torch

from oracle import kv_oracle as orc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("seed", range(4))
def test_calls_act_in_order(seed):
    from deserve_amd.kvcache import _native
    from deserve_amd.kvcache.paged.page_pool import GpuPagePool
    from deserve_amd.kvcache.pinned.pinned_memory import pinned_empty

    print("[case] swap order", seed, flush=True)
    L, P, num_pages, most = 3, 16, 40, 16
    pool = GpuPagePool(L, num_pages, P, "cuda", torch.bfloat16)
    rng = np.random.default_rng(seed)
    bits = lambda t: t.view(torch.int16).cpu().numpy()
    pool.pages.view(torch.int16).random_(0, 1 << 15)
    model = bits(pool.pages).copy()
    hosts = [pinned_empty((L * most,) + tuple(pool.pages.shape[2:]), torch.bfloat16) for _ in range(4)]
    for h in hosts:
        h.view(torch.int16).copy_(torch.from_numpy(rng.integers(0, 1 << 15, h.shape).astype(np.int16)))
    images = [bits(h).copy() for h in hosts]
    eng = _native.SwapEngine(1 << 20)
    for step in range(60):
        what = rng.choice(["out", "in", "exchange", "write"], p=[0.42, 0.42, 0.04, 0.12])
        n, a, b = int(rng.integers(1, most + 1)), int(rng.integers(4)), int(rng.integers(4))
        ids = rng.permutation(num_pages)[:n].astype(np.int32)
        tids = torch.from_numpy(ids)
        if what == "out":
            eng.swap_out(hosts[a][: L * n], pool, tids)
            images[a][: L * n] = orc.gather_pages(model, ids)
        elif what == "in":
            eng.swap_in(pool, hosts[a][: L * n], tids)
            orc.scatter_pages(model, ids, images[a][: L * n])
        elif what == "exchange":
            eng.exchange(hosts[a][: L * n], hosts[b][: L * n], pool, tids)
            out = orc.gather_pages(model, ids)
            if a != b:
                orc.scatter_pages(model, ids, images[b][: L * n])
            images[a][: L * n] = out
        else:
            eng.fence_pages()      # then the current stream may write pages
            pool.pages.view(torch.int16)[:, int(ids[0])] = step
            model[:, int(ids[0])] = step
    eng.wait()
    torch.cuda.synchronize()
    assert np.array_equal(bits(pool.pages), model)
    for h, image in zip(hosts, images):
        assert np.array_equal(bits(h), image)
    eng.close()


def test_work_on_an_offloaded_chunk_is_ordered_without_synchronize():
    """A device copy of handle.retrieve() enqueued right behind copy_gpu_to_cpu sees the pages
    (256 MB: ~5 ms on the link, the pages are packed long before)."""
    from deserve_amd.kvcache.manager import KVCacheManager
    from deserve_amd.kvcache.paged.chunk_pool import CpuChunkPool
    from deserve_amd.kvcache.paged.page_table import PageTableAllocator
    from deserve_amd.kvcache.virtual import VirtualPagedKVCache, VirtualPagePool

    print("[case] chunk read behind its offload", flush=True)
    L, P, n = 16, 16, 256
    pool = VirtualPagePool(L, n + 8, 8, P, torch.device("cuda"), torch.bfloat16)
    pool.pages.view(torch.int16).random_(0, 1 << 15)
    tables = PageTableAllocator(2, n * P, P, torch.device("cuda"))
    mgr = KVCacheManager(pool, CpuChunkPool(L, 9, P, torch.bfloat16), tables)
    cache = VirtualPagedKVCache.empty(tables, pool)
    cache.extend(n * P)
    want = orc.gather_pages(pool.pages.view(torch.int16).cpu().numpy(), cache.page_table.retrieve().numpy())
    handle = mgr.copy_gpu_to_cpu(cache, "task")
    got = handle.retrieve()[: L * n].to("cuda", non_blocking=True)
    cache.free()
    torch.cuda.current_stream().synchronize()
    assert np.array_equal(got.view(torch.int16).cpu().numpy(), want)
    mgr.synchronize()
    assert np.array_equal(handle.retrieve()[: L * n].view(torch.int16).numpy(), want)


@pytest.mark.parametrize("idle_between", [True, False])
def test_pages_fence_never_waits_for_the_link_however_many_offloads_went_before(idle_between):
    """fence_pages behind more offloads than the engine keeps host ranges of (256), all finished or
    still on their way: the current stream goes on while the last gigabyte (19 ms) travels."""
    from deserve_amd.kvcache import _native
    from deserve_amd.kvcache.paged.page_pool import GpuPagePool
    from deserve_amd.kvcache.pinned.pinned_memory import pinned_empty

    print("[case] pages fence behind 300 offloads", idle_between, flush=True)
    L, P, n = 16, 16, 1024                       # 1 MiB of all layers per page id
    pool = GpuPagePool(L, n, P, "cuda", torch.bfloat16)
    host = pinned_empty((L * n,) + tuple(pool.pages.shape[2:]), torch.bfloat16)
    every, one = torch.arange(n, dtype=torch.int32), torch.zeros(1, dtype=torch.int32)
    eng = _native.SwapEngine()
    assert eng.independent
    if not idle_between:
        for _ in range(2):                       # keep the link busy while the calls are made
            eng.swap_out(host, pool, every)
    for i in range(300):
        eng.swap_out(host[i * L: (i + 1) * L], pool, one)
    if idle_between:
        torch.cuda.synchronize()                 # the engine is not told
    eng.swap_out(host, pool, every)
    eng.fence_pages()
    event = torch.cuda.Event()
    event.record()
    event.synchronize()
    assert not eng.done()                        # the pages are free again, their copies on the link
    eng.wait()
    assert eng.done()
    eng.close()
