"""Copies into chunks travel behind the call that enqueued them; what uses the chunk's memory next is
ordered behind them, whoever holds it by then.  Swap engines are stood in for by recorders."""
import torch

from deserve_amd.kvcache.manager import KVCacheManager
from deserve_amd.kvcache.paged.chunk_pool import CpuChunkPool
from deserve_amd.kvcache.paged.page_table import PageTableAllocator
from deserve_amd.kvcache.virtual import VirtualPagedKVCache, VirtualPagePool

CPU = torch.device("cpu")


class Engine:
    staging_bytes = 128 << 20
    is_open = True

    def __init__(self, name, log):
        self.name, self.log, self.arrived = name, log, False

    def done(self):
        return self.arrived

    def __getattr__(self, call):
        if call not in ("swap_out", "swap_in", "fence", "fence_pages", "wait"):
            raise AttributeError(call)
        return lambda *args: self.log.append((self.name, call))


def _side(name, log, chunks):
    pool = VirtualPagePool(2, 40, 0, 16, CPU, torch.float16, n_kv_heads=1, head_dim=8)
    pool.engine = Engine(name, log)
    tables = PageTableAllocator(8, 4096, 16, CPU)

    def cache(tokens):
        c = VirtualPagedKVCache.empty(tables, pool)
        c.extend(tokens)
        return c

    return KVCacheManager(pool, chunks, tables), cache


def _chunks():
    return CpuChunkPool(2, 4, 16, torch.float16, n_kv_heads=1, head_dim=8)


def test_a_chunk_freed_and_handed_out_again_is_ordered_behind_the_copy_into_its_memory():
    log, chunks = [], _chunks()
    manager, cache = _side("a", log, chunks)
    first = manager.copy_gpu_to_cpu(cache(16 * 4), "t")
    first.free()                                       # cancelled while its pages travel
    other = [chunks.alloc(1) for _ in range(8)]        # all of the arena, the same memory among it
    log.clear()
    for h in other:
        h.retrieve()
    assert log == [("a", "fence")] * 4                 # the four units it spans, no more
    manager.synchronize()
    log.clear()
    for h in other:
        h.retrieve()
    assert log == []


def test_a_second_manager_with_an_engine_of_its_own_waits_for_the_first_ones_copies():
    log, chunks = [], _chunks()
    a, cache_a = _side("a", log, chunks)
    b, cache_b = _side("b", log, chunks)
    handle = a.copy_gpu_to_cpu(cache_a(16 * 2), "t")
    log.clear()
    b.copy_cpu_to_gpu(handle, "t")                     # reads the chunk on another engine's streams
    assert log == [("a", "fence"), ("b", "swap_in"), ("b", "fence_pages")]
    handle.free()
    log.clear()
    b.copy_gpu_to_cpu(cache_b(16 * 8), "u")            # writes the same memory
    assert log == [("a", "fence"), ("b", "swap_out"), ("b", "fence_pages")]
    log.clear()
    a.copy_cpu_to_gpu(handle, "t")                     # its own copies it keeps in order itself
    assert log == [("b", "fence"), ("a", "swap_in"), ("a", "fence_pages")]


def test_finished_copies_are_forgotten_without_anybody_waiting():
    log, chunks = [], _chunks()
    manager, cache = _side("a", log, chunks)
    one = cache(16)
    for i in range(100):
        manager.engine.arrived = i >= 80
        manager.copy_gpu_to_cpu(one, "t").free()
    assert len(chunks._writes) <= 64 and ("a", "wait") not in log
