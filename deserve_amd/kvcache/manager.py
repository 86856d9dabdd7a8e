"""Per-request offload / reload of scattered pages
(deserve_worker/kvcache/manager.py:12-89).

A request's pages are named by its block table and lie anywhere in the pool.
Offload packs them, all layers at once, into the request's pinned chunk in the
layout (L * n, 2, P, Hkv, D) - layer major, then block-table order - and reload
does the reverse into freshly allocated pages.  Both are enqueued on the swap
engine's side streams (gather/scatter kernel + one large copy per staging
chunk) instead of the reference's blocking advanced-index copy; ``synchronize``
blocks the host until they are done - a chunk holds its request's pages from
then on - and the compute stream is fenced behind what the copies do to the pool,
so a caller that keeps the reference's call order sees the same results.  Work of
that stream on a chunk (a copy of ``handle.retrieve()``) is ordered by ``retrieve``.
"""
from __future__ import annotations

import torch

from deserve_amd.kvcache import _native
from deserve_amd.kvcache.paged.chunk_pool import ChunkHandle, CpuChunkPool
from deserve_amd.kvcache.paged.kvcache import PagedKVCache
from deserve_amd.kvcache.paged.page_table import PageTableAllocator
from deserve_amd.kvcache.virtual import VirtualPagedKVCache, VirtualPagePool


class _Progress:
    """Copies out of one manager: enqueued so far; of these, waited for."""

    def __init__(self) -> None:
        self.enqueued = self.finished = 0


class _CopyOut:
    """A request's trip into its chunk (chunk_pool.PendingWrite)."""

    def __init__(self, engine: _native.SwapEngine, progress: _Progress) -> None:
        progress.enqueued += 1
        self.engine, self.progress, self.number = engine, progress, progress.enqueued

    def finished(self) -> bool:
        return self.number <= self.progress.finished or not self.engine.is_open   # closing one finishes its copies

    def poll(self) -> bool:
        return self.finished() or self.engine.done()

    def fence(self) -> None:
        self.engine.fence()


class KVCacheManager:
    def __init__(self, virtual_page_pool: VirtualPagePool, cpu_chunk_pool: CpuChunkPool,
                 page_table_allocator: PageTableAllocator, staging_bytes: int = 128 << 20):
        self.virtual_page_pool = virtual_page_pool
        self.cpu_chunk_pool = cpu_chunk_pool
        self.page_table_allocator = page_table_allocator
        # the pool's engine (its two streams also carry the bulk slice swap) unless another
        # staging size is asked for
        shared = getattr(virtual_page_pool, "engine", None)
        self.engine = shared if shared is not None and staging_bytes == shared.staging_bytes \
            else _native.SwapEngine(staging_bytes)
        self._progress = _Progress()

    def copy_gpu_to_cpu(self, paged_kvcache: PagedKVCache[VirtualPagePool],
                        task_id: str) -> ChunkHandle:
        """Only the copy; the caller frees the GPU pages and owns the handle."""
        table = paged_kvcache.page_table
        n = table.occupied
        handle = self.cpu_chunk_pool.alloc(n)
        rows = n * self.cpu_chunk_pool.num_layers
        # the engine keeps the order of its own copies; another manager's may still write this memory
        self.cpu_chunk_pool.order_behind_writes(handle, but=self.engine)
        self.engine.swap_out(handle.rows()[:rows], self.virtual_page_pool, table.retrieve())
        # pages may be handed to another request right after this returns: they have been packed
        # by the time the current stream goes on, and travel while it does
        self.engine.fence_pages()
        # not so work on the chunk's memory: retrieve() waits for the trip
        self.cpu_chunk_pool.note_write(handle, _CopyOut(self.engine, self._progress))
        return handle

    def copy_cpu_to_gpu(self, chunk_handle: ChunkHandle, task_id: str) -> VirtualPagedKVCache:
        """Only the copy; the caller frees the chunk and owns the new cache."""
        pool = self.virtual_page_pool
        n = chunk_handle.initial_size
        ids = pool.alloc(n)
        if ids is None:
            raise RuntimeError("Failed to allocate page tables")
        table = self.page_table_allocator.alloc()
        table.extend(ids)
        rows = n * self.cpu_chunk_pool.num_layers
        self.cpu_chunk_pool.order_behind_writes(chunk_handle, but=self.engine)
        self.engine.swap_in(pool, chunk_handle.rows()[:rows], ids)
        self.engine.fence_pages()   # attention on the current stream must see the pages
        isswap = torch.zeros((self.page_table_allocator.max_context_len,), dtype=torch.bool)
        isswap[:n] = ids >= pool.num_pages_main
        return VirtualPagedKVCache(page_table=table, isswap=isswap, pool=pool)

    def synchronize(self) -> None:
        enqueued = self._progress.enqueued
        self.engine.wait()
        self._progress.finished = enqueued
