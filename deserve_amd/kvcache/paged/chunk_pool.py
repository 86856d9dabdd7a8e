"""Pinned host arena for offloaded requests, carved by a buddy allocator whose
unit is one page of every layer (deserve_worker/kvcache/paged/chunk_pool.py:10-113).
A chunk of level k holds 2**k page-units laid out (L * n, 2, P, Hkv, D), layer
major - the layout KVCacheManager writes."""
from __future__ import annotations

import threading
from dataclasses import dataclass
from typing import List, Protocol, Tuple

import torch

from deserve_amd.kvcache._alloc import BuddyIndex
from deserve_amd.kvcache.pinned.pinned_memory import pinned_empty


@dataclass
class ChunkHandle:
    id: int
    level: int
    initial_size: int
    pool: "ChunkPool"

    def free(self) -> None:
        self.pool.free(self.id, self.level)

    def retrieve(self) -> torch.Tensor:
        """The chunk's rows, for work on the current stream: behind the copies that still write them."""
        self.pool.order_behind_writes(self)
        return self.rows()

    def rows(self) -> torch.Tensor:
        """The same for a caller that orders its accesses itself."""
        begin, end = BuddyIndex.span(self.id, self.level)
        return self.pool.chunks[begin * self.pool.num_layers: end * self.pool.num_layers]


class PendingWrite(Protocol):
    """A copy into a chunk that may still be on its way."""
    engine: object                    # what carries it; its copies keep their order among themselves

    def finished(self) -> bool: ...   # as far as the host knows
    def poll(self) -> bool: ...       # the same, with a look at the device; never waits
    def fence(self) -> None: ...      # orders the current stream behind it


_MANY_WRITES = 64


class ChunkPool:
    def __init__(self, num_layers: int, height: int, page_size: int, main_device: torch.device,
                 main_dtype: torch.dtype, n_kv_heads: int = 8, head_dim: int = 128):
        self.num_layers, self.height, self.page_size = num_layers, height, page_size
        self.main_device, self.main_dtype = torch.device(main_device), main_dtype
        self.mutex = threading.Lock()
        self.per_token_shape = (2, page_size, n_kv_heads, head_dim)
        self.chunks = pinned_empty(((1 << (height - 1)) * num_layers,) + self.per_token_shape,
                                   main_dtype)
        self._buddy = BuddyIndex(height)
        # copies that may still write, by the memory they write (a chunk can be freed and handed out
        # again while they do): first unit, end, copy
        self._writes: List[Tuple[int, int, PendingWrite]] = []

    def note_write(self, handle: ChunkHandle, write: PendingWrite) -> None:
        with self.mutex:
            self._writes = [w for w in self._writes if not w[2].finished()]
            if len(self._writes) >= _MANY_WRITES:     # nobody waits for them on the host
                self._writes = [w for w in self._writes if not w[2].poll()]
            self._writes.append(BuddyIndex.span(handle.id, handle.level) + (write,))

    def order_behind_writes(self, handle: ChunkHandle, but: object = None) -> None:
        """Orders the current stream behind the copies that still write the chunk's memory (not those
        of engine `but`)."""
        if not self._writes:
            return
        begin, end = BuddyIndex.span(handle.id, handle.level)
        with self.mutex:
            writes = [w for lo, hi, w in self._writes if lo < end and begin < hi]
        for w in writes:
            if w.engine is not but and not w.finished():
                w.fence()

    @property
    def available_ids(self) -> list:
        return self._buddy.levels

    def split(self, begin: int, end: int) -> None:
        """Public as in the reference (chunk_pool.py:51-59); like there, the caller holds
        the mutex or owns the pool."""
        self._buddy.split(begin, end)

    def alloc(self, size: int) -> ChunkHandle:
        with self.mutex:
            cid, level = self._buddy.alloc(size)   # RuntimeError when exhausted
        return ChunkHandle(cid, level, size, self)

    def free(self, id: int, level: int) -> None:
        with self.mutex:
            self._buddy.release(id, level)


class CpuChunkPool(ChunkPool):
    def __init__(self, num_layers: int, height: int, page_size: int, main_dtype: torch.dtype,
                 n_kv_heads: int = 8, head_dim: int = 128):
        super().__init__(num_layers, height, page_size, torch.device("cpu"), main_dtype,
                         n_kv_heads, head_dim)
