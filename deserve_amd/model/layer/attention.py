"""The KV part of one attention layer: RoPE -> KV append -> paged attention
(deserve_worker/model/layer/attention.py:160-193).  The q/k/v/o projections
around it are dense GEMMs of the model proper and are not part of this package;
``paged_forward`` takes the projected q, k, v and returns the attention output
in ragged (nnz, Hq * D) form, as the reference's method does before ``wo``."""
from __future__ import annotations

from typing import Optional

import torch

from deserve_amd.kvcache.paged.page_pool import PagePool
from deserve_amd.model.context.flash import FlashDecodeCtx, FlashForwardCtx, FlashPrefillCtx
from deserve_amd.paged_ops import (BatchDecodeWithPagedKVCacheWrapper, BatchPrefillWithPagedKVCacheWrapper,
                                   append_paged_kv_cache, apply_rope, rope_append_paged_kv_cache)


class PagedAttentionCore:
    def __init__(self, n_heads: int, n_kv_heads: int, head_dim: int, rope_theta: float = 500000.0,
                 use_rope: bool = True, fuse_rope_append: bool = True,
                 fuse_decode_append: bool = True) -> None:
        self.n_local_heads, self.n_local_kv_heads = n_heads, n_kv_heads
        self.head_dim, self.dim = head_dim, n_heads * head_dim
        self.rope_theta, self.use_rope = rope_theta, use_rope
        self.fuse_rope_append = fuse_rope_append
        self.fuse_decode_append = fuse_decode_append

    def paged_forward(self, xq: torch.Tensor, xk: torch.Tensor, xv: torch.Tensor,
                      ctx: FlashForwardCtx, out: Optional[torch.Tensor] = None) -> torch.Tensor:
        """out: where the result goes (contiguous, one row of Hq * D per token); None: a tensor of
        its own."""
        if torch.is_inference_mode_enabled():      # entering it again costs every layer 3 us
            return self._paged_forward(xq, xk, xv, ctx, out)
        with torch.inference_mode():
            return self._paged_forward(xq, xk, xv, ctx, out)

    def layers_forward(self, q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, ctx: FlashForwardCtx,
                       out: torch.Tensor) -> bool:
        """paged_forward for the layers ctx.layer_id .. of q, k, v and out, stacked: (L, tokens, heads, head_dim)
        each, launched by one call to the library - layer by layer from here a step of one request costs the
        host 13 us a layer, as long as the GPU works on it.  False, and nothing done, where the layers are not
        plain stacks for the launches that append as they attend (fp32 has none), or a method that a layer
        goes through has been replaced, on an object or its class: it is called for every layer then.
        ctx.layer_id counts on as it would."""
        if q.dtype is torch.float32 or q.dim() != 4 or _core_methods() != _CORE_METHODS or \
                not _CORE_NAMES.isdisjoint(vars(self)):
            return False
        n, first, pool = q.shape[0], ctx.layer_id, ctx.page_pool
        decode = type(ctx) is FlashDecodeCtx
        if not decode and type(ctx) is not FlashPrefillCtx:
            return False
        wrapper = ctx.decode_wrapper if decode else ctx.prefill_wrapper
        kind = BatchDecodeWithPagedKVCacheWrapper if decode else BatchPrefillWithPagedKVCacheWrapper
        if type(wrapper) is not kind or "forward" in vars(wrapper) or kind.forward is not _WRAPPER_FORWARD[kind] or \
                getattr(pool.get_layered_pages, "__func__", None) is not _LAYERED_PAGES or \
                not 0 <= first <= pool.pages.shape[0] - n:
            return False
        pages = pool.pages[first: first + n]
        with torch.inference_mode():
            if decode:
                taken = self.fuse_decode_append and k.shape[1] == ctx.bsz and wrapper.forward_layers(
                    q, pages, out, k, v, ctx.offsets if self.use_rope else None, self.rope_theta)
            else:
                if self.use_rope and not self.fuse_rope_append or not wrapper.fused_append_supported(q.dtype):
                    return False
                table = ctx.rope_table(q.shape[1], self.head_dim, self.rope_theta) if self.use_rope else None
                taken = wrapper.forward_layers(q, pages, out, k, v, table)
                if taken and table is not None:
                    ctx.rope_layer = first + n - 1     # the layer that would have asked for it last
        if taken:
            ctx.layer_id = first + n
        return taken

    def _rows(self, x: torch.Tensor, heads: int) -> torch.Tensor:
        """x as (tokens, heads, head_dim)."""
        s = x.shape
        return x if len(s) == 3 and s[1] == heads and s[2] == self.head_dim else x.view(-1, heads, self.head_dim)

    def _paged_forward(self, xq: torch.Tensor, xk: torch.Tensor, xv: torch.Tensor,
                       ctx: FlashForwardCtx, out: Optional[torch.Tensor]) -> torch.Tensor:
        if out is not None:
            out = self._rows(out, self.n_local_heads)
        xq = self._rows(xq, self.n_local_heads)
        xk = self._rows(xk, self.n_local_kv_heads)
        xv = self._rows(xv, self.n_local_kv_heads)
        pages = ctx.page_pool.get_layered_pages(ctx.layer_id)
        if (isinstance(ctx, FlashDecodeCtx) and self.fuse_decode_append and xk.shape[0] == ctx.bsz
                and ctx.decode_wrapper.fused_append_supported(xq.dtype)):
            # a decode step: the attention launch rotates q and the new k and writes the new
            # token into its page slot itself
            rope = dict(rope_offsets=ctx.offsets, rope_theta=self.rope_theta) if self.use_rope else {}
            out = ctx.decode_wrapper.forward(xq, pages, k_append=xk, v_append=xv, out=out, **rope)
            return out.view(-1, self.dim)
        if (isinstance(ctx, FlashPrefillCtx) and (self.fuse_rope_append or not self.use_rope)
                and ctx.prefill_wrapper.fused_append_supported(xq.dtype)):
            # k is rotated on its way into its slots, q as the attention loads it
            table = ctx.rope_table(xq.shape[0], self.head_dim, self.rope_theta) if self.use_rope else None
            out = ctx.prefill_wrapper.forward(xq, pages, causal=True, out=out, k_append=xk, v_append=xv,
                                              rope_table=table)
            return out.view(-1, self.dim)
        if self.use_rope and self.fuse_rope_append:
            # one kernel: rotated q comes back, rotated k and v go straight into their slots
            xq = rope_append_paged_kv_cache(xq, xk, xv, ctx.indptr, ctx.offsets, pages,
                                            ctx.kv_page_indices, ctx.kv_page_indptr,
                                            ctx.kv_last_page_lens, rope_theta=self.rope_theta)
        else:
            if self.use_rope:
                xq, xk = apply_rope(xq, xk, ctx.indptr, ctx.offsets, interleave=True,
                                    rope_theta=self.rope_theta)
            append_paged_kv_cache(xk, xv, ctx.indptr, pages, ctx.kv_page_indices,
                                  ctx.kv_page_indptr, ctx.kv_last_page_lens)
        if isinstance(ctx, FlashDecodeCtx):
            out = ctx.decode_wrapper.forward(xq, pages, out=out)
        elif isinstance(ctx, FlashPrefillCtx):
            out = ctx.prefill_wrapper.forward(xq, pages, causal=True, out=out)
        else:
            raise TypeError(f"unsupported forward context {type(ctx).__name__}")
        return out.view(-1, self.dim)


def _core_methods() -> tuple:
    """What paged_forward goes through."""
    return PagedAttentionCore.paged_forward, PagedAttentionCore._paged_forward, PagedAttentionCore._rows


# as they are here: see layers_forward
_CORE_NAMES = {"paged_forward", "_paged_forward", "_rows"}
_CORE_METHODS = _core_methods()
_WRAPPER_FORWARD = {kind: kind.forward for kind in (BatchDecodeWithPagedKVCacheWrapper, BatchPrefillWithPagedKVCacheWrapper)}
_LAYERED_PAGES = PagePool.get_layered_pages
