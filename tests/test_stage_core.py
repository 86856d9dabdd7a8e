"""A stage whose core, wrapper or pool has a replaced method - on the object or on its class, as a profiler or tracer
replaces it - calls it for every layer instead of taking all layers in one call (on the CPU: the calls are recorded)."""
import pytest
import torch

from deserve_amd.kvcache.paged.page_pool import PagePool
from deserve_amd.model.context.flash import FlashDecodeCtx
from deserve_amd.model.layer.attention import PagedAttentionCore
from deserve_amd.paged_ops import BatchDecodeWithPagedKVCacheWrapper
from deserve_amd.stage import KVStage, StageArgs

L, B = 3, 2


@pytest.fixture
def step(monkeypatch):
    """(stage, inputs, context, record of what ran): the attention itself is a stand-in."""
    record = []
    pool = PagePool(L, 4, 16, torch.device("cpu"), torch.bfloat16, 2, 128)
    ctx = object.__new__(FlashDecodeCtx)
    ctx.layer_id, ctx.page_pool, ctx.bsz, ctx.offsets = 0, pool, B, None
    ctx.decode_wrapper = BatchDecodeWithPagedKVCacheWrapper(torch.empty(16, dtype=torch.uint8))
    ctx.decode_wrapper.fused_append_supported = lambda dtype: True
    ctx.decode_wrapper.forward_layers = lambda *a: record.append("all layers") or True
    stage = KVStage(StageArgs(n_heads=4, n_kv_heads=2, dim=512, n_layers=L), use_rope=False)
    xs = tuple(torch.zeros(L, B, h, 128, dtype=torch.bfloat16) for h in (4, 2, 2))
    return stage, xs, ctx, record


def test_a_plain_stage_takes_all_layers_in_one_call(step):
    stage, xs, ctx, record = step
    stage.forward(xs, ctx)
    assert record == ["all layers"] and ctx.layer_id == L


@pytest.mark.parametrize("where", ["core class", "inner class", "core object", "wrapper class", "wrapper object",
                                   "pool class", "pool object"])
def test_a_replaced_method_is_called_for_every_layer(step, where, monkeypatch):
    stage, xs, ctx, record = step
    forward = lambda *a, **kw: record.append("layer") or kw["out"]
    core = lambda *a, **kw: record.append("layer")
    if where == "core class":
        monkeypatch.setattr(PagedAttentionCore, "paged_forward", core)
    elif where == "inner class":
        monkeypatch.setattr(PagedAttentionCore, "_paged_forward", core)
    elif where == "core object":
        stage.core._paged_forward = core
    elif where == "wrapper class":
        monkeypatch.setattr(BatchDecodeWithPagedKVCacheWrapper, "forward", forward)
    elif where == "wrapper object":
        ctx.decode_wrapper.forward = forward
    else:
        def pages(*a):
            record.append("layer")
            raise InterruptedError      # the wrapper itself is not planned

        if where == "pool class":
            monkeypatch.setattr(PagePool, "get_layered_pages", pages)
        else:
            ctx.page_pool.get_layered_pages = pages
        with pytest.raises(InterruptedError):
            stage.forward(xs, ctx)
        assert record == ["layer"]
        return
    stage.forward(xs, ctx)
    assert record == ["layer"] * L and ctx.layer_id == L
