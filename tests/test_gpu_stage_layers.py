"""A stage whose layers run in one call to the library, against the same layers called one by one (chunks with
their append as a launch in front): the same bits in the result and the pages, the same layer count.  What is
not a plain stack goes layer by layer, fp32 layers too, and a pool with too few layers is refused as it is there.
"""
import ctypes

import pytest
import torch

from deserve_amd import _lib
from deserve_amd.execution.exec import BatchDecode, BatchPrefill
from deserve_amd.stage import KVStage
from deserve_amd.synthetic import make_mixed_workload

pytestmark = pytest.mark.gpu

SHAPES = {
    "one_request": ([70], [], []),
    "decode": ([33, 600, 1, 16], [], []),
    "prompts": ([], [0, 40], [17, 5]),
    "chunks": ([], [500, 430], [30, 20]),      # whose launches append the rows themselves
    "shared_launch": ([30 + 40 * i for i in range(14)], [20], [12]),
}


def _run(shape, dtype, rope, together, q_of=lambda q: q, first=0, out_layers=3):
    """(result, pages, layer id, what layers_forward answered, whether flags were raised)."""
    wl = make_mixed_workload("t", *SHAPES[shape], 3, 16, 4, 128, 8, dtype, seed=5)
    stage = KVStage(wl.args, use_rope=rope)
    answers, layers_forward = [], stage.core.layers_forward

    def asked(*a):
        answers.append(layers_forward(*a) if together else False)
        return answers[-1]

    stage.core.layers_forward = asked
    kind = BatchPrefill if SHAPES[shape][2] else BatchDecode
    batch = kind(None, stage, wl.tasks, wl.caches)
    batch.prepare()
    ctx = batch.prefill_ctx if SHAPES[shape][2] else batch.decode_ctx
    flags = None
    if SHAPES[shape][2]:
        assert bool(ctx.prefill_wrapper._info.new_rows_late) == (shape == "chunks")
        flags = torch.zeros(_lib.lib().dskv_append_flags(), dtype=torch.int32, device="cuda") if together else None
        ctx.prefill_wrapper._flags = flags      # none: the append is a launch in front
    ctx.layer_id = first
    out = stage.forward((q_of(wl.q)[:out_layers], wl.k[:out_layers], wl.v[:out_layers]), ctx)
    torch.cuda.synchronize()
    return out, wl.pool.pages, ctx.layer_id, answers, flags is not None and bool(flags.any())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("rope", [False, True])
@pytest.mark.parametrize("shape", SHAPES)
def test_layers_in_one_call_match_layers_one_by_one(shape, rope, dtype):
    print("[case] stage layers", shape, rope, dtype, flush=True)
    for kw in ({}, {"first": 1, "out_layers": 2}):
        got, want = _run(shape, dtype, rope, True, **kw), _run(shape, dtype, rope, False, **kw)
        assert got[2] == want[2] == 3
        assert got[3] == [dtype is not torch.float32]
        assert got[4] == (shape == "chunks" and dtype is not torch.float32)
        for a, b in zip(got[:2], want[:2]):
            assert torch.equal(a.view(torch.uint8), b.view(torch.uint8))


def test_stacks_that_are_not_plain_go_layer_by_layer():
    print("[case] stage layers, strided q", flush=True)
    strided = lambda q: q.transpose(0, 1).contiguous().transpose(0, 1)
    flat = lambda q: q.reshape(q.shape[0], q.shape[1], -1)
    want = _run("decode", torch.bfloat16, True, False)
    for q_of in (strided, flat):
        got = _run("decode", torch.bfloat16, True, True, q_of)
        assert got[3] == [False]
        assert torch.equal(got[0].view(torch.int16), want[0].view(torch.int16))
        assert torch.equal(got[1].view(torch.int16), want[1].view(torch.int16))


@pytest.mark.parametrize("shape", ["decode", "prompts"])
def test_more_layers_than_the_pool_has_are_refused(shape):
    print("[case] stage layers beyond the pool", shape, flush=True)
    for together in (True, False):
        with pytest.raises(IndexError):
            _run(shape, torch.bfloat16, True, together, first=1)


@pytest.mark.parametrize("entry", ["mixed", "decode_fp32"])
def test_the_librarys_calls_for_layers_match_its_calls_for_one(entry):
    print("[case] stage layers, C entries", entry, flush=True)
    wl = make_mixed_workload("t", *SHAPES["shared_launch" if entry == "mixed" else "decode"], 3, 16, 4, 128, 8,
                             torch.bfloat16 if entry == "mixed" else torch.float32, seed=5)
    batch = (BatchPrefill if entry == "mixed" else BatchDecode)(None, KVStage(wl.args, use_rope=False), wl.tasks, wl.caches)
    batch.prepare()
    lib, pages, stream = _lib.lib(), wl.pool.pages, _lib.current_stream()
    ptrs = lambda *ts: [t.data_ptr() for t in ts]
    if entry == "mixed":
        step = _lib.MixedStep.from_buffer_copy(batch.prefill_ctx.prefill_wrapper._step)
        step.num_pages, step.causal, step.dtype, step.sm_scale = pages.shape[1], 1, _lib.BF16, 0.1
        one, all_layers, rows = lib.dskv_mixed_step, lib.dskv_mixed_layers, lambda l: ptrs(wl.k[l], wl.v[l])
    else:
        step = _lib.DecodeStep.from_buffer_copy(batch.decode_ctx.decode_wrapper._step)
        step.dtype, step.sm_scale = _lib.F32, 0.1
        one, all_layers, rows = lib.dskv_decode_step, lib.dskv_decode_layers, lambda l: [None, None]   # in the pages
    fresh, want, got = pages.clone(), torch.zeros_like(wl.q), torch.zeros_like(wl.q)
    for l in range(3):
        _lib.check(one(ctypes.byref(step), *ptrs(want[l], wl.q[l]), *rows(l), pages[l].data_ptr(), stream), "one")
    want_pages = pages.clone()
    pages.copy_(fresh)
    _lib.check(all_layers(ctypes.byref(step), 3, *ptrs(got, wl.q), *rows(slice(None)), pages.data_ptr(),
                          pages.stride(0) * pages.element_size(), stream), "layers")
    torch.cuda.synchronize()
    assert bool(torch.isfinite(want).all()) and bool(want.any())
    assert torch.equal(got.view(torch.uint8), want.view(torch.uint8))
    assert torch.equal(pages.view(torch.uint8), want_pages.view(torch.uint8))
