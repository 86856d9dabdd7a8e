"""The prefill / mixed step that rotates K on its way into the pages and q as the attention loads
it, against apply_rope + append + attention in separate calls: the same bits.  Edges: one token,
rows at the ends of tiles, tiles in parts, decode rows beside chunks in every layout, 63 and 64
requests (two ways to find a token's request), groups that do not divide a tile, pages from 2 tokens
to 32, KV rows of one head and of 17."""
import numpy as np
import pytest
import torch

from deserve_amd import _lib
from kvutil import make_scenario, to_torch

pytestmark = pytest.mark.gpu

AUTO, SHARED, TWO = _lib.ROUTE_AUTO, _lib.ROUTE_SHARED_LAUNCH, _lib.ROUTE_TWO_LAUNCHES
CASES = [
    # (name, kv_lens, qo_lens, P, Hq, Hkv, dtype, route)
    ("one_token", [1], [1], 16, 32, 8, "bf16", AUTO),
    ("short_prompts", [17, 203, 64], [17, 203, 64], 16, 32, 8, "bf16", AUTO),
    ("chunk_in_parts", [2100], [129], 16, 32, 8, "f16", AUTO),
    ("group3_page8", [300, 41], [65, 40], 8, 12, 4, "bf16", AUTO),
    ("group20_page2", [150, 9], [33, 2], 2, 40, 2, "f16", AUTO),
    ("one_kv_head_page32", [90, 33], [90, 1], 32, 8, 1, "bf16", AUTO),
    ("kv17", [50, 20], [50, 3], 16, 17, 17, "bf16", AUTO),
    ("shared_launch", [700, 1, 33, 250, 64], [130, 1, 1, 1, 30], 16, 64, 8, "bf16", SHARED),
    ("two_launches_page4", [700, 1, 33, 250], [130, 1, 1, 1], 4, 32, 8, "f16", TWO),
    ("63_requests", [20 + i for i in range(63)], [1] * 62 + [9], 8, 32, 8, "bf16", AUTO),
    ("64_requests", [20 + i for i in range(64)], [2] * 63 + [20], 16, 32, 8, "bf16", AUTO),
]


@pytest.mark.parametrize("case", CASES, ids=[c[0] for c in CASES])
def test_fused_rotation_matches_separate_calls(case):
    from deserve_amd.paged_ops import (BatchPrefillWithPagedKVCacheWrapper, append_paged_kv_cache, apply_rope,
                                       rope_table)

    name, kv, qo, P, Hq, Hkv, dtype, route = case
    print("[case] fused prefill", *case, flush=True)
    sc = make_scenario(62, kv_lens=kv, qo_lens=qo, P=P, Hq=Hq, Hkv=Hkv, D=128, dtype=dtype)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a, np.int32)).cuda()
    indptr, tab, tabptr, last = (dev(a) for a in (sc.qo_indptr, sc.kv_page_indices, sc.kv_page_indptr,
                                                  sc.kv_last_page_lens))
    offsets = dev(sc.kv_lens - sc.qo_lens)
    w = BatchPrefillWithPagedKVCacheWrapper(torch.empty(64 << 20, dtype=torch.uint8, device="cuda"))
    w.begin_forward(indptr, tabptr, tab, last, Hq, Hkv, 128, P, route_one_row_requests=route)
    q, k, v = (to_torch(a, dtype) for a in (sc.q, sc.k, sc.v))
    assert w.fused_append_supported(q.dtype) and not w.fused_append_supported(torch.float32)
    bits = lambda t: t.view(torch.int16)
    for rope in (True, False):
        pages, want_pages = to_torch(sc.pages, dtype), to_torch(sc.pages, dtype)
        qr, kr = apply_rope(q, k, indptr, offsets, interleave=True, rope_theta=5e5) if rope else (q, k)
        append_paged_kv_cache(kr, v, indptr, want_pages, tab, tabptr, last)
        want = w.forward(qr, want_pages, out=torch.full_like(q, float("nan")))
        table = rope_table(indptr, offsets, q.shape[0], 128, 5e5) if rope else None
        got = w.forward(q, pages, out=torch.full_like(q, float("nan")), k_append=k, v_append=v, rope_table=table)
        torch.cuda.synchronize()
        assert torch.equal(bits(pages), bits(want_pages))
        assert bool(torch.isfinite(got.float()).all()) and torch.equal(bits(got), bits(want))


def test_a_second_pass_over_the_layers_rotates_by_the_offsets_it_finds():
    """A context whose offsets are rewritten in place between two passes."""
    from deserve_amd.model.context.flash import FlashPrefillCtx
    from deserve_amd.paged_ops import rope_table

    print("[case] offsets rewritten between passes", flush=True)
    dev = lambda a: torch.tensor(a, dtype=torch.int32, device="cuda")
    ctx = FlashPrefillCtx(bsz=2, seqlens=dev([3, 4]), layer_id=0, page_pool=None, offsets=dev([0, 9]),
                          indptr=dev([0, 3, 7]), kv_page_indices=None, kv_page_indptr=None,
                          kv_last_page_lens=None, host={}, prefill_wrapper=None)
    first = ctx.rope_table(7, 128, 1e4)
    ctx.layer_id = 1
    assert ctx.rope_table(7, 128, 1e4) is first
    ctx.offsets.copy_(dev([5, 20]))
    ctx.layer_id = 0
    got = ctx.rope_table(7, 128, 1e4)
    assert torch.equal(got, rope_table(ctx.indptr, ctx.offsets, 7, 128, 1e4))
    assert not torch.equal(got, first)


def test_layers_on_another_stream_or_under_capture_have_a_table_of_their_own():
    """Layer 0 runs eagerly on the current stream.  A later layer on a side stream is not ordered behind
    it, and one that is captured has to find the offsets of the replay."""
    from deserve_amd.model.context.flash import FlashPrefillCtx
    from deserve_amd.paged_ops import rope_table

    print("[case] table per stream and capture", flush=True)
    dev = lambda a: torch.tensor(a, dtype=torch.int32, device="cuda")
    ctx = FlashPrefillCtx(bsz=2, seqlens=dev([3, 4]), layer_id=0, page_pool=None, offsets=dev([0, 9]),
                          indptr=dev([0, 3, 7]), kv_page_indices=None, kv_page_indptr=None,
                          kv_last_page_lens=None, host={}, prefill_wrapper=None)
    first = ctx.rope_table(7, 128, 1e4)
    torch.cuda.synchronize()
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        ctx.layer_id = 1
        other = ctx.rope_table(7, 128, 1e4)
    torch.cuda.synchronize()
    assert other is not first and torch.equal(other, first)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        ctx.layer_id = 2
        seen = ctx.rope_table(7, 128, 1e4).clone()
        ctx.layer_id = 3
        again = ctx.rope_table(7, 128, 1e4).clone()
    for offsets in ([5, 20], [0, 9], [700, 3]):
        ctx.offsets.copy_(dev(offsets))
        graph.replay()
        torch.cuda.synchronize()
        want = rope_table(ctx.indptr, ctx.offsets, 7, 128, 1e4)
        assert torch.equal(seen, want) and torch.equal(again, want)
    ctx.layer_id = 4
    assert ctx.rope_table(7, 128, 1e4) is first
