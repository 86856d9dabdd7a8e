"""The prefill launch whose tiles append the step's rows themselves, against the same step with the append as a
launch of its own: the same bits in pages and result.  Edges: the first new row at the ends of 32-token
blocks and of the four blocks between two waits, parts, one and two rounds of tokens per wave, empty shares, 63
requests, groups and head counts that leave waves idle, pages of 4 tokens; and what keeps the launch in front:
new rows within a walk's first twelve blocks, pages of 2 tokens, too many tokens, 64 requests, decode rows
beside, a pool that is not at a multiple of 256 bytes, a captured stream.  Tiles that find no flag raised -
every other plan entry does not look - append for themselves and walk again, beside tiles that wait."""
import ctypes
import math

import numpy as np
import pytest
import torch

from deserve_amd import _lib
from kvutil import make_scenario, to_torch

pytestmark = pytest.mark.gpu

AUTO, SHARED = _lib.ROUTE_AUTO, _lib.ROUTE_SHARED_LAUNCH
def _over(prior, new):   # (kv_lens, qo_lens)
    return [p + n for p, n in zip(prior, new)], list(new)


CASES = {   # kv_lens, qo_lens, page, Hq, Hkv, dtype, route, whether the tiles append
    "block_edges": (*_over([384, 385, 415, 416, 447, 480, 511], [5, 33, 1, 70, 2, 31, 3]), 16, 32, 8, "bf16", AUTO, True),
    "page4": (*_over([400, 390], [50, 9]), 4, 16, 4, "f16", AUTO, True),
    "too_near": (*_over([383, 500], [30, 20]), 16, 32, 8, "bf16", AUTO, False),
    "prompts": ([17, 203, 1], [17, 203, 1], 4, 32, 8, "f16", AUTO, False),
    "short_prompts": ([17, 30, 9], [17, 30, 9], 4, 32, 8, "f16", AUTO, False),
    "chunk": (*_over([4096], [512]), 16, 32, 8, "bf16", AUTO, True),
    "two_rounds": (*_over([3000], [901]), 8, 32, 8, "bf16", AUTO, True),
    "parts": (*_over([1700, 2360], [60, 40]), 16, 32, 8, "bf16", AUTO, True),
    "part_of_new_rows_only": (*_over([1100], [600]), 8, 32, 8, "bf16", AUTO, False),
    "many_tokens": (*_over([2300, 400], [2211, 70]), 16, 8, 2, "bf16", AUTO, False),
    "kv17": (*_over([400, 450], [20, 3]), 16, 17, 17, "f16", AUTO, True),
    "one_kv_head_group7": (*_over([400, 450], [40, 9]), 32, 7, 1, "bf16", AUTO, True),
    "63_requests": (*_over([400 + 3 * i for i in range(63)], [2] * 62 + [9]), 8, 32, 8, "bf16", AUTO, True),
    "64_requests": (*_over([400 + i for i in range(64)], [2] * 63 + [20]), 16, 32, 8, "bf16", AUTO, False),
    "no_rows_between": (*_over([700, 40, 400, 390], [30, 0, 9, 50]), 16, 32, 8, "bf16", AUTO, True),
    "shared": (*_over([600, 0, 32, 249, 400], [130, 1, 1, 1, 30]), 16, 64, 8, "bf16", SHARED, False),
    "page2": (*_over([500, 400], [33, 2]), 2, 40, 2, "f16", AUTO, False),
}


def _setup(case):
    from deserve_amd.paged_ops import BatchPrefillWithPagedKVCacheWrapper, rope_table

    kv, qo, P, Hq, Hkv, dtype, route, _ = CASES[case]
    sc = make_scenario(63, kv_lens=kv, qo_lens=qo, P=P, Hq=Hq, Hkv=Hkv, D=128, dtype=dtype)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a, np.int32)).cuda()
    indptr = dev(sc.qo_indptr)
    w = BatchPrefillWithPagedKVCacheWrapper(torch.empty(64 << 20, dtype=torch.uint8, device="cuda"))
    w.begin_forward(indptr, dev(sc.kv_page_indptr), dev(sc.kv_page_indices), dev(sc.kv_last_page_lens), Hq, Hkv, 128, P,
                    route_one_row_requests=route)
    q, k, v = (to_torch(a, dtype) for a in (sc.q, sc.k, sc.v))
    table = rope_table(indptr, dev(sc.kv_lens - sc.qo_lens), q.shape[0], 128, 5e5)
    return w, q, k, v, to_torch(sc.pages, dtype), table


def _call(w, q, k, v, pages, table, flags, polls):
    step = _lib.MixedStep.from_buffer_copy(w._step)
    step.rope_table = None if table is None else table.data_ptr()
    step.num_pages, step.causal, step.dtype, step.sm_scale = pages.shape[0], 1, _lib.dtype_code(q.dtype), 1 / math.sqrt(128)
    out = torch.full_like(q, float("nan"))
    if flags is None:
        _lib.check(_lib.lib().dskv_mixed_step(ctypes.byref(step), out.data_ptr(), q.data_ptr(), k.data_ptr(), v.data_ptr(),
                                              pages.data_ptr(), _lib.current_stream()), "step")
        return out
    _lib.check(_lib.lib().dskv_mixed_layers_flagged(
        ctypes.byref(step), flags.data_ptr(), flags.numel(), polls, 1, out.data_ptr(), q.data_ptr(), k.data_ptr(), v.data_ptr(), pages.data_ptr(), 0, _lib.current_stream()), "step")
    return out


def _bits(t):
    return t.view(torch.int16)


def _numbers(w):
    return w._flags.view(torch.int64).tolist()


@pytest.mark.parametrize("case", CASES)
def test_same_bits_as_an_append_in_front(case):
    print("[case] append rows", case, *CASES[case], flush=True)
    w, q, k, v, fresh, table = _setup(case)
    for tab in (table, None):
        want_pages = fresh.clone()
        want = _call(w, q, k, v, want_pages, tab, None, 0)
        assert bool(torch.isfinite(want.float()).all())
        for polls in (0, 0, 1, 1, 0):      # the flags of the call before are there, too
            pages = fresh.clone()
            got = _call(w, q, k, v, pages, tab, w._flags, polls)
            torch.cuda.synchronize()
            assert torch.equal(_bits(pages), _bits(want_pages)) and torch.equal(_bits(got), _bits(want)), polls
    assert bool(w._flags.any()) == CASES[case][-1]


def test_flags_are_64_bit_numbers_of_launches():
    """They do not come round: each launch's is the one before's plus one, in words of its own."""
    print("[case] append rows, numbers of launches", flush=True)
    w, q, k, v, fresh, table = _setup("block_edges")
    seen = []
    for _ in range(3):
        _call(w, q, k, v, fresh, table, w._flags, 0)
        raised = {n for n in _numbers(w)[:-1] if n}
        assert len(raised) == 1
        seen.append(raised.pop())
    assert seen == [seen[0], seen[0] + 1, seen[0] + 2] and 0 < seen[0] < 1 << 32
    odd = torch.zeros(w._flags.numel() + 1, dtype=torch.int32, device="cuda")[1:]
    _call(w, q, k, v, fresh, table, odd, 0)
    _call(w, q, k, v, fresh, table, odd[1:], 0)      # too few
    assert not bool(odd.any())


@pytest.mark.parametrize("case", [c for c in CASES if CASES[c][-1]])
def test_tiles_that_do_not_look_beside_tiles_that_wait(case):
    """The last number of the flags counts the second walks: one for each workgroup of an odd plan entry that
    meets new rows, none for the others."""
    print("[case] append rows, odd entries late", case, *CASES[case], flush=True)
    w, q, k, v, fresh, table = _setup(case)
    kv, qo, _, _, Hkv = CASES[case][:5]
    entries = w._tiles.cpu().numpy()[: 6 * w._n_tiles].reshape(-1, 6)
    meet = np.array([32 * int(e[3]) > kv[e[0]] - qo[e[0]] for e in entries])   # (whole walks end far beyond)
    want_pages = fresh.clone()
    want = _call(w, q, k, v, want_pages, table, None, 0)
    for polls in (_lib.APPEND_ODD_LATE, _lib.APPEND_ODD_LATE, _lib.APPEND_ODD_LATE | 1):
        pages, before = fresh.clone(), _numbers(w)[-1]
        got = _call(w, q, k, v, pages, table, w._flags, polls)
        torch.cuda.synchronize()
        assert torch.equal(_bits(pages), _bits(want_pages)) and torch.equal(_bits(got), _bits(want)), polls
        walks = _numbers(w)[-1] - before
        assert walks >= Hkv * int(meet[1::2].sum())
        if polls == _lib.APPEND_ODD_LATE:
            assert walks == Hkv * int(meet[1::2].sum())
    assert meet[1::2].any()


@pytest.mark.parametrize("case", ["too_near", "short_prompts", "part_of_new_rows_only"])
def test_walks_that_begin_with_new_rows_although_the_plan_says_late(case):
    """The lengths that count are the device's: such a walk leaves its share and appends for itself."""
    print("[case] append rows, not late", case, *CASES[case], flush=True)
    w, q, k, v, fresh, table = _setup(case)
    want_pages = fresh.clone()
    want = _call(w, q, k, v, want_pages, table, None, 0)
    assert not w._info.new_rows_late
    w._info.new_rows_late = 1
    pages = fresh.clone()
    got = _call(w, q, k, v, pages, table, w._flags, 0)
    torch.cuda.synchronize()
    assert torch.equal(_bits(pages), _bits(want_pages)) and torch.equal(_bits(got), _bits(want))
    # eight blocks are requested before the first look: 383 tokens of context are more
    assert bool(_numbers(w)[-1]) == (case != "too_near")


def test_one_sequence_handed_in_as_two_requests():
    """The second request attends to rows that the first one appends."""
    from deserve_amd.paged_ops import BatchPrefillWithPagedKVCacheWrapper

    print("[case] append rows, one sequence as two requests", flush=True)
    g = torch.Generator(device="cuda").manual_seed(3)
    rand = lambda *s: torch.randn(*s, generator=g, device="cuda").bfloat16()
    dev = lambda a: torch.tensor(a, dtype=torch.int32, device="cuda")
    table = torch.randperm(60, generator=g, device="cuda").int()
    w = BatchPrefillWithPagedKVCacheWrapper(torch.empty(64 << 20, dtype=torch.uint8, device="cuda"))
    w.begin_forward(dev([0, 60, 100]), dev([0, 48, 98]), torch.cat([table[:48], table[:50]]), dev([8, 16]), 32, 8, 128, 16)
    q, k, v, fresh = rand(100, 32, 128), rand(100, 8, 128), rand(100, 8, 128), rand(60, 2, 16, 8, 128)
    want_pages, pages = fresh.clone(), fresh.clone()
    want = _call(w, q, k, v, want_pages, None, None, 0)
    got = w.forward(q, pages, k_append=k, v_append=v)
    torch.cuda.synchronize()
    assert not bool(w._flags.any())
    assert torch.equal(_bits(pages), _bits(want_pages)) and torch.equal(_bits(got), _bits(want))
    one = BatchPrefillWithPagedKVCacheWrapper(torch.empty(64 << 20, dtype=torch.uint8, device="cuda"))
    one.begin_forward(dev([0, 100]), dev([0, 50]), table[:50], dev([16]), 32, 8, 128, 16)
    whole = one.forward(q, fresh.clone(), k_append=k, v_append=v)
    # the same sums in another order: two roundings to bf16 of values below 1
    assert float((whole.float() - got.float()).abs().max()) <= 2 * 2.0 ** -8


@pytest.mark.parametrize("where", ["k", "v", "workspace"])
def test_a_result_or_partials_that_lie_where_the_new_rows_do(where):
    """The new rows have been read before they are overwritten."""
    print("[case] append rows, overlapping", where, flush=True)
    w, q, k, v, fresh, table = _setup("kv17")
    want_pages, pages = fresh.clone(), fresh.clone()
    want = _call(w, q, k, v, want_pages, table, None, 0)
    if where == "workspace":
        v = w._workspace[: v.numel() * 2].view(v.dtype).view(v.shape).copy_(v)
    got = w.forward(q, pages, out={"k": k, "v": v}.get(where), k_append=k, v_append=v, rope_table=table)
    torch.cuda.synchronize()
    assert not bool(w._flags.any())
    assert torch.equal(_bits(pages), _bits(want_pages)) and torch.equal(_bits(got), _bits(want))


def test_a_pool_between_cache_lines_and_a_captured_stream():
    print("[case] append rows, odd pool and capture", flush=True)
    w, q, k, v, fresh, table = _setup("block_edges")
    want_pages = fresh.clone()
    want = _call(w, q, k, v, want_pages, table, None, 0)
    odd = torch.empty(fresh.numel() + 8, dtype=fresh.dtype, device="cuda")[8:].view(fresh.shape)
    odd.copy_(fresh)
    got = _call(w, q, k, v, odd, table, w._flags, 0)
    assert torch.equal(_bits(odd), _bits(want_pages)) and torch.equal(_bits(got), _bits(want))
    pages = fresh.clone()
    graph, side = torch.cuda.CUDAGraph(), torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.graph(graph, stream=side):
        got = _call(w, q, k, v, pages, table, w._flags, 0)
    for _ in range(3):
        pages.copy_(fresh)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(_bits(pages), _bits(want_pages)) and torch.equal(_bits(got), _bits(want))
