"""How many launches a scheduler that replays its decode steps has to capture: requests that grow by a token a step, end and are
replaced; and the plans that are filled up for it, against the ones that are not (256 compute units are assumed where there
is no GPU)."""
import ctypes

import numpy as np
import pytest
import torch

from deserve_amd import _lib
from deserve_amd.execution.graph import GraphedDecodeStep
from deserve_amd.paged_ops import BatchDecodeWithPagedKVCacheWrapper

PAGE, WORDS = 16, 1 << 17


class _Buffers:
    """A StagedUpload in host memory."""

    def __init__(self):
        self.dev, self.words = torch.zeros(WORDS, dtype=torch.int32), 0

    def staging(self):
        return self.dev

    def upload(self, words):
        self.words = words


def _plan(w, lens, n_kv, group=4, buffers=None, **more):
    n = -(-np.asarray(lens) // PAGE)
    indptr = torch.from_numpy(np.concatenate([[0], np.cumsum(n)]).astype(np.int32))
    last = torch.tensor([(x - 1) % PAGE + 1 for x in lens], dtype=torch.int32)
    buffers = buffers or _Buffers()
    w.begin_forward(indptr, torch.zeros(int(n.sum()), dtype=torch.int32), last, group * n_kv, n_kv, 128, PAGE,
                    plan_buffers=buffers, **more)
    return buffers


def _wrapper():
    return BatchDecodeWithPagedKVCacheWrapper(torch.empty(64 << 20, dtype=torch.uint8))


# (requests, shortest, longest, kv heads, captures): one for whole requests, one where some are cut, one of the other form
CASES = [(24, 20, 200, 8, 2), (20, 100, 300, 8, 2), (8, 50, 500, 8, 2), (32, 16, 400, 8, 2), (32, 64, 1024, 8, 3),
         (4, 64, 2000, 8, 2), (1, 1, 3000, 8, 3), (16, 16, 400, 16, 2), (24, 16, 400, 4, 2), (9, 30, 900, 12, 2)]


@pytest.mark.parametrize("batch,lo,hi,n_kv,most", CASES)
@pytest.mark.parametrize("turnover", [True, False])
def test_batches_that_grow_and_turn_over_need_few_captures(batch, lo, hi, n_kv, most, turnover):
    rng = np.random.default_rng(batch)
    w, buffers, keys = _wrapper(), _Buffers(), set()
    lens = rng.integers(lo, hi + 1, batch)
    for _ in range(600):
        lens = lens + 1
        if turnover:
            ended = rng.random(batch) < 0.02
            lens = np.where(ended, rng.integers(lo, hi + 1, batch), lens)
        lens = np.where(lens > hi, lo, lens)
        _plan(w, lens, n_kv, buffers=buffers)
        keys.add(GraphedDecodeStep.graph_key(batch, w._n_workgroups, w._n_items, [w._plan], True))
    assert len(keys) <= most, sorted((k[1:4]) for k in keys)


@pytest.mark.parametrize("lens", [[1], [60] * 4, [1777], [300, 20, 900], [5] * 70])
@pytest.mark.parametrize("n_kv,group", [(8, 4), (8, 8), (3, 2), (16, 1), (40, 1), (8, 9)])
def test_a_filled_plan_is_the_plan_with_empty_shares_behind(lens, n_kv, group):
    filled, plain = _wrapper(), _wrapper()
    a, b = _plan(filled, lens, n_kv, group), _Buffers()
    plain._fill_up = lambda plan, cap, words: words
    _plan(plain, lens, n_kv, group, b)
    x, y = a.dev[:a.words].numpy(), b.dev[:b.words].numpy()
    n, m, items = plain._n_workgroups, filled._n_workgroups, plain._n_items
    flag = ctypes.c_int32()
    _lib.lib().dskv_decode_launch(items, n, group * n_kv, n_kv, 128, _lib.BF16, ctypes.byref(flag))
    assert m == (max(n, 256 // n_kv) if flag.value else n) and filled._n_items == items and len(x) - len(y) == m - n
    _lib.lib().dskv_decode_launch(items, m, group * n_kv, n_kv, 128, _lib.BF16, ctypes.byref(flag2 := ctypes.c_int32()))
    assert flag2.value == flag.value                       # the same form
    assert x[1] == m and np.array_equal(np.delete(x[:4], 1), np.delete(y[:4], 1))
    assert np.array_equal(x[4: 5 + n], y[4: 5 + n]) and (x[5 + n: 5 + m] == items).all()
    assert np.array_equal(x[5 + m:], y[5 + n:])


def test_plans_that_are_not_filled_up():
    """A caller's own number of workgroups; 32 bits; an empty batch; too little room; what is no plan."""
    lib, w = _lib.lib(), _wrapper()
    for more, n in (({"target_workgroups": 5}, 5), ({}, 32)):
        _plan(w, [700] * 3, 8, **more)
        assert w._n_workgroups == n
    plain = _wrapper()
    plain._fill_up = lambda plan, cap, words: words
    for one in (w, plain):
        _plan(one, [100] * 3, 8, data_type=torch.float32)
    assert w._n_workgroups == plain._n_workgroups

    def fill(words, n_wgs, cap, heads=(32, 8), plan=None):
        plan = np.zeros(4096, np.int32) if plan is None else plan
        n, size = ctypes.c_int32(n_wgs), ctypes.c_int64(words)
        return lib.dskv_decode_plan_fill(plan.ctypes.data, cap, *heads, 128, _lib.BF16, ctypes.byref(n),
                                         ctypes.byref(size)), n.value, size.value

    assert fill(0, 0, 4096) == (0, 0, 0)
    b = _Buffers()
    _plan(plain, [60] * 4, 8, buffers=b)
    plan, n, words = b.dev.numpy()[:4096].copy(), plain._n_workgroups, b.words
    kept = plan.copy()
    assert fill(words, n, words + 31 - n, plan=plan) == (-2, n, words) and np.array_equal(plan, kept)
    assert fill(words, n + 1, 4096, plan=plan)[0] == -1 and fill(words, n, words - 1, plan=plan)[0] == -1
    assert fill(words, n, 4096, heads=(32, 7), plan=plan)[0] == -1 and np.array_equal(plan, kept)
    assert fill(words, n, words + 32 - n, plan=plan) == (0, 32, words + 32 - n)


@pytest.mark.gpu
def test_replays_of_batches_of_any_lengths_are_the_eager_step():
    """Four requests at a time out of twelve, from one share to 32, captured once for whole requests and once for cut ones."""
    from deserve_amd.execution.exec import get_wrappers
    from deserve_amd.model.context.flash import FlashDecodeCtx
    from deserve_amd.stage import KVStage, StageArgs
    from deserve_amd.synthetic import make_decode_workload

    dev, layers = torch.device("cuda:0"), 2
    lens = [5, 17, 30, 9, 100, 90, 120, 60, 1777, 900, 300, 2500]
    picks = [[0, 1, 2, 3], [4, 5, 6, 7], [8, 9, 10, 11], [0, 1, 2, 4], [8, 1, 2, 3], [4, 5, 6, 7], [10, 7, 4, 1]]
    eager, graphed = (make_decode_workload("k", lens, layers, 32, 8, 128, PAGE, torch.bfloat16, headroom_tokens=32,
                                           seed=4, fill=True) for _ in range(2))
    stage = KVStage(StageArgs(n_heads=32, n_kv_heads=8, dim=32 * 128, page_size=PAGE, n_layers=layers), use_rope=False)
    wrapper, _ = get_wrappers(dev)
    shape = dict(num_qo_heads=32, num_kv_heads=8, head_dim=128, page_size=PAGE)
    step = GraphedDecodeStep(stage, type(wrapper)(torch.empty(64 << 20, dtype=torch.uint8, device=dev)), max_batch=4,
                             max_pages=1024, device=dev, **shape)
    gen, counts = torch.Generator(device="cuda").manual_seed(2), set()
    for at, pick in enumerate(picks):
        print("[case] graph keys", pick, flush=True)
        xs = tuple(torch.randn((layers, 4, h, 128), device=dev, generator=gen).to(torch.bfloat16) for h in (32, 8, 8))
        take = lambda wl: ([wl.tasks[i] for i in pick], [wl.caches[i] for i in pick])
        ctx = FlashDecodeCtx.init_paged_decode_ctx(*take(eager), wrapper)
        wrapper.begin_forward(indptr=ctx.kv_page_indptr, indices=ctx.kv_page_indices, last_page_len=ctx.kv_last_page_lens,
                              indptr_host=ctx.host["kv_page_indptr"], last_page_len_host=ctx.host["kv_last_page_lens"],
                              indices_host=ctx.host["kv_page_indices"], **shape)
        counts.add(wrapper._n_workgroups)
        want = stage.forward(xs, ctx).clone()
        wrapper.end_forward()
        got = step.run(xs, *take(graphed)).clone()
        torch.cuda.synchronize()
        assert torch.equal(got.view(torch.int16), want.view(torch.int16)), at
        assert torch.equal(eager.pool.pages.view(torch.int16), graphed.pool.pages.view(torch.int16)), at
        for wl in (eager, graphed):
            for i in pick:
                wl.tasks[i].step()
    assert len(counts) > 3 and step.captures == 2
