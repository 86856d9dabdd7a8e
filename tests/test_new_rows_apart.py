"""Which prefill plans may leave the append to the attention launch's tiles: none in whose tables a page that takes
new rows occurs twice, since a tile waits for its own request's rows only (all on the CPU)."""
import numpy as np
import torch

from deserve_amd import _lib
from deserve_amd.paged_ops import BatchPrefillWithPagedKVCacheWrapper


def _i32(a):
    return np.ascontiguousarray(a, np.int32)


def _apart(qo, kv, tables, page):
    """(library's answer, by the definition)."""
    kv_ptr = _i32(np.r_[0, np.cumsum([len(t) for t in tables])])
    ids = _i32([i for t in tables for i in t])
    got = _lib.lib().dskv_new_rows_apart(
        _i32(np.r_[0, np.cumsum(qo)]).ctypes.data, kv_ptr.ctypes.data, _i32([(n - 1) % page + 1 for n in kv]).ctypes.data,
        ids.ctypes.data, len(qo), page)
    taking = {t[p // page] for n, m, t in zip(qo, kv, tables) for p in range(max(m - n, 0), m)}
    flat = ids.tolist()
    return bool(got), all(flat.count(i) == 1 for i in taking)


def test_named_cases():
    page = 16
    assert _apart([60, 40], [760, 800], [list(range(48)), list(range(50))], page) == (False, False)   # one sequence
    assert _apart([0, 40], [760, 800], [list(range(48)), list(range(50))], page) == (False, False)
    prefix = list(range(25))
    assert _apart([30, 9], [430, 409], [prefix + [30, 31], prefix + [40]], page) == (True, True)       # a shared prefix
    assert _apart([30, 9], [430, 405], [prefix + [30, 31], prefix + [30]], page) == (False, False)
    assert _apart([5], [32], [[7, 7]], page) == (False, False)       # its own old page again
    assert _apart([5], [48], [[7, 7, 8]], page) == (True, True)
    assert _apart([], [], [], page) == (True, True)
    assert _apart([3, 2], [3, 0], [[5], []], page) == (True, True)   # no pages
    assert _apart([40], [17], [[5, 6]], page) == (True, True)        # more rows than tokens


def test_against_the_definition():
    for seed in range(300):
        rng = np.random.default_rng(seed)
        page = int(rng.choice([1, 4, 16]))
        batch = int(rng.integers(1, 8))
        kv = rng.integers(1, 12 * page, batch)
        qo = np.minimum(rng.integers(0, 5 * page, batch), kv)
        pool = int(rng.choice([20, 200, 100000]))
        tables = [rng.integers(0, pool, -(-int(n) // page)).tolist() for n in kv]
        got, want = _apart(qo.tolist(), kv.tolist(), tables, page)
        assert got == want, seed


def _late(qo, kv, tables, page=16):
    w = BatchPrefillWithPagedKVCacheWrapper(torch.empty(64 << 20, dtype=torch.uint8))
    w._shape_args(32, 8, 128, page)
    t = lambda a: torch.from_numpy(_i32(a))
    h_qo, h_kv = t(np.r_[0, np.cumsum(qo)]), t(np.r_[0, np.cumsum([len(x) for x in tables])])
    h_last = t([(n - 1) % page + 1 for n in kv])
    cap = w._check_and_bound(h_qo, h_kv, h_last, t([i for x in tables for i in x]), None)
    w._plan_into(torch.zeros(cap, dtype=torch.int32), cap, h_qo, h_kv, h_last, 0)
    return bool(w._info.new_rows_late)


def test_a_plan_says_late_only_where_the_new_rows_are_apart():
    assert _late([60, 40], [760, 800], [list(range(48)), list(range(50, 100))])
    assert not _late([60, 40], [760, 800], [list(range(48)), list(range(50))])
    prefix = list(range(25))
    assert _late([30, 9], [430, 409], [prefix + [30, 31], prefix + [40]])
