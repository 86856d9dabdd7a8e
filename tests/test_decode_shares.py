"""How the planner lays out the shares of a small decode batch (host rules only; 256 compute units are assumed where
there is no GPU): requests whole or cut, rounds of a share's eight waves."""
import ctypes

import numpy as np
import pytest

from deserve_amd import _lib

WAVES = 8


def _shares(lens, n_kv, group=4, page=16):
    """(tiles of every share, shares each request is in, partial slots)."""
    lib = _lib.lib()
    n = -(-np.asarray(lens, np.int64) // page)
    indptr = np.concatenate([[0], np.cumsum(n)]).astype(np.int32)
    last = np.array([(x - 1) % page + 1 if x else 0 for x in lens], np.int32)
    cap = lib.dskv_decode_plan_bound(len(lens), int(n.sum()) * page)
    plan = np.zeros(cap, np.int32)
    items, wgs, words, ws = ctypes.c_int32(), ctypes.c_int32(), ctypes.c_int64(), ctypes.c_int64()
    rc = lib.dskv_decode_plan(indptr.ctypes.data, last.ctypes.data, len(lens), page, n_kv * group, n_kv, 128, 0,
                              plan.ctypes.data, cap, *[ctypes.byref(x) for x in (items, wgs, words, ws)])
    assert rc == 0, _lib.last_error()
    wg_ptr = plan[4: 4 + wgs.value + 1]
    table = plan[4 + wgs.value + 1 + 2 * len(lens): words.value].reshape(-1, 8)
    tiles = -(-(table[:, 2] - table[:, 1]) // 16)
    at = np.concatenate([np.concatenate([[0], np.cumsum(tiles[a:b])[:-1]]) for a, b in zip(wg_ptr, wg_ptr[1:]) if b > a])
    assert np.array_equal(at, table[:, 7])                     # tiles of the share in front of the item
    return [int(tiles[a:b].sum()) for a, b in zip(wg_ptr, wg_ptr[1:])], np.bincount(table[:, 0], minlength=len(lens)), int(plan[2])


def _needed(tiles, cap, cut):
    """Shares of at most `cap` tiles for the requests in order, longer ones cut (cut) or not allowed."""
    shares, filled = 0, 0
    for n in (int(n) for n in tiles if n):
        if filled and filled + n > cap:
            shares, filled = shares + 1, 0
        if n > cap:
            if not cut:
                return 1 << 30
            shares += -(-n // cap)
        else:
            filled += n
    return shares + (filled > 0)


@pytest.mark.parametrize("n_kv", [8, 16, 12, 5])
@pytest.mark.parametrize("seed", range(24))
def test_small_batches_are_cut_only_where_that_saves_rounds(n_kv, seed):
    rng = np.random.default_rng(seed)
    most = 256 // n_kv
    lens = rng.integers(0 if seed % 3 == 0 else 1, int(rng.choice([40, 260, 900])), int(rng.integers(1, 2 * most)))
    tiles = -(-lens // 16)
    if tiles.sum() > WAVES * most:
        lens = lens[: max(1, int(np.searchsorted(np.cumsum(tiles), WAVES * most * 0.9)))]
        tiles = -(-lens // 16)
    per_share, parts, slots = _shares(lens, n_kv)
    assert len(per_share) <= most and sum(per_share) == tiles.sum()
    assert slots == int(parts[parts > 1].sum()) < 2 * len(per_share) + 1
    if _needed(tiles, 2 * WAVES, False) <= most:        # whole in two rounds
        assert (parts == 1).all() and max(per_share) <= 2 * WAVES
    elif _needed(tiles, WAVES, True) <= most:           # one round, nothing cut that fits into a share
        assert max(per_share) <= WAVES and (tiles[parts > 1] > WAVES).all()


def test_whole_requests_need_no_workspace():
    for lens in ([256] * 16, [100] * 32, [16] * 200):
        per_share, parts, slots = _shares(lens, 8)
        assert slots == 0 and (parts == 1).all() and len(per_share) <= 32
