"""Mixed steps whose workspace cannot hold the form that the planner chooses (256 compute units are assumed where there is no
GPU): the next best one that fits, with nothing cut only where no partials fit at all."""
import numpy as np
import pytest
import torch

from deserve_amd import _lib
from deserve_amd.paged_ops import BatchPrefillWithPagedKVCacheWrapper

AUTO, OFF, SHARED = _lib.ROUTE_AUTO, _lib.ROUTE_OFF, _lib.LAYOUT_SHARED


def _plan(kv, qo, ws_bytes, route=True, target=0, page=16):
    at = lambda a: torch.from_numpy(np.concatenate([[0], np.cumsum(a)]).astype(np.int32))
    w = BatchPrefillWithPagedKVCacheWrapper(torch.empty(ws_bytes, dtype=torch.uint8))
    pages, last = -(-np.asarray(kv) // page), torch.tensor([(n - 1) % page + 1 for n in kv], dtype=torch.int32)
    h_qo, h_kv = at(qo), at(pages)
    w._shape_args(32, 8, 128, page)
    cap = w._check_and_bound(h_qo, h_kv, last, torch.zeros(int(pages.sum()), dtype=torch.int32), None)
    plan = torch.zeros(cap, dtype=torch.int32)
    words = w._plan_into(plan, cap, h_qo, h_kv, last, target, route)
    return w._info, plan[:words], w._info.tile_workspace_bytes + w._info.decode_workspace_bytes


FEW = [([8628, 4613, 8970, 8003, 7112, 2460, 7716, 1738], [1] * 7 + [28]), ([6307, 675, 1023, 2691, 2567], [1, 1, 1, 194, 206]),
       ([7958, 8789, 977, 773, 1353], [1] * 4 + [345]), ([9972, 8088, 9812, 3919, 6918, 2438], [1] * 5 + [487])]


@pytest.mark.parametrize("kv,qo", FEW)
def test_a_few_rows_become_tiles_in_parts_where_those_fit(kv, qo):
    chosen, _, need = _plan(kv, qo, 64 << 20)
    tiles, words, less = _plan(kv, qo, 64 << 20, route=OFF)
    assert chosen.layout == SHARED and tiles.n_splits > 1 and 0 < less < need
    got, at_hand, _ = _plan(kv, qo, less)
    assert bytes(got) == bytes(tiles) and torch.equal(at_hand, words)
    whole, words, none = _plan(kv, qo, 0, route=OFF, target=-1)
    got, at_hand, _ = _plan(kv, qo, less - 1)
    assert none == 0 and bytes(got) == bytes(whole) and torch.equal(at_hand, words)


def test_many_rows_stay_shared_beside_whole_tiles():
    kv, qo = [2000] * 40 + [4000], [1] * 40 + [300]
    chosen, _, need = _plan(kv, qo, 64 << 20)
    whole, words, less = _plan(kv, qo, 64 << 20, target=-1)
    assert chosen.layout == whole.layout == SHARED and less < need
    got, at_hand, _ = _plan(kv, qo, less)
    assert bytes(got) == bytes(whole) and torch.equal(at_hand, words)


def test_a_callers_own_number_and_its_limits_are_as_before():
    kv, qo = FEW[1]
    tiles, words, need = _plan(kv, qo, 64 << 20, target=512)
    assert tiles.layout != SHARED and tiles.n_splits > 1
    got, at_hand, _ = _plan(kv, qo, need, target=512)
    assert bytes(got) == bytes(tiles) and torch.equal(at_hand, words)
    whole, words, _ = _plan(kv, qo, 0, route=OFF, target=-1)
    for target in (512, -1):
        got, at_hand, _ = _plan(kv, qo, need - 1 if target > 0 else 0, target=target)
        assert bytes(got) == bytes(whole) and torch.equal(at_hand, words)
