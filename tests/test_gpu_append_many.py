"""The append kernel's form for launches of more than 4 MiB of K: one row set below and above that line, row sets of every
form, 63 and 64 requests, pages of any size, 32 bits, and rows rotated on their way.  Bit for bit, untouched bytes included."""
import numpy as np
import pytest
import torch

from kvutil import from_torch, make_scenario, to_torch
from oracle import kv_oracle as orc

pytestmark = pytest.mark.gpu


def _split(tokens, requests):
    """`tokens` over `requests`, one of them without any."""
    cuts = np.sort(np.random.default_rng(tokens).integers(0, tokens + 1, requests - 2))
    return np.insert(np.diff(np.concatenate([[0], cuts, [tokens]])), requests // 2, 0).astype(int).tolist()


CASES = [
    # (kv heads, tokens, requests, P, dtype)
    (8, 2048, 5, 16, "bf16"),      # 4 MiB: not yet
    (8, 2049, 5, 16, "bf16"),
    (8, 2500, 63, 8, "f16"),
    (8, 2500, 64, 16, "bf16"),
    (8, 2300, 200, 12, "bf16"),
    (4, 4097, 3, 12, "bf16"),
    (16, 1025, 3, 16, "bf16"),
    (5, 3277, 4, 16, "bf16"),      # 1280 bytes
    (17, 964, 7, 16, "bf16"),      # 4352 bytes: no lane holds its chunks
    (8, 1030, 64, 4, "f32"),
]


def _setup(case):
    heads, tokens, requests, P, dtype = case
    print("[case] append of many rows", *case, flush=True)
    qo = _split(tokens, requests)
    kv = [n + i * 7 % 40 + (n == 0) for i, n in enumerate(qo)]
    sc = make_scenario(31, kv_lens=kv, qo_lens=qo, P=P, Hq=heads, Hkv=heads, D=128, dtype=dtype)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a, np.int32)).cuda()
    return sc, [dev(a) for a in (sc.qo_indptr, sc.kv_page_indices, sc.kv_page_indptr, sc.kv_last_page_lens)]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "-".join(map(str, c)))
def test_append_of_many_rows(case):
    from deserve_amd.paged_ops import append_paged_kv_cache

    sc, (indptr, ids, ptr, last) = _setup(case)
    dtype = case[-1]
    want, pages = sc.pages.copy(), to_torch(sc.pages, dtype)
    orc.append_paged_kv(want, sc.k, sc.v, sc.qo_indptr, sc.kv_page_indices, sc.kv_page_indptr, sc.kv_last_page_lens)
    append_paged_kv_cache(to_torch(sc.k, dtype), to_torch(sc.v, dtype), indptr, pages, ids, ptr, last)
    word = np.uint32 if dtype == "f32" else np.uint16
    assert np.array_equal(from_torch(pages, dtype).view(word), want.view(word))


@pytest.mark.parametrize("case", [c for c in CASES if c[-1] != "f32" and c[3] != 12], ids=lambda c: "-".join(map(str, c)))
def test_append_of_many_rotated_rows(case):
    from deserve_amd.paged_ops import (BatchPrefillWithPagedKVCacheWrapper, append_paged_kv_cache, apply_rope,
                                       rope_table)

    sc, (indptr, ids, ptr, last) = _setup(case)
    heads, P, dtype = case[0], case[3], case[4]
    w = BatchPrefillWithPagedKVCacheWrapper(torch.empty(64 << 20, dtype=torch.uint8, device="cuda"))
    w.begin_forward(indptr, ptr, ids, last, heads, heads, 128, P)
    w._info.new_rows_late = 0      # the append in front of the attention
    q, k, v = (to_torch(a, dtype) for a in (sc.q, sc.k, sc.v))
    offsets = torch.from_numpy((sc.kv_lens - sc.qo_lens).astype(np.int32)).cuda()
    want, pages = to_torch(sc.pages, dtype), to_torch(sc.pages, dtype)
    _, k_rot = apply_rope(q, k, indptr, offsets, interleave=True, rope_theta=5e5)
    append_paged_kv_cache(k_rot, v, indptr, want, ids, ptr, last)
    w.forward(q, pages, k_append=k, v_append=v, rope_table=rope_table(indptr, offsets, q.shape[0], 128, 5e5))
    assert torch.equal(pages.view(torch.int16), want.view(torch.int16))
