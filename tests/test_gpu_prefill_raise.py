"""When query tiles raise their running maximum: scores that climb by less and by more than what a block may
hold under the old one, blocks that pass it by their sum alone, single spikes at the ends of blocks and lane
halves, scores that fall, and hundreds of powers of two either way - whole tiles, tiles in parts, and tiles
beside decode rows, against 64 bits."""
import numpy as np
import pytest
import torch

from deserve_amd import _lib
from kvutil import make_scenario, to_storage, to_torch

pytestmark = pytest.mark.gpu

T = 1300
t = np.arange(T)
spikes = np.zeros(T)
spikes[[31, 32, 36, 63, 100, 512, 703, 1299]] = [9, 18, 27, 5, 60, 61, 140, 200]
LEVELS = {   # log2 of a token's weight for the head with factor 1
    "climb": 9.0 * (t // 32),
    "climb_by_halves": 7.9 * (t // 16),
    "sum_alone": np.where(t < 32, 0.0, 6.9),
    "just_under": np.where(t < 32, 0.0, 3.9),
    "spikes": spikes,
    "fall": -50.0 * (t // 32),
    "far": np.where(t % 96 < 32, -300.0, 0.3 * t),
}
FACTORS = [1.0, -1.0, 0.25, 2.0]


@pytest.mark.parametrize("dtype", ["bf16", "f16"])
@pytest.mark.parametrize("levels", LEVELS)
def test_scores_that_move_the_maximum(levels, dtype):
    from deserve_amd.paged_ops import BatchPrefillWithPagedKVCacheWrapper

    print("[case] prefill maximum", levels, dtype, flush=True)
    qo, kv, P, Hq, Hkv, D = [100, 1], [T, 40], 16, 4, 1, 128
    sc = make_scenario(66, kv_lens=kv, qo_lens=qo, P=P, Hq=Hq, Hkv=Hkv, D=D, dtype=dtype)
    pages, q = to_torch(sc.pages, dtype), to_torch(sc.q, dtype)
    q[:100] = 0
    q[:100, :, 0] = torch.tensor([8 * f for f in FACTORS], dtype=q.dtype, device="cuda")
    k = np.zeros((T, D), np.float32)
    k[:, 0] = LEVELS[levels] / (8 * 1.4426950408889634 / np.sqrt(D))
    k = to_torch(to_storage(k, dtype), dtype)
    table = sc.kv_page_indices[: sc.kv_page_indptr[1]]
    for tok in range(0, T, P):
        n = min(P, T - tok)
        pages[int(table[tok // P]), 0, :n, 0] = k[tok: tok + n]
    v = torch.cat([pages[int(p), 1, :, 0] for p in table])[:T].double()
    s = torch.einsum("qhd,td->hqt", q[:100].double(), k.double()) / np.sqrt(D)
    s.masked_fill_(torch.arange(T, device="cuda") > T - 100 + torch.arange(100, device="cuda")[:, None], float("-inf"))
    want = (torch.softmax(s, -1) @ v).transpose(0, 1)
    # probabilities and results are rounded once each to 8 (f16: 11) bits, and a score in fp32 may be off by
    # 2^-22 of its size, of which exp2 makes as much of a weight
    eps = 2.0 ** (-8 if dtype == "bf16" else -11)
    bound = (2 * eps + float(s[s.isfinite()].abs().max()) * 2.0 ** -20) * float(v.abs().max())
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a, np.int32)).cuda()
    w = BatchPrefillWithPagedKVCacheWrapper(torch.empty(64 << 20, dtype=torch.uint8, device="cuda"))
    for route, target in ((False, -1), (False, 1024), (_lib.ROUTE_SHARED_LAUNCH, -1)):
        w.begin_forward(dev(sc.qo_indptr), dev(sc.kv_page_indptr), dev(sc.kv_page_indices), dev(sc.kv_last_page_lens),
                        Hq, Hkv, D, P, target_workgroups=target, route_one_row_requests=route)
        got = w.forward(q, pages)[:100].double()
        torch.cuda.synchronize()
        assert float((got - want).abs().max()) <= bound, (route, target)
