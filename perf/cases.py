"""The KV path's work as a stage of a serving pipeline does it, one case per kind and size.

Three kinds of pass, each through the calls an engine makes:

* ``step``: one step of a stage - ``BatchDecode`` when every request gets one token, else
  ``BatchPrefill`` (a prompt, a chunk of one, or a chunk beside running requests).  ``prepare()``
  builds the step's metadata and plans the attention, ``step()`` runs RoPE, the KV append and the
  paged attention of every layer.  Outputs: the attention output of all layers and the page pool.
* ``graph``: a decode step replayed by ``GraphedDecodeStep``; the graph is captured beforehand.
* ``swap``: the offloads and reloads of a step through ``KVCacheManager``, as the stage driver
  orders them: some requests leave for pinned host memory, others come back, ``synchronize()``.

A case fixes the lengths (``lens`` seeds them); values - pages, q, k, v, all N(0, 1) - and the
order in which the pool hands out its pages come from the seed.  Requests are 8 kv heads of 128
dims throughout: 32 q heads and 16 layers are half of an 8B-shaped model, 64 and 10 a 70B-shaped
stage.
"""
import math

import numpy as np
import torch

from deserve_amd.execution.exec import BatchDecode, BatchPrefill, get_wrappers
from deserve_amd.execution.graph import GraphedDecodeStep
from deserve_amd.kvcache.manager import KVCacheManager
from deserve_amd.kvcache.paged.chunk_pool import CpuChunkPool
from deserve_amd.kvcache.paged.page_table import PageTableAllocator
from deserve_amd.kvcache.virtual import VirtualPagedKVCache, VirtualPagePool
from deserve_amd.stage import KVStage
from deserve_amd.synthetic import fill_normal, make_mixed_workload, scatter_pool_order

KV_HEADS, HEAD_DIM = 8, 128
DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "fp32": torch.float32}
HALF_8B = {"layers": 16, "q_heads": 32}
STAGE_70B = {"layers": 10, "q_heads": 64}


def _step(layers, q_heads, dtype="bf16", page=16, rows=0, row_lo=1, row_hi=1, row_spread="uniform",
          chunks=0, new_lo=1, new_hi=1, prior_lo=0, prior_hi=0, rope=True, lens=0, kind="step"):
    """rows: running requests, one new token each over row_lo .. row_hi tokens of context;
    chunks: requests that get new_lo .. new_hi tokens over prior_lo .. prior_hi."""
    return {"kind": kind, "layers": layers, "q_heads": q_heads, "dtype": dtype, "page": page, "rows": rows,
            "row_lo": row_lo, "row_hi": row_hi, "row_spread": row_spread, "chunks": chunks, "new_lo": new_lo,
            "new_hi": new_hi, "prior_lo": prior_lo, "prior_hi": prior_hi, "rope": rope, "lens": lens}


def _swap(layers, out, back, lo, hi, dtype="bf16", page=16, lens=0):
    return {"kind": "swap", "layers": layers, "dtype": dtype, "page": page, "out": out, "back": back,
            "row_lo": lo, "row_hi": hi, "lens": lens}


def listed():
    cases = {
        # The smallest: one fp32 layer, 8 requests of 512 tokens with the new one.
        "one_layer_fp32": _step(1, 32, "fp32", rows=8, row_lo=511, row_hi=511, rope=False, lens=1),
        # A single user's decode step: nothing to batch, launches and host work count.
        "decode_1": _step(**HALF_8B, rows=1, row_lo=1777, row_hi=1777, lens=2),
        # A small batch of mid-length requests, replayed as a graph.
        "decode_8_graph": _step(**HALF_8B, rows=8, row_lo=300, row_hi=1100, lens=3, kind="graph"),
        # The ordinary decode step: 64 requests over U[256, 4096].
        "decode_64": _step(**HALF_8B, rows=64, row_lo=256, row_hi=4096, lens=2),
        # The deployed form of it: float16, pages of 8 tokens, microbatches of 75.
        "decode_75_page8_f16": _step(**HALF_8B, dtype="f16", page=8, rows=75, row_lo=256, row_hi=4096, lens=5),
        # The largest batch in bytes: 128 requests of lognormal length up to 32 k tokens, 70B-shaped.
        "decode_128_long": _step(**STAGE_70B, rows=128, row_lo=64, row_hi=32768, row_spread="lognormal", lens=5),
        # First steps of three short prompts, ragged.
        "prompts_short": _step(**HALF_8B, chunks=3, new_lo=17, new_hi=203, lens=7),
        # One scheduler step of a long prompt: 512 tokens over 4096 already there.
        "chunk_512": _step(**HALF_8B, chunks=1, new_lo=512, new_hi=512, prior_lo=4096, prior_hi=4096, lens=8),
        # The largest in operations: 16 chunks of 512 tokens over U[0, 8192].
        "chunks_16x512": _step(**HALF_8B, chunks=16, new_lo=512, new_hi=512, prior_lo=0, prior_hi=8192, lens=4),
        # The usual step under load: 75 running requests and a chunk up to 512 tokens in all.
        "mixed_75_437": _step(**HALF_8B, rows=75, row_lo=256, row_hi=4096, chunks=1, new_lo=437, new_hi=437,
                              prior_lo=2506, prior_hi=2506, lens=9),
        # The same, deployed on a 70B-shaped stage: float16, pages of 8.
        "mixed_75_437_70b": _step(**STAGE_70B, dtype="f16", page=8, rows=75, row_lo=256, row_hi=4096, chunks=1,
                                  new_lo=437, new_hi=437, prior_lo=0, prior_hi=4096, lens=10),
        # Page pressure on a 70B-shaped stage: four requests leave, four come back.
        "swap_4_4": _swap(10, 4, 4, 1024, 4096, lens=11),
    }
    return [dict(c, name=n) for n, c in cases.items()]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


# No drawn case costs more than the largest listed ones.
MOST_KV_BYTES, MOST_FLOPS = 15e9, 9e12


def draw(rng):
    while True:
        lens = rng.randrange(1 << 20)
        what = rng.choices(("decode", "graph", "chunks", "mixed", "fp32", "swap"), (35, 8, 25, 20, 6, 6))[0]
        if what == "swap":
            lo = _log_int(rng, 64, 2048)
            return _swap(rng.choice((10, 16)), rng.randint(1, 4), rng.randint(1, 4), lo, lo * 2,
                         rng.choice(("bf16", "f16")), rng.choice((8, 16)), lens)
        shape = dict(rng.choice((HALF_8B, STAGE_70B)), dtype=rng.choice(("bf16", "bf16", "f16")),
                     page=rng.choice((8, 16)), lens=lens)
        row_lo = _log_int(rng, 16, 2048)
        rows = {"row_lo": row_lo, "row_hi": row_lo * _log_int(rng, 1, 16)}
        new_lo = _log_int(rng, 2, 512)
        chunks = {"new_lo": new_lo, "new_hi": min(1024, new_lo * rng.randint(1, 3)), "prior_lo": 0,
                  "prior_hi": rng.choice((0, _log_int(rng, 16, 8192)))}
        if what == "fp32":
            c = _step(1, 32, "fp32", rng.choice((8, 16)), rows=_log_int(rng, 1, 64), rope=False, lens=lens, **rows)
        elif what == "chunks":
            c = _step(**shape, chunks=_log_int(rng, 1, 16), **chunks)
        elif what == "mixed":
            c = _step(**shape, rows=_log_int(rng, 2, 128), **rows, chunks=rng.randint(1, 3), **chunks)
        else:
            many = what == "decode"
            c = _step(**shape, rows=_log_int(rng, 1, 192 if many else 32), **rows, kind="step" if many else "graph")
            if many and rng.random() < 0.2:
                c["row_lo"], c["row_hi"], c["row_spread"] = 64, 32768, "lognormal"
        rows_ctx, prior, _ = _lengths(c)
        kv = (int(rows_ctx.sum()) + int(prior.sum())) * _token_bytes(c) * c["layers"]
        if kv <= MOST_KV_BYTES and work(c)["flops"] <= MOST_FLOPS:
            return c


def _token_bytes(case):
    return 2 * KV_HEADS * HEAD_DIM * DTYPES[case["dtype"]].itemsize


def _lengths(case):
    """(contexts of the running requests, priors of the chunks, their new tokens)."""
    rng = np.random.default_rng(case["lens"])
    if case["row_spread"] == "lognormal":
        rows = np.clip(np.exp(rng.normal(math.log(2048), 1.0, case["rows"])), case["row_lo"], case["row_hi"]).astype(np.int64)
    else:
        rows = rng.integers(case["row_lo"], case["row_hi"] + 1, case["rows"])
    prior = rng.integers(case["prior_lo"], case["prior_hi"] + 1, case["chunks"])
    return rows, prior, rng.integers(case["new_lo"], case["new_hi"] + 1, case["chunks"])


def _swap_lengths(case):
    rng = np.random.default_rng(case["lens"])
    return rng.integers(case["row_lo"], case["row_hi"] + 1, case["out"] + case["back"])


def prepare(case, seed):
    return _prepare_swap(case, seed) if case["kind"] == "swap" else _prepare_step(case, seed)


def _prepare_step(case, seed):
    rows, prior, new = _lengths(case)
    wl = make_mixed_workload("case", rows, prior, new, case["layers"], case["q_heads"], KV_HEADS, HEAD_DIM,
                             case["page"], DTYPES[case["dtype"]], seed=seed)
    state = {"kind": case["kind"], "wl": wl, "stage": KVStage(wl.args, use_rope=case["rope"]),
             "xs": (wl.q, wl.k, wl.v), "batch": BatchPrefill if case["chunks"] else BatchDecode}
    if case["kind"] == "graph":
        # a serving process captures a batch shape once and replays it from then on
        dev = wl.pool.main_device
        pages = sum(-(-(int(n) + 1) // case["page"]) for n in rows)
        state["graph"] = GraphedDecodeStep(state["stage"], get_wrappers(dev)[0], len(rows), pages, dev,
                                           case["q_heads"], KV_HEADS, HEAD_DIM, case["page"])
        state["graph"].run(state["xs"], wl.tasks, wl.caches)
    return state


def _prepare_swap(case, seed):
    lens, page, layers = _swap_lengths(case), case["page"], case["layers"]
    dev, dtype = torch.device("cuda"), DTYPES[case["dtype"]]
    pages = [-(-int(n) // page) for n in lens]
    pool = VirtualPagePool(layers, sum(pages) + 64, 16, page, dev, dtype, KV_HEADS, HEAD_DIM)
    fill_normal(pool.pages, seed + 1)
    scatter_pool_order(pool, seed + 2)
    tables = PageTableAllocator(2 * len(lens), max(pages) * page, page, dev)
    units = 2 * sum(1 << max(0, (n - 1).bit_length()) for n in pages)
    manager = KVCacheManager(pool, CpuChunkPool(layers, 1 + (units - 1).bit_length(), page, dtype, KV_HEADS, HEAD_DIM), tables)
    caches = []
    for n in lens:
        caches.append(VirtualPagedKVCache.empty(tables, pool))
        caches[-1].extend(int(n))
    away = [manager.copy_gpu_to_cpu(c, "task") for c in caches[case["out"]:]]
    manager.synchronize()
    for c in caches[case["out"]:]:
        c.free()
    return {"kind": "swap", "pool": pool, "manager": manager, "here": caches[: case["out"]], "away": away}


def run(state):
    if state["kind"] == "swap":
        return _run_swap(state)
    wl = state["wl"]
    if state["kind"] == "graph":
        out = state["graph"].run(state["xs"], wl.tasks, wl.caches)
    else:
        batch = state["batch"](state["xs"], state["stage"], wl.tasks, wl.caches)
        batch.prepare()
        out = batch.step(ignore_eos=True).all_xs
    return {"out": out, "pages": wl.pool.pages}


def _run_swap(state):
    manager = state["manager"]
    left = []
    for cache in state["here"]:
        left.append(manager.copy_gpu_to_cpu(cache, "task"))
        cache.free()
    back = []
    for handle in state["away"]:
        back.append(manager.copy_cpu_to_gpu(handle, "task"))
        handle.free()
    manager.synchronize()
    state["here"], state["away"] = back, left
    layers = state["pool"].num_layers
    return {"images": [h.retrieve()[: h.initial_size * layers] for h in left], "pages": state["pool"].pages}


def work(case):
    if case["kind"] == "swap":
        # every byte is read on one side of the host link and written on the other
        pages = [-(-int(n) // case["page"]) for n in _swap_lengths(case)]
        return {"bytes": 2 * sum(pages) * case["page"] * _token_bytes(case) * case["layers"], "flops": 0}
    rows, prior, new = _lengths(case)
    q_row = case["q_heads"] * HEAD_DIM * DTYPES[case["dtype"]].itemsize
    tokens = case["rows"] + int(new.sum())
    kv = (int(rows.sum()) + int(prior.sum())) * _token_bytes(case)
    # the pages' tokens once; the new tokens' k and v in and into their pages, q in, output out
    per_layer = kv + tokens * 2 * (_token_bytes(case) + q_row)
    pairs = int((rows + 1).sum()) + int((new * prior + new * (new + 1) // 2).sum())
    return {"bytes": per_layer * case["layers"], "flops": 4 * case["q_heads"] * HEAD_DIM * pairs * case["layers"]}


def tolerance(case):
    if case["kind"] == "swap":
        return "exact"
    # About four times what the largest cases show against the same rows in 64 bits (one fp32 layer
    # 1.7e-7; bf16 2.3e-3, 1.9e-2 at most; f16 2.7e-4, 1.5e-3 at most).
    if case["dtype"] == "fp32":
        return {"rel": 1e-6, "max": 8e-6}
    return {"rel": 1e-2, "max": 8e-2} if case["dtype"] == "bf16" else {"rel": 1.2e-3, "max": 1e-2}
