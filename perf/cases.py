"""The work this framework is used for, as cases that can be timed and compared: embedding rows looked up through
`collcache.torch`, the PyTorch surface, at the sizes its configurations, tests and benchmark use.

A case names a table (rows x dim of a type, the share of it cached in HBM), how its keys are distributed and one step
of a program that uses it:

  lookup   coll_torch_lookup_key_t_val_ret: the blocking lookup of a batch
  async    coll_torch_lookup_async: the same enqueued on torch's stream
  forward  coll_torch_forward: a serving step, which also records the hotness of a prefix of the batch
  pooled   coll_torch_lookup_pooled: a multi-hot feature looked up and combined per sample
  unique   coll_torch_lookup_unique, then the rows back at every position: the sparse layer's unique -> lookup -> gather
  refresh  two steps of a loop that refreshes the cache behind every lookup, counted and placed on the device

The library serves one cache per process, so the cache a case needs is built once (`_cache`) and stays until a case
needs another one; what a seed changes are the batches.  Tables hold N(0, 1) values, keys are drawn from a Zipf law
over the ranks of a random permutation of the rows (0: uniform), and hotness is recorded from batches of the same law.
"""
import math
import os
import sys

import numpy as np
import torch

import ugache_amd

sys.path.insert(0, os.path.dirname(os.path.abspath(ugache_amd.__file__)))
import collcache.torch as co  # noqa: E402
from collcache.common import _basics  # noqa: E402

_ELEM = {"fp32": 4, "fp16": 2, "bf16": 2}
_TYPE = {"fp32": torch.float32, "fp16": torch.float16, "bf16": torch.bfloat16}
# what makes a cache another one; the rest of a case describes its batches
_CACHE_FIELDS = ("rows", "dim", "dtype", "share", "zipf", "sparse_ids", "device_refresh")
_MUL, _BITS = 0x9E3779B97F4A7C15, 40  # sparse ids: id of row r = r * _MUL mod 2^40
_PRESAMPLE_KEYS = 8 << 20
# the share of a batch whose hotness the serving loop records
_RECORDED = 0.05


def _case(name, path, **kw):
    c = {"name": name, "path": path, "rows": 1_000_000, "dim": 128, "dtype": "fp32", "share": 1.0, "zipf": 0.0,
         "keys": 65_536, "int64": True, "sparse_ids": False, "device_refresh": False, "bag": 0, "ragged": False,
         "combiner": "sum", "weighted": False}
    c.update(kw)
    return c


def listed():
    # a recommendation table of 26 sparse fields, 40 % of it cached (the share of the DLR configuration, 40 of 106 GB)
    dlr = dict(rows=4_160_000, dim=128, dtype="fp32", share=0.4, zipf=1.2)
    # node features, a quarter of them cached (the GNN configuration at a fifth of its rows)
    gnn = dict(rows=20_000_000, dim=128, dtype="fp32", share=0.25, zipf=0.9)
    # sparse 64-bit ids over short fp16 rows, a tenth cached behind the hash table (at a twelfth of its rows)
    ids = dict(rows=40_000_000, dim=64, dtype="fp16", share=0.1, zipf=1.05, sparse_ids=True)
    return [
        # an inference request of 64 samples: what counts is how soon the call returns
        _case("request_1664", "lookup", keys=64 * 26, **dlr),
        # a serving step of 1,024 samples with its hotness recorded
        _case("serving_step_26k", "forward", keys=1024 * 26, **dlr),
        # a training batch of 8,192 samples, enqueued like any torch op
        _case("dlr_batch_async", "async", keys=8192 * 26, **dlr),
        # one multi-hot feature of 16 weighted ids per sample, averaged
        _case("bag16_mean", "pooled", keys=65_536 * 16, bag=16, combiner="mean", weighted=True, **dlr),
        # short rows and few ids per sample: 26 fields of 1 to 4 ids, the whole table in HBM, bfloat16
        _case("bag4_short_rows", "pooled", keys=8192 * 26 * 5 // 2, bag=4, ragged=True, rows=20_000_000, dim=32,
              dtype="bf16", zipf=1.05),
        # node features, all of them in HBM: the all-hit configuration
        _case("features_full", "lookup", keys=262_144, int64=False, rows=10_000_000, dim=128),
        # feature widths and batches as sampling graphs makes them, no power of two in sight
        _case("features_odd_full", "lookup", keys=200_003, rows=1_500_000, dim=301, zipf=0.5),
        _case("features_odd_half", "lookup", keys=150_001, int64=False, rows=6_000_000, dim=50, share=0.5, zipf=1.2),
        # a large sampled batch with a quarter of the table cached: the host link bounds it
        _case("features_mixed_1m", "lookup", keys=1 << 20, **gnn),
        # the same table, the distinct nodes of a batch looked up once and spread over its positions
        _case("features_unique", "unique", keys=262_144, **gnn),
        # a large batch of hashed ids
        _case("hashed_ids_1m", "lookup", keys=1 << 20, **ids),
        # ... and of a program that refreshes its cache behind every batch
        _case("refresh_each_step", "refresh", keys=262_144, device_refresh=True, **ids),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    path = rng.choice(["lookup"] * 8 + ["async"] * 2 + ["forward"] * 2 + ["pooled"] * 5 + ["unique"] * 2 + ["refresh"])
    dtype = rng.choice(["fp32", "fp32", "fp16", "bf16"])
    elem = _ELEM[dtype]
    if path == "pooled" or rng.random() < 0.5:
        dim = rng.choice([16, 32, 64, 96, 128, 200, 256, 384, 512])
    else:  # an odd width: any number of 4-byte words
        dim = rng.randint(3, 600) * (4 // elem)
    row = dim * elem
    rows = min(_log_int(rng, 300_000, 24_000_000), 6_000_000_000 // row)
    share = rng.choice([1.0, 1.0, round(rng.uniform(0.1, 0.6), 3)]) if path != "refresh" else round(rng.uniform(0.1, 0.4), 3)
    zipf = rng.choice([0.0, 0.5, 0.8, 1.05, 1.2]) if share == 1.0 else rng.choice([0.9, 1.05, 1.2])
    sparse = share < 1.0 and path != "pooled" and rng.random() < 0.4
    # keys: any size, bounded by what the largest listed case writes and by what it takes over the host link
    most = min(1 << 20, (400 << 20) // row)
    if share < 1.0:
        miss = 1.0 - _cdf(share * rows, rows, zipf)
        most = min(most, int((48 << 20) / (row * (miss + 0.01))))
    if path in ("unique", "refresh"):
        most = min(most, 300_000)
    keys = _log_int(rng, 512, max(most, 1024))
    if path == "refresh":  # the device places from its counters: a batch observes fewer rows than the cache holds
        keys = min(keys, int(share * rows) // 4)
    more = {}
    if path == "pooled":
        more = dict(bag=rng.choice([1, 2, 4, 8, 16, 40]), ragged=rng.random() < 0.5,
                    combiner=rng.choice(["sum", "mean", "sqrtn"]), weighted=rng.random() < 0.5)
    c = _case("", path, rows=rows, dim=dim, dtype=dtype, share=share, zipf=zipf, keys=keys,
              int64=sparse or rng.random() < 0.5, sparse_ids=sparse, device_refresh=path == "refresh", **more)
    del c["name"]
    return c


# ---- keys ------------------------------------------------------------------------------------------------------------
def _cdf(rank, rows, s):
    """share of the draws that fall on the first `rank` ranks (the continuous bounded law the keys are drawn from)"""
    if s == 0.0:
        return rank / rows
    return ((rank + 1.0) ** (1.0 - s) - 1.0) / ((rows + 1.0) ** (1.0 - s) - 1.0)


def _ranks(n, rows, s, gen):
    u = torch.rand(n, generator=gen, device="cuda", dtype=torch.float64)
    if s == 0.0:
        r = (u * rows).to(torch.int64)
    else:
        e = 1.0 - s
        r = ((((rows + 1.0) ** e - 1.0) * u + 1.0) ** (1.0 / e)).to(torch.int64) - 1
    return r.clamp_(0, rows - 1)


def _distinct(case, n):
    """how many rows n draws of the case's law are expected to touch"""
    rows, s = case["rows"], case["zipf"]
    edges = np.unique(np.concatenate([np.arange(0, min(rows, 4096) + 1), np.geomspace(1, rows, 4096).astype(np.int64),
                                      [rows]])).astype(np.float64)
    mass = np.diff(_cdf(edges, rows, s))
    count = np.diff(edges)
    return float(np.sum(count * -np.expm1(n * np.log1p(-np.minimum(mass / count, 1.0 - 1e-12)))))


def _keys_of(case, rows_t):
    if case["sparse_ids"]:
        mul = torch.tensor(_MUL - (1 << 64), dtype=torch.int64, device=rows_t.device)
        rows_t = (rows_t * mul) & ((1 << _BITS) - 1)
    return rows_t if case["int64"] else rows_t.to(torch.int32)


# ---- the cache a case looks keys up in -------------------------------------------------------------------------------
_open = {"key": None, "perm": None}
_REFRESH_ENV = {"COLL_GPU_RECORD": "1", "COLL_GPU_REFRESH": "1", "COLL_MISS_STAGE_ROWS": str(1 << 20)}


def _cache(case):
    """builds the cache of the case unless it is the one this process has; returns row number by rank"""
    key = tuple(case[f] for f in _CACHE_FIELDS)
    if _open["key"] == key:
        return _open["perm"]
    if _open["key"] is not None:
        co.coll_torch_shutdown()
        _open.update(key=None, perm=None)
        torch.cuda.empty_cache()
    rows, dim, share, s = case["rows"], case["dim"], case["share"], case["zipf"]
    for name, value in _REFRESH_ENV.items():
        os.environ.pop(name, None)
        if case["device_refresh"]:
            os.environ[name] = value
    co.config({"cache_percentage": share, "_cache_policy": co.kCollCacheAsymmLink, "num_device": 1,
               "num_global_step_per_epoch": 1000, "num_epoch": 1, "num_total_item": rows, "omp_thread_num": 8})
    if case["sparse_ids"]:
        _basics.set_key_map(_MUL, _BITS)
    co.coll_cache_record_init(0)
    gen = torch.Generator(device="cuda").manual_seed(1)
    perm = torch.randperm(rows, generator=gen, device="cuda", dtype=torch.int64)
    if share < 1.0:
        for _ in range(4):
            batch = _keys_of(case, perm[_ranks(_PRESAMPLE_KEYS // 4, rows, s, gen)])
            co.coll_torch_record(0, batch.cpu())
    emb = co.coll_torch_create_emb_shm(0, rows, dim, _TYPE[case["dtype"]])
    step = max(1, (256 << 20) // (dim * 4))
    for r0 in range(0, rows, step):
        part = torch.randn((min(step, rows - r0), dim), generator=gen, device="cuda")
        emb[r0 : r0 + step].copy_(part.to(emb.dtype))
    _basics.C_LIB_CTYPES.coll_cache_set_max_num_keys(max(1 << 20, case["keys"]))
    co.coll_torch_init_t(0, 0, emb, share)
    # every serving step records a prefix, none of them starts a refresh
    co.coll_torch_forward_config(True, 0, _RECORDED, False)
    _open.update(key=key, perm=perm)
    return perm


def prepare(case, seed):
    perm = _cache(case)
    gen = torch.Generator(device="cuda").manual_seed(1_000_003 + seed)
    n, state = case["keys"], {"path": case["path"]}
    if case["path"] == "pooled":
        samples = max(1, n * (2 if case["ragged"] else 1) // (case["bag"] + (1 if case["ragged"] else 0)))
        if case["ragged"]:
            length = torch.randint(1, case["bag"] + 1, (samples,), generator=gen, device="cuda")
        else:
            length = torch.full((samples,), case["bag"], dtype=torch.int64, device="cuda")
        state["offsets"] = torch.cat([torch.zeros(1, dtype=torch.int64, device="cuda"), length.cumsum(0)])
        n = int(state["offsets"][-1])
        state["combiner"] = case["combiner"]
        state["weights"] = (torch.rand(n, generator=gen, device="cuda") + 0.5) if case["weighted"] else None
    state["keys"] = _keys_of(case, perm[_ranks(n, case["rows"], case["zipf"], gen)])
    if case["path"] == "refresh":
        state["next_keys"] = _keys_of(case, perm[_ranks(n, case["rows"], case["zipf"], gen)])
    return state


def run(state):
    path, keys = state["path"], state["keys"]
    if path == "lookup":
        return co.coll_torch_lookup_key_t_val_ret(0, keys, pad_to_8=False)
    if path == "async":
        return co.coll_torch_lookup_async(0, keys, pad_to_8=False)
    if path == "forward":
        return co.coll_torch_forward(0, keys, pad_to_8=False)
    if path == "pooled":
        return co.coll_torch_lookup_pooled(0, keys, state["offsets"], state["weights"], state["combiner"])
    if path == "unique":
        emb, inverse = co.coll_torch_lookup_unique(0, keys)
        return {"rows": emb.index_select(0, inverse), "distinct": emb.size(0)}
    # refresh: the second step's rows, and how many of them the refreshed cache served
    co.coll_torch_lookup_key_t_val_ret(0, keys, pad_to_8=False)
    co.coll_torch_refresh(0, foreground=True)
    out = co.coll_torch_lookup_key_t_val_ret(0, state["next_keys"], pad_to_8=False)
    hits = _basics.last_group_offset(0)[1]
    co.coll_torch_refresh(0, foreground=True)
    return {"rows": out, "hits": hits}


def work(case):
    """bytes: keys, weights and offsets read, every row the batch touches read once, every output row written once;
    flops: a multiply and an add per looked-up value of a pooled case"""
    n, row = case["keys"], case["dim"] * _ELEM[case["dtype"]]
    key = 8 if case["int64"] else 4
    touched = _distinct(case, n)
    if case["path"] == "pooled":
        samples = n / ((case["bag"] + 1) / 2.0 if case["ragged"] else case["bag"])
        per_id = key + (4 if case["weighted"] else 0)
        return {"bytes": n * per_id + samples * 8 + touched * row + samples * row, "flops": 2.0 * n * case["dim"]}
    one = n * key + touched * row + n * row
    if case["path"] == "unique":
        return {"bytes": one + 4.0 * n, "flops": 0}
    if case["path"] == "refresh":
        # per step: the batch, a counter per touched row, the rows that come in read and written, two membership bitmaps
        moved = _distinct(case, 2 * n) - touched
        return {"bytes": 2.0 * (one + 4.0 * touched + 2.0 * moved * row + case["rows"] / 4.0), "flops": 0}
    return {"bytes": one, "flops": 0}


def tolerance(case):
    """rows are copied, so they are the same bytes; a combination is an fp32 sum over the ids of a sample, rounded to
    the table's type at the end"""
    if case["path"] != "pooled":
        return "exact"
    # about four times the largest difference from the same combination in float64 over bags of 1 to 40 ids: fp32
    # rel 1.3e-7, max 8e-7; fp16 rel 2.1e-4, max 4.9e-4; bf16 rel 1.7e-3, max 3.9e-3 (half an ulp of the rounding)
    return {"fp32": {"rel": 6e-7, "max": 4e-6}, "fp16": {"rel": 8e-4, "max": 2e-3}, "bf16": {"rel": 6.6e-3, "max": 1.6e-2}}[
        case["dtype"]]
