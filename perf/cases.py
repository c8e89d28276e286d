"""The sorts that this framework is timed on: calls a program makes through the
public entry points, from latency-bound ones to the largest configuration.

A case names the call (`op`), the key type (`kind`), the number of keys (`n`) and
what the keys hold (`data`):

  op     sort      GpuSorter.encode(OP_SORT): keys in HBM, sorted in place
         argsort   GpuSorter.encode(OP_ARGSORT): the stable order of keys in HBM
         pairs     GpuSorter.encode(OP_PAIRS): keys and u32 values in HBM, in place
         order_by  argsort, then GpuGather.encode_gather of a u64 column by it
         slice     argsort_<kind>(array): host keys in, host indices out
  data   uniform   every bit random
         normal    floats N(0, 1e3); of f32 keys 2% are zeros, infinities,
                   subnormals and NaNs
         ties      floats quantised to 4,096 values in [-1, 1)
         zipf      integers: Zipf(1.1) ranks below 2^20 and a tenth of the keys
                   one run of a single key
         records   u64 (file index << 32 | offset): few files with many records
         narrow    integers below 2^20 (ids, small counters)

Calls are stream-ordered on torch's current stream, as a program that keeps its
columns in torch tensors makes them; nothing waits between them.  An in-place sort
begins with a copy of the column it sorts, since the program still needs the
unsorted one.  Results are compared as bit patterns, so -0.0, NaN payloads and the
order of ties count.
"""
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if os.path.join(ROOT, "gpu-forge_amd") not in sys.path:
    sys.path.insert(0, os.path.join(ROOT, "gpu-forge_amd"))

from forge_sort import NP_DTYPES, OP_ARGSORT, OP_PAIRS, OP_SORT, GpuGather, GpuSorter  # noqa: E402

M = 1 << 20


def listed():
    return [
        # a query's few results put in order: one call's latency
        {"name": "sort_u32_1k", "op": "sort", "kind": "u32", "n": 1_000, "data": "uniform"},
        # a small table sorted by a score, its row ids carried along
        {"name": "pairs_f32_10k", "op": "pairs", "kind": "f32", "n": 10_007, "data": "normal"},
        # search results ordered by their (file, offset) key, a column fetched in that order
        {"name": "order_by_u64_100k", "op": "order_by", "kind": "u64", "n": 100_003, "data": "records"},
        # a host program's array through the slice API: copies both ways
        {"name": "slice_argsort_f32_1m", "op": "slice", "kind": "f32", "n": 1_000_003, "data": "normal"},
        # the smallest benchmark configuration, device resident
        {"name": "sort_u32_1m", "op": "sort", "kind": "u32", "n": M, "data": "uniform"},
        # the size most sorts of the benchmark are quoted at
        {"name": "sort_u32_16m", "op": "sort", "kind": "u32", "n": 16 * M, "data": "uniform"},
        # ordering by a quantised score: every key value occurs thousands of times
        {"name": "argsort_f32_16m_ties", "op": "argsort", "kind": "f32", "n": 16 * M, "data": "ties"},
        # 64-bit signed keys (timestamps, hashes) with row ids, an odd length
        {"name": "pairs_i64_16m", "op": "pairs", "kind": "i64", "n": 16_000_057, "data": "uniform"},
        # skewed ids with row ids: grouping a log by a hot key
        {"name": "pairs_u32_64m_zipf", "op": "pairs", "kind": "u32", "n": 64 * M, "data": "zipf"},
        # float columns with every special value
        {"name": "sort_f32_64m", "op": "sort", "kind": "f32", "n": 64 * M, "data": "normal"},
        # the largest 64-bit configuration
        {"name": "sort_f64_128m", "op": "sort", "kind": "f64", "n": 128 * M, "data": "normal"},
        # the headline configuration
        {"name": "sort_u32_256m", "op": "sort", "kind": "u32", "n": 256 * M, "data": "uniform"},
    ]


DATA = {"u32": ("uniform", "zipf", "narrow"), "i32": ("uniform", "narrow"), "f32": ("normal", "ties"),
        "u64": ("uniform", "records", "narrow"), "i64": ("uniform", "narrow"), "f64": ("normal", "ties")}


def draw(rng):
    """One more case: every op, key type and kind of data, sizes from 1,000 keys
    to 512 MiB of keys and values (4 MiB of host keys), odd ones among them."""
    op = rng.choice(("sort", "sort", "sort", "argsort", "pairs", "order_by", "slice"))
    kind = rng.choice(sorted(DATA))
    most = (4 << 20 if op == "slice" else 512 << 20) // (key_bytes(kind) + (0 if op == "sort" else 4))
    n = int(math.exp(rng.uniform(math.log(1_000), math.log(most))))
    if rng.random() < 0.25:
        n = max(1_000, n & ~1023)
    return {"op": op, "kind": kind, "n": n, "data": rng.choice(DATA[kind])}


def key_bytes(kind):
    return 8 if kind.endswith("64") else 4


_made = {}


def sorter():
    """The program's one sorter, on torch's current stream."""
    if "sorter" not in _made:
        _made["sorter"] = GpuSorter.with_context(0, torch.cuda.current_stream().cuda_stream)
    return _made["sorter"]


def gatherer():
    if "gather" not in _made:
        _made["gather"] = GpuGather.with_context(0, torch.cuda.current_stream().cuda_stream)
    return _made["gather"]


def make_keys(case, seed):
    """The keys' bit patterns: int32 or int64 on the GPU."""
    kind, n, data = case["kind"], case["n"], case["data"]
    g = torch.Generator(device="cuda").manual_seed(seed)
    wide = key_bytes(kind) == 8
    bits = torch.int64 if wide else torch.int32

    def integers(low, high, dtype=torch.int64):
        return torch.randint(low, high, (n,), generator=g, device="cuda", dtype=dtype)

    if data == "uniform":
        if wide:
            return integers(-(1 << 62), 1 << 62) * 2 + integers(0, 2)
        return integers(-(1 << 31), 1 << 31, torch.int32)
    if data == "narrow":
        return integers(0, 1 << 20, bits)
    if data == "records":
        files = torch.clamp(torch.rand(n, generator=g, device="cuda", dtype=torch.float64).pow_(-1 / 0.3), max=2e5).to(torch.int64) - 1
        return (files << 32) | integers(0, 1 << 24)
    if data == "zipf":
        ranks = 1 << 20
        cdf = torch.arange(1, ranks + 1, device="cuda", dtype=torch.float64).pow_(-1.1).cumsum_(0)
        cdf /= cdf[-1].clone()
        keys = torch.empty(n, device="cuda", dtype=bits)
        for at in range(0, n, 16 * M):
            u = torch.rand(min(16 * M, n - at), generator=g, device="cuda", dtype=torch.float64)
            keys[at:at + u.numel()] = torch.searchsorted(cdf, u).clamp_(max=ranks - 1).to(bits)
        start, hot = torch.randint(0, n - n // 10, (1,), generator=g, device="cuda"), torch.randint(0, ranks, (1,), generator=g, device="cuda")
        start = int(start)
        keys[start:start + n // 10] = hot.to(bits)
        return keys
    fl = torch.float64 if wide else torch.float32
    if data == "ties":
        x = torch.rand(n, generator=g, device="cuda", dtype=torch.float32)
        return (torch.floor(x * 4096).to(fl) / 2048 - 1).view(bits)
    keys = (torch.randn(n, generator=g, device="cuda", dtype=fl) * 1e3).view(bits)
    if not wide:
        where = torch.randint(0, 300, (n,), generator=g, device="cuda", dtype=torch.int32)
        special = torch.tensor([-(1 << 31), 0, 0x7F800000, -0x800000], dtype=torch.int64, device="cuda").to(torch.int32)
        for i in range(4):
            keys[where == i] = special[i]
        payload = torch.randint(1, 1 << 22, (n,), generator=g, device="cuda", dtype=torch.int32)
        keys = torch.where(where == 4, payload, keys)                    # subnormal
        keys = torch.where(where == 5, payload | 0x7FC00000, keys)       # NaN
    return keys


def prepare(case, seed):
    op, n = case["op"], case["n"]
    keys = make_keys(case, seed)
    if op == "slice":
        return {"case": case, "sorter": sorter(), "keys": keys.cpu().numpy().view(NP_DTYPES[case["kind"]])}
    st = {"case": case, "sorter": sorter(), "src": keys}
    if op == "sort":
        st["keys"] = torch.empty_like(keys)
    elif op == "pairs":
        st["rows"] = torch.arange(n, device="cuda", dtype=torch.int32)
        st["keys"], st["vals"] = torch.empty_like(keys), torch.empty_like(st["rows"])
    else:
        st["index"] = torch.empty(n, device="cuda", dtype=torch.int32)
        if op == "order_by":
            g = torch.Generator(device="cuda").manual_seed(seed + 1)
            st["gather"] = gatherer()
            st["column"] = torch.randint(0, 1 << 62, (n,), generator=g, device="cuda", dtype=torch.int64)
            st["out"] = torch.empty_like(st["column"])
    return st


def run(st):
    case, s = st["case"], st["sorter"]
    op, kind, n = case["op"], case["kind"], case["n"]
    if op == "slice":
        return getattr(s, "argsort_" + kind)(st["keys"])
    if op == "sort":
        st["keys"].copy_(st["src"])
        s.encode(OP_SORT, kind, st["keys"].data_ptr(), None, n)
        return st["keys"]
    if op == "pairs":
        st["keys"].copy_(st["src"])
        st["vals"].copy_(st["rows"])
        s.encode(OP_PAIRS, kind, st["keys"].data_ptr(), st["vals"].data_ptr(), n)
        return st["keys"], st["vals"]
    s.encode(OP_ARGSORT, kind, st["src"].data_ptr(), st["index"].data_ptr(), n)
    if op == "argsort":
        return st["index"]
    st["gather"].encode_gather(st["column"].data_ptr(), st["index"].data_ptr(), st["out"].data_ptr(), n, True, n)
    return st["index"], st["out"]


def work(case):
    """Keys (and values, or the column) read once, results written once: the
    sort itself has no arithmetic to speak of."""
    k, n = key_bytes(case["kind"]), case["n"]
    per = {"sort": 2 * k, "pairs": 2 * (k + 4), "argsort": k + 4, "slice": k + 4, "order_by": k + 4 + 16}[case["op"]]
    return {"bytes": n * per, "flops": 0}


def tolerance(case):
    return "exact"


def exact(case, seed):
    """Keys, indices and columns are moved, not computed: bit patterns, compared exactly."""
    return None
