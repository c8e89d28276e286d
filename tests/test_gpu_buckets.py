"""The bucket path (one block, or a sample, a partition and a block per bucket)
against the oracle: bit-identical keys, the stable order of equal keys, at the
sizes where its kernels change (rows, tiles, a block's keys, the samples), on
the data that its branches are for."""
import numpy as np
import pytest

import oracle
from test_gpu_parity import BITS, KINDS, NP, bits_equal, first_diff

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def sorter():
    from forge_sort import GpuSorter
    s = GpuSorter.new()
    yield s
    s.close()


def keys_of(kind, n, data, seed):
    g = np.random.Generator(np.random.PCG64(seed))
    u, wide = BITS[kind], BITS[kind] == np.uint64
    if kind.startswith("f") and data in ("normal", "quantised", "specials"):
        x = (g.standard_normal(n) * 1e3).astype(NP[kind])
        if data == "quantised":
            x = (np.floor(x / 100) * 100).astype(NP[kind])
        if data == "specials":
            at = g.random(n) < 0.1
            x[at] = g.choice(np.array([-0.0, 0.0, np.inf, -np.inf, np.nan, -np.nan, 1e-40], dtype=NP[kind]), int(at.sum()))
        return x
    if data in ("normal", "uniform"):
        b = g.integers(0, 1 << (64 if wide else 32), size=n, dtype=u, endpoint=False)
    elif data == "quantised":                     # 40 values, far apart
        b = g.choice(g.integers(0, 1 << (64 if wide else 32), size=40, dtype=u, endpoint=False), size=n)
    elif data == "specials":                      # half the keys one value, the greatest and the least among the rest
        b = g.integers(0, 1 << (64 if wide else 32), size=n, dtype=u, endpoint=False)
        b[g.random(n) < 0.5] = u(0x1234567)
        b[g.random(n) < 0.05] = ~u(0)
        b[g.random(n) < 0.05] = u(0)
    elif data == "clusters":                      # two narrow ranges far apart, and a lone key between
        b = g.integers(0, 1 << 12, size=n, dtype=u) + np.where(g.random(n) < 0.5, u(0), ~u(0) - u(1 << 13)).astype(u)
        b[n // 2] = u(1) << u(20)
    elif data == "sorted":
        b = np.sort(g.integers(0, 1 << (64 if wide else 32), size=n, dtype=u, endpoint=False))
    else:
        b = np.full(n, 0x80000001, dtype=u)       # "same"
    return b.view(NP[kind])


def check(sorter, op, kind, keys):
    n = keys.size
    if op == "sort":
        got = keys.copy()
        getattr(sorter, f"sort_{kind}")(got)
        exp = oracle.sort(kind, keys)
        assert bits_equal(got, exp, kind), first_diff(got, exp, kind)
    elif op == "argsort":
        got, exp = getattr(sorter, f"argsort_{kind}")(keys), oracle.argsort(kind, keys)
        assert np.array_equal(got, exp), first_diff(got, exp, "u32")
    else:
        vals = np.random.Generator(np.random.PCG64(n)).integers(0, 1 << 32, size=n, dtype=np.uint32)
        gk, gv = keys.copy(), vals.copy()
        getattr(sorter, f"sort_pairs_{kind}")(gk, gv)
        ek, ev = oracle.sort_pairs(kind, keys, vals)
        assert bits_equal(gk, ek, kind), first_diff(gk, ek, kind)
        assert np.array_equal(gv, ev), first_diff(gv, ev, "u32")


# (buckets, n): one block from two keys to its last; 8 buckets on the least
# sizes; tile edges of the partition; oversized buckets (two and four of many
# keys: sorted by their blocks through device memory)
SHAPES = [("one", 2), ("one", 63), ("one", 512), ("one", 513), ("one", 4095), ("one", 6144), ("by size", 8193),
          ("buckets", 64), ("buckets", 1025), ("buckets", 20_000), ("buckets", 262_145), ("two", 40_001), ("four", 60_000)]


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("op", ["sort", "argsort", "pairs"])
@pytest.mark.parametrize("shape,n", SHAPES)
def test_bucket_path(sorter, op, kind, shape, n):
    from forge_sort import BUCKETS_ALWAYS, BUCKETS_BY_SIZE, BUCKETS_ONE_BLOCK, TEST_BUCKETS
    mode = {"one": BUCKETS_ONE_BLOCK, "by size": BUCKETS_BY_SIZE, "buckets": BUCKETS_ALWAYS,
            "two": BUCKETS_ALWAYS + (1 << 8), "four": BUCKETS_ALWAYS + (2 << 8)}[shape]
    sorter.set_test_option(TEST_BUCKETS, mode)
    try:
        for i, data in enumerate(("normal", "quantised", "specials", "clusters", "sorted", "same")):
            check(sorter, op, kind, keys_of(kind, n, data, seed=7000 + i))
    finally:
        sorter.set_test_option(TEST_BUCKETS, BUCKETS_BY_SIZE)


@pytest.mark.parametrize("kind,op", [("u32", "sort"), ("f32", "argsort"), ("i64", "sort"), ("f64", "pairs")])
@pytest.mark.parametrize("data", ["normal", "quantised", "specials", "clusters"])
def test_bucket_path_largest(sorter, kind, op, data):
    """The largest sizes that take the path by size (512 buckets, the most
    samples), and one key more (the digit passes)."""
    n = 1_100_000 if kind == "f64" else 1_500_000
    for m in (n, n + 1):
        check(sorter, op, kind, keys_of(kind, m, data, seed=7100 + m % 2))
