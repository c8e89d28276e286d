"""The bucket path (one block, or a sample, a partition and a block per bucket)
against the oracle: bit-identical keys, the stable order of equal keys, at the
sizes where its kernels change (rows, tiles, a block's keys, the samples), on
the data that its branches are for."""
import numpy as np
import pytest

import oracle
from test_gpu_parity import BITS, KINDS, NP, bits_equal, first_diff, hip_stream  # noqa: F401

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
    elif data == "narrow":                        # 20 varying bits
        b = g.integers(0, 1 << 20, size=n, dtype=u)
    elif data == "lone":                          # 12, but for one key that a sample misses
        b = g.integers(0, 1 << 12, size=n, dtype=u)
        b[n // 3 + 1] = ~u(0)
    elif data == "runs":                          # random keys, each five times in a row
        b = np.repeat(g.integers(0, 1 << (64 if wide else 32), size=n // 5 + 1, dtype=u, endpoint=False), 5)[:n]
    elif data == "records":                       # (file index << 32 | offset), most keys in few files
        b = (np.minimum(g.random(n) ** (-1 / 0.3), 2e5).astype(np.uint64) - u(1)) << u(32) | g.integers(0, 1 << 24, size=n, dtype=u)
    elif data == "cluster":                       # half of them in a range that quantiles' top bits share
        b = np.where(g.random(n) < 0.5, g.integers(0, 1 << 10, size=n), g.integers(0, 1 << 50, size=n)).astype(u)
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


@pytest.mark.parametrize("kind", ["u64", "i64", "f64"])
@pytest.mark.parametrize("op", ["sort", "argsort", "pairs"])
@pytest.mark.parametrize("lnb,n", [(0, 64), (0, 5121), (1, 30_000), (0, 300_001), (2, 150_000)])
def test_two_levels(sorter, op, kind, lnb, n):
    """Two levels of buckets, or the digit passes where few digits vary: least
    size, tile edges, few buckets (children larger than a block), every kind of
    data that takes another branch."""
    from forge_sort import BUCKETS_BY_SIZE, BUCKETS_TWO_LEVELS, PATH_DIGITS, PATH_TWO_LEVELS, TEST_BUCKETS
    sorter.set_test_option(TEST_BUCKETS, BUCKETS_TWO_LEVELS + (lnb << 8))
    try:
        for i, data in enumerate(("normal", "quantised", "specials", "clusters", "sorted", "same", "narrow", "lone", "runs")):
            keys = keys_of(kind, n, data, seed=7200 + i)
            check(sorter, op, kind, keys)
            b = keys.view(np.uint64)
            top = np.uint64(1 << 63)
            b = np.where(b & top, ~b, b | top) if kind == "f64" else b
            varying = int(np.bitwise_or.reduce(b ^ b[0]))
            assert sorter.last_pass_info()[1] == sum(1 << j for j in range(8) if varying >> (8 * j) & 0xFF)
            path, overflows = sorter.last_bucket_info()
            digits = bin(sorter.last_pass_info()[1]).count("1")
            assert path == PATH_TWO_LEVELS if digits > 4 else path in (PATH_TWO_LEVELS, PATH_DIGITS), (path, digits)
            assert overflows == 0
    finally:
        sorter.set_test_option(TEST_BUCKETS, BUCKETS_BY_SIZE)


@pytest.mark.parametrize("kind,op,n", [("f64", "sort", 1_500_001), ("f64", "argsort", 1_000_001), ("f64", "argsort", 1 << 20),
                                       ("f64", "pairs", 1 << 20), ("i64", "pairs", 12_000_000)])
@pytest.mark.parametrize("data", ["normal", "quantised", "narrow", "lone"])
def test_two_levels_by_size(sorter, kind, op, n, data):
    """The least sizes that take two levels by size, and one below (f64 with
    values between the one level's largest and 2^20 keys)."""
    from forge_sort import PATH_DIGITS, PATH_TWO_LEVELS
    check(sorter, op, kind, keys_of(kind, n, data, seed=7300))
    if n == 1_000_001:
        assert sorter.last_bucket_info()[0] == PATH_DIGITS
    elif data == "normal":
        assert sorter.last_bucket_info() == (PATH_TWO_LEVELS, 0)


@pytest.mark.parametrize("kind,op,n,values,lnb", [
    ("f64", "sort", 1_600_000, 256, 0), ("f64", "argsort", 4_000_000, 190, 0), ("u64", "pairs", 12_000_000, 192, 0),
    ("u32", "sort", 1_000_000, 400, 0), ("i64", "pairs", 900_001, 300, 0),
    ("f64", "sort", 850_000, 384, 1), ("u64", "argsort", 850_000, 384, 1)])      # (two buckets of 192 values each)
def test_repeated_values(sorter, kind, op, n, values, lnb):
    """Evenly spaced values, every one in a group of the sample's own, so that
    a bucket between two splitters can hold two: exact, and no region too small."""
    from forge_sort import BUCKETS_BY_SIZE, BUCKETS_TWO_LEVELS, PATH_BUCKETS, PATH_TWO_LEVELS, TEST_BUCKETS
    sorter.set_test_option(TEST_BUCKETS, BUCKETS_TWO_LEVELS + (lnb << 8) if lnb else BUCKETS_BY_SIZE)
    try:
        for seed in (1, 2, 3):
            k = np.random.Generator(np.random.PCG64(seed)).integers(0, values, size=n, dtype=BITS[kind])
            keys = k / (values - 1) if kind == "f64" else (k * (~BITS[kind](0) // BITS[kind](values))).view(NP[kind])
            check(sorter, op, kind, keys)
            assert sorter.last_bucket_info() == (PATH_TWO_LEVELS if lnb or n > 1_500_000 else PATH_BUCKETS, 0)
    finally:
        sorter.set_test_option(TEST_BUCKETS, BUCKETS_BY_SIZE)


@pytest.mark.parametrize("op,n", [("sort", 1_500_000), ("argsort", 1_000_000), ("pairs", 8_193), ("pairs", 13_000_001)])
@pytest.mark.parametrize("data", ["records", "cluster"])
def test_crowded_samples(sorter, op, n, data):
    """64-bit samples that their top bits do not order."""
    check(sorter, op, "u64", keys_of("u64", n, data, seed=7600))
    assert sorter.last_bucket_info()[1] == 0


@pytest.mark.parametrize("kind,op", [("u32", "sort"), ("i32", "pairs"), ("f32", "argsort"), ("i64", "sort"),
                                     ("f64", "pairs")])
@pytest.mark.parametrize("data", ["normal", "quantised", "specials", "clusters", "runs"])
def test_bucket_path_largest(sorter, kind, op, data):
    """The largest sizes that take the path by size (512 buckets, the most
    samples), and one key more (the digit passes; f64: two levels)."""
    n = {"u32": 1_100_000, "i32": 600_000, "f32": 190_000, "i64": 1_500_000, "f64": 1_000_000}[kind]
    for m in (n, n + 1):
        check(sorter, op, kind, keys_of(kind, m, data, seed=7100 + m % 2))


@pytest.mark.parametrize("kind,op,n,reserved", [("u32", "sort", 790_000, 1_000_000), ("u64", "pairs", 380_001, 400_000),
                                                ("f64", "pairs", 1_200_001, 1_300_000), ("f64", "sort", 1_600_001, 1_700_000),
                                                # (more look-back entries than the reserved sort: smaller tiles)
                                                ("u32", "sort", 2_000_000, 2_200_000), ("f64", "pairs", 1_040_000, 1_300_000)])
def test_bucket_path_captured(hip_stream, kind, op, n, reserved):  # noqa: F811
    """Scratch reserved for more keys holds the sort of fewer (a smaller sort's
    regions may be larger); captured into a HIP graph and replayed on data that
    takes other branches (two levels: the buckets, the digit passes, and back),
    eager sorts between the replays."""
    import ctypes
    from forge_sort import OP_PAIRS, OP_SORT, GpuSorter
    hip = ctypes.CDLL("libamdhip64.so.7")
    st = ctypes.c_void_p(hip_stream)
    s = GpuSorter.with_context(0, hip_stream)
    code = OP_PAIRS if op == "pairs" else OP_SORT
    graph, exe = ctypes.c_void_p(), ctypes.c_void_p()
    vals = np.arange(n, dtype=np.uint32)
    try:
        kb, vb = s.alloc_sort_buffer(kind, n), s.alloc_sort_buffer("u32", n)
        s.reserve(code, kind, reserved)
        assert hip.hipStreamBeginCapture(st, 0) == 0
        s.encode(code, kind, kb.device_ptr(), vb.device_ptr(), n, stream=hip_stream)
        assert hip.hipStreamEndCapture(st, ctypes.byref(graph)) == 0
        assert hip.hipGraphInstantiate(ctypes.byref(exe), graph, None, None, ctypes.c_size_t(0)) == 0
        for r, data in enumerate(("uniform", "narrow", "lone", "quantised", "same", "normal")):
            keys = keys_of(kind, n, data, seed=7400 + r)
            kb.copy_from_slice(keys)
            vb.copy_from_slice(vals)
            assert hip.hipGraphLaunch(exe, st) == 0
            assert hip.hipStreamSynchronize(st) == 0
            ek, ev = oracle.sort_pairs(kind, keys, vals)
            assert bits_equal(kb.as_slice(), ek, kind), f"replay {r} ({data})"
            assert op == "sort" or np.array_equal(vb.as_slice(), ev), f"replay {r} ({data})"
            check(s, "sort", kind, keys_of(kind, n // 3, "normal", seed=7500 + r))
        kb.free()
        vb.free()
    finally:
        if exe.value:
            hip.hipGraphExecDestroy(exe)
        if graph.value:
            hip.hipGraphDestroy(graph)
        s.close()
