"""The bucket path's kernels on the CPU emulator against the oracle: small blocks
and tiles, so that a few thousand keys fill many buckets; one wave at a time,
which turns a missing barrier into a wrong result; the sanitizers; a region
that overflows."""
import os
import subprocess

import pytest

from test_cpu_emulation import emulator, pytestmark, run_cases  # noqa: F401

CASES = [
    # one block: every op and key width, one key more than the rows of a wave,
    # few values, quantised and special floats, every key equal
    "one_sort:u32:500:uniform:1", "one_sort:f32:768:few:2", "one_argsort:u32:300:few:3", "one_pairs:f64:512:uniform:4",
    "one_sort:i64:511:uniform:5", "one_sort:u32:2:uniform:6", "one_sort:u64:400:low12:7", "one_argsort:i32:65:same:8",
    # buckets: uniform, few values (buckets of one value larger than a block),
    # skewed, narrow, equal keys; look-back over many tiles
    "bk_sort:u32:3000:uniform:9", "bk_sort:u32:3000:few:10", "bk_sort:i64:2000:uniform:11", "bk_argsort:f32:2000:few:12",
    "bk_pairs:u64:1500:uniform:13", "bk_pairs:u32:3000:zipf:14", "bk_argsort:f64:3000:low12:15", "bk_sort:f64:3000:same:16",
    "bk_argsort:u32:5000:same:17", "bk_sort:u32:64:uniform:18", "bk_offset:f32:3001:uniform:19",
    # few buckets of many keys: blocks that sort theirs through device memory
    "bk2_sort:u32:5000:uniform:20", "bk2_pairs:f64:4000:few:21", "bk2_argsort:u32:4000:uniform:22",
]
# two levels: uniform, buckets and children of one value, larger than a block,
# the least size; the digit passes for one, two and no varying digit; a sample
# that shows two digits of eight
TWO = [
    "two_sort:u64:9000:uniform:1", "two_sort:i64:6000:uniform:2", "two_pairs:u64:6000:uniform:3",
    "two_argsort:f64:9000:uniform:4", "two_sort:f64:9000:few:5", "two_pairs:f64:9000:few:6", "two_sort:u64:64:uniform:10",
    "two2_sort:i64:9000:uniform:12", "two2_argsort:u64:12000:uniform:13",
    "two_sort:u64:5000:same:8", "two_argsort:i64:5000:same:9", "two_argsort:u64:9000:low12:14", "two_pairs:u64:5000:byte0:3",
    "two_sort:u64:5000:byte1:3", "two_pairs:u64:9000:lone:1", "two_sort:i64:9000:lone:1",
]


def test_emulated_buckets(emulator):  # noqa: F811
    run_cases("small", CASES + TWO, parallel=4)
    run_cases("prod", ["two4_sort:f64:60000:uniform:6", "two4_pairs:u64:50000:lone:7", "one_sort:u32:8192:uniform:1", "one_pairs:f64:6144:few:2", "bk_sort:u32:40000:uniform:3",
                       "bk_argsort:f32:30000:few:4", "bk_pairs:u64:20000:zipf:5"], parallel=3, env={"EMU_CUS": "8"})


def test_emulated_buckets_of_repeated_values(emulator):  # noqa: F811
    """Evenly spaced values, each in a group of the sample's own, so that a
    bucket between two splitters can hold two of them: no region of either
    level overflows (256 values each of a bucket: steps384 of two buckets)."""
    run_cases("prod", ["two_sort:f64:200000:steps256:1", "two_pairs:f64:200000:tenths190:2",
                       "two_sort:u64:200000:steps192:1", "two_argsort:i64:200000:steps256:1",
                       "two1_sort:f64:850000:steps384:2", "two1_sort:u64:850000:steps384:3",
                       "bk_sort:u32:200000:steps400:1", "bk_pairs:u64:200000:steps300:2"], parallel=4, env={"EMU_CUS": "8"})


SAMPLES = ["bk_sort:u64:3000:records:1", "bk_argsort:u64:3000:records:2", "bk_pairs:i64:3000:cluster:3",
           "two_sort:u64:9000:records:4", "two_pairs:u64:6000:cluster:5", "bk2_sort:u64:4000:cluster:6"]


def test_emulated_crowded_samples(emulator):  # noqa: F811
    """Samples of 64-bit keys that their top bits do not order: splitters from
    the top bits alone, or, where quantiles share them, from all bits."""
    run_cases("small", SAMPLES, parallel=2)
    run_cases("small", SAMPLES, env={"EMU_SCHED": "wave"}, parallel=2)
    run_cases("prod", ["bk_argsort:u64:60000:records:1", "bk_sort:u64:60000:cluster:2", "two_pairs:u64:100000:records:3",
                       "two_sort:u64:100000:cluster:4"], parallel=4, env={"EMU_CUS": "8"})


@pytest.mark.parametrize("order", ["wave", "wave_rev"])
def test_emulated_buckets_wave_serial(emulator, order):  # noqa: F811
    run_cases("small", CASES + TWO, timeout=900, env={"EMU_SCHED": order}, parallel=4)


def test_emulated_buckets_overflow(emulator):  # noqa: F811
    """A region with room for one row only: its keys do not fit, and every
    bucket's block gathers its keys from the caller's instead (the
    fault-injection build): every op, few values, buckets larger than a block
    and of one value, an odd start."""
    run_cases("faults", ["bkover_sort:u32:3000:uniform:1", "bkover_pairs:u64:2000:few:2", "bkover_argsort:f32:3000:uniform:3",
                         "bkover_sort:i64:2000:uniform:4", "bkover_pairs:f64:3001:uniform:5", "bkover_sort:f32:3000:few:6",
                         "bkover_argsort:u64:3000:few:1", "bkover2_sort:u32:5000:uniform:2", "bkover2_pairs:u64:5000:uniform:3",
                         "bkover2_argsort:i32:5000:few:3", "bkover_pairs:u32:5000:zipf:9", "bkover_sort:u32:5000:zipf:9",
                         "bkover_offset:i64:3001:uniform:7",
                         # two levels: of the first (every bucket gathered by its block) or of every bucket's second child
                         "twoover_sort:u64:9000:uniform:1", "twoover_pairs:u64:6000:few:3", "twoover_argsort:f64:9000:uniform:2",
                         "twoover2_sort:i64:9000:uniform:5", "twoover_pairs:f64:9000:uniform:6", "twoover_sort:f64:9000:few:1",
                         "twosecond_sort:u64:9000:uniform:3", "twosecond_pairs:f64:9000:uniform:4"],
              env={"EMU_WORKERS": "1", "EMU_XCDS": "1"})   # (tiles in order: this build soon gives up a look-back wait)


def test_emulated_paths_by_size(emulator):  # noqa: F811
    """The product's limits: one block, one level of buckets, two (k / 255, whose
    regions must hold), the digit passes beyond; capture and the static scratch."""
    run_cases("limits", ["size1_sort:u32:8192:uniform:1", "size2_sort:u32:8193:few:2", "size1_pairs:i64:6144:few:3",
                         "size2_argsort:f64:6145:uniform:4", "size2_pairs:f32:20001:uniform:5", "size0_sort:f32:190001:uniform:6",
                         "size3_sort:f64:1600000:steps256:1", "capture:u32:20000:uniform:7", "capture:f64:20000:uniform:8",
                         "noalloc:i32:9000:few:9", "noalloc:u64:6000:uniform:10"], parallel=4, env={"EMU_CUS": "8"})


@pytest.mark.parametrize("kind", ["u32", "i32", "f32", "u64", "i64", "f64"])
def test_reserve_holds_smaller_sorts(emulator, kind):  # noqa: F811
    """fs_reserve(n), then captured sorts of every smaller size, by the
    product's limits: paths, tiles and regions change with the size, and none
    may need more scratch than was reserved."""
    run_cases("limits", [f"reserve:{kind}:4294967295:uniform:1"], env={"EMU_CUS": "256"})


def test_buckets_without_memory(emulator):  # noqa: F811
    """The bucket path needs more scratch than the digit passes: where that
    much cannot be had they sort instead, by the product's limits (one level
    for u32 and i64, two for f64)."""
    run_cases("limits", ["memory:u32:590000:uniform:1", "memory:i64:990000:uniform:2", "memory:f64:1600000:uniform:3"],
              env={"EMU_CUS": "256"}, parallel=3)


def test_emulated_buckets_sanitizers(emulator):  # noqa: F811
    libasan = subprocess.run(["g++", "-print-file-name=libasan.so"], capture_output=True, text=True).stdout.strip()
    if not os.path.isabs(libasan):
        pytest.skip("libasan not found")
    run_cases("san", CASES[::2] + TWO[::2], timeout=600, env={"LD_PRELOAD": libasan, "EMU_NO_SEGV_HANDLER": "1", "EMU_CUS": "4",
                                                  "ASAN_OPTIONS": "detect_leaks=0:detect_stack_use_after_return=0"}, parallel=3)
