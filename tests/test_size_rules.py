"""The library's rules on sizes, compiled for the CPU."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def rule(tmp_path_factory):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ not found")
    exe = tmp_path_factory.mktemp("rules") / "size_rules"
    subprocess.run([gxx, "-O1", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    os.path.join(ROOT, "tests", "native", "size_rules.cpp"), "-o", str(exe)],
                   check=True, capture_output=True)

    def call(name, *args):
        r = subprocess.run([str(exe), name, *map(str, args)], capture_output=True, text=True, check=True)
        v = [int(x) for x in r.stdout.split()]
        return v[0] if len(v) == 1 else v
    return call


# sub-cells of these tile counts, chunk length, keys a pair
@pytest.mark.parametrize("tiles,tch,kp", [([64] * 98, 16, 10), ([64] * 98, 32, 16), ([64] * 98, 48, 32),
                                          ([96, 33, 64, 1] * 40, 16, 10), ([64] * 20, 16, 10),
                                          ([500] + [3] * 60, 48, 32), ([64] * 900, 65536, 10), ([16] * 70, 16, 10)])
def test_first_pairs_hold_what_the_queries_reach(rule, tiles, tch, kp):
    """Queries that reach every sub-cell, or the longest half of them: their
    chunks and the seed's fit the first lists, also (short of the size that is
    quick to free) if the queries looked at reach a sixth less than the others."""
    Q, n, seed_tiles = 300, 64, 16
    for reached in (sorted(tiles)[len(tiles) // 2:], tiles):
        chunks = sum(-(-t // tch) for t in reached)
        seed = -(-max(tiles) // seed_tiles)
        assert Q * (chunks + seed) <= rule("first_pairs", Q, n * chunks, n, max(tiles), seed_tiles, kp)
        if Q * (chunks + seed) * kp * 8 <= 64 << 20:
            less = n * chunks * 5 // 6 + 1
            assert Q * (chunks + seed) <= rule("first_pairs", Q, less, n, max(tiles), seed_tiles, kp) + Q


def test_first_pairs_are_bounded(rule):
    """64 pairs a query at least, one GiB of partial results at most, the
    former where they conflict."""
    assert rule("first_pairs", 1000, 0, 64, 96, 16, 10) == 64_000
    assert rule("first_pairs", 1000, 64 * 40, 64, 96, 16, 10) == 64_000
    assert rule("first_pairs", 4000, 64 * 180, 64, 72, 16, 10) * 10 * 8 <= 64 << 20
    assert rule("first_pairs", 4000, 64 * 220, 64, 72, 16, 10) == 4000 * 225 * 6 // 5
    assert rule("first_pairs", 50_000, 64 * 400, 64, 96, 128, 32) * 32 * 8 == 1 << 30
    assert rule("first_pairs", 200_000, 64 * 400, 64, 96, 128, 32) == 200_000 * 64


@pytest.mark.parametrize("half", [0, 1])
def test_float_items_are_whole_where_many_and_even(rule, half):
    """Whole sub-cells from 14001 items up if none is more than twice the
    mean, chunks of 128 tiles for binary16 rows if the longest has 512, of 48
    otherwise."""
    whole, chunk = 65536, 48
    assert rule("float_item_tiles", half, 1024, 62500, 511, 10_000) == chunk
    assert rule("float_item_tiles", half, 1024, 62500, 512, 10_000) == (128 if half else chunk)
    assert rule("float_item_tiles", half, 100, 62500, 977, 6400) == chunk
    assert rule("float_item_tiles", half, 140, 140 * 64, 96, 6400) == chunk
    assert rule("float_item_tiles", half, 140, 140 * 64, 96, 6401) == whole
    assert rule("float_item_tiles", half, 976, 976 * 64, 128, 10_000) == whole
    assert rule("float_item_tiles", half, 976, 976 * 64, 129, 10_000) == chunk
    assert rule("float_item_tiles", half, 976, 976 * 64, 96, 64) == chunk


@pytest.mark.parametrize("D,dim,elem", [(4, 64, 1), (100, 128, 1), (100, 128, 4), (264, 512, 2), (520, 768, 2)])
def test_pad_records_leave_room_for_the_index(rule, D, dim, elem):
    """Records at a padded dimension are made only where a full graph of 64
    edges a row, the largest array behind them, and its scratch still fit."""
    N = 1_000_000
    rec = N // 16 * (dim * 16 * elem + 16 * 4 * 4)   # rows, norms, row ids and attribute words
    assert rule("pad_records_fit", rec, 5 * rec) == 1
    assert rule("pad_records_fit", rec, 5 * rec - 1) == 0
    for free in (rec, rec + 260 * N - 1):
        assert rule("pad_records_fit", rec, free) == 0 or free - rec >= 260 * N
