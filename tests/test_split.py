"""The launches' splits (crit_amd/csrc/pkv_split.hpp, compiled here for the host): every piece of work is somebody's, once,
and no XCD is left with much more of it than the others."""
import ctypes
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
UNITS = 32      # compute units an XCD


@pytest.fixture(scope="module")
def split(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("no g++")
    where = tmp_path_factory.mktemp("split")
    (where / "split.cpp").write_text("""#include "pkv_split.hpp"
extern "C" int xcds_log2(int64_t pairs, int64_t tiles, int64_t units, int64_t held) { return pkv::xcds_of_pair_log2(pairs, tiles, units, held); }
extern "C" int64_t workgroups(int64_t pairs, int64_t tiles, int l) { return pkv::dealt_workgroups(pairs, tiles, l); }
extern "C" int window_tiles(int64_t tiles, int full, int64_t places, int64_t units) { return pkv::window_tiles_16bit(tiles, full != 0, places, units); }
extern "C" int window_tiles_8bit(int scaled, int64_t tiles, int full, int64_t places, int64_t units) { return pkv::window_tiles_8bit(scaled != 0, tiles, full != 0, places, units); }
extern "C" int apart(int value_dim, int64_t triples, int64_t partitions, int64_t units) { return pkv::merge_dims_apart(value_dim, triples, partitions, units); }
extern "C" void rows(uint32_t workgroups, uint32_t p0, uint32_t p1, uint32_t parts, uint32_t per_row, int* row, uint32_t* partition, uint32_t* place) {
    for (uint32_t w = 0; w < workgroups; ++w) {
        const pkv::RowPlace at = pkv::row_place(w, p0, p1, parts, per_row, 256, [=](uint32_t x) { return x / per_row; });
        row[w] = at.row, partition[w] = at.partition, place[w] = at.place;
    }
}
extern "C" void deal(int64_t pairs, int64_t tiles, int l, int* pair, int* tile) {
    const int64_t n = pkv::dealt_workgroups(pairs, tiles, l);
    for (int64_t w = 0; w < n; ++w) {
        const pkv::DealtTile d = pkv::dealt_tile((uint32_t)w, (uint32_t)pkv::tiles_of_share(tiles, l), l);
        pair[w] = d.pair, tile[w] = d.tile;
    }
}
""")
    out = str(where / "split.so")
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-O1", "-shared", "-fPIC", "-I", os.path.join(ROOT, "crit_amd", "csrc"),
                    str(where / "split.cpp"), "-o", out], check=True)
    lib = ctypes.CDLL(out)
    lib.xcds_log2.argtypes, lib.workgroups.argtypes = [ctypes.c_int64] * 4, [ctypes.c_int64, ctypes.c_int64, ctypes.c_int]
    lib.window_tiles.argtypes = [ctypes.c_int64, ctypes.c_int, ctypes.c_int64, ctypes.c_int64]
    lib.window_tiles_8bit.argtypes = [ctypes.c_int, ctypes.c_int64, ctypes.c_int, ctypes.c_int64, ctypes.c_int64]
    lib.workgroups.restype = ctypes.c_int64
    lib.apart.argtypes = [ctypes.c_int, ctypes.c_int64, ctypes.c_int64, ctypes.c_int64]
    lib.rows.argtypes = [ctypes.c_uint32] * 5 + [ctypes.c_void_p] * 3
    lib.deal.argtypes = [ctypes.c_int64, ctypes.c_int64, ctypes.c_int, ctypes.c_void_p, ctypes.c_void_p]
    return lib


def dealt(split, pairs, tiles, l):
    """[(xcd, pair, tile)] of the launch's workgroups that have one."""
    n = split.workgroups(pairs, tiles, l)
    pair, tile = (ctypes.c_int * n)(), (ctypes.c_int * n)()
    split.deal(pairs, tiles, l, pair, tile)
    return [(w % 8, pair[w], tile[w]) for w in range(n) if pair[w] < pairs and tile[w] < tiles]


def test_every_tile_of_every_pair_is_dealt_once(split):
    for pairs in list(range(1, 35)) + [63, 64, 65, 66, 70]:
        for tiles in (1, 2, 3, 7, 8, 9, 16, 33, 73):
            for l in range(4):
                work = dealt(split, pairs, tiles, l)
                assert sorted((p, t) for _, p, t in work) == [(p, t) for p in range(pairs) for t in range(tiles)], (pairs, tiles, l)


@pytest.mark.parametrize("held", [UNITS, 2 * UNITS])
def test_the_busiest_xcd_has_no_more_than_with_whole_pairs(split, held):
    for pairs in range(1, 71):
        for tiles in (1, 2, 3, 7, 8, 9, 10, 16, 32, 48, 64, 73, 128, 192):
            l = split.xcds_log2(pairs, tiles, UNITS, held)
            whole = -(-pairs // 8) * tiles
            load = [0] * 8
            for xcd, _, _ in dealt(split, pairs, tiles, l):
                load[xcd] += 1
            assert max(load) <= whole and (l == 0 or 10 * max(load) <= 11 * whole)
            assert split.workgroups(pairs, tiles, l) <= -(-pairs // 8) * 8 * tiles      # no wider a launch than with whole pairs
            assert l == 0 or (pairs % 8 != 0 and tiles > 1)
    # a few pairs fill the card
    assert [split.xcds_log2(n, 64, UNITS, held) for n in (1, 2, 4, 8)] == [3, 2, 1, 0]


@pytest.mark.parametrize("pairs", [1, 2, 4, 9, 18, 20, 33, 63, 66])
@pytest.mark.parametrize("live", [1, 2, 3])
def test_short_chunks_of_a_long_launch_do_not_meet_on_one_xcd(split, pairs, live):
    # the launch is sized for its longest chunk; the others' few tiles are spread over the XCDs however their pairs are dealt
    for tiles in (16, 48):
        for l in range(4):
            load = [0] * 8
            for xcd, _, tile in dealt(split, pairs, tiles, l):
                load[xcd] += tile < live
            assert max(load) <= -(-pairs // 8) * live, (tiles, l, load)


@pytest.mark.parametrize("pairs,tiles,held", [(17, 16, 32), (21, 16, 32), (33, 16, 32), (65, 16, 32), (63, 1, 64), (66, 1, 64), (7, 64, 32), (64, 8, 32)])
def test_many_even_pairs_and_short_chunks_stay_whole(split, pairs, tiles, held):
    assert split.xcds_log2(pairs, tiles, UNITS, held) == 0


def test_a_row_of_four_tiles_is_not_read_twice_in_a_large_launch(split):
    # 64 rows of 4 head pairs and 16 partitions on 256 compute units: a launch sized for 5, 6 or 9 tiles whose rows may have
    # fewer keeps them four a workgroup; where every row has them all, three hold them in as few workgroups
    for tiles in range(1, 33):
        for full in (0, 1):
            for places in (1, 16, 128, 256, 257, 4096):
                held = split.window_tiles(tiles, full, places, 256)
                assert held == min(tiles, 2) if tiles < 3 else held in (3, 4)
                assert tiles < 3 or -(-tiles // held) == -(-tiles // 4)      # never more workgroups for full rows
                if not full and places > 256:
                    for row in range(1, tiles + 1):      # a row of fewer tiles: no more workgroups than four a workgroup
                        assert -(-row // held) <= max(1, -(-row // 4)) or tiles < 3, (tiles, row)
    assert [split.window_tiles(t, 1, 4096, 256) for t in (3, 4, 5, 6, 7, 8, 9, 10)] == [3, 4, 3, 3, 4, 4, 3, 4]
    assert [split.window_tiles(t, 0, 4096, 256) for t in (3, 4, 5, 6, 7, 8, 9, 10)] == [3, 4, 4, 4, 4, 4, 4, 4]
    # one row of 4 head pairs and 64 partitions: its second workgroups run beside its first
    assert [split.window_tiles(t, 0, 256, 256) for t in (5, 6, 9)] == [3, 3, 4] and split.window_tiles(9, 0, 42, 256) == 3


def test_8_bit_windows_of_three_tiles(split):
    # three in one workgroup only where they are a whole full row of scaled rows in a launch past two workgroups a compute unit;
    # FP8 with its multipliers goes in twos whatever the tables have room for (3 rows in tables of 8,192 pages: 1,536 places)
    for tiles in range(2, 10):
        for full in (0, 1):
            for places in (1, 511, 512, 513, 1536, 1 << 20):
                assert split.window_tiles_8bit(0, tiles, full, places, 256) == 2
                assert split.window_tiles_8bit(1, tiles, full, places, 256) == (3 if tiles == 3 and full and places > 512 else 2)


@pytest.mark.parametrize("per_row", [1, 2, 3, 4, 5, 8, 14, 16, 28])
@pytest.mark.parametrize("parts", [1, 64, 1000])
def test_two_rows_without_a_list(split, per_row, parts):
    for p0, p1 in ((0, 0), (1, 0), (0, 1), (40, 0), (0, 17), (1, 1), (59, 64), (64, 59), (20, 33), (7, 59), (64, 64), (30, 88), (88, 30), (196, 196), (1, 200),
                   (118, 196), (196, 40), (40, 66), (128, 64), (64, 128), (0, 70), (70, 0)):
        n0, n1 = min(p0, parts), min(p1, parts)
        live = per_row * (n0 + n1)
        row, partition, place = (ctypes.c_int * live)(), (ctypes.c_uint32 * live)(), (ctypes.c_uint32 * live)()
        split.rows(live, p0, p1, parts, per_row, row, partition, place)
        units = list(zip(row, partition, place))
        # every unit of both rows once, on the first workgroups, none without work between them
        assert sorted(units) == [(r, b, x) for r, n in ((0, n0), (1, n1)) for b in range(n) for x in range(per_row)], (p0, p1)
        for r in (0, 1):      # a row is on every XCD alike
            load = [0] * 8
            for w in range(live):
                load[w % 8] += row[w] == r
            assert max(load) - min(load) <= 12, (p0, p1, load)
        pieces = [(p0, p1)[r] // parts + (b < (p0, p1)[r] % parts) for r, b, _ in units]
        if max(p0, p1) <= parts:      # the rows' last partitions end the launch
            assert all(b == (n0, n1)[r] - 1 for r, b, _ in units[live - per_row * (bool(n0) + bool(n1)):])
        elif live <= 512 and p0 // parts != p1 // parts:      # two of the longest share a compute unit only where no shorter one is alone
            worst = max((a + b for a, b in zip(pieces, pieces[256:])), default=0)
            assert worst < 2 * max(pieces) or min(pieces[:256]) == max(pieces), (p0, p1)


def test_merges_of_many_long_rows_take_their_dims_apart(split):
    # 128-wide values: 20 to 63 rows of 32 heads and more than 8 partitions; small launches, few partitions and 256-wide values do not
    assert all(split.apart(128, rows * 32, parts, 256) for rows in (20, 32, 63, 64, 128) for parts in (9, 17, 64))
    assert not any(split.apart(128, rows * 32, parts, 256) for rows in (1, 16, 19) for parts in (4, 17, 64))
    assert not any(split.apart(128, rows * 32, parts, 256) for rows in (20, 63) for parts in (1, 4, 8))
    assert not any(split.apart(256, triples, 64, 256) for triples in (24, 640, 2047))
