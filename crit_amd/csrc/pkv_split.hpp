// How the launches split their work: plain arithmetic over sizes, without device code, so that it can be checked apart
// from the kernels (tests/test_split.py compiles it for the host).
#pragma once
#include <stdint.h>

#ifdef __HIPCC__
#define PKV_SPLIT_FN __host__ __device__ static inline
#else
#define PKV_SPLIT_FN static inline
#endif

namespace pkv {

constexpr int kXcds = 8;      // dies with an L2 of their own; workgroups go to them round robin by linear id

// -- prompt chunks: the tiles of a (chunk, KV head) pair over the XCDs ----------------------------------------------------
// A pair's tiles read the same keys, so they belong on one XCD, unless the pairs are too few or too uneven to keep all of
// them busy: a launch of `pairs` pairs of `tiles` tiles each, a pair dealt to 1 << l XCDs, leaves its busiest XCD
// ceil(pairs << l / 8) * ceil(tiles >> l) tiles. Taken is the smallest l within a tenth of the least load: splitting
// costs the L2s another copy of the keys. Pairs that are a multiple of 8 are even as they are. `units` compute units an
// XCD, `held` workgroups it holds at once.
//   - A tenth less load is the least that measured as less time; 8 XCDs a pair is for a lone pair (more pairs of which
//     each XCD has an eighth start the later pairs' longest tiles last: 7 pairs of 64 tiles 86 -> 120 us; 5 pairs of 2,048
//     tokens after 2,048: 206 us as they are, 190 on four XCDs, 197 on eight).
//   - Where an XCD has more tiles than it holds, but none of its pairs alone, less than half a tile a compute unit is not
//     worth the copies (17 pairs of 16 tiles of 256 rows: 39 us, 42 / 48 / 45 on 2 / 4 / 8 XCDs; 33: 57, 61 / 73 / 67; 65:
//     83, 89 / 106 / 95). Half a tile is: 20 pairs of 32 tiles 144 -> 123 us, 18 pairs of 48 tiles (256 wide) 485 -> 392.
//   - Few pairs: 2 of 192 tiles (256 wide, 2,048 tokens after 2,048) 762 -> 262 us on four XCDs, 4 of 64 tiles 209 -> 129
//     on two, 1 of 128 tiles 182 -> 81 on eight. Pairs of one tile stay as they are whatever their count.
PKV_SPLIT_FN int64_t busiest_xcd(int64_t pairs, int64_t tiles, int l) {
    return ((pairs << l) + kXcds - 1) / kXcds * ((tiles + (1 << l) - 1) >> l);
}
PKV_SPLIT_FN int xcds_of_pair_log2(int64_t pairs, int64_t tiles, int64_t units, int64_t held) {
    const int most = pairs == 1 ? 3 : 2;
    const int64_t whole = busiest_xcd(pairs, tiles, 0);
    int64_t least = whole;
    for (int l = 1; l <= most; ++l) least = busiest_xcd(pairs, tiles, l) < least ? busiest_xcd(pairs, tiles, l) : least;
    int l = 0;
    while (10 * busiest_xcd(pairs, tiles, l) > 11 * least) ++l;
    if (tiles <= held && whole > held && 2 * (whole - busiest_xcd(pairs, tiles, l)) < units) l = 0;
    return l;
}
// Tiles of a pair one of its XCDs takes at most, and the workgroups of the launch.
PKV_SPLIT_FN int64_t tiles_of_share(int64_t tiles, int l) { return (tiles + (1 << l) - 1) >> l; }
PKV_SPLIT_FN int64_t dealt_workgroups(int64_t pairs, int64_t tiles, int l) {
    return tiles_of_share(tiles, l) * (((pairs << l) + kXcds - 1) / kXcds * kXcds);
}
// The pair and the tile of a workgroup; a pair from `pairs` on or a tile from `tiles` on is nobody's. Shares (a pair's
// part on one XCD) are numbered round by round, one a XCD; a pair's shares lie in one round, and which of its tiles the
// first of them takes moves on by one every round: otherwise the few tiles of short chunks all meet on the same XCDs.
// Later tiles see more keys: they start first.
struct DealtTile {
    int pair, tile;
};
PKV_SPLIT_FN DealtTile dealt_tile(uint32_t workgroup, uint32_t share_tiles, int l) {
    const uint32_t xcd = workgroup % kXcds, q = workgroup / kXcds, round = q / share_tiles;
    return DealtTile{(int)((xcd + kXcds * round) >> l),
                     (int)(((share_tiles - 1 - (q - round * share_tiles)) << l) + ((xcd + round) & ((1u << l) - 1)))};
}

// -- windows over 16-bit pages of 128-wide heads: query tiles a workgroup holds --------------------------------------------
// `tiles` of a row with every column; `full`: every row has them all, as far as the caller says; `places`: (row, KV heads
// of a wavefront, partition) triples of the launch; `units`: the card's compute units.
//   - Three tiles instead of four wherever they take no more workgroups (3, 5, 6 and 9 tiles): a step is bound by its
//     matrix and softmax work, which tiles that no row fills cost as well. 64 rows ~U[1024, 8192], 32 / 8 heads x 128,
//     BF16, three against four: 5 columns (3 tiles) 280 us against 314, 9 columns (5) 476 / 557, 12 columns (6) 494 / 582;
//     64 / 8 heads, 9 columns (9) 714 / 853.
//   - But a row of four tiles in a launch sized for five, six or nine has one workgroup of four, and two of three, each
//     of which reads the row: 56 / 8 heads, a launch of 5 columns, rows of 4: 459 us in threes, 329 in fours. So those
//     launches take threes only where every row is full, or where the launch is small enough that the second workgroup
//     runs beside the first: up to two workgroups a compute unit where a row has two of them (one row of 32,768: 66 us
//     against 77; 3 rows of 32,768, three times as many: 159 against 120), one where it has three.
PKV_SPLIT_FN int window_tiles_16bit(int64_t tiles, bool full, int64_t places, int64_t units) {
    if (tiles <= 2) return (int)tiles;
    const int64_t threes = (tiles + 2) / 3;
    if (threes != (tiles + 3) / 4) return 4;
    return threes == 1 || full || (threes - 1) * threes * places <= 2 * units ? 3 : 4;
}

// The same over 8-bit pages, for windows of three tiles or more: two tiles a workgroup, two workgroups a compute unit. Pages of
// scaled rows (a step pair has one maximum there, half the softmax and value products): three in one workgroup, one a
// compute unit, where that holds a row whole and the tables have room for more of them than two a compute unit: a row is
// then read and converted once instead of twice. 64 rows ~U[1024, 8192], 32 / 8 heads x 128, 5 columns: INT8 217 -> 189 us,
// fp8:row 216 -> 177; 16 rows of 4,600 in tables of 8,192 pages 74 -> 62. Small launches miss the second workgroup (3 rows
// of up to 4,000 in tables of their own length: 38 us in twos, 49 in threes; in tables of 8,192 pages, which the rule cannot
// tell from long rows, 53 and 57), and four tiles in one wavefront are too long a step (8 columns of one row of 50,000, 56
// / 8 heads, 99 and 126). FP8 with its multipliers gains nothing by threes (64 rows 203 and 200, 32 rows 116 and 118, 3
// rows in tables of 8,192 pages 51 and 60, 32 rows of 700 there 37 and 43).
PKV_SPLIT_FN int window_tiles_8bit(bool scaled_rows, int64_t tiles, bool full, int64_t places, int64_t units) {
    return scaled_rows && tiles == 3 && full && places > 2 * units ? 3 : 2;
}

// -- windows of two rows without a list of units: the place a workgroup takes ------------------------------------------------
// Rows of `p0` and `p1` pieces in up to `parts` partitions each (piece i in partition i % parts), `per_row` places (heads, tiles) a
// partition, by_row(x) = x / per_row, `units` compute units. Workgroups from per_row * (both rows' partitions) on have none. With
// those between the others (a row's places by the tables' partitions, the rows beside each other) the hardware, which deals
// workgroups out round by round and counts them too, left some compute units with twice the work of others. For the same
// reason workgroups `units` apart share a unit, and so:
//   - Both rows' partitions beside each other while both have them, then the longer one's others, the rows' last ones, which
//     are parts of pieces, at the end. Which row comes first changes every eight workgroups: they go to the XCDs by number, and
//     a row would be on half of the XCDs.
//   - Partitions of more pieces in one row than in the other: a row after the other. In a launch of two rounds at most the
//     shorter one first: the longest places are then the first round's last, which share with none or with the second's last
//     (where the first row takes a round by itself, the other's p % parts partitions of a piece more come last, or they would
//     share with that row's). In a longer launch the longer one first.
// 32 / 8 heads x 128, BF16 / FP8 / fp8:row / INT8, from a list of units, by the tables' partitions, and so: 2 rows of 30,000 and
// 50,000 67.5 / 41.0 / 41.0 / 43.5 us, 72 / 44.0 / 47.3 / 46.8, 63.8 / 37.5 / 38.7 / 41.0; of 10,000 and 90,000 87 / 54.2 / 56 / 56,
// 96 / 55.8 / 61 / 62, 83.5 / 51.3 / 53.8 / 53.6; of 60,000 and 100,000 131 / 72.6 / 74 / 79, 125 / 82.5 / 87 / 89, 108 / 67.5 / 70 /
// 74.5; in splits of 1,024, 30,000 and 90,000, 84 / 56 / 57.5 / 58, 95 / 60.7 / 65 / 66, 79.5 / 50.5 / 53 / 53.8; alike, 100,000 160 /
// 98.5 / 101 / 103.7, 146 / 93 / 95.5 / 98.5, 147 / 94.5 / 96 / 99.
struct RowPlace {
    int row;
    uint32_t partition, place;
};
template <typename DIV>
PKV_SPLIT_FN RowPlace row_place(uint32_t workgroup, uint32_t p0, uint32_t p1, uint32_t parts, uint32_t per_row, uint32_t units, DIV by_row) {
    const uint32_t n0 = p0 < parts ? p0 : parts, n1 = p1 < parts ? p1 : parts;
    if ((p0 > parts || p1 > parts) && p0 / parts != p1 / parts) {
        const bool two_rounds = per_row * (n0 + n1) <= 2 * units;
        const uint32_t head = (p0 < p1) == two_rounds ? 0 : 1, taken = per_row * (head ? n1 : n0);
        if (workgroup < taken) {
            const uint32_t b = by_row(workgroup);
            return RowPlace{(int)head, b, workgroup - b * per_row};
        }
        const uint32_t p = head ? p0 : p1, n = head ? n0 : n1, rest = workgroup - taken, q = by_row(rest);
        const uint32_t b = two_rounds && taken >= units && p > parts ? q + p % parts : q;
        return RowPlace{(int)(head ^ 1), b < n ? b : b - n, rest - q * per_row};
    }
    const uint32_t whole0 = n0 ? n0 - 1 : 0, whole1 = n1 ? n1 - 1 : 0, both = whole0 < whole1 ? whole0 : whole1;
    if (workgroup < 2 * per_row * both) {
        const uint32_t b = by_row(workgroup / 2), x = workgroup - 2 * per_row * b;
        return RowPlace{(int)((x >= per_row ? 1u : 0u) ^ ((b * per_row / 4) & 1u)), b, x >= per_row ? x - per_row : x};
    }
    if (workgroup < per_row * (whole0 + whole1)) {
        const uint32_t rest = workgroup - 2 * per_row * both, q = by_row(rest);
        return RowPlace{whole1 > whole0 ? 1 : 0, both + q, rest - q * per_row};
    }
    const uint32_t rest = workgroup - per_row * (whole0 + whole1);
    const bool second = !n0 || rest >= per_row;
    return RowPlace{second ? 1 : 0, second ? whole1 : whole0, rest < per_row ? rest : rest - per_row};
}

// -- merges: which value dims a wavefront's lanes take -------------------------------------------------------------------
// Side by side (a load of 8 or 16 bytes a partition in place of two or four of 4) where a wavefront's own time is the launch's;
// but 128-wide values of more than two wavefronts a compute unit with batches of 32 partitions in flight (rows of more than 8
// partitions) come 64 apart. Triples of 128-wide values of 4 / 12 / 32 partitions, side by side and 64 apart: 512 3.0 / 4.27 / 4.65 us
// and 3.1 / 4.4 / 4.8; 640 3.1 / 4.55 / 5.0 and 3.2 / 4.5 / 4.9; 896 3.2 / 4.95 / 5.45 and 3.3 / 4.6 / 5.05; 1,536 3.6 / 6.2 / 6.7 and 3.7 /
// 5.6 / 6.2; 2,016 3.85 / 6.9 / 8.0 and 3.9 / 5.95 / 7.0. 256-wide values (batches of 16) gain side by side at every size (1,512 of
// 4 / 12 / 32 4.1 / 9.4 / 19.0 and 4.3 / 9.9 / 19.7). 8 wavefronts a compute unit and more (batches of 8): 64 apart (10,240 triples of
// up to 17, behind their split launch: 276.2 us side by side, 274.5 so).
PKV_SPLIT_FN bool merge_dims_apart(int value_dim, int64_t triples, int64_t partitions, int64_t units) {
    return triples >= 8 * units || (value_dim == 128 && 2 * triples >= 5 * units && partitions > 8);
}

}   // namespace pkv
