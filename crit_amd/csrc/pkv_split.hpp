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

}   // namespace pkv
