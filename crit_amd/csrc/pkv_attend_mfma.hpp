// Paged decode / verify-window attention for 128-wide heads over pages of a multiple of 16 positions: the bandwidth
// path of the split and fused launches.
//
// The kernel is bound by HBM reads of K and V; everything else is arranged so that nothing but those reads limits it.
// The two products of a step run on the matrix pipe, which a decode kernel otherwise leaves idle, because the vector
// pipe cannot keep up with 8-bit pages at HBM rate (one v_dot2 per two multiply-adds, plus the conversions, was two
// thirds of its cycles): a step is 16 positions of one KV head, and steps are taken in pairs,
//   S^T[16 positions][16 query rows] = K[16][128] . Q^T      4 x v_mfma_f32_16x16x32 a step (bf16 / f16 operands)
//   O^T[128 dims][16 query rows]    += V^T[128][16] . P^T    8 x v_mfma_f32_16x16x16 a step, or
//                                   += V^T[128][32] . P^T    8 x v_mfma_f32_16x16x32 a pair (pages of scaled rows)
// with operands laid out so that nothing is shuffled between the two products:
//   keys    lane (p = lane % 16, u = lane / 16) holds 16-byte pieces of the row of position p; piece c holds dims
//           32 c + 8 u .. + 7, the eight contraction elements the first product's A operand wants from that lane
//           (8-bit pages: two pieces of 16 codes, converted to 16-bit pairs, exactly);
//   scores  come out with lane (c = lane % 16, u) holding query row c at positions 4 u .. 4 u + 3, which is the B operand
//           of a step's second product, or half of a pair's: the probabilities go from the softmax to the matrix pipe as
//           packed registers, no LDS, no shuffle;
//   values  lane (i, u) holds a dim of the rows of positions 4 u .. 4 u + 3 of a step, as two 16-bit pairs.
// Which of the two: G, below.
// The 16 query rows of a tile are rows of the flattened (column, group head) list, so the GQA group's heads share
// every K/V byte read once. A wavefront serves HW adjacent KV heads (2 where the head count is even) in ONE matrix tile:
// a step is then 8 positions of both heads (rows 0 .. 7 of the tile the first head's positions, rows 8 .. 15 the
// second's, columns 0 .. 7 the first head's query rows, 8 .. 15 the second's; the products of one head's keys with the
// other head's queries are masked), so a load instruction fetches both heads' rows of a position, 512 contiguous bytes
// of 16-bit pages: what the HBM system streams best from randomly placed pages.
// Softmax state: the running maximum of a query row is kept equal in the four lanes that hold the row (two
// v_permlane swaps a maximum), the sums per lane until the unit's end.
//
// How a step's rows reach their operands. With one or two query tiles over 16-bit pages a wavefront loads them straight
// into the operands' registers, a pair in flight beside the one in use, two workgroups a compute unit. A key operand's lanes
// lie in 16 different rows, so such a load is 64 requests of 16 bytes to the cache instead of 16 of 64 (5.7 requests a
// 128-byte line over the kernel, by its counters), and the registers of several tiles, of 256-wide heads or of converted
// codes leave no room for loads in flight. So all other kernels have the memory pipe write a wavefront's rows into its
// own ring in LDS (global_load_lds: no register holds them, a request takes 64 adjacent bytes) and read the operands from
// there, values transposed by the LDS itself (ds_read_b64_tr_b16). Nothing is shared between wavefronts, so no barrier
// orders the ring: the waits count loads. Against the same kernels with all rows in registers: 64 rows ~U[1024, 8192], 32
// / 8 heads x 128, 5 columns BF16 331 -> 284 us; 8 rows of 16,000, 24 / 4 x 256, fp8:row 74 -> 67; one row of 50,000, 56 /
// 8, 8 columns, INT8 116 -> 98.
//
// Row-exactness: position n is always read in the same step of the same pair of the same wavefront of its unit (pairs do
// not cross pieces), at the same place of the matrix operands; the matrix pipe computes each output element from its own row and column only; every other
// reduction is a fixed tree. So a column's bits depend on its own query and keys, `piece`, `partitions`, the page kind
// and the cache geometry only: not on the rows beside it, the launch's width, the tile it falls in, which workgroup
// served it, or `fused`.
#pragma once
#include "pkv_attend_args.hpp"
#include "pkv_dma.hpp"
#include "pkv_split.hpp"

namespace pkv {

template <bool F16>
PKV_DEV f32x4 mfma_k32(u32x4 a, u32x4 b, f32x4 c) {
    if constexpr (F16) {
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
    } else {
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
    }
}
template <bool F16>
PKV_DEV f32x4 mfma_k16(u32x2 a, u32x2 b, f32x4 c) {
    typedef __attribute__((ext_vector_type(4))) short s16x4;
    typedef __attribute__((ext_vector_type(4))) _Float16 f16x4;
    if constexpr (F16) {
        return __builtin_amdgcn_mfma_f32_16x16x16f16(__builtin_bit_cast(f16x4, a), __builtin_bit_cast(f16x4, b), c, 0, 0, 0);
    } else {
        return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(__builtin_bit_cast(s16x4, a), __builtin_bit_cast(s16x4, b), c, 0, 0, 0);
    }
}

// The values of one step, or of a pair's two, as the second product's operand: two 16-bit pairs a step.
template <bool F16>
PKV_DEV f32x4 mfma_steps(const uint32_t (&a)[2], const uint32_t (&b)[2], f32x4 c) { return mfma_k16<F16>(u32x2{a[0], a[1]}, u32x2{b[0], b[1]}, c); }
template <bool F16>
PKV_DEV f32x4 mfma_steps(const uint32_t (&a)[4], const uint32_t (&b)[4], f32x4 c) {
    return mfma_k32<F16>(u32x4{a[0], a[1], a[2], a[3]}, u32x4{b[0], b[1], b[2], b[3]}, c);
}

template <bool F16>
PKV_DEV uint32_t pair16(float a, float b) {      // two FP32 values as one 16-bit pair, round to nearest even
    if constexpr (F16) return pack_f16(a, b);
    typedef __attribute__((ext_vector_type(2))) __bf16 pair_t;
    const pair_t r = {(__bf16)a, (__bf16)b};
    return __builtin_bit_cast(uint32_t, r);
}

// Four codes of one word as two packed 16-bit pairs (x: codes 0,1; y: codes 2,3), exactly.
template <int KIND>
PKV_DEV u32x2 codes4_to_pairs(uint32_t w) {
    if constexpr (KIND == 3) {
        const float f0 = (float)(int8_t)w, f1 = (float)(int8_t)(w >> 8), f2 = (float)(int8_t)(w >> 16), f3 = (float)(int8_t)(w >> 24);
        return u32x2{__builtin_amdgcn_perm(f2u(f1), f2u(f0), 0x07060302), __builtin_amdgcn_perm(f2u(f3), f2u(f2), 0x07060302)};
    } else {
        return u32x2{__builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8((int)w, 1.0f, false)),
                     __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8((int)w, 1.0f, true))};
    }
}

// The maximum (sum) of x over the four lanes 16 apart that hold one tile column: two v_permlane swaps.
PKV_DEV float max_across_quarters(float x) {
    const int v = (int)f2u(x);
    auto a = __builtin_amdgcn_permlane16_swap(v, v, false, false);      // rows (0,1) and (2,3) meet
    const float y = __builtin_fmaxf(u2f((uint32_t)a[0]), u2f((uint32_t)a[1]));
    const int w = (int)f2u(y);
    auto b = __builtin_amdgcn_permlane32_swap(w, w, false, false);      // halves meet
    return __builtin_fmaxf(u2f((uint32_t)b[0]), u2f((uint32_t)b[1]));
}
PKV_DEV float sum_across_quarters(float x) {      // (row 0 + row 1) + (row 2 + row 3), the same bits in all four lanes
    const int v = (int)f2u(x);
    auto a = __builtin_amdgcn_permlane16_swap(v, v, false, false);
    const float y = u2f((uint32_t)a[0]) + u2f((uint32_t)a[1]);
    const int w = (int)f2u(y);
    auto b = __builtin_amdgcn_permlane32_swap(w, w, false, false);
    return u2f((uint32_t)b[0]) + u2f((uint32_t)b[1]);
}

typedef float f32x4_any __attribute__((ext_vector_type(4), aligned(4)));      // four floats of a workspace that is any floats

struct Tile {      // a step in registers (16-bit pages, 128-wide heads)
    u32x4 k[4];      // the lane's pieces of its position's key row
    u32x4 v[4];      // the lane's 8 dims of the value rows of its quarter's four positions
};

// Piece c of a lane's key row as the first product's A operand: 16-bit values as they are, codes as 16-bit pairs, exactly.
template <int KIND>
PKV_DEV u32x4 key_operand(const u32x4* k, int c) {
    if constexpr (KIND == 0) {
        return k[c];
    } else {
        const uint32_t w0 = c % 2 ? k[c / 2].z : k[c / 2].x, w1 = c % 2 ? k[c / 2].w : k[c / 2].y;
        const u32x2 lo = codes4_to_pairs<KIND>(w0), hi = codes4_to_pairs<KIND>(w1);
        return u32x4{lo.x, lo.y, hi.x, hi.y};
    }
}

// Launches without a list of units, a workgroup a place of the tables (the launcher's rule): with more of its steps in flight, or as
// the list's; of two rows, the place by row_place() (a kernel of its own: with both in one, a lone row's window of two tiles of INT8
// pages took 97.6 us in place of 96.8).
constexpr int kPlacesNone = 0, kPlacesDeep = 1, kPlacesPlain = 2, kPlacesTwo = 3;
constexpr int kMaskNone = 0, kMaskTree = 1, kMaskSliding = 2;
constexpr int kTileRows = 16;      // query rows (columns of S^T) a tile holds
constexpr int kLdsRows = 512;      // batch rows whose descriptors a workgroup keeps in LDS (the others are read from memory)

// Workgroups a compute unit holds where one or two tiles a wavefront leave the registers for them. Measured on MI355X:
// three of them (fewer registers each) and four steps in flight a wavefront both stream less (the memory system is
// saturated by two and two; more concurrent streams cost DRAM locality).
constexpr int kMfmaWaves = 2;

// Where a kernel keeps the steps in flight. 16-bit pages of 128-wide heads with one query tile or two: in registers, two
// workgroups a compute unit. Everything else: in LDS, sent there by the memory pipe itself (a ring of a wavefront's own).
// DEEP: the same in a launch of no more units than compute units, which has LDS and time to spare: no second workgroup hides
// a wavefront's wait for its one pair in flight, so it has two, in a ring, and its queries before its rows; and a unit's place
// is the workgroup's, which reads that one row's numbers and makes no list (3 rows of 3,584, 32 / 8 heads, from a graph: 19.7
// -> 15.7 us, 1.0 of it the list; of 512 18.4 -> 13.9; one row of 512 16.9 -> 12.5). A lone wavefront issues an instruction
// every four clocks, so what the list's kernels keep in spilled scalar registers shows as well: FP8 29.2 -> 24.8 us, of 512
// 14.9 -> 11.6 (four pairs in flight beside the list: 28.2).
template <int KIND, int DH, int QT, int PLACES>
struct MfmaShape {
    static constexpr bool DEEP = PLACES == kPlacesDeep;
    static constexpr bool kRing = KIND != 0 || DH == 2 || QT > 2 || DEEP;
    static constexpr int kGroups = DH == 2 || QT > 2 || DEEP ? 1 : kMfmaWaves;      // workgroups a compute unit
    static constexpr int kPairs = kRing && kGroups == 1 && !(DH == 2 && KIND == 0) ? 2 : 1;      // pairs of steps in flight a wavefront
};

// The launch: as many workgroups as the card holds at once, each working through units of the list (row, KV head
// group, query tile, partition) until it is exhausted. The hardware's own dispatcher binds a workgroup to an XCD by its
// id and starts workgroups strictly in order, so with units as uneven as ragged contexts make them it leaves slots
// idle behind a busy one; resident workgroups that pull the next unit themselves from the launch's counter (the
// caller's memory) keep every slot busy to the end. A workgroup knows its next unit while it works on the current one
// (its first two units are its index and that plus the grid; a ticket names the unit after the next): the next unit's
// page table entries are requested before the current unit's steps, its first keys, values and queries right after the
// current unit's last step, so the current unit's fold, its partials' stores and the draw of the following ticket
// happen while the next unit's rows are already on their way. A drawn unit without work (the list is a grid over rows
// of different lengths) is passed over by the drawing thread at once. The last workgroup to finish zeroes the counters
// for the next launch that uses them. Without counters the units are dealt in turn.
// MASK: what hides positions of a column beside its own end: nothing, a draft tree, or a sliding window (with or
// without a tree). Trees and windows are kernels of their own: a tree's short mask (in the step) is of no use to a
// window, whose kernels it cost registers and time (when all rows went through registers: 64 rows ~U[1024, 8192], 32 / 8
// heads, a window of 1,024, 3 columns: BF16 174 us in one kernel, 154 apart, INT8 194 and 184; a tree's kernels without a
// window, INT8, 5 columns, 305 -> 283).
// DH: 128-wide halves of a head (1: heads of 128; 2: heads of 256, whose rows
// are 512 bytes of 16-bit pages by themselves, so a wavefront serves one KV head: HW 1): twice the key pieces, query
// pieces, score products and output tiles, the same layouts otherwise; twice the registers too, so one workgroup a
// compute unit, which keeps as many bytes in flight as two of the narrower ones (a step's rows are twice as long).
// QT: query tiles a wavefront holds (windows of several columns, wide GQA groups): a step's keys and values, once in
// the registers, are multiplied with each tile's queries and probabilities in turn, every tile with its own softmax
// state and accumulators, so a tile's bits are what they are alone and the rows are read once for QT tiles instead of
// once a tile. More than one tile takes the registers of a second workgroup on the compute unit (one stays). Built for
// four or three tiles (or a window's two) of 128-wide heads over 16-bit pages, two over 8-bit pages and three over scaled
// rows (pairs still fit two workgroups a compute unit) or of 256-wide heads, where it measured faster (64 rows ~U[1024,
// 8192] of 32 / 8 heads, 8 columns, a tile at a time and so: 663 and 333 us, FP8 342 and 222); four tiles of 8-bit pages
// measured slower.
// NARROW: 64-wide heads, read as 128-wide ones. Two adjacent KV heads' rows of a position are 128 contiguous values,
// which is what a 128-wide head's row is: the launcher hands the kernel half the KV heads at twice the width and GQA
// groups twice as large (a group's first half the query heads of the even KV head, its second half the odd one's: the
// query heads' own order). A query row enters the first product with zeros in the other head's 64 dims (exact: the
// products with them are zeros), so its scores are its own head's; the second product gives it 128 output dims of
// which its own head's 64 are kept. Twice the matrix work a byte, on a pipe this kernel leaves nine tenths idle, for
// the 128-wide kernel's loads: 512 contiguous bytes a position and wavefront. What follows a KV head (row scales, an
// FP8 pool's multipliers) is looked up by the column's own head.
template <int KIND, bool F16, int HW, bool FUSED, int MASK, int DH = 1, int QT = 1, bool NARROW = false, int PLACES = kPlacesNone>
__global__ __launch_bounds__(256, (MfmaShape<KIND, DH, QT, PLACES>::kGroups)) void attend_mfma_kernel(AttendArgs a) {
    constexpr bool ALONE = PLACES != kPlacesNone;      // a place a workgroup
    static_assert(!ALONE || (!FUSED && MASK != kMaskSliding), "small launches: the split launch, without a sliding window");
    static_assert(!NARROW || (DH == 1 && QT == 1), "64-wide heads: one 128-wide pair a tile row, one tile a workgroup");
    constexpr bool RING = MfmaShape<KIND, DH, QT, PLACES>::kRing;
    constexpr int NP = MfmaShape<KIND, DH, QT, PLACES>::kPairs, NT = 2 * NP;      // pairs of steps in flight, steps
    // The next unit's queries wait in registers, where a unit is long enough for it: what is requested among its first rows
    // makes the waits on those coarser (256-wide heads, 376 units of at most six pairs, INT8: 45.4 us, 46.5 so).
    constexpr bool AHEAD = ALONE || (RING && DH == 1 && QT > 2);
    constexpr int D = 128 * DH;
    static_assert(DH == 1 || (DH == 2 && HW == 1), "heads of 128 or 256; one KV head a wavefront at 256");
    static_assert(QT == 1 || !FUSED, "several query tiles: the split launch");
    constexpr int EB = KIND == 0 ? 2 : 1;
    constexpr int CPH = kTileRows / HW;      // tile columns a KV head holds
    constexpr int SPW = kTileRows / HW;      // positions a wavefront's step covers (tile rows a KV head holds)
    // Steps that share one maximum, factor and sum, and one product for their values. Both of a pair where a row's scale is
    // multiplied into the probability before it is rounded to 16 bits. Elsewhere a step has its own: its largest
    // probability, where it moves the maximum, is then 1, which 16 bits hold, and one maximum for both leaves the first
    // step's below 1 (16 rows ~U[1024, 8192], FP32 results, from 64 bits: BF16 1.237e-3 in place of 1.253e-3, 256-wide heads
    // 1.171e-3 in place of 1.215e-3, FP8 1.364e-3 in place of 1.372e-3; row-scaled FP8 and INT8 1.609e-3 and 1.589e-3
    // either way). One maximum is the cheaper (5 columns of 64 such rows, the queries' signs then still set here, see lane_values: BF16 289
    // us, each its own 303; FP8 174 and 207).
    constexpr int G = KIND >= 2 ? 2 : 1;
    constexpr int FW = RING ? 64 : D;        // output dims folded at a time
    constexpr int FG = FW / 64;              // groups of four of them a thread folds: dims 64 i + 4 (tid % 16) .. + 3 of column tid / 16
    constexpr int ROWB = D * EB;             // bytes of a key or value row
    constexpr int CPR = ROWB / 16;           // its 16-byte chunks
    constexpr int HALF = 16 * ROWB;          // a step's keys (its values follow)
    constexpr int NKI = HALF / 1024;         // loads of a wavefront they take
    constexpr int SCI = KIND >= 2 ? 1 : 0;   // ... and their rows' scales
    constexpr int NK = 2 * (NKI + SCI), NV = 2 * NKI;      // ... a pair's keys with all scales, its values
    constexpr int SCN = NARROW ? 64 : 32;    // scales of a step: keys', values' (NARROW: the even heads', the odd ones', twice)
    __shared__ __align__(16) float s_acc[4][kTileRows][FW];
    __shared__ __align__(1024) uint8_t s_ring[RING ? 4 : 1][RING ? NT : 1][RING ? 2 * HALF : 16];
    __shared__ __align__(16) float s_scales[RING && KIND >= 2 ? 4 : 1][RING && KIND >= 2 ? NT : 1][RING && KIND >= 2 ? SCN : 4];
    __shared__ float s_m[4][kTileRows], s_l[4][kTileRows];
    __shared__ int s_rows[kLdsRows][5];      // count, first position, table row, first token, first partial row
    __shared__ int s_before[kLdsRows + 1];   // the dense list: partitions but the last of the rows before row r
    __shared__ int s_wave_sum[4];
    __shared__ uint16_t s_order[kLdsRows];   // the dense list: the rows by the size of their last partition
    int* const s_key = reinterpret_cast<int*>(&s_acc[0][0][0]);      // ... (while the list is made)
    static_assert(sizeof(s_acc) >= (kLdsRows + 256) * sizeof(int), "the list's keys lie in the fold's array");
    __shared__ unsigned s_unit;

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int c16 = lane & 15, u4 = lane >> 4;
    const unsigned grid = gridDim.x;
    const bool pulled = !ALONE && a.ticket != nullptr;
    const int hgroups = a.hkv / HW;
    // The list of units. Launches of up to kLdsRows rows take the dense list: every row's partitions but its last, row
    // by row (each for every head group and tile), then every row's last partition (usually a partial piece: the
    // smallest units go last) - no unit without work beyond tiles a short window row does not fill. Larger launches
    // take the grid units_x x units_y, whose units without work are passed over as they are drawn.
    const bool dense = !ALONE && a.n_rows <= kLdsRows;      // (ALONE: a unit a workgroup, which asks memory for its own row)
    const unsigned per_row = (unsigned)(hgroups * a.tiles);
    const int slot_bytes = a.hkv * D * EB;
    const bool tree = MASK == kMaskTree || (MASK == kMaskSliding && (a.parents != nullptr || a.parents64 != nullptr));
    const int win = MASK == kMaskSliding ? a.sliding : 0;      // (a tree's launch has no window)

    // Quotients by the launch's own numbers (none of them a power of two in general: a division is forty instructions).
    auto by_group = [&](int x) __attribute__((always_inline)) -> int { return (int)div32(a.group_div, (uint32_t)x); };
    auto pieces_of = [&](int n_keys) __attribute__((always_inline)) -> int { return (int)div32(a.piece_div, (uint32_t)(n_keys + a.piece - 1)); };

    // -- every row's descriptors, once per workgroup
    auto row_from_memory = [&](int r, int (&d)[5]) __attribute__((always_inline)) {
        const int count = a.counts ? a.counts[r] : a.columns;
        const int64_t first64 = a.firsts[r];
        d[0] = min(count, a.columns);
        d[1] = (int)(first64 < 0 ? 0 : (first64 > (int64_t)0x3fffffff ? (int64_t)0x3fffffff : first64));
        d[2] = a.rows[(int64_t)r * a.rows_step];
        d[3] = a.starts[r];
        d[4] = a.offsets ? a.offsets[r] - a.offsets[0] : r * a.columns;
    };
    if constexpr (!ALONE) {
        for (int r = tid; r < min(a.n_rows, kLdsRows); r += 256) {
            int d[5];
            row_from_memory(r, d);
#pragma unroll
            for (int i = 0; i < 5; ++i) s_rows[r][i] = d[i];
        }
        lds_barrier();
    }
    // Partitions that hold positions of row r (of its last column): what its units divide.
    auto row_partitions = [&](int r) __attribute__((always_inline)) -> int {
        const int count = s_rows[r][0];
        if (count <= 0) return 0;
        if constexpr (FUSED) return 1;
        const int n_keys = min(s_rows[r][1] + count, a.max_keys);
        return min(pieces_of(n_keys), a.parts);
    };
    if (dense) {      // s_before[r] = sum over r' < r of max(partitions(r') - 1, 0): thread i sums rows 2 i and 2 i + 1
        const int r0 = 2 * tid, r1 = 2 * tid + 1;
        const int c0 = r0 < a.n_rows ? max(row_partitions(r0) - 1, 0) : 0, c1 = r1 < a.n_rows ? max(row_partitions(r1) - 1, 0) : 0;
        const int run = (int)wave_inclusive_sum((unsigned)(c0 + c1));      // inclusive prefix over the threads
        if (lane == 63) s_wave_sum[wave] = run;
        lds_barrier();
        int base = 0;
        for (int w = 0; w < wave; ++w) base += s_wave_sum[w];
        const int upto = base + run - (c0 + c1);      // rows before 2 i
        if (r0 <= a.n_rows) s_before[r0] = upto;
        if (r1 <= a.n_rows) s_before[r1] = upto + c0;
        if (tid == 255 && kLdsRows <= a.n_rows) s_before[kLdsRows] = upto + c0 + c1;
        // The rows' last partitions are taken largest first (a launch's tail is as long as its last units): positions
        // the last partition holds (more than a piece where partitions hold several pieces), ties by row. A row's place is the
        // number of rows before it. Up to 256 rows, in launches of more units than workgroups; more rows cost more to rank
        // than it returns.
        const bool ranked = a.n_rows <= 256 && (unsigned)a.units_x * (unsigned)a.units_y > grid;
        int* const s_rank = s_key + kLdsRows;
        for (int r = tid; r < (ranked ? 256 : a.n_rows); r += 256) {
            const int count = r < a.n_rows ? s_rows[r][0] : 0;
            unsigned key = 0;      // a size of 23 bits, then the row: no two alike, and none above those past the last row
            if (count > 0) {
                const int n_keys = min(s_rows[r][1] + count, a.max_keys);
                const int n_pieces = pieces_of(n_keys);
                const int size = FUSED ? n_keys : (n_pieces > a.parts ? a.piece + 1 : n_keys - (n_pieces - 1) * a.piece);
                key = (unsigned)min(size, 0x7ffffe) + 1u;
            }
            if (ranked) s_key[r] = (int)(r < a.n_rows ? (key << 8) + (unsigned)(255 - r) : 0u), s_rank[r] = 0;
            else s_order[r] = (uint16_t)r;
        }
        lds_barrier();
        if (ranked) {
            // 64 rows a wavefront, a lane each, four others a read; the wavefronts that 64 or 128 rows leave over share the
            // others. (One other at a time, by v_readlane, and ties by a comparison of rows were 5 us of a launch of 128 rows: of
            // 40 to 300 positions, 24 / 3 heads x 128, BF16 27.8 us, 22.6 so; 64 rows ~U[1024, 8192], 32 / 8 heads, one column
            // BF16 215.7 and 211.6, FP8 119.0 and 115.3.)
            const int shares = a.n_rows <= 64 ? 4 : a.n_rows <= 128 ? 2 : 1, row = 64 * (wave / shares) + lane;
            if (64 * (wave / shares) < a.n_rows) {
                const unsigned key = (unsigned)s_key[row];
                int rank = 0;
#pragma unroll 4
                for (int o = 4 * (wave % shares); o < a.n_rows; o += 4 * shares) {
                    const u32x4 others = *reinterpret_cast<const u32x4*>(s_key + o);
#pragma unroll
                    for (int i = 0; i < 4; ++i) rank += others[i] > key ? 1 : 0;
                }
                atomicAdd(&s_rank[row], rank);
            }
            lds_barrier();
            if (tid < a.n_rows) s_order[s_rank[tid]] = (uint16_t)tid;
        }
        lds_barrier();
    }
    const unsigned phase1 = dense ? (unsigned)__builtin_amdgcn_readfirstlane(s_before[a.n_rows]) * per_row : 0u;
    const unsigned total = dense ? phase1 + (unsigned)a.n_rows * per_row : (unsigned)a.units_x * (unsigned)a.units_y;

    // -- a unit of the list, decoded (everything uniform over the workgroup)
    struct Unit {
        bool valid;
        int kvh0, j0, b, count, first, n_keys, n_pieces, start, c_lo, prow;
        int64_t trow;
    };
    auto decode = [&](unsigned unit) __attribute__((always_inline)) -> Unit {
        Unit un;
        un.valid = false;
        if (!ALONE && unit >= total) return un;
        int bx, b, r;
        bool last = false;      // dense list: the row's last partition
        int d[5];
        if constexpr (PLACES == kPlacesTwo) {      // (both rows' numbers in one round trip to memory)
            int d1[5];
            row_from_memory(0, d), row_from_memory(1, d1);
            auto pieces_of_row = [&](const int (&n)[5]) __attribute__((always_inline)) -> uint32_t {
                return (uint32_t)__builtin_amdgcn_readfirstlane(n[0] > 0 ? pieces_of(min(n[1] + n[0], a.max_keys)) : 0);
            };
            const uint32_t p0 = pieces_of_row(d), p1 = pieces_of_row(d1), mine = blockIdx.y * grid + blockIdx.x;
            if (mine >= per_row * (min(p0, (uint32_t)a.parts) + min(p1, (uint32_t)a.parts))) return un;
            const RowPlace at = row_place(mine, p0, p1, (uint32_t)a.parts, per_row, (uint32_t)a.cus,
                                          [&](uint32_t x) __attribute__((always_inline)) -> uint32_t { return div32(a.row_div, x); });
            r = at.row, b = (int)at.partition, bx = (int)at.place;
#pragma unroll
            for (int i = 0; i < 5; ++i) d[i] = r ? d1[i] : d[i];
        } else if constexpr (ALONE) {
            r = (int)div32(a.row_div, blockIdx.x), b = (int)blockIdx.y;
            bx = (int)blockIdx.x - r * (int)per_row;
        } else if (dense) {
            if (unit < phase1) {
                const int q = (int)div32(a.row_div, unit);      // the q-th of all rows' partitions but their last
                bx = (int)(unit - (unsigned)q * per_row);
                int n = 0;      // the row: the last with s_before[r] <= q (64 rows a look)
                for (int r0 = 0; r0 < a.n_rows; r0 += 64)
                    n += __builtin_popcountll(__builtin_amdgcn_ballot_w64(r0 + lane < a.n_rows && s_before[min(r0 + lane, kLdsRows)] <= q));
                r = n - 1, b = q - __builtin_amdgcn_readfirstlane(s_before[r]);
            } else {
                const unsigned rest = unit - phase1;
                const unsigned at = div32(a.row_div, rest);
                r = __builtin_amdgcn_readfirstlane(s_order[at]), bx = (int)(rest - at * per_row), b = 0, last = true;
            }
        } else {
            bx = (int)(unit % (unsigned)a.units_x);
            b = (int)(unit / (unsigned)a.units_x);
            r = (int)div32(a.row_div, (uint32_t)bx);
            bx -= r * (int)per_row;
        }
        const int tiles_before = (int)div32(a.tiles_div, (uint32_t)bx), tile = bx - tiles_before * a.tiles;
        un.kvh0 = tiles_before * HW;      // the first of the wavefronts' KV heads
        if constexpr (PLACES != kPlacesTwo) {
            if (!ALONE && r < kLdsRows) {
#pragma unroll
                for (int i = 0; i < 5; ++i) d[i] = s_rows[r][i];
            } else {
                row_from_memory(r, d);
            }
        }
#pragma unroll
        for (int i = 0; i < 5; ++i) d[i] = __builtin_amdgcn_readfirstlane(d[i]);
        un.count = d[0], un.first = d[1], un.start = d[3], un.prow = d[4];
        un.trow = (int64_t)d[2] * a.tab_stride;
        un.j0 = tile * (QT * CPH);           // the first row of the unit's tiles in the flattened (column, group head) list
        if (un.j0 >= un.count * a.g) return un;
        un.c_lo = by_group(un.j0);
        const int c_hi = min(un.count, by_group(un.j0 + QT * CPH - 1) + 1);
        un.n_keys = min(un.first + c_hi, a.max_keys);
        un.n_pieces = pieces_of(un.n_keys);
        if constexpr (!FUSED) {
            // Units are taken in list order, y slowest, and a launch's tail is as long as its last units: the row's
            // last partition (usually a partial piece, the smallest unit of work) is listed after every other
            // partition, in kTailClasses rows of y by its size (a whole piece or more first, the smallest last).
            const int np = min(un.n_pieces, a.parts);
            if (np <= 0) return un;
            if (dense) {
                if (last) b = np - 1;
                else if (b >= np - 1) return un;      // (a tile of earlier columns that holds fewer pieces than the row's last)
            } else if constexpr (ALONE) {
                if (b >= np) return un;
            } else {
                int cls = 0;
                if (np == un.n_pieces) cls = min(kTailClasses - 1, (np * a.piece - un.n_keys) * kTailClasses / a.piece);
                if (b >= a.units_y - kTailClasses) {
                    if (b - (a.units_y - kTailClasses) != cls) return un;
                    b = np - 1;
                } else if (b >= np - 1) {
                    return un;
                }
            }
        } else if (dense && !last) {
            return un;
        }
        un.b = b;
        un.valid = true;
        return un;
    };

    // -- what a lane holds for the whole launch
    // Tile rows: row i is position i % SPW of the step, of head i / SPW. This lane's places in the three layouts:
    //   keys    its row c16;  values and scores  rows 4 u4 .. 4 u4 + 3.
    const int hsel = c16 / CPH;                                     // the head (of the wavefront's HW) of this lane's tile column
    const int k_head = c16 / SPW, k_pos = c16 % SPW;
    const int r_head = (4 * u4) / SPW, r_pos = (4 * u4) % SPW;      // (SPW is 8 or 16: a lane's four rows lie in one head)
    const bool mine = hsel == r_head;                               // this lane's scores are of its own column's head
    // Byte offsets of what this lane reads in a step, from the step's first slot and the unit's first head.
    const uint32_t kvo = (uint32_t)(k_pos * slot_bytes + k_head * D * EB + u4 * 16);
    uint32_t vvo[4];
#pragma unroll
    for (int p = 0; p < 4; ++p) vvo[p] = (uint32_t)((r_pos + p) * slot_bytes + r_head * D * EB + c16 * 8 * EB);
    // A ring's step in LDS: the tile's 16 key rows (row i: position i % SPW of head i / SPW), then its value rows. The memory
    // pipe writes lane i's 16 bytes at byte 16 i of a kilobyte, whatever it fetched for that lane, so a load's lanes take
    // adjacent chunks of a row (four lanes a 64-byte request, where the operand's own layout would be a request a lane)
    // and the chunks of a row are stored permuted, chunk c of row i at place c ^ turn(i) (in its low four bits), which
    // spreads the operands' reads (16 rows, one chunk each) over all banks. 8-bit values are not permuted, but row
    // 4 u + p lies in place 4 p + u: a read takes rows p, 4 + p, 8 + p, 12 + p.
    auto turn = [](int row) __attribute__((always_inline)) -> int { return CPR == 8 ? (row >> 1) & 7 : 2 * (row & 7) + (row >> 3); };
    uint32_t k_from[NKI], v_from[NKI];
    if constexpr (RING) {
#pragma unroll
        for (int j = 0; j < NKI; ++j) {
            const int place = 64 * j + lane, row = place / CPR, c = place % CPR;
            k_from[j] = (uint32_t)((row % SPW) * slot_bytes + (row / SPW) * ROWB + 16 * (c ^ turn(row)));
            if constexpr (KIND == 0) {
                v_from[j] = k_from[j];
            } else {
                const int vrow = 4 * (row & 3) + (row >> 2);
                v_from[j] = (uint32_t)((vrow % SPW) * slot_bytes + (vrow / SPW) * ROWB + 16 * c);
            }
        }
    }
    const unsigned ring_at = (unsigned)__builtin_amdgcn_readfirstlane((int)(uintptr_t)&s_ring[RING ? wave : 0][0][0]);
    const unsigned scales_at = (unsigned)__builtin_amdgcn_readfirstlane((int)(uintptr_t)&s_scales[RING && KIND >= 2 ? wave : 0][0][0]);
    const uint32_t k_read = (uint32_t)(c16 * ROWB + 16 * (u4 ^ turn(c16)));      // chunk 4 l + u4 of row c16: ^ 64 l (+ 256 from l = 4 on)
    const int t_row = 4 * u4 + (c16 >> 2);      // 16-bit values, transposed: four values of row t_row, of every 16 dims
    const uint32_t t_read = (uint32_t)(t_row * ROWB + 8 * (c16 & 1)), t_turn = (uint32_t)(16 * (((c16 & 3) >> 1) ^ turn(t_row)));
    // the scale this lane sends to LDS: of which head's keys or values, and of which row of the tile
    const int sc_row = lane & 15, sc_odd = NARROW ? (lane >> 4) & 1 : 0;
    const float* sc_from = (lane >> (NARROW ? 5 : 4)) & 1 ? a.vs : a.ks;
    if constexpr (RING && KIND >= 2)
        sc_from += NARROW ? (sc_row % SPW) * 2 * a.hkv + 2 * (sc_row / SPW) + sc_odd : (sc_row % SPW) * a.hkv + sc_row / SPW;

    // -- a wavefront's steps of a partition: steps wave, wave + 4, ... of pieces part, part + parts, ..., taken in pairs
    // within a piece (a piece's last pair may lack its second step). Lane 2 i + r holds the first position and the table
    // entry of step r of pair from + i, for 32 pairs at a time: one load of the page table, and no wait on it in the loop.
    // A step that is not there has position -1 and the entry of one that is.
    struct Steps {
        int base, entry, in_page, from, first_piece;
        uint32_t slot;
    };
    const int steps_a_piece = a.piece / SPW;
    const int pairs_a_piece = ((steps_a_piece - wave + 3) / 4 + 1) / 2;      // this wavefront's (0: too short a piece for it)
    auto hold = [&](const Unit& un, int first_piece, int from) __attribute__((always_inline)) -> Steps {
        Steps s;
        s.from = from, s.first_piece = first_piece;
        const int n = from + (lane >> 1), r = lane & 1;
        const int turns = n < pairs_a_piece ? 0 : n / max(pairs_a_piece, 1), k = n - turns * pairs_a_piece;
        const int piece = first_piece + turns * a.parts;
        const int st = wave + 8 * k;
        const bool there = pairs_a_piece > 0 && piece < un.n_pieces;
        const int at = there ? piece * a.piece + st * SPW : 0x7fffffff - 8 * SPW;      // (pieces of the row: positions below 2^31)
        const bool one = at < un.n_keys, two = one && st + 4 < steps_a_piece && at + 4 * SPW < un.n_keys;
        s.base = r == 0 ? (one ? at : -1) : (two ? at + 4 * SPW : -1);
        const int of = s.base >= 0 ? s.base : (one ? at : 0);
        const int page = of >> a.page_shift;
        s.entry = a.tables[un.trow + (page < a.tab_width ? page : a.tab_width - 1)];
        s.in_page = of & (a.page - 1);
        s.slot = 0u;
        return s;
    };
    auto resolve = [&](Steps& s) __attribute__((always_inline)) { s.slot = (uint32_t)s.entry * (uint32_t)a.page + (uint32_t)s.in_page; };
    auto steps_of = [&](const Unit& un, int part) __attribute__((always_inline)) -> Steps {
        int first_piece = part;
        if (win > 0) {      // pieces wholly below the tile's window are skipped (no row sees them)
            const int wlo = un.first + un.c_lo - win + 1;
            const int below = (wlo > 0 ? wlo : 0) / a.piece - part;
            if (below > 0) first_piece = part + (below + a.parts - 1) / a.parts * a.parts;
        }
        return hold(un, first_piece, 0);
    };
    struct Pair {
        int base, second;      // the steps' first positions; -1: no such step
        uint32_t s0, s1;       // their first slots (of a step that is not there: another's)
    };
    auto pair_no = [&](const Unit& un, Steps& s, int n) __attribute__((always_inline)) -> Pair {
        if (n - s.from >= 32) s = hold(un, s.first_piece, s.from + 32), resolve(s);
        const int l = 2 * (n - s.from);
        Pair p;
        p.base = __builtin_amdgcn_readlane(s.base, l), p.second = __builtin_amdgcn_readlane(s.base, l + 1);
        p.s0 = (uint32_t)__builtin_amdgcn_readlane((int)s.slot, l), p.s1 = (uint32_t)__builtin_amdgcn_readlane((int)s.slot, l + 1);
        return p;
    };
    // Loads of one step from its first slot. Every lane loads its place of the step whether the row holds that
    // position or not (the page does; a step past the row's keys is never listed): what such a place holds is dropped
    // where it is used (keys: the score is masked; values and scales: zeroed, see sanitize()).
    // (NARROW: `odd`, whether this lane's column is a query row of the pair's odd KV head; the scales are per KV head)
    Tile t[RING ? 1 : NT];
    auto fetch_k = [&](const Unit& un, uint32_t slot0, int i) __attribute__((always_inline)) {
        const uint8_t* sbase = a.kp + (int64_t)slot0 * slot_bytes + un.kvh0 * ROWB;
        if constexpr (RING) {
#pragma unroll
            for (int j = 0; j < NKI; ++j) dma_rows<false>(k_from[j], sbase, ring_at + (unsigned)(i * 2 * HALF + 1024 * j));
            if constexpr (KIND >= 2) {
                if (SCN == 64 || lane < SCN)
                    dma_words(sc_from + ((int64_t)slot0 * a.hkv + un.kvh0) * (NARROW ? 2 : 1), scales_at + (unsigned)(i * SCN * 4));
            }
        } else {
#pragma unroll
            for (int c = 0; c < 4; ++c) t[i].k[c] = *reinterpret_cast<const u32x4*>(sbase + kvo + 64 * c);
        }
    };
    // NARROW: whether this lane's tile column (a query row of the flattened list) belongs to the pair's odd KV head.
    auto odd_of = [&](const Unit& un) __attribute__((always_inline)) -> int {
        if constexpr (!NARROW) return 0;
        const int j = un.j0 + c16 % CPH;
        return j - by_group(j) * a.g >= (a.g >> 1) ? 1 : 0;
    };
    auto fetch_v = [&](const Unit& un, uint32_t slot0, int i) __attribute__((always_inline)) {
        const uint8_t* sbase = a.vp + (int64_t)slot0 * slot_bytes + un.kvh0 * ROWB;
        if constexpr (RING) {
#pragma unroll
            for (int j = 0; j < NKI; ++j) dma_rows<true>(v_from[j], sbase, ring_at + (unsigned)(i * 2 * HALF + HALF + 1024 * j));
        } else {
#pragma unroll
            for (int p = 0; p < 4; ++p) t[i].v[p] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(sbase + vvo[p]));
        }
    };

    // -- what a lane holds for one unit: its tile column's token, query head, last visible position, ancestors, scale,
    // and the query operand (its column's row, piece c = the dims the keys' piece c holds; zeros in a dead column)
    int col[QT], lim[QT];
    unsigned long long anc[QT];
#pragma unroll
    for (int q = 0; q < QT; ++q) col[q] = 0, lim[q] = -1, anc[q] = 0ull;
    float sscale = a.sscale;
    float vm_cur[HW], vm_nxt[HW];      // FP8 pages: the value multipliers of the unit's heads
    float km_nxt = 1.0f;               // ... and the key multiplier of this lane's column's
    uint32_t link_lo = 0u, link_hi = 0u;      // draft trees: the parent of column `lane` of the unit's row
#pragma unroll
    for (int h = 0; h < HW; ++h) vm_cur[h] = vm_nxt[h] = 1.0f;
    u32x4 qb[QT][4 * DH], qb_nxt[QT][4 * DH];
    auto load_queries = [&](const Unit& un, int odd, int q, int jr, int cl, bool live, u32x4 (&to)[QT][4 * DH]) __attribute__((always_inline)) {
        const int qhead = (un.kvh0 + hsel) * a.g + jr - cl * a.g;
        const uint8_t* row = a.q + ((int64_t)(un.start + cl) * a.q_st + (int64_t)qhead * a.q_sh) * 2;
#pragma unroll
        for (int c = 0; c < 4 * DH; ++c) {
            // 16-bit pages: dims 32 c + 8 u4 ..; 8-bit pages: dims 64 (c / 2) + 16 u4 + 8 (c % 2) .. (the codes a lane's two loads hold)
            const int dim = KIND == 0 ? 32 * c + 8 * u4 : 64 * (c / 2) + 16 * u4 + 8 * (c % 2);
            to[q][c] = u32x4{0, 0, 0, 0};
            if constexpr (NARROW) {      // the column's own head's 64 dims, zeros in the other head's
                if (live && (dim >> 6) == odd) to[q][c] = *reinterpret_cast<const u32x4*>(row + (dim & 63) * 2);
            } else {
                if (live) to[q][c] = *reinterpret_cast<const u32x4*>(row + dim * 2);
            }
        }
    };
    // What a unit needs beside its rows is requested with its page table entries, a unit ahead, and is there when its rows are
    // sent for. A wait on any of it behind the unit's rows would wait for those too, and behind the fold for the partials'
    // stores as well, which the compiler cannot count; a workgroup alone on its compute unit has nothing to do meanwhile
    // (64 rows ~U[1024, 8192], 32 / 8 heads x 128 BF16, 5 columns: 277.2 and 274.4 us, which is as much as two runs differ). A
    // tree's links, walked a load at a time for every tile, were most of what a lone row gained (one of 50,000, 56 / 8 heads,
    // INT8, a tree of 8: 98.9 -> 96.5).
    auto request = [&](const Unit& un) __attribute__((always_inline)) {
        if constexpr (KIND == 1) {
#pragma unroll
            for (int h = 0; h < HW; ++h) vm_nxt[h] = a.hm ? a.hm[a.hkv + un.kvh0 + h] : a.v_mult;
            km_nxt = a.hm ? a.hm[NARROW ? 2 * (un.kvh0 + hsel) + odd_of(un) : un.kvh0 + hsel] : a.k_mult;
        }
        if constexpr (MASK != kMaskNone) {
            if (tree && lane < un.count) {
                if (a.parents) {
                    link_lo = (uint32_t)a.parents[un.start + lane];
                } else {
                    const u32x2 link = *reinterpret_cast<const u32x2*>(a.parents64 + un.start + lane);
                    link_lo = link.x, link_hi = link.y;
                }
            }
        }
        if constexpr (AHEAD) {
            const int odd = odd_of(un);
#pragma unroll
            for (int q = 0; q < QT; ++q) {
                const int jr = un.j0 + q * CPH + c16 % CPH, cl = by_group(jr);
                load_queries(un, odd, q, jr, cl, cl < un.count, qb_nxt);
            }
        }
    };
    auto requested_here = [&](const Steps& s) __attribute__((always_inline)) {
        if constexpr (!RING) return;      // (rows in registers: the compiler's count knows them all)
        asm volatile("" ::"v"(s.entry), "v"(km_nxt), "v"(link_lo), "v"(link_hi));
#pragma unroll
        for (int h = 0; h < HW; ++h) asm volatile("" ::"v"(vm_nxt[h]));
        if constexpr (AHEAD) {
#pragma unroll
            for (int q = 0; q < QT; ++q)
#pragma unroll
                for (int c = 0; c < 4 * DH; ++c) asm volatile("" ::"v"(qb_nxt[q][c].x), "v"(qb_nxt[q][c].y), "v"(qb_nxt[q][c].z), "v"(qb_nxt[q][c].w));
        }
    };
    // (Nothing is done to the queries here: without AHEAD they are the youngest loads, and a wait on them waits for all rows
    // requested before. A negative scale's sign set in them: 64 rows ~U[1024, 8192], 5 columns BF16 303 us, 284 so; 16 rows of 4
    // columns, 24 / 4 x 256, 113 and 101; 64 rows of 24 / 2 x 256, one column, 156 and 147.)
    auto lane_values = [&](const Unit& un) __attribute__((always_inline)) {
        if constexpr (KIND == 1) sscale = a.sscale * km_nxt;
        // Draft trees: lane c makes column c's ancestors and itself: what it has, and what the furthest of them has, until the
        // farthest is the root (as ancestors(); a link that does not point at an earlier column is none).
        uint32_t seen_lo = 0u, seen_hi = 0u;
        if constexpr (MASK != kMaskNone) {
            if (tree) {
                seen_lo = lane < 32 ? 1u << lane : 0u, seen_hi = lane < 32 ? 0u : 1u << (lane - 32);
                int up = lane < un.count && link_hi == 0u && link_lo < (uint32_t)lane ? (int)link_lo : lane;
                for (int reach = 1; reach < un.count; reach *= 2) {
                    seen_lo |= (uint32_t)__shfl((int)seen_lo, up), seen_hi |= (uint32_t)__shfl((int)seen_hi, up);
                    up = __shfl(up, up);
                }
            }
        }
        const int odd = odd_of(un);
#pragma unroll
        for (int q = 0; q < QT; ++q) {
            const int jr = un.j0 + q * CPH + c16 % CPH;
            col[q] = by_group(jr);
            const bool live = col[q] < un.count;
            lim[q] = live ? min(un.first + col[q], un.n_keys - 1) : -1;
            if constexpr (MASK != kMaskNone) {
                if (tree) {
                    const uint32_t lo = (uint32_t)__shfl((int)seen_lo, col[q] & 63), hi = (uint32_t)__shfl((int)seen_hi, col[q] & 63);
                    anc[q] = live ? ((unsigned long long)hi << 32) | lo : 0ull;
                }
            }
            if constexpr (AHEAD) {
#pragma unroll
                for (int c = 0; c < 4 * DH; ++c) qb[q][c] = qb_nxt[q][c];
            } else {
                load_queries(un, odd, q, jr, col[q], live, qb);
            }
        }
    };
    auto queries_here = [&]() __attribute__((always_inline)) {      // (a ring's loads are not the compiler's: its count knows only these)
#pragma unroll
        for (int q = 0; q < QT; ++q)
#pragma unroll
            for (int c = 0; c < 4 * DH; ++c) asm volatile("" ::"v"(qb[q][c].x), "v"(qb[q][c].y), "v"(qb[q][c].z), "v"(qb[q][c].w));
    };

    auto fill = [&](const Unit& un, Steps& s) __attribute__((always_inline)) {      // a partition's first NP pairs
#pragma unroll
        for (int i = 0; i < NP; ++i) {
            const Pair p = pair_no(un, s, i);
            fetch_k(un, p.s0, 2 * i), fetch_k(un, p.s1, 2 * i + 1);
            fetch_v(un, p.s0, 2 * i), fetch_v(un, p.s1, 2 * i + 1);
        }
    };

    unsigned u_next = blockIdx.x + grid;
    Unit cur = decode(blockIdx.x);
    Steps steps = {};
    if (cur.valid) {
        steps = steps_of(cur, FUSED ? 0 : cur.b);
        request(cur);
        requested_here(steps);
        resolve(steps);
        fill(cur, steps);
        lane_values(cur);
#pragma unroll
        for (int h = 0; h < HW; ++h) vm_cur[h] = vm_nxt[h];
    }
    for (;;) {
        // The next unit: its first steps' page table entries are requested now and wait in registers.
        const Unit nxt = [&]() __attribute__((always_inline)) -> Unit { if constexpr (ALONE) return Unit{}; else return decode(u_next); }();
        Steps steps_nxt = {};
        if (nxt.valid) {
            steps_nxt = steps_of(nxt, FUSED ? 0 : nxt.b);
            request(nxt);
        }
        // The ticket of the unit after the next is looked at after the current unit's fold. It is drawn when the current
        // unit's steps are done (rows in registers: a returning atomic in flight beside them makes the waits on them
        // coarser), or a ring of two pairs before that: there it has returned before the next unit's rows are sent for,
        // and no wait on it waits for those.
        unsigned drawn = 0;
        bool asked = false, sent = false;      // the ticket is drawn; the next unit's first loads are out
        auto draw = [&]() __attribute__((always_inline)) {
            if (pulled && (!AHEAD || !asked) && tid == 0) drawn = atomicAdd(a.ticket, 1u);
            asked = true;
        };
        auto hand_over = [&]() __attribute__((always_inline)) {
            draw();
            if constexpr (AHEAD) asm volatile("" ::"v"(drawn));
            if (nxt.valid) {
                requested_here(steps_nxt);
                resolve(steps_nxt);
                fill(nxt, steps_nxt);
                lane_values(nxt);
            }
            sent = true;
        };

        if (cur.valid) {
            const int part_lo = FUSED ? 0 : cur.b;
            const int part_hi = FUSED ? min(a.parts, cur.n_pieces) : cur.b + 1;
            float run_m = -INFINITY, run_l = 0.0f;
            f32x4 run_a[FUSED ? D / 64 : 1];
#pragma unroll
            for (int i = 0; i < (FUSED ? D / 64 : 1); ++i) run_a[i] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
            for (int part = part_lo; part < part_hi; ++part) {
                float m[QT], l[QT];                  // the lane's column of each tile: running maximum (the same in its four lanes), the lane's share of the sum
                f32x4 acc[QT][8 * DH];               // O^T: acc[q][8 h + j][i] = dim 128 h + 32 u4 + 8 i + j of the lane's column of tile q
#pragma unroll
                for (int q = 0; q < QT; ++q) {
                    m[q] = -INFINITY, l[q] = 0.0f;
#pragma unroll
                    for (int j = 0; j < 8 * DH; ++j) acc[q][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
                }

                const int odd_cur = odd_of(cur);
                // A pair of steps, in places 2 i and 2 i + 1: positions base .. + SPW - 1 and second .. + SPW - 1 (second < 0: no such
                // step). keys_here and values_here wait until the pair's have landed, refill_k and refill_v send for what comes to a
                // step's place next. Both steps' scores come first, then their probabilities, then the values; two query tiles
                // in registers go step by step (both steps' scores and probabilities at once are 76 bytes of scratch a lane
                // more: 64 rows ~U[1024, 8192], 32 / 8 heads, a tree of 4, 279 us, 266 so; one tile 215.7 and 217.8).
                constexpr bool APART = !RING && QT > 1;
                auto step = [&](int base, int second, int i, auto&& keys_here, auto&& values_here, auto&& refill_k, auto&& refill_v) __attribute__((always_inline)) {
                    const int base_b = second >= 0 ? second : 0x3fffff00;      // (past every column's last position)
                    // Both steps wholly seen by every column of the tiles (a draft tree's: before the window's first
                    // position): nothing is asked of a position.
                    const bool whole = MASK != kMaskSliding && win <= 0 &&
                                       base_b + SPW <= min(MASK == kMaskTree ? cur.first : cur.first + cur.c_lo + 1, cur.n_keys);
                    const uint8_t* const places[2] = {&s_ring[RING ? wave : 0][RING ? 2 * i : 0][0], &s_ring[RING ? wave : 0][RING ? 2 * i + 1 : 0][0]};
                    // -- scores of steps lo .. hi - 1. A step of its own maximum sums the keys' even pieces and the odd ones apart.
                    f32x4 s0[2][QT], s1[2][QT];
                    u32x4 held[2][RING ? CPR / 4 : 1];
                    auto scores = [&](int lo, int hi) __attribute__((always_inline)) {
#pragma unroll
                        for (int r = lo; r < hi; ++r)
#pragma unroll
                            for (int q = 0; q < QT; ++q) s0[r][q] = f32x4{0.0f, 0.0f, 0.0f, 0.0f}, s1[r][q] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                        for (int c = 0; c < 4 * DH; ++c) {
                            u32x4 k[2];
#pragma unroll
                            for (int r = lo; r < hi; ++r) k[r] = key_operand<KIND>(RING ? held[r] : t[RING ? 0 : 2 * i + r].k, c);
#pragma unroll
                            for (int q = 0; q < QT; ++q) {
#pragma unroll
                                for (int r = lo; r < hi; ++r) {
                                    f32x4& sum = G == 1 && c % 2 ? s1[r][q] : s0[r][q];
                                    sum = mfma_k32<F16>(k[r], qb[q][c], sum);
                                }
                            }
                        }
                    };
                    float ks8[8], vs8[8];
                    // -- the lane's probabilities: its column at positions base + r_pos + i, second + r_pos + i of head r_head. Another
                    // head's column (a lane that is not `mine`) sees nothing: its scores stay out of the maximum, its
                    // probabilities become zeros (chosen, not multiplied: the other head's values may be anything).
                    uint32_t pb[2][QT][2 * G];
                    float alpha[2][QT];
                    bool rescale[2];
                    auto soften = [&](int r) __attribute__((always_inline)) {      // step r, or with G 2 both
                        rescale[r] = false;
#pragma unroll
                        for (int q = 0; q < QT; ++q) {
                            float x[4 * G];
#pragma unroll
                            for (int i = 0; i < 4 * G; ++i) {
                                const int st = G == 1 ? r : i / 4;
                                const float raw = G == 1 ? s0[st][q][i & 3] + s1[st][q][i & 3] : s0[st][q][i & 3];
                                x[i] = raw * (KIND >= 2 ? sscale * ks8[4 * st + (i & 3)] : sscale);
                            }
                            if (!whole) {
                                const int room = lim[q] - r_pos;      // position n (of the step's first) is visible while n + i <= room
#pragma unroll
                                for (int i = 0; i < 4 * G; ++i) {
                                    const int at = ((G == 1 ? r : i / 4) == 0 ? base : base_b) + (i & 3);
                                    bool vis = at <= room;
                                    if constexpr (MASK != kMaskNone) {
                                        const int n = at + r_pos;
                                        if (tree) vis = vis && (n < cur.first || ((anc[q] >> ((n - cur.first) & 63)) & 1ull) != 0);
                                        if (win > 0) vis = vis && n > cur.first + col[q] - win;
                                    }
                                    x[i] = vis ? x[i] : -INFINITY;
                                }
                            }
                            float y = __builtin_fmaxf(__builtin_fmaxf(x[0], x[1]), __builtin_fmaxf(x[2], x[3]));
                            if constexpr (G == 2) y = __builtin_fmaxf(y, __builtin_fmaxf(__builtin_fmaxf(x[4], x[5]), __builtin_fmaxf(x[6], x[7])));
                            if constexpr (HW > 1) y = mine ? y : -INFINITY;
                            const float m_new = __builtin_fmaxf(m[q], max_across_quarters(y));
                            const float sub = m_new == -INFINITY ? 0.0f : m_new;
                            alpha[r][q] = m[q] == -INFINITY ? 1.0f : exp2_fast(m[q] - sub);      // (nothing summed yet: nothing to rescale)
                            rescale[r] = rescale[r] || alpha[r][q] != 1.0f;
                            m[q] = m_new;
                            float p[4 * G];
#pragma unroll
                            for (int i = 0; i < 4 * G; ++i) p[i] = exp2_fast(x[i] - sub);
                            float sum = (p[0] + p[1]) + (p[2] + p[3]);
                            if constexpr (G == 2) sum += (p[4] + p[5]) + (p[6] + p[7]);
                            sum = HW == 1 || mine ? sum : 0.0f;
                            l[q] = G == 1 ? __builtin_fmaf(l[q], alpha[r][q], sum) : l[q] * alpha[r][q] + sum;
#pragma unroll
                            for (int i = 0; i < 2 * G; ++i) {
                                const uint32_t w = KIND >= 2 ? pair16<F16>(p[2 * i] * vs8[2 * i], p[2 * i + 1] * vs8[2 * i + 1]) : pair16<F16>(p[2 * i], p[2 * i + 1]);
                                pb[r][q][i] = HW == 1 || mine ? w : 0u;
                            }
                        }
                    };
                    auto move = [&](int r) __attribute__((always_inline)) {
                        if (__builtin_amdgcn_ballot_w64(rescale[r]) != 0) {      // some column's maximum moved
#pragma unroll
                            for (int q = 0; q < QT; ++q)
#pragma unroll
                                for (int j = 0; j < 8 * DH; ++j) acc[q][j] *= alpha[r][q];
                        }
                    };
                    // The row's last steps: what lies past its keys may be anything, and a probability of zero times a NaN is a
                    // NaN. Such values become zeros.
                    auto clean = [&](int r) __attribute__((always_inline)) {
                        const int at = r == 0 ? base : base_b;
                        if (at + SPW > cur.n_keys) {
                            if constexpr (RING) {
                                uint8_t* values = &s_ring[wave][2 * i + r][HALF];
                                for (int row = 0; row < 16; ++row) {
                                    if (at + row % SPW < cur.n_keys) continue;
                                    uint8_t* to = values + (KIND == 0 ? row : 4 * (row & 3) + (row >> 2)) * ROWB;
                                    for (int b = lane * 4; b < ROWB; b += 256) *reinterpret_cast<uint32_t*>(to + b) = 0u;
                                }
                            } else {
#pragma unroll
                                for (int p = 0; p < 4; ++p)
                                    if (at + r_pos + p >= cur.n_keys) t[RING ? 0 : 2 * i + r].v[p] = u32x4{0, 0, 0, 0};
                            }
                        }
                    };
                    // -- values: the lane's dims of a step's four rows as two 16-bit pairs, then O^T += V^T P^T
                    auto values = [&](int r) __attribute__((always_inline)) {      // step r, or with G 2 both
                        if constexpr (!RING) {      // dims {8 i + j}: a v_perm a pair
                            const Tile& tl = t[RING ? 0 : 2 * i + r];
#pragma unroll
                            for (int w = 0; w < 4; ++w) {
                                const uint32_t lo[2] = {__builtin_amdgcn_perm(tl.v[1][w], tl.v[0][w], 0x05040100), __builtin_amdgcn_perm(tl.v[3][w], tl.v[2][w], 0x05040100)};
                                const uint32_t hi[2] = {__builtin_amdgcn_perm(tl.v[1][w], tl.v[0][w], 0x07060302), __builtin_amdgcn_perm(tl.v[3][w], tl.v[2][w], 0x07060302)};
#pragma unroll
                                for (int q = 0; q < QT; ++q) {
                                    acc[q][2 * w] = mfma_steps<F16>(lo, pb[r][q], acc[q][2 * w]);
                                    acc[q][2 * w + 1] = mfma_steps<F16>(hi, pb[r][q], acc[q][2 * w + 1]);
                                }
                            }
                        } else if constexpr (KIND == 0) {      // dims 16 b + (0 .. 15): transposed by the LDS
#pragma unroll
                            for (int b = 0; b < 8 * DH; ++b) {
                                const u32x2 v = read_transposed(places[r] + (uint32_t)HALF + t_read + (t_turn ^ (uint32_t)(32 * (b & 7))) + (uint32_t)(256 * (b >> 3)));
                                const uint32_t va[2] = {v.x, v.y};
#pragma unroll
                                for (int q = 0; q < QT; ++q) acc[q][b] = mfma_steps<F16>(va, pb[r][q], acc[q][b]);
                            }
                        } else {      // dims {8 i + j}: codes of adjacent rows side by side, then as 16-bit pairs
#pragma unroll
                            for (int h = 0; h < DH; ++h) {
                                u32x2 v[G][4];
#pragma unroll
                                for (int p = 0; p < 4; ++p) {
                                    const uint32_t at = (uint32_t)(HALF + (4 * p + u4) * ROWB + 128 * h + 8 * c16);
#pragma unroll
                                    for (int g = 0; g < G; ++g) v[g][p] = *reinterpret_cast<const u32x2*>(places[r + g] + at);
                                }
#pragma unroll
                                for (int w = 0; w < 2; ++w) {
                                    uint32_t va[4][2 * G];
#pragma unroll
                                    for (int g = 0; g < G; ++g) {
                                        // bytes (a0 b0 a1 b1) and (a2 b2 a3 b3): two rows' codes of one dim side by side
                                        const uint32_t lo01 = __builtin_amdgcn_perm(v[g][1][w], v[g][0][w], 0x05010400), hi01 = __builtin_amdgcn_perm(v[g][1][w], v[g][0][w], 0x07030602);
                                        const uint32_t lo23 = __builtin_amdgcn_perm(v[g][3][w], v[g][2][w], 0x05010400), hi23 = __builtin_amdgcn_perm(v[g][3][w], v[g][2][w], 0x07030602);
                                        // (dims 4 w + 0, 1 from the low halves, 2, 3 from the high ones; .x: rows 0, 1; .y: rows 2, 3)
                                        const u32x2 a01 = codes4_to_pairs<KIND>(lo01), a23 = codes4_to_pairs<KIND>(lo23);
                                        const u32x2 b01 = codes4_to_pairs<KIND>(hi01), b23 = codes4_to_pairs<KIND>(hi23);
                                        va[0][2 * g] = a01.x, va[0][2 * g + 1] = a23.x, va[1][2 * g] = a01.y, va[1][2 * g + 1] = a23.y;
                                        va[2][2 * g] = b01.x, va[2][2 * g + 1] = b23.x, va[3][2 * g] = b01.y, va[3][2 * g + 1] = b23.y;
                                    }
#pragma unroll
                                    for (int q = 0; q < QT; ++q) {
#pragma unroll
                                        for (int j = 0; j < 4; ++j) acc[q][8 * h + 4 * w + j] = mfma_steps<F16>(va[j], pb[r][q], acc[q][8 * h + 4 * w + j]);
                                    }
                                }
                            }
                        }
                    };
                    if constexpr (APART) {
#pragma unroll
                        for (int r = 0; r < 2; ++r) scores(r, r + 1), refill_k(r), clean(r), soften(r), move(r), values(r), refill_v(r);
                        return;
                    }
                    keys_here();
                    if constexpr (RING) {
#pragma unroll
                        for (int l = 0; l < CPR / 4; ++l) {
                            const uint32_t at = (k_read ^ (uint32_t)(64 * (l & 3))) + (uint32_t)(256 * (l >> 2));
                            held[0][l] = *reinterpret_cast<const u32x4*>(places[0] + at);
                            held[1][l] = *reinterpret_cast<const u32x4*>(places[1] + at);
                        }
                    }
                    scores(0, 2);
                    if constexpr (KIND >= 2) {
                        const int first = NARROW ? 16 * odd_cur : 0;
#pragma unroll
                        for (int r = 0; r < 2; ++r) {
                            const float* sc = s_scales[wave][2 * i + r];
                            const f32x4 k4 = *reinterpret_cast<const f32x4*>(sc + first + 4 * u4), v4 = *reinterpret_cast<const f32x4*>(sc + SCN / 2 + first + 4 * u4);
#pragma unroll
                            for (int p = 0; p < 4; ++p) ks8[4 * r + p] = k4[p], vs8[4 * r + p] = v4[p];
                        }
                        if (base_b + SPW > cur.n_keys) {      // (scales past the row's keys may be anything)
#pragma unroll
                            for (int p = 0; p < 8; ++p) vs8[p] = (p < 4 ? base : base_b) + r_pos + (p & 3) < cur.n_keys ? vs8[p] : 0.0f;
                        }
                    }
                    if constexpr (RING) wait_lds();
                    refill_k(0), refill_k(1);      // (the keys' places are free: the loads of NP pairs ahead go out)
                    soften(0);
                    if constexpr (G == 1) soften(1);
                    move(0);
                    values_here();
                    clean(0), clean(1);
                    values(0);
                    if constexpr (G == 1) move(1), values(1);
                    if constexpr (RING) wait_lds();
                    refill_v(0), refill_v(1);
                };

                if (part != part_lo) {
                    steps = steps_of(cur, part);
                    resolve(steps);
                    fill(cur, steps);
                }
                Pair at[NP];
#pragma unroll
                for (int i = 0; i < NP; ++i) at[i] = pair_no(cur, steps, i);
                int n = NP;      // the next pair to send for
                if constexpr (RING) {
                    // A pair's keys are sent for again (NP pairs ahead) as soon as its scores are issued, its values as soon as
                    // its second product is; loads return in order, so a wait counts the younger ones that are surely there.
                    queries_here();
                    bool alive = true;
                    while (alive) {
#pragma unroll
                        for (int i = 0; i < NP; ++i) {
                            if (at[i].base < 0) {
                                alive = false;
                                break;
                            }
                            const Pair ahead = pair_no(cur, steps, n);
                            const bool more = ahead.base >= 0;
                            if constexpr (AHEAD) {
                                if (!more && part == part_hi - 1) draw();
                            }
                            const bool follows = NP == 2 && at[NP - 1 - i].base >= 0;
                            step(at[i].base, at[i].second, i,
                                 [&]() __attribute__((always_inline)) { if (follows) wait_dma<NV + NK + NV>(); else wait_dma<NV>(); },
                                 [&]() __attribute__((always_inline)) {
                                     if constexpr (NP == 2) { if (more) wait_dma<NK + NV + NK>(); else if (follows) wait_dma<NK + NV>(); else wait_dma<0>(); }
                                     else { if (more) wait_dma<NK>(); else wait_dma<0>(); }
                                 },
                                 [&](int r) __attribute__((always_inline)) { if (more) fetch_k(cur, r == 0 ? ahead.s0 : ahead.s1, 2 * i + r); },
                                 [&](int r) __attribute__((always_inline)) { if (more) fetch_v(cur, r == 0 ? ahead.s0 : ahead.s1, 2 * i + r); });
                            at[i] = ahead, ++n;
                        }
                    }
                } else if (at[0].base >= 0) {
                    // In registers the compiler counts the loads: the loop's are unconditional (exact waits), the last pair is peeled.
                    static_assert(RING || NP == 1, "one pair in registers");
                    const auto none = [](auto...) {};
                    Pair ahead = pair_no(cur, steps, n);
                    while (ahead.base >= 0) {
                        step(at[0].base, at[0].second, 0, none, none,
                             [&](int r) __attribute__((always_inline)) { fetch_k(cur, r == 0 ? ahead.s0 : ahead.s1, r); },
                             [&](int r) __attribute__((always_inline)) { fetch_v(cur, r == 0 ? ahead.s0 : ahead.s1, r); });
                        at[0] = ahead;
                        ahead = pair_no(cur, steps, ++n);
                    }
                    step(at[0].base, at[0].second, 0, none, none, none, none);
                }
                // The unit's steps are done: the next unit's first keys, values and queries go out before the fold.
                const int fold_col_j0 = cur.j0, fold_kvh0 = cur.kvh0;
                if (part == part_hi - 1) hand_over();

                // A tile's column sums over its four lanes, then the four wavefronts through LDS, in wavefront order; tile
                // after tile (and FW dims after FW dims) through the same arrays. A thread folds FG groups of four dims of one
                // column: what follows the column (its place, the maximum, the four factors) is made once a thread. Four
                // adjacent dims lie together, group g of column c at place g ^ c (the columns' rows start in one bank).
#pragma unroll
                for (int q = 0; q < QT; ++q) {
                    const float l_col = sum_across_quarters(l[q]);
                    const int cc = tid >> 4, g0 = tid & 15;
                    const int head_i = cc / CPH;
                    const int j = fold_col_j0 + q * CPH + cc % CPH;
                    const int c = by_group(j), in_group = j - c * a.g;
                    const int odd = NARROW ? (in_group >= (a.g >> 1) ? 1 : 0) : 0;      // NARROW: the 64 dims of the column's own KV head are kept
                    float M = 0.0f, L = 0.0f, fw[4];
                    float vm = 1.0f;
                    if constexpr (KIND == 1) {
                        if constexpr (NARROW) vm = a.hm ? a.hm[2 * a.hkv + 2 * (fold_kvh0 + head_i) + odd] : a.v_mult;
                        else vm = HW == 1 ? vm_cur[0] : (head_i == 0 ? vm_cur[0] : vm_cur[HW - 1]);
                    }
                    Fold fo = {};
                    // A column folds the partitions that hold its positions, as the merge does.
                    const int held = FUSED ? min(a.parts, pieces_of(min(cur.first + c + 1, a.max_keys))) : 0;
                    auto group = [&](int w, int col_, int g) __attribute__((always_inline)) -> f32x4* { return reinterpret_cast<f32x4*>(&s_acc[w][col_][4 * (g ^ col_)]); };
#pragma unroll
                    for (int sl = 0; sl < D / FW; ++sl) {
                        if (part != part_lo || q > 0 || sl > 0) lds_barrier();      // the fold before has read the LDS
                        if constexpr (RING && KIND == 0) {      // (acc[b][i] = dim 16 b + 4 u4 + i)
#pragma unroll
                            for (int b = 0; b < 4; ++b) *group(wave, c16, 4 * b + u4) = acc[q][4 * sl + b];
                        } else if constexpr (RING) {            // (acc[8 h + j][i] = dim 128 h + 32 u4 + 8 i + j)
                            if ((u4 >> 1) == (sl & 1)) {
#pragma unroll
                                for (int i = 0; i < 4; ++i) {
                                    const f32x4* x = &acc[q][8 * (sl >> 1)];
                                    *group(wave, c16, 8 * (u4 & 1) + 2 * i) = f32x4{x[0][i], x[1][i], x[2][i], x[3][i]};
                                    *group(wave, c16, 8 * (u4 & 1) + 2 * i + 1) = f32x4{x[4][i], x[5][i], x[6][i], x[7][i]};
                                }
                            }
                        } else {
#pragma unroll
                            for (int i = 0; i < 4; ++i) {
                                *group(wave, c16, 8 * u4 + 2 * i) = f32x4{acc[q][0][i], acc[q][1][i], acc[q][2][i], acc[q][3][i]};
                                *group(wave, c16, 8 * u4 + 2 * i + 1) = f32x4{acc[q][4][i], acc[q][5][i], acc[q][6][i], acc[q][7][i]};
                            }
                        }
                        if (sl == 0 && u4 == 0) s_m[wave][c16] = m[q], s_l[wave][c16] = l_col;
                        lds_barrier();
                        if (sl == 0) {
                            M = s_m[0][cc];
#pragma unroll
                            for (int w = 1; w < 4; ++w) M = __builtin_fmaxf(M, s_m[w][cc]);
                            const float sub = M == -INFINITY ? 0.0f : M;
#pragma unroll
                            for (int w = 0; w < 4; ++w) {
                                fw[w] = exp2_fast(s_m[w][cc] - sub);
                                L = __builtin_fmaf(s_l[w][cc], fw[w], L);
                            }
                            if (FUSED && c < cur.count && part < held) {
                                fo = fold(run_m, run_l, M, L);
                                run_m = fo.m, run_l = fo.l;
                            }
                        }
                        f32x4 A[FG];
#pragma unroll
                        for (int i = 0; i < FG; ++i) {
                            A[i] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                            for (int w = 0; w < 4; ++w) {
                                const f32x4 x = *group(w, cc, 16 * i + g0);
#pragma unroll
                                for (int k = 0; k < 4; ++k) A[i][k] = __builtin_fmaf(x[k], fw[w], A[i][k]);
                            }
                            if constexpr (KIND == 1) A[i] *= vm;
                        }
                        if (c >= cur.count) continue;
                        if constexpr (FUSED) {
                            if (part < held) {
#pragma unroll
                                for (int i = 0; i < FG; ++i)
#pragma unroll
                                    for (int k = 0; k < 4; ++k) run_a[FG * sl + i][k] = __builtin_fmaf(run_a[FG * sl + i][k], fo.keep, A[i][k] * fo.take);
                            }
                        } else {
                            const int64_t at = ((int64_t)(cur.prow + c) * a.hq + (fold_kvh0 + head_i) * a.g + in_group) * a.parts + cur.b;
#pragma unroll
                            for (int i = 0; i < FG; ++i) {
                                const int d = FW * sl + 64 * i;      // (NARROW: the half d / 64 of the pair)
                                if (!NARROW || d / 64 == odd) *reinterpret_cast<f32x4_any*>(a.po + at * (NARROW ? 64 : D) + (NARROW ? 0 : d) + 4 * g0) = A[i];
                            }
                            if (sl == 0 && g0 == 0) a.pm[at] = M, a.pl[at] = L;
                        }
                    }
                }
            }
            if constexpr (FUSED) {
                const int cc = tid >> 4, d0 = 4 * (tid & 15);
                const int j = cur.j0 + cc % CPH;
                const int c = by_group(j), in_group = j - c * a.g;
                const int odd = NARROW ? (in_group >= (a.g >> 1) ? 1 : 0) : 0;
                if (c < cur.count) {
                    const int head = (cur.kvh0 + cc / CPH) * a.g + in_group;
                    float M = run_m, L = run_l, keep = 1.0f;
                    if (a.sinks) {
                        const Fold fo = fold(M, L, a.sinks[head] * kLog2e, 1.0f);
                        keep = fo.keep, M = fo.m, L = fo.l;
                    }
                    const int64_t to = (int64_t)(cur.start + c) * a.o_st + (int64_t)head * a.o_sh + d0;
#pragma unroll
                    for (int i = 0; i < D / 64; ++i) {
                        if (NARROW && i != odd) continue;
#pragma unroll
                        for (int k = 0; k < 4; ++k) {
                            const float A = a.sinks ? run_a[i][k] * keep : run_a[i][k];
                            store_out(a.out, a.out_dtype, to + (NARROW ? 0 : 64 * i) + k, L != 0.0f ? A / L : 0.0f);
                        }
                    }
                    if (a.lse && d0 == 0) a.lse[(int64_t)(cur.start + c) * a.hq + head] = L != 0.0f ? __builtin_fmaf(M, kLn2, __logf(L)) : -INFINITY;
                }
            }
        }
        if constexpr (ALONE) break;      // (a unit a workgroup)
        if (!sent) hand_over();      // (nothing to do in this round: the next unit's first rows go out all the same)

        // The unit after the next: the ticket drawn above, or, while it names a unit without work, the ones after it.
        unsigned u_after = u_next + grid;
        if (pulled) {
            if (wave == 0) {      // (the whole wavefront: decode() looks at 64 rows at once)
                unsigned found = 2 * grid + (unsigned)__builtin_amdgcn_readfirstlane((int)drawn);
                while (found < total && !decode(found).valid) {
                    if (lane == 0) drawn = atomicAdd(a.ticket, 1u);
                    found = 2 * grid + (unsigned)__builtin_amdgcn_readfirstlane((int)drawn);
                }
                if (lane == 0) s_unit = found;
            }
            lds_barrier();      // (and every thread is done with the fold's shared arrays)
            u_after = (unsigned)__builtin_amdgcn_readfirstlane((int)s_unit);
        } else {
            lds_barrier();
        }
        if (!nxt.valid && u_next >= total && u_after >= total) break;
        cur = nxt, steps = steps_nxt;
#pragma unroll
        for (int h = 0; h < HW; ++h) vm_cur[h] = vm_nxt[h];
        u_next = u_after;
        lds_barrier();      // every thread has read s_unit before the next round's draw is published
    }
    if constexpr (RING) wait_dma<0>();      // (LDS must not be written for a workgroup that has gone)
    if (!pulled) return;
    if (threadIdx.x == 0) {
        if (atomicAdd(a.ticket + 1, 1u) == grid - 1) {
            atomicExch(a.ticket, 0u);
            atomicExch(a.ticket + 1, 0u);
        }
    }
}

}   // namespace pkv
