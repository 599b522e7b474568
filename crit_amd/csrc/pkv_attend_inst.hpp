// Launch of the split (or fused) kernels for ONE page kind; each pkv_attend_k*.hip instantiates one kind so the
// kinds compile in parallel.
#pragma once
#include "pkv_attend_mfma.hpp"
#include "pkv_attend128.hpp"
#include "pkv_attend_generic.hpp"
#include "pkv_launch.hpp"

namespace pkv {

template <int KIND, bool F16, int QR, bool FUSED>
static int launch_one(const AttendArgs& a, int lpr, bool page16, dim3 grid, hipStream_t stream) {
    // (which tile heights each variant is built for: launch_attend picks among them)
    constexpr bool LISTS = QR == 1 || QR == 4, SPECIAL = QR == 2 || QR == 8;
    if (a.blocks && (FUSED || !LISTS)) return CRIT_PKV_E_GEOMETRY;
    if ((a.derive_table || a.fv) && !SPECIAL) return CRIT_PKV_E_GEOMETRY;
    if constexpr (!FUSED && LISTS) {
        if (a.blocks && a.fast128) {
            // block lists whose steps lie in one block and one page: the bandwidth path walking each column's list
            AttendArgs u = a;
            u.units_x = (int)grid.x, u.units_y = (int)grid.y + kTailClasses - 1;
            const int64_t units = (int64_t)u.units_x * u.units_y;
            if (units > 0x7fffffff) return CRIT_PKV_E_GEOMETRY;
            const int64_t resident = (int64_t)compute_units() * attend_waves(KIND, QR);
            const dim3 pgrid((unsigned)(units < resident ? units : resident));
            if (units <= resident) u.ticket = nullptr;      // (a unit a workgroup: nothing to draw, no counter touched)
            switch (a.heads_per_wave) {
                case 1: hipLaunchKernelGGL((attend128_kernel<KIND, F16, QR, 1, false, true>), pgrid, dim3(256), 0, stream, u); break;
                case 2: hipLaunchKernelGGL((attend128_kernel<KIND, F16, QR, 2, false, true>), pgrid, dim3(256), 0, stream, u); break;
                default: return CRIT_PKV_E_GEOMETRY;
            }
            return hip_code(hipGetLastError());
        }
        if (a.blocks) {      // other block lists: the generic kernel, each position looked up on its own
            switch (lpr) {
                case 2: hipLaunchKernelGGL((attend_generic_kernel<KIND, F16, 2, QR, false, true>), grid, dim3(256), 0, stream, a); break;
                case 4: hipLaunchKernelGGL((attend_generic_kernel<KIND, F16, 4, QR, false, true>), grid, dim3(256), 0, stream, a); break;
                case 8: hipLaunchKernelGGL((attend_generic_kernel<KIND, F16, 8, QR, false, true>), grid, dim3(256), 0, stream, a); break;
                case 16: hipLaunchKernelGGL((attend_generic_kernel<KIND, F16, 16, QR, false, true>), grid, dim3(256), 0, stream, a); break;
                case 32: hipLaunchKernelGGL((attend_generic_kernel<KIND, F16, 32, QR, false, true>), grid, dim3(256), 0, stream, a); break;
                default: return CRIT_PKV_E_GEOMETRY;
            }
            return hip_code(hipGetLastError());
        }
    }
    if constexpr (SPECIAL && KIND == 3 && FUSED) {
        if (a.iqk) {      // INT8 queries against INT8 keys: a prompt chunk's window rows (with or without its own fresh rows)
            switch (a.fv ? lpr : -lpr) {
#define PKV_IQK(L) \
    case L: hipLaunchKernelGGL((attend_generic_kernel<KIND, F16, L, QR, true, false, true, false, true>), grid, dim3(256), 0, stream, a); break; \
    case -L: hipLaunchKernelGGL((attend_generic_kernel<KIND, F16, L, QR, true, false, false, false, true>), grid, dim3(256), 0, stream, a); break;
                PKV_IQK(2) PKV_IQK(4) PKV_IQK(8) PKV_IQK(16) PKV_IQK(32)
#undef PKV_IQK
                default: return CRIT_PKV_E_GEOMETRY;
            }
            return hip_code(hipGetLastError());
        }
    }
    if (a.iqk) return CRIT_PKV_E_GEOMETRY;
    if constexpr (SPECIAL) {
    if (a.derive_table && a.fv) {      // derived keys over pages and fresh value rows
        switch (lpr) {
            case 2: if constexpr (QR == 8) { hipLaunchKernelGGL((attend_generic_kernel<KIND, F16, 2, QR, FUSED, false, true, true>), grid, dim3(256), 0, stream, a); break; } return CRIT_PKV_E_GEOMETRY;
            case 4: if constexpr (QR == 8) { hipLaunchKernelGGL((attend_generic_kernel<KIND, F16, 4, QR, FUSED, false, true, true>), grid, dim3(256), 0, stream, a); break; } return CRIT_PKV_E_GEOMETRY;
            case 8: hipLaunchKernelGGL((attend_generic_kernel<KIND, F16, 8, QR, FUSED, false, true, true>), grid, dim3(256), 0, stream, a); break;
            case 16: hipLaunchKernelGGL((attend_generic_kernel<KIND, F16, 16, QR, FUSED, false, true, true>), grid, dim3(256), 0, stream, a); break;
            case 32: if constexpr (QR == 8) { hipLaunchKernelGGL((attend_generic_kernel<KIND, F16, 32, QR, FUSED, false, true, true>), grid, dim3(256), 0, stream, a); break; } return CRIT_PKV_E_GEOMETRY;
            default: return CRIT_PKV_E_GEOMETRY;
        }
    } else if (a.derive_table) {      // keys derived from the value rows: the generic kernel's variant (any head width; the widths other than 64 and 128 in tiles of 8 rows only)
        switch (lpr) {
            case 2: if constexpr (QR == 8) { hipLaunchKernelGGL((attend_generic_kernel<KIND, F16, 2, QR, FUSED, false, false, true>), grid, dim3(256), 0, stream, a); break; } return CRIT_PKV_E_GEOMETRY;
            case 4: if constexpr (QR == 8) { hipLaunchKernelGGL((attend_generic_kernel<KIND, F16, 4, QR, FUSED, false, false, true>), grid, dim3(256), 0, stream, a); break; } return CRIT_PKV_E_GEOMETRY;
            case 8: hipLaunchKernelGGL((attend_generic_kernel<KIND, F16, 8, QR, FUSED, false, false, true>), grid, dim3(256), 0, stream, a); break;
            case 16: hipLaunchKernelGGL((attend_generic_kernel<KIND, F16, 16, QR, FUSED, false, false, true>), grid, dim3(256), 0, stream, a); break;
            case 32: if constexpr (QR == 8) { hipLaunchKernelGGL((attend_generic_kernel<KIND, F16, 32, QR, FUSED, false, false, true>), grid, dim3(256), 0, stream, a); break; } return CRIT_PKV_E_GEOMETRY;
            default: return CRIT_PKV_E_GEOMETRY;
        }
    } else if (a.fv) {       // fresh rows beside the pages: the generic kernel's variant that reads both (any head width; the widths other than 64 and 128 in tiles of 8 rows only)
        switch (lpr) {
            case 2: hipLaunchKernelGGL((attend_generic_kernel<KIND, F16, 2, QR, FUSED, false, true>), grid, dim3(256), 0, stream, a); break;
            case 4: hipLaunchKernelGGL((attend_generic_kernel<KIND, F16, 4, QR, FUSED, false, true>), grid, dim3(256), 0, stream, a); break;
            case 8: hipLaunchKernelGGL((attend_generic_kernel<KIND, F16, 8, QR, FUSED, false, true>), grid, dim3(256), 0, stream, a); break;
            case 16: hipLaunchKernelGGL((attend_generic_kernel<KIND, F16, 16, QR, FUSED, false, true>), grid, dim3(256), 0, stream, a); break;
            case 32: hipLaunchKernelGGL((attend_generic_kernel<KIND, F16, 32, QR, FUSED, false, true>), grid, dim3(256), 0, stream, a); break;
            default: return CRIT_PKV_E_GEOMETRY;
        }
    }
    if (a.derive_table || a.fv) return hip_code(hipGetLastError());
    }
    if (lpr == 16) {
        hipLaunchKernelGGL((attend_generic_kernel<KIND, F16, 16, QR, FUSED>), grid, dim3(256), 0, stream, a);
    } else if (lpr == 8) {
        hipLaunchKernelGGL((attend_generic_kernel<KIND, F16, 8, QR, FUSED>), grid, dim3(256), 0, stream, a);
    } else if (lpr == 32) {
        hipLaunchKernelGGL((attend_generic_kernel<KIND, F16, 32, QR, FUSED>), grid, dim3(256), 0, stream, a);
    } else if (lpr == 4) {
        hipLaunchKernelGGL((attend_generic_kernel<KIND, F16, 4, QR, FUSED>), grid, dim3(256), 0, stream, a);
    } else if (lpr == 2) {
        hipLaunchKernelGGL((attend_generic_kernel<KIND, F16, 2, QR, FUSED>), grid, dim3(256), 0, stream, a);
    } else {
        return CRIT_PKV_E_GEOMETRY;
    }
    return hip_code(hipGetLastError());
}

// The bandwidth path's kernel for one kind of mask, by the KV heads a wavefront serves, the heads' width and the query
// tiles a workgroup holds.
template <int KIND, bool F16, int MASK>
static int launch_mfma_masked(const AttendArgs& u, bool fused, dim3 grid, hipStream_t stream) {
#define PKV_MFMA(...) hipLaunchKernelGGL((attend_mfma_kernel<KIND, F16, __VA_ARGS__>), grid, dim3(256), 0, stream, u)
    const bool pair = u.heads_per_wave == 2;
    if (fused) {
        if (u.query_tiles != 1) return CRIT_PKV_E_GEOMETRY;
        if (u.narrow) {      // 64-wide heads in pairs
            if (pair) PKV_MFMA(2, true, MASK, 1, 1, true);
            else PKV_MFMA(1, true, MASK, 1, 1, true);
        } else if (u.dk == 256) {
            PKV_MFMA(1, true, MASK, 2);
        } else if (pair) {
            PKV_MFMA(2, true, MASK);
        } else {
            PKV_MFMA(1, true, MASK);
        }
        return hip_code(hipGetLastError());
    }
    if constexpr (MASK != kMaskSliding) {
        if (u.places == kPlacesDeep) {      // (two KV heads a wavefront, or 256-wide ones)
            if (u.dk == 256) {
                if (u.query_tiles == 1) PKV_MFMA(1, false, MASK, 2, 1, false, kPlacesDeep);
                else PKV_MFMA(1, false, MASK, 2, 2, false, kPlacesDeep);
            } else if (u.narrow) {
                PKV_MFMA(2, false, MASK, 1, 1, true, kPlacesDeep);
            } else if (u.query_tiles == 1) {
                PKV_MFMA(2, false, MASK, 1, 1, false, kPlacesDeep);
            } else if (u.query_tiles == 2) {
                PKV_MFMA(2, false, MASK, 1, 2, false, kPlacesDeep);
            } else if constexpr (KIND == 0) {
                if (u.query_tiles == 3) PKV_MFMA(2, false, MASK, 1, 3, false, kPlacesDeep);
                else PKV_MFMA(2, false, MASK, 1, 4, false, kPlacesDeep);
            }
            return hip_code(hipGetLastError());
        }
        if (u.places == kPlacesPlain) {
            if (u.narrow) PKV_MFMA(2, false, MASK, 1, 1, true, kPlacesPlain);
            else if (u.query_tiles == 1) PKV_MFMA(2, false, MASK, 1, 1, false, kPlacesPlain);
            else PKV_MFMA(2, false, MASK, 1, 2, false, kPlacesPlain);
            return hip_code(hipGetLastError());
        }
        if (u.places == kPlacesTwo) {
            if (u.narrow) PKV_MFMA(2, false, MASK, 1, 1, true, kPlacesTwo);
            else if (u.query_tiles == 1) PKV_MFMA(2, false, MASK, 1, 1, false, kPlacesTwo);
            else PKV_MFMA(2, false, MASK, 1, 2, false, kPlacesTwo);
            return hip_code(hipGetLastError());
        }
    }
    if (u.narrow) {
        if (u.query_tiles != 1) return CRIT_PKV_E_GEOMETRY;
        if (pair) PKV_MFMA(2, false, MASK, 1, 1, true);
        else PKV_MFMA(1, false, MASK, 1, 1, true);
        return hip_code(hipGetLastError());
    }
    switch (u.query_tiles) {
        case 1:
            if (u.dk == 256) PKV_MFMA(1, false, MASK, 2);
            else if (pair) PKV_MFMA(2, false, MASK);
            else PKV_MFMA(1, false, MASK);
            return hip_code(hipGetLastError());
        case 2:      // two workgroups a compute unit still (256-wide heads: one)
            if (u.dk == 256) PKV_MFMA(1, false, MASK, 2, 2);
            else if (pair) PKV_MFMA(2, false, MASK, 1, 2);
            else PKV_MFMA(1, false, MASK, 1, 2);
            return hip_code(hipGetLastError());
        case 3:      // split launches of 128-wide heads, one workgroup a compute unit, over 16-bit pages and scaled rows
            if constexpr (KIND != 1) {
                if (u.dk == 256) return CRIT_PKV_E_GEOMETRY;
                if (pair) PKV_MFMA(2, false, MASK, 1, 3);
                else PKV_MFMA(1, false, MASK, 1, 3);
                return hip_code(hipGetLastError());
            }
            break;
        case 4:      // ... over 16-bit pages
            if constexpr (KIND == 0) {
                if (u.dk == 256) return CRIT_PKV_E_GEOMETRY;
                if (pair) PKV_MFMA(2, false, MASK, 1, 4);
                else PKV_MFMA(1, false, MASK, 1, 4);
                return hip_code(hipGetLastError());
            }
            break;
    }
    return CRIT_PKV_E_GEOMETRY;
#undef PKV_MFMA
}

// 128- and 256-wide heads over pages of a multiple of 16 positions: the bandwidth path, resident workgroups pulling units.
template <int KIND, bool F16>
static int launch_mfma(const AttendArgs& a, bool fused, dim3 grid, hipStream_t stream) {
    AttendArgs u = a;
    // (a split launch lists a row's last partition once more for each size class it may fall in)
    u.units_x = (int)grid.x, u.units_y = fused ? (int)grid.y : (int)grid.y + kTailClasses - 1;
    const int64_t units = (int64_t)u.units_x * u.units_y;
    if (units > 0x7fffffff) return CRIT_PKV_E_GEOMETRY;
    u.group_div = make_div32((uint32_t)a.g), u.piece_div = make_div32((uint32_t)a.piece), u.tiles_div = make_div32((uint32_t)a.tiles);
    u.row_div = make_div32((uint32_t)(a.hkv / a.heads_per_wave * a.tiles));
    const int64_t resident = (int64_t)compute_units() * (a.dk == 256 || a.query_tiles > 2 ? 1 : kMfmaWaves);
    dim3 pgrid((unsigned)(units < resident ? units : resident));
    // A unit a workgroup at most: nothing to draw, and no counter touched (a draw's round trip and the count of the
    // finished workgroups are a few microseconds at the end of a launch that is one unit long).
    if (units <= resident) u.ticket = nullptr;
    const int mask = a.sliding > 0 ? kMaskSliding : (a.parents != nullptr || a.parents64 != nullptr ? kMaskTree : kMaskNone);
    // A workgroup a place of the tables ((row, heads, tiles) times partitions), no list of units. Up to a compute unit a place:
    // one workgroup a compute unit, more of its steps in flight (tables longer than their rows have places without work, and
    // more places than compute units may be any launch). One row or two of more places: the ordinary kernels' steps, three
    // workgroups a compute unit of one tile (160 registers and fewer without the list) and two of two tiles, two rows' units
    // by row_place(). One of 200,000, 40 / 8 heads x 128, in splits of 1,024, BF16 166 -> 160 us, FP8 96 -> 89, INT8 101 -> 95; one
    // of 50,000, 56 / 8 heads, a tree of 5, FP8 69 -> 65; 2 rows of 100,000 160 -> 147, of 30,000 and 50,000 67.5 -> 63.8, of
    // 2,000 in tables of 8,192 pages 30.0 -> 17.5, FP8 40.1 -> 28.3. More rows keep the list: by the tables' places, rows that are
    // alike gain and uneven ones lose (3 of 50,000, BF16 / FP8, 116 / 68.5 us, 101 / 63 without it; 4 of 30,000 to 60,000 144 / 74
    // and 145 / 87; 64 of 1,024 to 8,192 209.9 / 113.6 and 239.3 / 120.7). An odd number of KV heads, a wavefront a head, and
    // sliding windows have no such kernels and were not measured.
    const bool places = !fused && (a.dk == 256 || a.heads_per_wave == 2) && (KIND == 0 || a.query_tiles <= 2) && mask != kMaskSliding && grid.y <= 65535;
    u.places = kPlacesNone, u.cus = compute_units();
    if (places && (int64_t)grid.x * grid.y <= compute_units()) u.places = kPlacesDeep;
    else if (places && a.n_rows <= 2 && a.dk == 128 && a.query_tiles <= 2) u.places = a.n_rows == 1 ? kPlacesPlain : kPlacesTwo;
    if (u.places != kPlacesNone) pgrid = grid;
    switch (mask) {
        case kMaskNone: return launch_mfma_masked<KIND, F16, kMaskNone>(u, fused, pgrid, stream);
        case kMaskTree: return launch_mfma_masked<KIND, F16, kMaskTree>(u, fused, pgrid, stream);
        default: return launch_mfma_masked<KIND, F16, kMaskSliding>(u, fused, pgrid, stream);
    }
}

template <int KIND, bool F16>
static int launch_kind_impl(const AttendArgs& a, int lpr, int qr, bool fused, bool page16, dim3 grid, hipStream_t stream) {
    if (a.fast128 && !a.blocks) return launch_mfma<KIND, F16>(a, fused, grid, stream);
    switch (qr) {
#define PKV_CASE(Q)                                                                               \
    case Q:                                                                                       \
        return fused ? launch_one<KIND, F16, Q, true>(a, lpr, page16, grid, stream)               \
                     : launch_one<KIND, F16, Q, false>(a, lpr, page16, grid, stream);
        PKV_CASE(1) PKV_CASE(2) PKV_CASE(4) PKV_CASE(8)
#undef PKV_CASE
    }
    return CRIT_PKV_E_GEOMETRY;
}

}   // namespace pkv
