// solve_plan.hpp -- host-side choices of the line solves: the shape of a tile
// and what it takes of LDS.  Arithmetic only (no HIP calls), so that the
// choices can be checked without a device.
#pragma once

#include <algorithm>

#include "kernels.hpp"

namespace intp_amd {

constexpr int kTileThreads = 256;
constexpr int kMaxTileThreads = 512;
constexpr int kTileLines = 32;
constexpr int kMaxTileLines = 64;
constexpr int kSegRows = 8;  // segments and warm-ups are multiples of this

// LDS of a workgroup on gfx950, and of one of two workgroups that share a CU.
constexpr int64_t kLdsBytes = 160 * 1024;
constexpr int64_t kTileLdsBudget = 80 * 1024;
// Static LDS of the kernels that call solve_tile, at most: one offset a
// line and two flags, a pair for each variant that the batch's merged kernel
// holds; rounded up to the 16 bytes at which the dynamic part (the tile)
// starts.
constexpr int64_t kTileStaticLds = kMaxTileLines * 8 + 16;
constexpr int64_t kBatchStaticLds = kMaxTileLines * 8 + 128;

// Row stride of a tile in elements: odd on the contiguous axis, so that
// the coalesced runs along a line spread over the LDS banks, and for
// kTileLines lines on any axis.
constexpr int kTileStep = kTileLines + 1;
__host__ __device__ inline int64_t tile_step(int64_t lpb, int64_t inner) {
    return inner == 1 || lpb == kTileLines ? lpb | 1 : lpb;
}
// Rows before and after a tile cut into segments, zeroed: a segment's first
// or last batch can read and write past the line's ends.
constexpr int64_t kTilePad = kSegRows;
__host__ __device__ inline int64_t tile_pad(int segs) { return segs > 0 ? kTilePad : 0; }
__host__ __device__ inline int64_t tile_elements(int64_t n, int64_t lpb, int64_t inner, int segs) {
    return (n + 2 * tile_pad(segs)) * tile_step(lpb, inner);
}

// Factors of the rows outside [flo, fhi) and [blo, bhi), with one row of
// each range for the rest, staged in LDS after the tile: a few rows on a
// uniform grid.  On grids where that is more than kEdgeMax elements (the
// non-uniform ones) nothing is staged and every row reads global memory.
constexpr int kEdgeMax = 1024;

__host__ __device__ inline int edge_elements(int64_t n, int bw, const SolveParams& sp) {
    const int64_t e = (sp.flo + 1 + n - sp.fhi) * bw + (sp.blo + 1 + n - sp.bhi) * (bw + 1);
    return sp.segs > 0 && e <= kEdgeMax ? static_cast<int>(e) : 0;
}

// Dynamic LDS of a tile of p.lines_per_block lines.
inline int64_t tile_lds(const SolveParams& p, int bw, int compute_bytes) {
    return (tile_elements(p.n, p.lines_per_block, p.inner, p.segs) + edge_elements(p.n, bw, p)) * compute_bytes;
}

// Workgroups whose LDS a CU holds: it is given out in 1280-byte granules (a
// contiguous cubic axis in whole lines, 32 a tile: at 200 rows with 53,328
// bytes, three a CU, 66 us; with 53,840, two, 89).
inline int64_t resident_by_lds(int64_t lds) { return kLdsBytes / ((lds + 1279) / 1280 * 1280); }

// Estimated time of one axis, us, by the ways to solve its lines: plain
// tiles, tiles of one segment a line, tiles cut into segments, the same where comparisons fail in every
// tile (which are then solved again in one piece), and in place in HBM with
// a lane a line.  Fitted to kernel times of 190 axes (both element types,
// orders 2 to 7, 16 to 4000 rows, 500 to 10^5 lines; most within 15 %): a
// tile of up to 32 lines takes its rows' chain, so what counts is the rounds
// of tiles that the chip takes at once; in place, a launch of few
// lines waits for its chain from HBM, and one of many moves the table four
// times.
struct LineTimes {
    double plain = 0, one = 0, cut = 0, failed = 0, in_place = 0;
};

inline LineTimes line_times(const SolveParams& p, int bw, bool cyclic, int compute_bytes) {
    const bool f64 = compute_bytes == 8;
    const double n = static_cast<double>(p.n);
    // workgroups a CU: by LDS and, 256 threads each, by the kernels' registers
    auto rounds = [&](int segs, int threads) {
        const int by_registers = segs == 0 ? (f64 && (bw == 4 || (cyclic && bw == 2)) ? 2 : f64 && bw == 3 && !cyclic ? 3 : 4)
                                 : f64     ? (cyclic || bw >= 3 ? 2 : 3)
                                           : (cyclic || bw >= 3 ? 3 : 4);
        SolveParams q = p;
        q.segs = segs;
        const int64_t lds = tile_lds(q, bw, compute_bytes) + kTileStaticLds;
        const int64_t resident = std::max<int64_t>(1, std::min<int64_t>(by_registers * 256 / threads, resident_by_lds(lds)));
        const int64_t tiles = (p.nlines + p.lines_per_block - 1) / p.lines_per_block;
        // a last round that is not full overlaps the one before in part
        const int64_t whole = (tiles + 256 * resident - 1) / (256 * resident);
        return std::max(1.0, 0.5 * (static_cast<double>(whole) + static_cast<double>(tiles) / (256.0 * resident)));
    };
    LineTimes t;
    const double copy = (p.inner == 1 ? 4.0 : 0.0) + (p.lines_per_block > kTileLines ? 0.08 * n : 0.0);
    const double row = f64 ? (cyclic ? 0.13 + 0.055 * bw : 0.12 + 0.01 * bw) : (cyclic ? 0.1 + 0.04 * bw : 0.09 + 0.008 * bw);
    t.plain = rounds(0, kTileThreads) * (3.5 + copy + row * n);
    t.one = rounds(1, kTileThreads) * (3.5 + copy + (cyclic ? 0.78 : 0.88) * row * n);
    if (p.segs > 1) {
        const double rows = p.warm + (n + p.segs - 1) / p.segs;
        const double cut_row = (f64 ? (cyclic ? 0.1 + 0.03 * bw : 0.07 + 0.012 * bw) : (cyclic ? 0.07 + 0.03 * bw : 0.06 + 0.01 * bw)) +
                               (p.fast_divide ? 0.0 : 0.06);
        t.cut = rounds(p.segs, std::max(64, p.segs * p.lines_per_block)) *
                ((f64 || cyclic ? 9.0 : 6.0) + copy + 0.012 * n + cut_row * rows);
        t.failed = t.cut + 0.6 * t.plain;
    }
    const double chain = f64 ? 0.2 * (cyclic ? 0.75 + 0.3 * bw : 0.82 + 0.09 * bw) : 0.105 * (cyclic ? 1.0 + 0.4 * bw : 0.66 + 0.18 * bw);
    const double table = n * static_cast<double>(p.nlines) * compute_bytes;
    t.in_place = std::max(4.0 + chain * n, 5.0 + 4.0 * table / 7.2e6);
    // sums to add elsewhere are a pass of their own
    if (p.accum) t.in_place += 4.0 + 3.0 * table / 5e6;
    return t;
}

// How the lines of p (n, nlines, inner and the segment fields set, and accum
// where the results are added) are solved where a workgroup may have max_lds
// bytes of LDS.
inline TilePlan plan_tile(const SolveParams& p, int bw, bool cyclic, int compute_bytes, int64_t max_lds) {
    TilePlan plan;
    const int64_t n = p.n, inner = p.inner;
    // lines long enough for rows of equal factors (and, cyclic, for the
    // strips' prefix) to matter; shorter ones are substituted plainly
    // (one axis, one segment against plain: n = 97, order 4 20.6 / 17.8 us;
    // n = 150, order 3 28 / 29 us)
    SolveParams cut = p;
    const bool can_cut = (p.warm > 0 || bw == 0) && n >= kMinSegmentRows && (!cyclic || n >= 2 * p.warm);
    cut.segs = can_cut ? 1 : 0;
    auto bytes = [&](int64_t lpb) {
        cut.lines_per_block = static_cast<int32_t>(lpb);
        return tile_lds(cut, bw, compute_bytes) + kTileStaticLds;
    };
    // Segments for a tile of lpb lines: one per thread and line of 256
    // threads, halved while that costs few rows (fewer warm-ups), and one
    // where the warm-ups would not pay.
    auto rows = [&](int64_t segs) { return segs == 1 ? n : p.warm + ((n + segs - 1) / segs + 7) / 8 * 8; };
    auto segments = [&](int64_t lpb) -> int64_t {
        int64_t segs = kTileThreads / lpb;
        while (segs > 1 && (segs * 8 > n || rows(segs / 2) <= rows(segs) + rows(segs) / 8)) segs /= 2;
        return segs > 1 && segs >= bw && 4 * rows(segs) <= 3 * n ? segs : 1;
    };
    // Lines per tile: the least estimated time over the rounds of resident
    // workgroups.  A round copies its tiles (20 B/ns per CU; strided rows
    // move whole 64-byte sectors) and substitutes rows(segs) rows twice at
    // about 25 ns (60 cycles), workgroups on one CU sharing its SIMDs.
    // Measured against every choice from 4 to 32 lines on the grids of 1 to
    // 3 dimensions from 700 x 900 to 256^3: within 5 % of the fastest.
    double best = 0.0;
    for (int lpb = kTileLines; lpb >= 1; lpb /= 2) {
        const int64_t lds = bytes(lpb);
        if (lds > std::min(kLdsBytes, max_lds)) continue;
        if (inner >= 64 && lpb < 4) continue;  // in HBM instead
        const int64_t tiles = (p.nlines + lpb - 1) / lpb;
        const int64_t resident = std::min<int64_t>(std::min<int64_t>(3, resident_by_lds(lds)), (tiles + 255) / 256);
        const int64_t rounds = (tiles + 256 * resident - 1) / (256 * resident);
        const int64_t width = inner == 1 ? lpb * compute_bytes : std::max<int64_t>(lpb * compute_bytes, 64);
        const int64_t segs = can_cut ? segments(lpb) : 1;
        const double t = rounds * resident * (2.0 * width * n / 20.0 + rows(segs) * 50.0);
        if (plan.lines == 0 || t < best) {
            best = t;
            plan.lines = lpb;
            plan.segs = can_cut ? static_cast<int>(segs) : 0;
        }
    }
    if (plan.lines == 0) return plan;
    // uncut tiles that the chip holds at once: nothing is faster
    if (!can_cut && p.nlines <= 256 * plan.lines) return plan;
    cut.lines_per_block = plan.lines;
    cut.segs = plan.segs;
    const LineTimes t = line_times(cut, bw, cyclic, compute_bytes);
    // Segments start from states that the rows before them must reproduce.
    // Data decides whether they do: fields that decay faster than the factors
    // fade (a Gaussian, zeros after a box) fail in many tiles, which are then
    // solved twice.  Lines are cut where that gains though every second tile
    // fails (256^3 cubic, the contiguous axis, us: plain 146, cut 92 on noise
    // and 179 on a Gaussian; order 5: 167, 150, 244, so plain).  In FP32 every
    // fourth: half of those solves are corrections, whose right-hand sides are
    // rounding errors, and noise does not fail (order 5, 256^3 refined, the
    // build, us: plain 575 on any data, cut 535 on noise, 574 on a Gaussian).
    const double fails = compute_bytes == 4 ? 0.25 : 0.5;
    const double expected = t.cut + fails * (t.failed - t.cut);
    const bool cut_pays = plan.segs > 1 && expected < t.plain;
    double tiled = cut_pays ? expected : t.plain;
    if (!cut_pays) {
        // uncut, a tile keeps one lane a line busy: as many lines as take the
        // fewest rounds (order 5, 144 rows, 20736 contiguous lines: 32 lines
        // 53 us, 64 lines 48)
        SolveParams whole = p;
        for (int lpb = plan.lines * 2; lpb <= kMaxTileLines; lpb *= 2) {
            whole.lines_per_block = lpb;
            if (tile_lds(whole, bw, compute_bytes) + kTileStaticLds > std::min(kLdsBytes, max_lds)) break;
            const double plain = line_times(whole, bw, cyclic, compute_bytes).plain;
            if (plain < 0.93 * tiled) {
                tiled = plain;
                plan.lines = lpb;
            }
        }
        // one segment has nothing to compare, and its rows of equal factors
        // and its division are cheaper; wide bands lose that to the kernel's
        // registers
        plan.segs = 0;
        if (can_cut && plan.lines <= kTileLines && (cyclic || (p.fast_divide && bw <= 2))) {
            whole.lines_per_block = plan.lines;
            const double one = line_times(whole, bw, cyclic, compute_bytes).one;
            if (one < tiled) {
                tiled = one;
                plan.segs = 1;
            }
        }
    }
    // 64 or more lines side by side make in-place rows coalesced
    // (order 5, 64 rows, 65536 lines: tiles 46 us, in place 22; cubic, 256
    // rows, 65536 lines: 78 and 77, and 149 where the tiles fail; 100 rows,
    // 10^4 lines: 17.6 and 25.5)
    if (inner >= 64 && t.in_place < tiled) {
        plan.lines = plan.segs = 0;
        plan.in_place = true;
        return plan;
    }
    plan.threads = plan.segs <= 1 ? kTileThreads : std::max(64, plan.segs * plan.lines);
    return plan;
}

// Lines too long for a tile, in chunks (solve_long.hip): lines per workgroup
// and its threads, segments of len rows per line, rows and number of chunks.
// lpb 0: not even one line fits.
struct LongShape {
    int lpb = 0, threads = 0, segs = 0, len = 0, rows = 0, chunks = 0;
};

constexpr int kLongThreads = 128;  // contiguous lines (lpb 1); 256 for lines side by side
constexpr int kStridedLen = 32;
// Static LDS of the chunk kernels, at most: three arrays of an entry a line
// and a flag.
constexpr int64_t kLongStaticLds = 3 * kMaxTileLines * 8 + 16;

// Dynamic LDS of a chunk's workgroup: its rows, the warm-up before them and a
// pad on both sides, and the staged factors.
inline int64_t long_lds(const SolveParams& p, int bw, const LongShape& s, int compute_bytes) {
    SolveParams cut = p;
    cut.segs = s.segs;
    return ((s.rows + p.warm + 2 * kTilePad) * tile_step(s.lpb, p.inner) + edge_elements(p.n, bw, cut)) * compute_bytes;
}

inline LongShape plan_long(const SolveParams& p, int bw, bool cyclic, int compute_bytes) {
    int lpb = 1;
    if (p.inner > 1)
        while (lpb < kTileLines && 2 * lpb <= p.inner) lpb *= 2;
    // fewer lines side by side where a long warm-up (352 rows on nodes graded
    // by 5 % a cell, order 7; at most 400) leaves no room for 32
    for (; lpb >= 1; lpb /= 2) {
        LongShape s;
        s.lpb = lpb;
        s.threads = lpb == 1 ? kLongThreads : 256;
        s.segs = s.threads / lpb;
        s.len = s.segs <= 8 ? kStridedLen : kSegRows;
        s.rows = s.segs * s.len;
        const int64_t H = cyclic ? p.n - bw : p.n;
        s.chunks = static_cast<int>((H + s.rows - 1) / s.rows);
        if (long_lds(p, bw, s, compute_bytes) + kLongStaticLds <= kLdsBytes) return s;
    }
    return LongShape{};
}

}  // namespace intp_amd
