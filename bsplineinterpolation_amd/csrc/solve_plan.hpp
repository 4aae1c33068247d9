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
// Static LDS of the kernels that call solve_tile, at most: two offsets a
// line and, for each variant the kernel holds, two flags; rounded up to the 16
// bytes at which the dynamic part (the tile) starts.
constexpr int64_t kTileStaticLds = 2 * kMaxTileLines * 8 + 128;

// Row stride of a tile in elements: odd on the contiguous axis, so that
// the coalesced runs along a line spread over the LDS banks, and for
// kTileLines lines on any axis.
constexpr int kTileStep = kTileLines + 1;
__host__ __device__ inline int64_t tile_step(int64_t lpb, int64_t inner) {
    return inner == 1 || lpb == kTileLines ? lpb | 1 : lpb;
}
// Rows before and after the tile, zeroed: a segment's first or last batch
// can read and write past the line's ends.
constexpr int64_t kTilePad = kSegRows;
__host__ __device__ inline int64_t tile_elements(int64_t n, int64_t lpb, int64_t inner) {
    return (n + 2 * kTilePad) * tile_step(lpb, inner);
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
    return (tile_elements(p.n, p.lines_per_block, p.inner) + edge_elements(p.n, bw, p)) * compute_bytes;
}

// The tile for the lines of p (n, nlines, inner and the segment fields set)
// where a workgroup may have max_lds bytes of LDS.
inline TilePlan plan_tile(const SolveParams& p, int bw, bool cyclic, int compute_bytes, int64_t max_lds) {
    TilePlan plan;
    const int64_t n = p.n, inner = p.inner;
    // lines long enough for rows of equal factors (and, cyclic, for the
    // strips' prefix) to matter; shorter ones are substituted plainly
    // (one axis, one segment against plain: n = 97, order 4 20.6 / 17.8 us;
    // n = 150, order 3 28 / 29 us)
    SolveParams cut = p;
    cut.segs = (p.warm > 0 || bw == 0) && n >= kMinSegmentRows && (!cyclic || n >= 2 * p.warm) ? 1 : 0;
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
        const int64_t resident = std::min<int64_t>(std::min<int64_t>(3, kLdsBytes / lds), (tiles + 255) / 256);
        const int64_t rounds = (tiles + 256 * resident - 1) / (256 * resident);
        const int64_t width = inner == 1 ? lpb * compute_bytes : std::max<int64_t>(lpb * compute_bytes, 64);
        const int64_t segs = cut.segs > 0 ? segments(lpb) : 1;
        const double t = rounds * resident * (2.0 * width * n / 20.0 + rows(segs) * 50.0);
        if (plan.lines == 0 || t < best) {
            best = t;
            plan.lines = lpb;
            plan.segs = cut.segs > 0 ? static_cast<int>(segs) : 0;
        }
    }
    if (plan.lines == 0) return plan;
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
