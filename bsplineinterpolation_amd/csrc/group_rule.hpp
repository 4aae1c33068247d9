// group_rule.hpp -- whether a batch of points is grouped by brick before
// evaluation (abi.hip).  Arithmetic only, so that the choice can be checked
// without a device.
#pragma once

#include <algorithm>
#include <cstdint>

namespace intp_amd {

struct GroupCase {
    int dim = 0, order = 0, elem_bytes = 0;  // elements as the evaluation reads them (gradient cells: 16 bytes)
    int64_t elements = 0;                    // of the table
    int64_t npts = 0;
    int launches = 0, results = 0;
    bool one_pass = false;                   // grouped by the one counting pass, not by radix passes
    bool staged = true;                      // radix passes: the bricks' patches fit LDS
    int64_t bricks = 0;
};

// Estimated times, us, in caller order and grouped, of a 3D batch.  In caller
// order a point costs the cache lines of its stencil rows: 4 ps a line from
// L2 (6 ps of gradient cells), 14 ps more for the share of the table beyond it and 1.6 ps beyond the
// 256 MB Infinity Cache.  Grouped, it costs the moving of its record, its results in
// random order, its stencil's elements from LDS (or rows from L2, where the
// patches do not fit), and the caller-order cost of the points that share
// their brick with too few others.  Fitted to 765 pairs of measured times
// (tables of 30^3 to 512^3, orders 0 to 5, both element types, 40,000 to 17M
// points): choosing by them costs 0.6 % over the better of each pair on
// average (us, caller order / grouped: cubic 512^3, 2^24 points, value and
// partials 6274 / 3059; order 1, 256^3, 2^20 points, value 94 / 137; order 5, 100^3,
// 131,072 points, value and partials 63 / 98, 400,000 points 185 / 134).
struct GroupTimes {
    double caller_order, grouped;
};

inline GroupTimes group_times(const GroupCase& c) {
    const double table = static_cast<double>(c.elements) * c.elem_bytes, n = static_cast<double>(c.npts) * 1e-6;
    auto beyond = [&](double bytes) { return table > bytes ? 1.0 - bytes / table : 0.0; };
    const double l2 = beyond(0x1.4p22), cache = beyond(0x1p28);
    const int row = c.order + 1;
    const double lines = static_cast<double>(row) * row * (1.0 + c.order * c.elem_bytes / 128.0);
    const double stencil = static_cast<double>(c.launches) * c.elem_bytes * row * row * row;
    const double share = static_cast<double>(c.bricks) / static_cast<double>(std::max<int64_t>(1, c.npts));
    const bool cells = c.elem_bytes == 16;
    GroupTimes t;
    t.caller_order = 10.0 + n * c.launches * lines *
                                (4.05 * (cells ? 1.4 : 1.0) + 14.1 * l2 + 1.65 * cache) * (cells ? 1.1 : 1.0);
    if (c.one_pass)
        t.grouped = 45.0 + n * (20.3 + 6.8 * c.results + 0.057 * stencil + 11.7 * l2 + 92.0 * cache) +
                    0.02 * static_cast<double>(c.bricks) + t.caller_order * std::min(1.0, 26.0 * share);
    else
        t.grouped = 49.0 + n * (41.0 + 6.9 * c.results + 0.018 * stencil + 21.0 * l2 + 44.0 * cache +
                                (c.staged ? 0.0 : c.launches * 6.3 * lines - 28.0)) +
                    t.caller_order * std::min(1.0, 8.2 * share);
    return t;
}

// Batches that group_pays is asked about: at 2.1 ns a point, the most it can
// cost, fewer do not pay.  Calls on the fixed buffer use it from 2^20 points
// on; smaller ones leave it alone.
inline bool group_considered(int64_t npts, int launches, bool fixed_buffer) {
    return npts * launches >= 32768 && (!fixed_buffer || npts >= (int64_t{1} << 20));
}

// 2D stencils have k + 1 rows only: 2D tables gain beyond the 256 MB
// Infinity Cache, from 2^20 points on (2^24 points on 1024^2, cubic: 0.87
// ms in caller order, 2.15 ms grouped).
inline bool group_pays(const GroupCase& c) {
    if (c.dim != 3) return c.npts >= (int64_t{1} << 20) && static_cast<double>(c.elements) * c.elem_bytes >= 0x1p28;
    const GroupTimes t = group_times(c);
    return t.caller_order > t.grouped;
}

}  // namespace intp_amd
