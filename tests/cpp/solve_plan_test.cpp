// The host-side choices of the line solves (solve_plan.hpp): no plan may ask
// for more LDS than a workgroup has.

#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <vector>

#include "grid.hpp"
#include "solve_plan.hpp"

using namespace intp_amd;

namespace {

int failures = 0;

void check(bool ok, const char* what, int order, int periodic, int bytes, int64_t n, int64_t inner, int64_t value) {
    if (ok) return;
    if (++failures <= 20)
        std::printf("%s: order %d periodic %d bytes %d n %lld inner %lld: %lld\n", what, order, periodic, bytes,
                    static_cast<long long>(n), static_cast<long long>(inner), static_cast<long long>(value));
}

// Solve parameters of a dimension of n points, from the setup of a shorter
// one: on a uniform grid the rows of unequal factors at both ends stay as
// they are.
SolveParams stretched(const DimSetup& s, bool f32, int64_t n, int64_t inner, int64_t nlines) {
    SolveParams p{};
    set_segment_params(f32 ? s.lu.seg32 : s.lu.seg64, &p);
    const int more = static_cast<int>(n - s.n);
    if (p.fhi > p.flo + 1) p.fhi += more;
    if (p.bhi > p.blo + 1) p.bhi += more;
    p.n = n;
    p.inner = inner;
    p.nlines = nlines;
    return p;
}

// Static LDS the kernels are built with is at most `static_lds` (read from
// the code objects by the caller).
void tiles(int64_t static_lds) {
    for (int order = 1; order <= 7; ++order)
        for (int periodic = 0; periodic < 2; ++periodic)
            for (int f32 = 0; f32 < 2; ++f32) {
                const int bytes = f32 ? 4 : 8;
                DimSetup s;
                if (!setup_dimension(order, periodic != 0, 3000, 0.0, 1.0, nullptr, s, true).empty()) std::abort();
                const struct { int64_t inner, nlines; } lines[] = {{1, 1}, {1, 3}, {1, 70}, {3, 3}, {17, 34}, {64, 640}, {300, 300}};
                for (const auto& l : lines)
                    for (int64_t n = 3000; n < 42000; ++n) {
                        const SolveParams base = stretched(s, f32 != 0, n, l.inner, l.nlines);
                        SolveParams p = base;
                        const TilePlan plan = plan_tile(p, s.lu.p, s.lu.cyclic, bytes, kLdsBytes);
                        if (plan.lines == 0) continue;
                        p.lines_per_block = plan.lines;
                        p.segs = plan.segs;
                        const int64_t lds = (tile_lds(p, s.lu.p, bytes) + 15) / 16 * 16 + static_lds;
                        check(lds <= kLdsBytes, "tile LDS", order, periodic, bytes, n, l.inner, lds);
                    }
            }
}

// Lines too long for a tile: every warm-up that segment_plan can give (at
// most 400 rows), and nodes whose factors fade slowly.
void chunks(int64_t static_lds) {
    for (int bw = 0; bw <= 6; ++bw)
        for (int cyclic = 0; cyclic < 2; ++cyclic)
            for (int bytes : {4, 8})
                for (int64_t inner : {1, 2, 3, 15, 16, 31, 32, 63, 64, 70, 1000})
                    for (int warm = 0; warm <= 400; warm += 8)
                        for (int edge = 1; edge < 200; edge += 11) {
                            SolveParams p{};
                            p.warm = warm;
                            p.inner = inner;
                            p.nlines = inner * 2;
                            p.n = 30000;
                            p.flo = p.blo = edge;
                            p.fhi = p.bhi = 30000 - edge;
                            const LongShape s = plan_long(p, bw, cyclic != 0, bytes);
                            check(s.lpb > 0 && s.rows % kSegRows == 0 && s.threads == s.segs * s.lpb, "chunk shape", bw, cyclic, bytes,
                                  warm, inner, s.lpb);
                            const int64_t lds = (long_lds(p, bw, s, bytes) + 15) / 16 * 16 + static_lds;
                            check(lds <= kLdsBytes, "chunk LDS", bw, cyclic, bytes, warm, inner, lds);
                        }
    std::vector<double> x;
    for (int i = 0; i < 6000; ++i) x.push_back(i == 0 ? 0.0 : x.back() + std::pow(1.05, std::min(i % 400, 400 - i % 400)));
    DimSetup s;
    if (!setup_dimension(7, false, 6000, 0.0, 1.0, x.data(), s, true).empty()) std::abort();
    check(s.lu.seg64.warm > 340, "warm-up of graded nodes", 7, 0, 8, 6000, 64, s.lu.seg64.warm);
}

// How lines are solved where the fastest way is clear from measurement: cut
// where few lines leave the chip idle, in place where many lie side by side.
void choices() {
    enum { kCut, kWhole, kInPlace };
    const struct {
        int order, periodic;
        int64_t n, nlines, inner;
        int want;
        bool f32 = false;
    } cases[] = {
        {3, 0, 8192, 1, 1, kCut},         {6, 1, 8192, 1, 1, kCut},         {3, 0, 2000, 2000, 1, kCut},
        {3, 0, 2000, 2000, 2000, kCut},   {5, 0, 1021, 769, 769, kCut},     {3, 0, 1000, 4096, 64, kCut},
        {3, 0, 256, 65536, 1, kCut},      {5, 0, 256, 65536, 1, kWhole},    {7, 0, 200, 40000, 1, kWhole},
        {3, 0, 256, 65536, 256, kInPlace}, {5, 0, 256, 65536, 65536, kInPlace}, {7, 0, 180, 32400, 180, kInPlace},
        {6, 1, 180, 32400, 180, kInPlace}, {5, 0, 64, 65536, 65536, kInPlace}, {5, 0, 100, 50000, 100, kInPlace},
        {3, 0, 20, 90000, 300, kInPlace},  {3, 0, 100, 10000, 100, kWhole},  {5, 0, 80, 6400, 80, kWhole},
        {3, 0, 64, 64, 64, kWhole},        {3, 0, 64, 4096, 64, kWhole},
        {3, 0, 200, 40000, 1, kWhole},      {3, 0, 204, 41616, 1, kCut},
        {5, 0, 256, 65536, 1, kCut, true}, {5, 0, 256, 65536, 256, kInPlace, true},
    };
    for (const auto& c : cases) {
        DimSetup s;
        if (!setup_dimension(c.order, c.periodic != 0, c.n, 0.0, 1.0, nullptr, s, true).empty()) std::abort();
        SolveParams p{};
        set_segment_params(c.f32 ? s.lu.seg32 : s.lu.seg64, &p);
        p.n = c.n;
        p.nlines = c.nlines;
        p.inner = c.inner;
        const TilePlan plan = plan_tile(p, s.lu.p, s.lu.cyclic, c.f32 ? 4 : 8, kLdsBytes);
        const int got = plan.in_place ? kInPlace : plan.lines == 0 ? -1 : plan.segs > 1 ? kCut : kWhole;
        check(got == c.want, "choice", c.order, c.periodic, 8, c.n, c.inner, got);
    }
}

}  // namespace

// Lines that are never cut get no segment plan; others do, also where their
// factors differ from row to row.
void segment_plans() {
    for (int order = 2; order <= 7; ++order)
        for (int periodic = 0; periodic < 2; ++periodic)
            for (int uniform = 0; uniform < 2; ++uniform)
                for (int64_t n : {int64_t{20}, kMinSegmentRows - 1, kMinSegmentRows, int64_t{1000}}) {
                    std::vector<double> x(static_cast<size_t>(n + 1));
                    for (int64_t i = 0; i <= n; ++i) x[static_cast<size_t>(i)] = 0.3 * i + 0.1 * ((i * 7) % 3);
                    DimSetup s;
                    if (!setup_dimension(order, periodic != 0, n, -0.4, 1.7, uniform ? nullptr : x.data(), s, true).empty())
                        std::abort();
                    for (const SegmentPlan* seg : {&s.lu.seg64, &s.lu.seg32})
                        check((seg->warm > 0) == (n >= kMinSegmentRows) && seg->warm % 8 == 0, "warm-up", order, periodic,
                              seg == &s.lu.seg64 ? 8 : 4, n, uniform, seg->warm);
                }
}

int main(int argc, char** argv) {
    tiles(argc > 1 ? std::atoll(argv[1]) : kTileStaticLds);
    choices();
    segment_plans();
    chunks(argc > 2 ? std::atoll(argv[2]) : kLongStaticLds);
    check(argc < 4 || std::atoll(argv[3]) <= kBatchStaticLds, "batch kernels' static LDS", 0, 0, 0, 0, 0, argc < 4 ? 0 : std::atoll(argv[3]));
    if (failures) std::printf("%d failures\n", failures);
    return failures ? 1 : 0;
}
