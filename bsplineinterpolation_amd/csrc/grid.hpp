// grid.hpp -- kernel parameters of one grid dimension from its host setup
// (shared by the single-spline and the batched entry points).
#pragma once

#include "kernels.hpp"
#include "setup.hpp"

namespace intp_amd {

// `stride`: elements between neighbouring control points along the
// dimension; the table pointers (knots, reciprocals, polynomials) are the
// caller's device copies.
inline DimParams make_dim_params(const DimSetup& s, int order, int64_t stride, const double* knots,
                                 const double* recip, const double* poly) {
    DimParams p{};
    p.knots = knots;
    p.recip = recip;
    p.n = s.n;
    p.stride = stride;
    p.nt = static_cast<int32_t>(s.knots.size());
    p.periodic = s.periodic ? 1 : 0;
    p.uniform = s.uniform ? 1 : 0;
    p.lo = s.lo;
    p.hi = s.hi;
    p.period = s.hi - s.lo;
    p.inv_dx = s.uniform ? 1.0 / s.dx : 0.0;
    p.shift = s.periodic ? 1.0 : 0.5 * static_cast<double>(order + 1);
    p.xmin = s.xmin;
    p.xmax = s.xmax;
    p.dx = s.dx;
    p.half = s.half;
    p.poly = poly;
    p.nleft = s.nleft;
    p.nright = s.nright;
    p.nclass = s.nclass;
    return p;
}

// The segment fields of a line solve.
#ifdef __HIPCC__
__host__ __device__
#endif
inline void set_segment_params(const SegmentPlan& seg, SolveParams* sp) {
    sp->warm = seg.warm;
    sp->flo = seg.flo;
    sp->fhi = seg.fhi;
    sp->blo = seg.blo;
    sp->bhi = seg.bhi;
    sp->fast_divide = seg.fast_divide ? 1 : 0;
    sp->zh = seg.zh;
    sp->zl = seg.zl;
    sp->strip_rest = seg.strip_rest;
    for (int m = 0; m < kMaxOrder; ++m) {
        sp->eq_lower[m] = seg.eq_lower[m];
        sp->eq_upper[m] = seg.eq_upper[m];
    }
}

}  // namespace intp_amd
