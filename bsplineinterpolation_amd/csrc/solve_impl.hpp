// solve_impl.hpp -- control-point solve on gfx950 (device code shared by
// solve.hip and the batched kernels of batch.hip): every grid line of one axis
// is an independent band (or cyclic band) system sharing one LU
// factorization (InterpolationTemplate.hpp:448-580).
//
// solve_tile: a workgroup copies up to 64 lines into LDS with coalesced
// loads, substitutes them there, whole or cut into segments of one lane
// each (solve_segments), and writes the tile back.  The first pass reads
// the caller's values with the periodic index shift applied
// (InterpolationTemplate.hpp:452-462), so no separate copy precedes it.
// Lines too long for LDS are cut into chunks first (solve_long.hip); strided
// axes with many lines are substituted in HBM, one line per lane.
//
// What bounds it.  Substituting a line is a chain of dependent rows: 16
// cycles forward (order 3), and backward 16 and an IEEE division of 70.
// With one lane per line a CU held at most 64 chains (its LDS full of
// lines), and one 1D line kept one lane of the chip busy.  Segments put 8
// lanes or more on a line; the division by a pivot that repeats takes two
// operations (KnownDivisor); rows whose factors repeat take them from
// scalar registers.  Whole solves, before -> after:
//   1D 8192 cubic 643 -> 50 us (clamped), order 6 periodic FP32 storage,
//   two solves, 3314 -> 199 us; 2D 1021 x 769 order 5 364 -> 72 us, 2000^2
//   cubic 655 -> 83 us; 3D 128^3 cubic 102 -> 81 us, 256^3 cubic 300 -> 256
//   us (the contiguous axis 101 us, of which copying the tile in and out is
//   44, 6.1 TB/s; the strided ones 75 us each in place).
//
// The substitution is the reference's (BandLU.hpp:121-143, 216-259)
// reordered by rows: each entry receives the same updates in the same
// order.  Built without FMA contraction and with correctly rounded
// divisions, the result is bit-identical to the reference's.
#pragma once

#include <hip/hip_runtime.h>

#include "solve_plan.hpp"

namespace intp_amd {

namespace {

constexpr int kSolveBlock = 256;

// Elements a lane moves per batch: their loads (values and factor
// coefficients) are issued together, then substituted in order, then
// stored.
constexpr int kBatch = 8;
// Loads of a tile copy in flight per thread.
constexpr int kCopyBatch = 8;

template <int BW, bool CYC, typename C>
struct LineState {
    C hist[BW + 1];    // forward: hist[m-1] = y[j-m]
    C acc[BW + 1];     // forward: rows n-BW+r of a cyclic matrix, strip-updated
    C nxt[BW + 1];     // backward: nxt[m-1] = x[j+m]
    C corner[BW + 1];  // backward: x[n-BW+c]
};

// A zero the compiler cannot see through, held in a vector register.  The
// factor coefficients are the same for every lane, so without it they
// would be read with scalar loads, whose completion counter is shared with
// LDS reads and not ordered: every batch would then wait for all loads in
// flight, including the next batch's.  Offset by this zero they are
// vector loads, which complete in order, so the next batch stays in
// flight while the current one is substituted.
__device__ __forceinline__ int32_t lane_zero() {
    int32_t z;
    asm volatile("v_mov_b32 %0, 0" : "=v"(z));
    return z;
}

// Factor coefficients live in global memory.  Pointers read from a
// spline record (the batched kernels) are generic, and generic loads are
// flat loads, which count on the LDS counter as well: the same waits as
// scalar loads.  The explicit address space keeps them global loads.
template <typename C>
using GlobalPtr = const __attribute__((address_space(1))) C*;

template <typename C>
__device__ __forceinline__ GlobalPtr<C> factor_ptr(const void* p, int32_t z) {
    return (GlobalPtr<C>)(p) + z;
}

// Registers of one batch of forward rows: the loaded right-hand sides and
// the factor coefficients of those rows.
template <int BW, bool CYC, typename C, int B>
struct ForwardBatch {
    C xb[B];
    C lc[B][BW + 1];
    C sc[B][BW + 1];
};

// Registers of one batch of backward rows.
template <int BW, bool CYC, typename C, int B>
struct BackwardBatch {
    C xb[B];
    C uc[B][BW + 1];
    C rc[B][BW + 1];
    C dg[B];
};

template <int BW, bool CYC, typename C, typename P, int B>
__device__ __forceinline__ void load_forward(ForwardBatch<BW, CYC, C, B>& r, const P* __restrict__ x, int64_t step,
                                             int64_t n, int64_t j0, const SolveParams& sp, int32_t z) {
    const GlobalPtr<C> __restrict__ lower = factor_ptr<C>(sp.lower, z);
    const GlobalPtr<C> __restrict__ bottom = factor_ptr<C>(sp.bottom, z);
#pragma unroll
    for (int u = 0; u < B; ++u) {
        r.xb[u] = static_cast<C>(x[(j0 + u) * step]);
#pragma unroll
        for (int m = 0; m < BW; ++m) r.lc[u][m] = lower[(j0 + u) * BW + m];
        if constexpr (CYC) {
#pragma unroll
            for (int q = 0; q < BW; ++q) r.sc[u][q] = bottom[q * n + j0 + u];
        }
    }
}

// Forward substitution of rows j0 .. j0+B-1 (unit lower triangle, plus
// the bottom strip of a cyclic matrix) from loaded registers; stores the
// rows.
template <int BW, bool CYC, typename C, typename P, int B>
__device__ __forceinline__ void run_forward(ForwardBatch<BW, CYC, C, B>& r, P* __restrict__ x, int64_t step,
                                            int64_t n, int64_t j0, LineState<BW, CYC, C>& st) {
#pragma clang fp contract(off)
#pragma unroll
    for (int u = 0; u < B; ++u) {
        const int64_t j = j0 + u;
        C v = r.xb[u];
        if constexpr (CYC) {
#pragma unroll
            for (int q = 0; q < BW; ++q)
                if (j == n - BW + q) v = st.acc[q];
        }
#pragma unroll
        for (int m = BW; m >= 1; --m) v = v - r.lc[u][m - 1] * st.hist[m - 1];
        r.xb[u] = v;
#pragma unroll
        for (int m = BW; m >= 2; --m) st.hist[m - 1] = st.hist[m - 2];
        if (BW > 0) st.hist[0] = v;
        if constexpr (CYC) {
#pragma unroll
            for (int q = 0; q < BW; ++q)
                if (j < n - BW + q - BW) st.acc[q] = st.acc[q] - r.sc[u][q] * v;
        }
    }
#pragma unroll
    for (int u = 0; u < B; ++u) x[(j0 + u) * step] = static_cast<P>(r.xb[u]);
}

template <int BW, bool CYC, typename C, typename P, int B>
__device__ __forceinline__ void load_backward(BackwardBatch<BW, CYC, C, B>& r, const P* __restrict__ x, int64_t step,
                                              int64_t n, int64_t j0, const SolveParams& sp, int32_t z) {
    const GlobalPtr<C> __restrict__ upper = factor_ptr<C>(sp.upper, z);
    const GlobalPtr<C> __restrict__ diag = factor_ptr<C>(sp.diag, z);
    const GlobalPtr<C> __restrict__ right = factor_ptr<C>(sp.right, z);
#pragma unroll
    for (int u = 0; u < B; ++u) {
        const int64_t j = j0 - u;
        r.xb[u] = static_cast<C>(x[j * step]);
#pragma unroll
        for (int m = 0; m < BW; ++m) r.uc[u][m] = upper[j * BW + m];
        r.dg[u] = diag[j];
        if constexpr (CYC) {
#pragma unroll
            for (int c = 0; c < BW; ++c) r.rc[u][c] = right[c * n + j];
        }
    }
}

// Backward substitution of rows j0, j0-1, .., j0-B+1 (upper triangle,
// plus the right strip of a cyclic matrix) from loaded registers; stores
// the rows.
template <int BW, bool CYC, typename C, typename P, int B>
__device__ __forceinline__ void run_backward(BackwardBatch<BW, CYC, C, B>& r, P* __restrict__ x, int64_t step,
                                             int64_t n, int64_t j0, LineState<BW, CYC, C>& st) {
#pragma clang fp contract(off)
#pragma unroll
    for (int u = 0; u < B; ++u) {
        const int64_t j = j0 - u;
        C v = r.xb[u];
        if constexpr (CYC) {
#pragma unroll
            for (int c = BW - 1; c >= 0; --c)
                if (j < n - BW + c - BW) v = v - r.rc[u][c] * st.corner[c];
        }
#pragma unroll
        for (int m = BW; m >= 1; --m) v = v - r.uc[u][m - 1] * st.nxt[m - 1];
        v = v / r.dg[u];
        r.xb[u] = v;
#pragma unroll
        for (int m = BW; m >= 2; --m) st.nxt[m - 1] = st.nxt[m - 2];
        if (BW > 0) st.nxt[0] = v;
        if constexpr (CYC) {
#pragma unroll
            for (int c = 0; c < BW; ++c)
                if (j == n - BW + c) st.corner[c] = v;
        }
    }
#pragma unroll
    for (int u = 0; u < B; ++u) x[(j0 - u) * step] = static_cast<P>(r.xb[u]);
}

// Rows per batch: two batches are in registers at once (the one being
// substituted and the next one loading), so wide cyclic bands use 4.
// Kernels that merge many band widths pass 4 to bound their registers.
template <int BW, bool CYC>
constexpr int batch_rows() {
    return BW * (CYC ? 2 : 1) <= 4 ? kBatch : kBatch / 2;
}

// Forward substitution of rows a .. e-1 of a line from state `st`
// (software-pipelined: the loads of the next batch of rows, right-hand
// sides and factor coefficients, are in flight while the current batch is
// substituted, so one lane's chain of dependent rows does not wait for
// memory every batch; each row receives the same updates in the same
// order as without pipelining).
template <int BW, bool CYC, typename C, typename P, int B>
__device__ __forceinline__ void forward_range(P* __restrict__ x, int64_t step, int64_t n, int64_t a, int64_t e,
                                              const SolveParams& sp, LineState<BW, CYC, C>& st, int32_t z) {
    const int64_t nb = (e - a) / B;  // full batches
    if (nb > 0) {
        ForwardBatch<BW, CYC, C, B> ba, bb;
        load_forward<BW, CYC, C, P, B>(ba, x, step, n, a, sp, z);
        int64_t t = 0;
        for (; t + 2 <= nb; t += 2) {
            load_forward<BW, CYC, C, P, B>(bb, x, step, n, a + (t + 1) * B, sp, z);
            run_forward<BW, CYC, C, P, B>(ba, x, step, n, a + t * B, st);
            // batch t + 2, or (past the end) a harmless reload of batch nb - 1
            load_forward<BW, CYC, C, P, B>(ba, x, step, n, a + min(t + 2, nb - 1) * B, sp, z);
            run_forward<BW, CYC, C, P, B>(bb, x, step, n, a + (t + 1) * B, st);
        }
        if (t < nb) run_forward<BW, CYC, C, P, B>(ba, x, step, n, a + t * B, st);
    }
    for (int64_t j = a + nb * B; j < e; ++j) {
        ForwardBatch<BW, CYC, C, 1> r;
        load_forward<BW, CYC, C, P, 1>(r, x, step, n, j, sp, z);
        run_forward<BW, CYC, C, P, 1>(r, x, step, n, j, st);
    }
}

// Backward substitution of rows e-1 down to a from state `st` (pipelined
// like forward_range).
template <int BW, bool CYC, typename C, typename P, int B>
__device__ __forceinline__ void backward_range(P* __restrict__ x, int64_t step, int64_t n, int64_t a, int64_t e,
                                               const SolveParams& sp, LineState<BW, CYC, C>& st, int32_t z) {
    const int64_t nb = (e - a) / B;
    if (nb > 0) {
        BackwardBatch<BW, CYC, C, B> ba, bb;
        load_backward<BW, CYC, C, P, B>(ba, x, step, n, e - 1, sp, z);
        int64_t t = 0;
        for (; t + 2 <= nb; t += 2) {
            load_backward<BW, CYC, C, P, B>(bb, x, step, n, e - 1 - (t + 1) * B, sp, z);
            run_backward<BW, CYC, C, P, B>(ba, x, step, n, e - 1 - t * B, st);
            load_backward<BW, CYC, C, P, B>(ba, x, step, n, e - 1 - min(t + 2, nb - 1) * B, sp, z);
            run_backward<BW, CYC, C, P, B>(bb, x, step, n, e - 1 - (t + 1) * B, st);
        }
        if (t < nb) run_backward<BW, CYC, C, P, B>(ba, x, step, n, e - 1 - t * B, st);
    }
    for (int64_t j = e - 1 - nb * B; j >= a; --j) {
        BackwardBatch<BW, CYC, C, 1> r;
        load_backward<BW, CYC, C, P, 1>(r, x, step, n, j, sp, z);
        run_backward<BW, CYC, C, P, 1>(r, x, step, n, j, st);
    }
}

// Solves one line x[0], x[step], ..., x[(n-1)*step] in place, computing
// in C (elements of x have type P).
template <int BW, bool CYC, typename C, typename P, int B = batch_rows<BW, CYC>()>
__device__ __forceinline__ void substitute(P* __restrict__ x, int64_t step, int64_t n, const SolveParams& sp) {
    LineState<BW, CYC, C> st;
#pragma unroll
    for (int m = 0; m <= BW; ++m) st.hist[m] = st.nxt[m] = st.corner[m] = st.acc[m] = C(0);
    if constexpr (CYC) {
#pragma unroll
        for (int q = 0; q < BW; ++q) st.acc[q] = static_cast<C>(x[(n - BW + q) * step]);
    }
    const int32_t z = lane_zero();
    forward_range<BW, CYC, C, P, B>(x, step, n, 0, n, sp, st, z);
    backward_range<BW, CYC, C, P, B>(x, step, n, 0, n, sp, st, z);
}

// A launch of a few long lines (lines beyond a tile whose factors fade too
// slowly to be cut, or without room for the chunks' table) substitutes each
// line with one lane whose factor loads run one batch of rows ahead: from
// HBM every batch would wait a full memory latency.  When the launch has
// at most kWarmLines lines and the factors fit kWarmBytes, every thread of
// the workgroup first reads the factor arrays once (one 4-byte word per
// 64 bytes), so that the substitution finds them in L2, or past its 4 MB in
// the device's last-level cache (one cubic line of 100,000 rows: 12.8 ms at
// a limit of 2 MB, 12.0).  The arithmetic is unchanged.
constexpr int64_t kWarmLines = 8;
constexpr int64_t kWarmBytes = int64_t{32} << 20;

template <int BW, bool CYC, typename C, int NT>
__device__ __forceinline__ void warm_factors(const SolveParams& sp, int64_t n) {
    if (sp.nlines > kWarmLines) return;
    const int64_t per = static_cast<int64_t>(sizeof(C)) * n;
    const int64_t bytes = per * (2 * BW + 1) + (CYC ? per * 2 * BW : 0);
    if (bytes > kWarmBytes) return;
    uint32_t acc = 0;
    auto touch = [&](const void* p, int64_t nbytes) {
        const uint32_t* w = static_cast<const uint32_t*>(p);
        const int64_t lines = nbytes / 64;
        for (int64_t i = threadIdx.x; i < lines; i += NT * 4) {
            uint32_t v[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) v[u] = i + u * NT < lines ? w[(i + u * NT) * 16] : 0u;
#pragma unroll
            for (int u = 0; u < 4; ++u) acc ^= v[u];
        }
    };
    touch(sp.lower, per * BW);
    touch(sp.upper, per * BW);
    touch(sp.diag, per);
    if constexpr (CYC) {
        touch(sp.bottom, per * BW);
        touch(sp.right, per * BW);
    }
    asm volatile("" ::"v"(acc));  // the loads' results are used
}

// ---- segmented substitution ---------------------------------------------
//
// A line's substitution is one dependent chain of rows, but the chain
// forgets: an interpolating spline's LU recurrences contract (0.27 per row
// at order 3, 0.54 at order 7), so started `warm` rows early from a zero
// state they arrive at the very bits of the full recurrence (measured over
// all orders, 2 to 7, clamped, periodic and graded, on noise and on smooth
// data: 27 to 38 rows at the worst for orders 2 and 3 in FP64, 97 at order
// 7; the median is 22, 30 and 66).  So the line is cut into segments, one
// lane each.  Every lane warms up on the rows before its segment without
// storing, then substitutes its own rows.  Afterwards each lane compares
// the state it started from with the rows its neighbour stored, bit for
// bit.  Equal states mean equal rows, so a line that passes holds exactly
// the sequential result.  If any comparison of a workgroup fails, the tile
// is loaded again and solved in one piece.  That happens on
// exactly constant lines (two starts can settle on neighbouring fixed
// points: 0.7 to 16 % of the boundaries for orders 3 and 4, up to 40 % at
// order 5) and where data decays faster than the factors fade (a Gaussian's
// flanks, zeros after data: a true state there is a tail of the data).
//
// The strips of a cyclic matrix are the other chain: x[n-BW+q] minus
// bottom[q][j] * y[j] over all j.  The strip decays like the recurrence, so
// after a prefix of `warm` rows, summed in order, the remaining terms are
// below the rounding of the sum A.  That is checked too: with t the
// largest remaining strip entry (strip_rest) times the largest |y|,
// A - t == A and A + t == A make every later subtraction a no-op
// (rounding is monotonic).  Where they do not hold, the other rows are
// summed too.
//
// Numerators too small for the two-operation division, infinities and NaN
// are found after each batch of rows, which is then divided in full: a field
// of 1e-290 costs 0.27 ms at 256^3 cubic, 0.25 at ordinary values (0.85 where
// a tile that met one was solved again, twice).
//
// Rows whose factors repeat bit for bit (the interior of a uniform grid,
// all but the first ~8 * order rows and the last few) take them from
// registers instead of memory: [flo, fhi) for the forward sweep and [blo,
// bhi) for the backward one.
__device__ __forceinline__ bool same_bits(double a, double b) {
    return __double_as_longlong(a) == __double_as_longlong(b);
}
__device__ __forceinline__ bool same_bits(float a, float b) { return __float_as_int(a) == __float_as_int(b); }

// Row of the staged table that stands for row r, and its inverse.
__device__ __forceinline__ int edge_row(int r, int lo, int hi) { return r < hi ? min(r, lo) : r - hi + lo + 1; }
__device__ __forceinline__ int edge_source(int i, int lo, int hi) { return i <= lo ? i : i - lo - 1 + hi; }

template <typename C>
struct EdgeTable {
    const C* lower = nullptr;  // LDS, or null
    const C* upper = nullptr;
    const C* diag = nullptr;
};

template <int BW, typename C>
__device__ __forceinline__ EdgeTable<C> stage_edges(const SolveParams& sp, C* lds, int tid, int NT) {
    const int n = static_cast<int>(sp.n);
    EdgeTable<C> t;
    if (edge_elements(n, BW, sp) == 0) return t;
    const int ef = sp.flo + 1 + n - sp.fhi, eb = sp.blo + 1 + n - sp.bhi;
    const GlobalPtr<C> lower = (GlobalPtr<C>)(sp.lower);
    const GlobalPtr<C> upper = (GlobalPtr<C>)(sp.upper);
    const GlobalPtr<C> diag = (GlobalPtr<C>)(sp.diag);
    C* el = lds;
    C* eu = el + ef * BW;
    C* ed = eu + eb * BW;
    for (int i = tid; i < ef; i += NT) {
        const int r = edge_source(i, sp.flo, sp.fhi);
#pragma unroll
        for (int m = 0; m < BW; ++m) el[i * BW + m] = r < n ? lower[r * BW + m] : C(0);
    }
    for (int i = tid; i < eb; i += NT) {
        const int r = edge_source(i, sp.blo, sp.bhi);
#pragma unroll
        for (int m = 0; m < BW; ++m) eu[i * BW + m] = r < n ? upper[r * BW + m] : C(0);
        ed[i] = r < n ? diag[r] : C(1);
    }
    t.lower = el;
    t.upper = eu;
    t.diag = ed;
    return t;
}

// The batches t (multiples of B) of a sweep in which every lane of the
// wave is on rows of equal factors, as one scalar range.  The lane of
// segment s covers rows len * s - before + t .. + B - 1 (sweep order), of
// which [lo, hi) have equal factors and rows from `end` on do not count;
// the wave holds the segments first .. last.  The first segment of a wave
// reaches `lo` last and its last segment leaves `hi` first.
struct BatchRange {
    int lo, hi;
};

__device__ __forceinline__ BatchRange equal_batches(int first, int last, int len, int before, int count, int lo,
                                                    int hi, int end, int B) {
    const int a = lo - (first * len - before), b = hi - (last * len - before);
    BatchRange r;
    r.lo = a > 0 ? (a + B - 1) / B * B : 0;
    r.hi = hi >= end ? count : b < 0 ? 0 : min(b / B * B, count);
    if (first > last) r = {0, 0};
    return r;
}

// One batch of forward rows (row u at x + u * step) from right-hand sides
// xb; lc(u, m) gives the factors.
template <int BW, bool CYC, bool STORE, typename C, int B, typename L>
__device__ __forceinline__ void seg_forward_rows(const C (&xb)[B], C* x, int step, C (&hist)[BW + 1], C& vmax, L lc) {
#pragma clang fp contract(off)
#pragma unroll
    for (int u = 0; u < B; ++u) {
        C v = xb[u];
#pragma unroll
        for (int m = BW; m >= 1; --m) v = v - lc(u, m - 1) * hist[m - 1];
#pragma unroll
        for (int m = BW; m >= 2; --m) hist[m - 1] = hist[m - 2];
        if (BW > 0) hist[0] = v;
        if constexpr (STORE) {
            x[u * step] = v;
            if constexpr (CYC) vmax = fmax(vmax, fabs(v));
        }
    }
}

// Rows j0 .. j0+count-1 (both multiples of B; batches below row 0 or from
// `end` on are skipped) of one lane; row j sits at line[(j - origin) * step],
// with rows origin - B .. limit + B - 1 there to read.  The batches of equal factors run in a
// loop of their own, the next batch's right-hand sides in flight while one
// is substituted; the few others before and after it in a second.  A batch
// that crosses `end` also stores up to B - 1 rows after it.
template <int BW, bool CYC, bool STORE, typename C, int B>
__device__ __forceinline__ void seg_forward(C* line, int step, int origin, int limit, int j0, int count, int end,
                                            bool mine, BatchRange eq, const SolveParams& sp,
                                            const EdgeTable<C>& edge, C (&hist)[BW + 1], C& vmax) {
    const GlobalPtr<C> __restrict__ lower = (GlobalPtr<C>)(sp.lower);
    C kl[BW + 1];
#pragma unroll
    for (int m = 0; m < BW; ++m) kl[m] = static_cast<C>(sp.eq_lower[m]);
    const int stride = B * step, low = -B * step, high = (limit - origin) * step;
    int t = 0;
#pragma unroll 1
    for (int part = 0; part < 2; ++part) {
        const int stop = part == 0 ? min(eq.lo, count) : count;
#pragma unroll 1
        for (; t < stop; t += B) {
            const int j = j0 + t;
            if (!(mine && j >= 0 && j < end)) continue;
            C xb[B], lb[B][BW + 1];
            C* x = line + (j - origin) * step;
#pragma unroll
            for (int u = 0; u < B; ++u) xb[u] = x[u * step];
            if (edge.lower) {
#pragma unroll
                for (int u = 0; u < B; ++u) {
                    const int r = edge_row(min(j + u, end - 1), sp.flo, sp.fhi);
#pragma unroll
                    for (int m = 0; m < BW; ++m) lb[u][m] = edge.lower[r * BW + m];
                }
            } else {
#pragma unroll
                for (int u = 0; u < B; ++u)
#pragma unroll
                    for (int m = 0; m < BW; ++m) lb[u][m] = lower[min(j + u, end - 1) * BW + m];
            }
            seg_forward_rows<BW, CYC, STORE, C, B>(xb, x, step, hist, vmax, [&](int u, int m) { return lb[u][m]; });
        }
        if (part == 1 || t >= eq.hi) continue;
        // batches outside the held rows read the ones next to them
        int at = (j0 + t - origin) * step;
        C xa[B], xb[B];
        auto load = [&](C (&xv)[B], int i) {
            i = min(max(i, low), high);
#pragma unroll
            for (int u = 0; u < B; ++u) xv[u] = line[i + u * step];
        };
        auto run = [&](const C (&xv)[B]) {
            const int j = j0 + t;
            if (mine && j >= 0 && j < end)
                seg_forward_rows<BW, CYC, STORE, C, B>(xv, line + at, step, hist, vmax,
                                                       [&](int, int m) { return kl[m]; });
            t += B;
            at += stride;
            asm volatile("" : "+v"(at));  // one running index, not one per row
        };
        load(xa, at);
#pragma unroll 1
        while (true) {
            load(xb, at + stride);
            run(xa);
            if (t >= eq.hi) break;
            load(xa, at + stride);
            run(xb);
            if (t >= eq.hi) break;
        }
    }
}

// v / d for the pivot d of the rows [blo, bhi) in two operations, RN(v zh
// + RN(v zl)) with zh + zl the reciprocal of d (Brisebarre, Muller and
// Raina, "Accelerating correctly rounded floating-point division when the
// divisor is known in advance", IEEE Transactions on Computers 53(8),
// 2004).  The host has checked every numerator whose quotient lies near
// enough to a rounding boundary, so the result is the correctly rounded
// quotient (zl >= 0 keeps the sign of a zero) unless v zl underflows,
// which `least` finds, or v is infinite, which leaves a NaN in every later
// row.  The caller looks for both after a batch of rows and divides that
// batch in full.
template <typename C>
struct KnownDivisor {
    C zh, zl, d;
    // least: the smallest exponent of a numerator so far (a zero, an infinity
    // and a NaN count as 0)
    __device__ __forceinline__ C divide(C v, int& least) const {
#pragma clang fp contract(off)
        if constexpr (sizeof(C) == 8) {
            least = min(least, __builtin_amdgcn_frexp_exp(v));
            return __builtin_fma(v, zh, v * zl);
        } else {
            least = min(least, __builtin_amdgcn_frexp_expf(v));
            return __builtin_fmaf(v, zh, v * zl);
        }
    }
    __device__ __forceinline__ static bool underflows(int least) { return least < (sizeof(C) == 8 ? -900 : -90); }
};

template <typename C>
__device__ __forceinline__ KnownDivisor<C> known_pivot(const SolveParams& sp) {
    KnownDivisor<C> k{static_cast<C>(sp.zh), static_cast<C>(sp.zl), C(1)};
    if (sp.fast_divide) k.d = ((GlobalPtr<C>)(sp.diag))[sp.blo];
    return k;
}

// One batch of backward rows (row u at x - u * step, u downward from row j).
template <int BW, bool CYC, bool STORE, typename C, int B, typename U, typename D, typename R>
__device__ __forceinline__ void seg_backward_rows(const C (&xb)[B], C* x, int step, int n, int j,
                                                  const C (&corner)[BW + 1], C (&nxt)[BW + 1], U uc, D divide, R rc) {
#pragma clang fp contract(off)
#pragma unroll
    for (int u = 0; u < B; ++u) {
        C v = xb[u];
        if constexpr (CYC) {
#pragma unroll
            for (int c = BW - 1; c >= 0; --c)
                if (j - u < n - BW + c - BW) v = v - rc(u, c) * corner[c];
        }
#pragma unroll
        for (int m = BW; m >= 1; --m) v = v - uc(u, m - 1) * nxt[m - 1];
        v = divide(u, v);
#pragma unroll
        for (int m = BW; m >= 2; --m) nxt[m - 1] = nxt[m - 2];
        if (BW > 0) nxt[0] = v;
        if constexpr (STORE) x[-u * step] = v;
    }
}

// Rows j0, j0-1, .., j0-count+1 of one lane (batches below row 0 or from
// `end` on are skipped; j0 + 1 - end and count are multiples of B), in two
// loops like seg_forward.  A batch that crosses row 0 also stores up to
// B - 1 rows before it.
template <int BW, bool CYC, bool STORE, typename C, int B>
__device__ __forceinline__ void seg_backward(C* line, int step, int origin, int n, int j0, int count, int end,
                                             bool mine, BatchRange eq, const SolveParams& sp, const EdgeTable<C>& edge,
                                             const KnownDivisor<C>& kz, const C (&corner)[BW + 1], C (&nxt)[BW + 1]) {
    const GlobalPtr<C> __restrict__ upper = (GlobalPtr<C>)(sp.upper);
    const GlobalPtr<C> __restrict__ diag = (GlobalPtr<C>)(sp.diag);
    const GlobalPtr<C> __restrict__ right = (GlobalPtr<C>)(sp.right);
    C ku[BW + 1];
#pragma unroll
    for (int m = 0; m < BW; ++m) ku[m] = static_cast<C>(sp.eq_upper[m]);
    if (!sp.fast_divide) eq.hi = eq.lo = 0;
    const int stride = B * step, low = -step, high = (end + B - 1 - origin) * step;
    auto load_strips = [&](C (&rb)[B][BW + 1], int j) {
        if constexpr (CYC) {
#pragma unroll
            for (int u = 0; u < B; ++u)
#pragma unroll
                for (int c = 0; c < BW; ++c) rb[u][c] = right[c * n + min(max(j - u, 0), n - 1)];
        }
    };
    int t = 0;
#pragma unroll 1
    for (int part = 0; part < 2; ++part) {
        const int stop = part == 0 ? min(eq.lo, count) : count;
#pragma unroll 1
        for (; t < stop; t += B) {
            const int j = j0 - t;
            if (!(mine && j >= 0 && j < end)) continue;
            C xb[B], rb[B][BW + 1], ub[B][BW + 1], db[B];
            C* x = line + (j - origin) * step;
#pragma unroll
            for (int u = 0; u < B; ++u) xb[u] = x[-u * step];
            load_strips(rb, j);
            if (edge.lower) {
#pragma unroll
                for (int u = 0; u < B; ++u) {
                    const int r = edge_row(max(j - u, 0), sp.blo, sp.bhi);
#pragma unroll
                    for (int m = 0; m < BW; ++m) ub[u][m] = edge.upper[r * BW + m];
                    db[u] = edge.diag[r];
                }
            } else {
#pragma unroll
                for (int u = 0; u < B; ++u) {
#pragma unroll
                    for (int m = 0; m < BW; ++m) ub[u][m] = upper[max(j - u, 0) * BW + m];
                    db[u] = diag[max(j - u, 0)];
                }
            }
            seg_backward_rows<BW, CYC, STORE, C, B>(xb, x, step, n, j, corner, nxt,
                                                    [&](int u, int m) { return ub[u][m]; },
                                                    [&](int u, C v) { return v / db[u]; },
                                                    [&](int u, int c) { return rb[u][c]; });
        }
        if (part == 1 || t >= eq.hi) continue;
        int at = (j0 - t - origin) * step;
        C xa[B], xb[B], ra[B][BW + 1], rb[B][BW + 1];
        auto load = [&](C (&xv)[B], C (&rv)[B][BW + 1], int i, int j) {
            i = min(max(i, low), high);
#pragma unroll
            for (int u = 0; u < B; ++u) xv[u] = line[i - u * step];
            load_strips(rv, j);
        };
        auto run = [&](const C (&xv)[B], const C (&rv)[B][BW + 1]) {
            const int j = j0 - t;
            if (mine && j >= 0 && j < end) {
                auto rows = [&](auto divide) {
                    seg_backward_rows<BW, CYC, STORE, C, B>(xv, line + at, step, n, j, corner, nxt,
                                                            [&](int, int m) { return ku[m]; }, divide,
                                                            [&](int u, int c) { return rv[u][c]; });
                };
                C before[BW + 1];
                int least = 0;
#pragma unroll
                for (int m = 0; m < BW; ++m) before[m] = nxt[m];
                auto finite = [&]() { return nxt[0] - nxt[0] == C(0); };
                const bool fast = finite();  // (infinities and NaN stay in every row)
                if (fast) rows([&](int, C v) { return kz.divide(v, least); });
                if (!fast || kz.underflows(least) || !finite()) {
#pragma unroll
                    for (int m = 0; m < BW; ++m) nxt[m] = before[m];
                    rows([&](int, C v) { return v / kz.d; });
                }
            }
            t += B;
            at -= stride;
            asm volatile("" : "+v"(at));  // one running index, not one per row
        };
        load(xa, ra, at, j0 - t);
#pragma unroll 1
        while (true) {
            load(xb, rb, at - stride, j0 - t - B);
            run(xa, ra);
            if (t >= eq.hi) break;
            load(xa, ra, at - stride, j0 - t - B);
            run(xb, rb);
            if (t >= eq.hi) break;
        }
    }
}

// Substitutes the lines of one tile (rows of `step` elements, line l at
// tile + l) in `segs` segments each, thread tid taking segment tid / lpb of
// line tid % lpb.  False: a comparison failed and the tile's contents are
// undefined.  Every thread of the workgroup takes part.
template <int BW, bool CYC, typename C, int B>
__device__ __forceinline__ bool solve_segments(const SolveParams& sp, C* tile, int step, int nl, int lpb, int segs,
                                               const EdgeTable<C>& edge, int tid, int (&failed)[2]) {
    const int n = static_cast<int>(sp.n);
    const int shift = __builtin_ctz(static_cast<unsigned>(lpb));
    const int line = tid & (lpb - 1), seg = tid >> shift;
    const int H = CYC ? n - BW : n;  // the last BW rows of a cyclic matrix follow the strips
    const int len = ((H + segs - 1) / segs + kSegRows - 1) / kSegRows * kSegRows;
    const int warm = sp.warm;
    const bool mine = line < nl && seg < segs && seg * len < H;
    // the wave's segments (a wave is 64 threads in a row of tid)
    const int wave = __builtin_amdgcn_readfirstlane(tid) & ~63;
    const int seg0 = wave >> shift, seg1 = min((wave + 63) >> shift, (H + len - 1) / len - 1);
    C* x = tile + line;
    C hist[BW + 1], start[BW + 1], corner[BW + 1];
    C vmax = C(0);
#pragma unroll
    for (int m = 0; m <= BW; ++m) hist[m] = start[m] = corner[m] = C(0);
    // whether any thread's `bad` is set (LDS flag, cleared below between
    // barriers)
    auto any_bad = [&](bool bad) {
        if (__any(bad) && (threadIdx.x & 63) == 0) failed[0] = 1;
        __syncthreads();
        return failed[0] != 0;
    };
    if (tid < 2) failed[tid] = 0;
    // forward
    const int a = seg * len;
    C strip_row = C(0);  // x[n-BW+q] of the thread that sums strip q (the forward sweep stores past row H)
    if constexpr (CYC && BW > 0) {
        if (line < nl && seg < BW) strip_row = x[(H + seg) * step];
    }
    if (segs > 1) {
        seg_forward<BW, CYC, false, C, B>(x, step, 0, H, a - warm, warm, H, mine && seg > 0,
                                          equal_batches(max(seg0, 1), seg1, len, warm, warm, sp.flo, sp.fhi, H, B),
                                          sp, edge, hist, vmax);
#pragma unroll
        for (int m = 0; m < BW; ++m) start[m] = hist[m];
    }
    __syncthreads();
    seg_forward<BW, CYC, true, C, B>(x, step, 0, H, a, len, H, mine,
                                     equal_batches(seg0, seg1, len, 0, len, sp.flo, sp.fhi, H, B), sp, edge, hist,
                                     vmax);
    __syncthreads();
    bool bad = false;
    if (mine && seg > 0) {
#pragma unroll
        for (int m = 0; m < BW; ++m) bad = bad || !same_bits(start[m], x[(a - 1 - m) * step]);
    }
    if constexpr (CYC && BW > 0) {
#pragma clang fp contract(off)
        // x[n-BW+q] minus the terms of rows a .. e - 1, by thread q of a line
        const GlobalPtr<C> __restrict__ bottom = (GlobalPtr<C>)(sp.bottom);
        auto strip = [&](C acc, int a, int e) {
#pragma unroll 8
            for (int j = a; j < e; ++j) acc = acc - bottom[seg * n + j] * x[j * step];
            x[(H + seg) * step] = acc;
        };
        const int rows = n - 2 * BW + seg, prefix = min(warm, rows);
        if (line < nl && seg < BW) strip(strip_row, 0, prefix);
        __syncthreads();
        // terms that are not below the rounding of the sums, infinities and
        // NaN: the rest of the rows are summed too
        bool rest = false;
        if (mine) {
            rest = !(hist[0] - hist[0] == C(0));
#pragma unroll
            for (int q = 0; q < BW; ++q) {
                const C A = x[(H + q) * step];
                const C t = static_cast<C>(sp.strip_rest) * vmax;
                rest = rest || !(A - t == A && A + t == A) || same_bits(A, C(-0.0));
            }
        }
        if (__any(rest) && (threadIdx.x & 63) == 0) failed[1] = 1;
        if (any_bad(bad)) return false;
        if (failed[1]) {
            if (line < nl && seg < BW) strip(x[(H + seg) * step], prefix, rows);
            __syncthreads();
        }
        if (line < nl && seg == 0) {
            // the last rows, then the backward rows that fix the corners
            LineState<BW, CYC, C> st;
#pragma unroll
            for (int m = 0; m <= BW; ++m) st.hist[m] = st.nxt[m] = st.corner[m] = st.acc[m] = C(0);
#pragma unroll
            for (int m = 0; m < BW; ++m) {
                st.hist[m] = x[(H - 1 - m) * step];
                st.acc[m] = x[(H + m) * step];
            }
            const int32_t z = lane_zero();
            forward_range<BW, CYC, C, C, 1>(x, step, n, H, n, sp, st, z);
            backward_range<BW, CYC, C, C, 1>(x, step, n, H, n, sp, st, z);
        }
        __syncthreads();
#pragma unroll
        for (int c = 0; c < BW; ++c) corner[c] = x[(H + c) * step];
    } else {
        if (segs > 1 && any_bad(bad)) return false;
    }
    // backward: segment `seg` from the end; in sweep order row r is H - 1 - r
    const int top = H - seg * len;
    const int blo = H - min(sp.bhi, H), bhi = H - sp.blo;
    const KnownDivisor<C> kz = known_pivot<C>(sp);
    C nxt[BW + 1];
    nxt[BW] = C(0);
#pragma unroll
    for (int m = 0; m < BW; ++m) nxt[m] = CYC && top + warm >= H ? corner[m] : C(0);
    if (segs > 1) {
        seg_backward<BW, CYC, false, C, B>(x, step, 0, n, top + warm - 1, warm, H, mine && seg > 0,
                                           equal_batches(max(seg0, 1), seg1, len, warm, warm, blo, bhi, H, B), sp,
                                           edge, kz, corner, nxt);
#pragma unroll
        for (int m = 0; m < BW; ++m) start[m] = nxt[m];
        __syncthreads();
    }
    seg_backward<BW, CYC, true, C, B>(x, step, 0, n, top - 1, len, H, mine,
                                      equal_batches(seg0, seg1, len, 0, len, blo, bhi, H, B), sp, edge, kz, corner,
                                      nxt);
    __syncthreads();
    if (segs == 1) return true;
    bad = false;
    if (mine && seg > 0) {
#pragma unroll
        for (int m = 0; m < BW; ++m) bad = bad || !same_bits(start[m], x[(top + m) * step]);
    }
    return !any_bad(bad);
}

// One workgroup: lines [first, first + lpb) staged through LDS in the
// compute type C; the table holds T.  Row j of line l sits at
// tile[j * step + l].  With sp.accum set, the solved lines are added into
// accum instead of being stored to x.
// tid: the thread's place in the workgroup of NT threads, whole waves of it
// in any order (the callers rotate the waves: where one wave substitutes,
// neighbouring workgroups on a CU then use different SIMDs).
// SEG false: plain substitution (sp.segs 0), without the segments' pad rows.
// SEG true with sp.segs 0 (the batch's 256-thread kernel): plain, with them.  FIXED: with a copy of the
// segment code for the row stride kTileStep.  ONE: lines of known pivots that
// fail are solved as one segment at any band width.
template <int BW, bool CYC, typename T, typename C, int B = batch_rows<BW, CYC>(), bool SEG = true,
          bool FIXED = true, bool ONE = false>
__device__ __forceinline__ void solve_tile(const SolveParams& sp, int64_t first, unsigned char* tile_bytes,
                                           int64_t* line_base, int tid, int NT) {
    const int lpb = sp.lines_per_block;
    const int64_t n = sp.n, inner = sp.inner;
    const int step = static_cast<int>(tile_step(lpb, inner));
    C* tile = reinterpret_cast<C*>(tile_bytes) + (SEG ? kTilePad : 0) * step;
    T* __restrict__ X = static_cast<T*>(sp.x);
    const int nl = static_cast<int>(min(static_cast<int64_t>(lpb), sp.nlines - first));
    if (tid < nl) {
        const int64_t line = first + tid;
        const int64_t o = line / inner, ii = line - o * inner;
        // the line's place in the values (first pass, contiguous lines), or in
        // the table
        if (!sp.src) {
            line_base[tid] = o * n * inner + ii;
        } else {
            // inner == 1: o runs over the outer dims in C order
            // constant indices (a runtime-indexed loop would force a
            // SolveParams built in registers out to scratch memory)
            int64_t rem = o, off = 0, mul = n;
#pragma unroll
            for (int d = kMaxDim - 1; d >= 0; --d) {
                if (d >= sp.outer_dims) continue;
                const int64_t nd = sp.outer_n[d];
                const int64_t id = rem % nd;
                rem /= nd;
                int64_t w = id - sp.outer_shift[d];
                if (w < 0) w += nd;
                off += w * mul;
                mul *= nd;
            }
            line_base[tid] = off;
        }
    }
    __syncthreads();

    // Contiguous lines: tile element e is (line e / n, row e % n).
    // Strided lines: (line e % lpb, row e / lpb); as NT % lpb == 0 a
    // thread keeps one line.  Pairs (FP64) or quads (FP32) of strided lines
    // that are adjacent and aligned in memory move as 16-byte vectors.  A
    // batch of kCopyBatch loads is in flight at once: a tile is a round
    // trip or two, not one per few elements.
    typedef T VecT __attribute__((ext_vector_type(16 / sizeof(T))));
    constexpr int V = 16 / sizeof(T);
    const uint32_t un = static_cast<uint32_t>(n);
    const int lshift = __builtin_ctz(static_cast<unsigned>(lpb));
    const uint32_t count = static_cast<uint32_t>(inner == 1 ? nl * n : lpb * n);
    const uint32_t my_l = static_cast<uint32_t>(tid) & static_cast<uint32_t>(lpb - 1);
    const bool vec = inner > 1 && lpb >= V && inner % V == 0 && (reinterpret_cast<uintptr_t>(X) & 15) == 0 &&
                     (reinterpret_cast<uintptr_t>(sp.accum) & 15) == 0;
    const int vshift = lshift - __builtin_ctz(static_cast<unsigned>(V));
    const uint32_t my_v = (static_cast<uint32_t>(tid) & ((1u << max(vshift, 0)) - 1u)) * V;
    auto load = [&]() {
        if (sp.src) {
            for (uint32_t e0 = tid; e0 < count; e0 += NT * kCopyBatch) {
                // the values are read once: non-temporal loads keep them from
                // evicting the factors and the lines being written
                C v[kCopyBatch];
                uint32_t at[kCopyBatch];
#pragma unroll
                for (int u = 0; u < kCopyBatch; ++u) {
                    const uint32_t e = min(e0 + u * NT, count - 1);
                    const uint32_t l = fast_div(e, sp.div_n), jj = e - l * un;
                    int64_t js = static_cast<int64_t>(jj) - sp.shift_last;
                    if (js < 0) js += n;
                    v[u] = static_cast<C>(__builtin_nontemporal_load(&sp.src[line_base[l] + js]));
                    at[u] = jj * static_cast<uint32_t>(step) + l;
                }
#pragma unroll
                for (int u = 0; u < kCopyBatch; ++u)
                    if (e0 + u * NT < count) tile[at[u]] = v[u];
            }
        } else if (inner == 1) {
            const T* __restrict__ base = X + first * n;
            for (uint32_t e0 = tid; e0 < count; e0 += NT * kCopyBatch) {
                C v[kCopyBatch];
#pragma unroll
                for (int u = 0; u < kCopyBatch; ++u) v[u] = static_cast<C>(base[min(e0 + u * NT, count - 1)]);
#pragma unroll
                for (int u = 0; u < kCopyBatch; ++u) {
                    const uint32_t e = e0 + u * NT;
                    if (e < count) {
                        const uint32_t l = fast_div(e, sp.div_n), jj = e - l * un;
                        tile[jj * static_cast<uint32_t>(step) + l] = v[u];
                    }
                }
            }
        } else if (vec) {
            if (static_cast<int>(my_v) < nl) {
                const T* __restrict__ line = X + line_base[my_v];
                const uint32_t rows = NT >> vshift;
                for (uint32_t j0 = static_cast<uint32_t>(tid) >> vshift; j0 < un; j0 += rows * kCopyBatch) {
                    VecT v[kCopyBatch];
#pragma unroll
                    for (int u = 0; u < kCopyBatch; ++u)
                        v[u] = *reinterpret_cast<const VecT*>(
                            line + static_cast<int64_t>(min(j0 + u * rows, un - 1)) * inner);
#pragma unroll
                    for (int u = 0; u < kCopyBatch; ++u)
                        if (j0 + u * rows < un) {
#pragma unroll
                            for (int i = 0; i < V; ++i)
                                tile[(j0 + u * rows) * static_cast<uint32_t>(step) + my_v + i] = static_cast<C>(v[u][i]);
                        }
                }
            }
        } else if (static_cast<int>(my_l) < nl) {
            const T* __restrict__ line = X + line_base[my_l];
            for (uint32_t e0 = tid; e0 < count; e0 += NT * kCopyBatch) {
                C v[kCopyBatch];
#pragma unroll
                for (int u = 0; u < kCopyBatch; ++u) {
                    const uint32_t jj = min(e0 + u * NT, count - 1) >> lshift;
                    v[u] = static_cast<C>(line[static_cast<int64_t>(jj) * inner]);
                }
#pragma unroll
                for (int u = 0; u < kCopyBatch; ++u) {
                    const uint32_t e = e0 + u * NT;
                    if (e < count) tile[(e >> lshift) * static_cast<uint32_t>(step) + my_l] = v[u];
                }
            }
        }
        __syncthreads();
    };
    bool done = false;
    if constexpr (SEG) {
        __shared__ int failed[2];
        EdgeTable<C> edge;
        if (sp.segs > 0) {
            const int pad = static_cast<int>(kTilePad) * step;
            for (int i = tid; i < pad; i += NT) tile[i - pad] = tile[static_cast<int>(n) * step + i] = C(0);
            edge = stage_edges<BW, C>(sp, reinterpret_cast<C*>(tile_bytes) + tile_elements(n, lpb, inner, 1), tid, NT);
        }
        load();
        // segmented; then, if a comparison failed, in one piece: as one
        // segment, which has nothing to compare, or plainly where the rows of
        // equal factors do not make up for its steps (plan_tile)
        const bool one = CYC || (sp.fast_divide && (BW <= 2 || ONE));
#pragma unroll 1
        for (int segs = sp.segs; segs > 0 && !done; segs = segs > 1 && one ? 1 : 0) {
            // the usual row stride of many lines as a constant: row offsets
            // become immediates of the LDS instructions
            if (FIXED && step == kTileStep)
                done = solve_segments<BW, CYC, C, B>(sp, tile, kTileStep, nl, lpb, segs, edge, tid, failed);
            else
                done = solve_segments<BW, CYC, C, B>(sp, tile, step, nl, lpb, segs, edge, tid, failed);
            if (!done) load();
        }
    } else {
        load();
    }
    if (!done) {
        if (tid < nl) substitute<BW, CYC, C, C, B>(tile + tid, step, n, sp);
        __syncthreads();
    }

    // ---- store ----
    T* __restrict__ Y = sp.accum ? static_cast<T*>(sp.accum) : X;
    const bool add = sp.accum != nullptr;
    if (inner == 1) {
        T* __restrict__ base = Y + first * n;
        for (uint32_t e0 = tid; e0 < count; e0 += NT * kCopyBatch) {
            C v[kCopyBatch];
#pragma unroll
            for (int u = 0; u < kCopyBatch; ++u) {
                const uint32_t e = min(e0 + u * NT, count - 1);
                const uint32_t l = fast_div(e, sp.div_n), jj = e - l * un;
                v[u] = tile[jj * static_cast<uint32_t>(step) + l];
            }
#pragma unroll
            for (int u = 0; u < kCopyBatch; ++u)
                if (e0 + u * NT < count) {
                    T* at = base + e0 + u * NT;
                    *at = add ? static_cast<T>(*at + static_cast<T>(v[u])) : static_cast<T>(v[u]);
                }
        }
    } else if (vec) {
        if (static_cast<int>(my_v) < nl) {
            T* __restrict__ line = Y + line_base[my_v];
            const uint32_t rows = NT >> vshift;
#pragma unroll 4
            for (uint32_t j = static_cast<uint32_t>(tid) >> vshift; j < un; j += rows) {
                VecT* at = reinterpret_cast<VecT*>(line + static_cast<int64_t>(j) * inner);
                VecT v;
#pragma unroll
                for (int i = 0; i < V; ++i) v[i] = static_cast<T>(tile[j * static_cast<uint32_t>(step) + my_v + i]);
                if (add) v = *at + v;
                *at = v;
            }
        }
    } else if (static_cast<int>(my_l) < nl) {
        T* __restrict__ line = Y + line_base[my_l];
        for (uint32_t e0 = tid; e0 < count; e0 += NT * kBatch) {
            C v[kBatch];
#pragma unroll
            for (int u = 0; u < kBatch; ++u)
                v[u] = tile[(min(e0 + u * NT, count - 1) >> lshift) * static_cast<uint32_t>(step) + my_l];
#pragma unroll
            for (int u = 0; u < kBatch; ++u) {
                const uint32_t e = e0 + u * NT;
                if (e < count) {
                    T* at = line + static_cast<int64_t>(e >> lshift) * inner;
                    *at = add ? static_cast<T>(*at + static_cast<T>(v[u])) : static_cast<T>(v[u]);
                }
            }
        }
    }
}

}  // namespace

}  // namespace intp_amd
