// setup.cpp -- knot vectors, collocation matrices and their band LU.
//
// Follows the reference's construction so the factors match it bit for bit
// (compiled without FMA contraction): knots Interpolation.hpp:322-464,
// range BSpline.hpp:224-226, collocation rows InterpolationTemplate.hpp:
// 254-426, no-pivot LU BandLU.hpp:103-118,159-213.  The LU here runs over
// the fill pattern of a cyclic band matrix (band + right columns + bottom
// rows); every entry receives the reference's updates in the reference's
// order (pivot step ascending), which is what fixes its rounding.
#include "setup.hpp"

#include <algorithm>
#include <cmath>
#include <cstring>

namespace intp_amd {

namespace {

// The fill pattern of a (cyclic) band matrix and its LU.
class PatternMatrix {
   public:
    PatternMatrix(int64_t n, int p, int q, bool cyclic)
        : n_(n), p_(p), q_(q), w_(p + q + 1), cyclic_(cyclic),
          band_(static_cast<size_t>(n * w_), 0.0),
          right_(cyclic ? static_cast<size_t>(n * p) : 0, 0.0),
          bottom_(cyclic ? static_cast<size_t>(q * n) : 0, 0.0) {}

    bool in_band(int64_t i, int64_t j) const { return j - i <= q_ && i - j <= p_; }

    double& at(int64_t i, int64_t j) {
        if (in_band(i, j)) return band_[static_cast<size_t>(i * w_ + (j - i + p_))];
        if (cyclic_ && j >= n_ - p_) return right_[static_cast<size_t>(i * p_ + (j - (n_ - p_)))];
        // cyclic bottom rows
        return bottom_[static_cast<size_t>((i - (n_ - q_)) * n_ + j)];
    }
    bool stored(int64_t i, int64_t j) const {
        if (i < 0 || j < 0 || i >= n_ || j >= n_) return false;
        if (in_band(i, j)) return true;
        return cyclic_ && (j >= n_ - p_ || i >= n_ - q_);
    }

    // Right-looking LU without pivoting over the fill pattern.  Step k leaves
    // row k final and the p rows below it partly updated.  Where the matrix
    // rows [first_alike, last_alike] are equal (the interior of a uniform
    // grid), these p + 1 rows settle, bit for bit, after a few dozen steps,
    // and every later step up to the last equal row leaves the same: they
    // are copied, and only the strips of a cyclic matrix are computed.
    // Whole dimension without the tables of refined builds, every step
    // computed -> settled rows copied: cubic, n = 100,000, 4.71 -> 1.58 ms
    // (most of the rest is first touches of 9 MB); periodic order 6, n =
    // 8192, 1.20 -> 0.44 ms; order 5, n = 1000, 63 -> 18 us; cubic, n = 256,
    // 10.1 -> 4.9 us.
    void factor(int64_t first_alike, int64_t last_alike) {
        // steps whose rows and columns all lie clear of the corner blocks
        const int64_t clear = std::max<int64_t>(0, std::min(n_ - 1, cyclic_ ? n_ - 4 * p_ - 1 : n_ - 2 * p_ - 1));
        const size_t window = static_cast<size_t>((p_ + 1) * w_);
        std::vector<double> before(window);
        int64_t k = 0;
        for (; k < clear; ++k) {
            clear_step(k, &band_[static_cast<size_t>((k + 1) * w_)], &band_[static_cast<size_t>(k * w_)]);
            const double* now = &band_[static_cast<size_t>(k * w_)];
            const int64_t stop = std::min(clear - 1, last_alike - p_);
            if (k + p_ > first_alike && stop > k + p_ &&
                std::memcmp(before.data(), now, window * sizeof(double)) == 0) {
                const double* w = before.data();  // rows k .. k + p as step k left them
                for (int64_t i = k + 1; i <= stop; ++i) std::copy_n(w, w_, &band_[static_cast<size_t>(i * w_)]);
                std::copy_n(w, window, &band_[static_cast<size_t>(stop * w_)]);
                if (cyclic_)
                    for (int64_t i = k + 1; i <= stop; ++i) strip_step(i, w + w_, w);
                settled_lo_ = k;
                settled_hi_ = stop;
                k = stop;
                first_alike = n_;  // once
                continue;
            }
            if (k + p_ <= last_alike) std::copy_n(now, window, before.begin());
        }
        for (; k + 1 < n_; ++k) step(k);
    }

    // Rows with equal factors found by factor(): [lo, hi] (lo > hi: none).
    int64_t settled_lo() const { return settled_lo_; }
    int64_t settled_hi() const { return settled_hi_; }

    // The rows of the matrix as 2w+1 = 2p+1 entries A(i, i-p) .. A(i, i+p),
    // columns modulo n on a cyclic matrix (before factor()).
    void rows(std::vector<double>& out) {
        out = band_;
        if (!cyclic_) return;
        for (int64_t i = 0; i < n_; ++i) {
            if (i >= p_ && i + q_ < n_) {
                i = std::max(i, n_ - q_ - 1);
                continue;
            }
            for (int m = -p_; m <= q_; ++m) {
                const int64_t j = ((i + m) % n_ + n_) % n_;
                out[static_cast<size_t>(i * w_ + (m + p_))] = stored(i, j) ? at(i, j) : 0.0;
            }
        }
    }

    void export_factors(LineFactors& f) {
        f.n = n_;
        f.p = p_;
        f.q = q_;
        f.cyclic = cyclic_;
        f.lower.assign(static_cast<size_t>(n_ * p_), 0.0);
        f.upper.assign(static_cast<size_t>(n_ * q_), 0.0);
        f.diag.assign(static_cast<size_t>(n_), 0.0);
        for (int64_t i = 0; i < n_; ++i) {
            const double* row = &band_[static_cast<size_t>(i * w_)];
            f.diag[static_cast<size_t>(i)] = row[p_];
            for (int m = 1; m <= p_; ++m)
                if (i - m >= 0) f.lower[static_cast<size_t>(i * p_ + m - 1)] = row[p_ - m];
            for (int m = 1; m <= q_; ++m)
                if (i + m < n_) f.upper[static_cast<size_t>(i * q_ + m - 1)] = row[p_ + m];
        }
        if (cyclic_) {
            f.bottom.assign(static_cast<size_t>(q_ * n_), 0.0);
            f.right.assign(static_cast<size_t>(p_ * n_), 0.0);
            for (int r = 0; r < q_; ++r) {
                const int64_t i = n_ - q_ + r;
                if (i > p_)
                    std::copy_n(&bottom_[static_cast<size_t>(r * n_)], static_cast<size_t>(i - p_),
                                &f.bottom[static_cast<size_t>(r * n_)]);
            }
            for (int c = 0; c < p_; ++c) {
                const int64_t j = n_ - p_ + c;
                for (int64_t i = 0; i < j - q_; ++i)
                    f.right[static_cast<size_t>(c * n_ + i)] = right_[static_cast<size_t>(i * p_ + c)];
            }
        }
    }

    // Entry (i, j) of row i inside the band, for filling.
    double* band_row(int64_t i) { return &band_[static_cast<size_t>(i * w_)]; }
    int width() const { return w_; }

   private:
    // One step over the whole pattern.
    void step(int64_t k) {
        const int64_t r0 = k + 1, r1 = std::min<int64_t>(k + p_, n_ - 1);
        const int64_t b0 = cyclic_ ? std::max<int64_t>(n_ - q_, k + p_ + 1) : n_;
        const int64_t c0 = k + 1, c1 = std::min<int64_t>(k + q_, n_ - 1);
        const int64_t s0 = cyclic_ ? std::max<int64_t>(n_ - p_, k + q_ + 1) : n_;
        const double pivot = at(k, k);
        for (int64_t i = r0; i <= r1; ++i) at(i, k) /= pivot;
        for (int64_t i = b0; i < n_; ++i) at(i, k) /= pivot;
        auto update_row = [&](int64_t i) {
            const double lik = at(i, k);
            for (int64_t j = c0; j <= c1; ++j) at(i, j) -= lik * at(k, j);
            for (int64_t j = s0; j < n_; ++j) at(i, j) -= lik * at(k, j);
        };
        for (int64_t i = r0; i <= r1; ++i) update_row(i);
        for (int64_t i = b0; i < n_; ++i) update_row(i);
    }

    // step() where rows k .. k + p and their band columns lie clear of the
    // last p columns and q rows: the same updates in the same order.  rk:
    // row k, below: the p rows below it.
    void clear_step(int64_t k, double* below, const double* rk) {
        const double* bk = rk + p_;
        for (int a = 1; a <= p_; ++a) {
            double* row = below + (a - 1) * w_ + (p_ - a);  // column k
            row[0] /= bk[0];
            const double l = row[0];
            for (int m = 1; m <= q_; ++m) row[m] -= l * bk[m];
        }
        if (cyclic_) strip_step(k, below, rk);
    }

    // The strips' share of such a step (p == q): the right columns of the p
    // rows below row k, and the bottom rows.
    void strip_step(int64_t k, const double* below, const double* rk) {
        const double* right = &right_[static_cast<size_t>(k * p_)];
        for (int a = 1; a <= p_; ++a) {
            const double l = below[(a - 1) * w_ + (p_ - a)];
            double* ri = &right_[static_cast<size_t>((k + a) * p_)];
            for (int c = 0; c < p_; ++c) ri[c] -= l * right[c];
        }
        const double* bk = rk + p_;
        for (int r = 0; r < q_; ++r) {
            double* row = &bottom_[static_cast<size_t>(r * n_ + k)];
            row[0] /= bk[0];
            const double l = row[0];
            for (int m = 1; m <= q_; ++m) row[m] -= l * bk[m];
            double* corner = &band_[static_cast<size_t>((n_ - q_ + r) * w_ + (p_ - r))];  // column n - p
            for (int c = 0; c < p_; ++c) corner[c] -= l * right[c];
        }
    }

    int64_t settled_lo_ = 1, settled_hi_ = 0;
    int64_t n_;
    int p_, q_, w_;
    bool cyclic_;
    std::vector<double> band_, right_, bottom_;
};

// Rows until the recurrence of either sweep, started from a state of size 1 with
// zero right-hand sides, falls below 2^-24 and below 2^-53 (the largest over
// a few starts: the unit states at the middle row on a uniform grid, whose
// interior rows are alike; elsewhere eight rows, and one state of alternating
// signs, which the recurrences, whose poles are negative, keep longest);
// kMaxForget if it does not.  Every unit state at eight rows took 14 us of a
// build of 130 (order 7, 200 non-uniform points).
constexpr int kMaxForget = 128;

void forget_rows(const LineFactors& f, bool uniform, int* rows24, int* rows53) {
    const int bw = f.p;
    const int64_t starts = uniform ? 1 : std::min<int64_t>(8, f.n);
    *rows24 = *rows53 = 0;
    for (int64_t s = 0; s < 2 * starts; ++s)
        for (int unit = 0; unit < (uniform ? bw : 1); ++unit) {
            const bool forward = s < starts;
            double h[16] = {};
            h[unit] = 1.0;
            for (int m = 1; !uniform && m < bw; ++m) h[m] = -h[m - 1];
            const int64_t j0 = uniform ? f.n / 2 : (s % starts) * f.n / starts;
            int rows = 0, r24 = kMaxForget, r53 = kMaxForget;
            for (int64_t j = forward ? j0 : f.n - 1 - j0; j >= 0 && j < f.n; j += forward ? 1 : -1) {
                double v = 0.0, big = 0.0;
                const double* c = forward ? &f.lower[static_cast<size_t>(j * bw)] : &f.upper[static_cast<size_t>(j * bw)];
                for (int m = 0; m < bw; ++m) v -= c[m] * h[m];
                if (!forward) v /= f.diag[static_cast<size_t>(j)];
                for (int m = bw - 1; m > 0; --m) h[m] = h[m - 1];
                h[0] = v;
                for (int m = 0; m < bw; ++m) big = std::max(big, std::fabs(h[m]));
                ++rows;
                if (big <= 0x1p-24) r24 = std::min(r24, rows);
                if (big <= 0x1p-53) r53 = rows;
                if (r53 < kMaxForget || rows >= kMaxForget) break;
            }
            // a start that runs out of rows says nothing
            if (r53 == kMaxForget && rows < kMaxForget) continue;
            *rows24 = std::max(*rows24, r24);
            *rows53 = std::max(*rows53, r53);
        }
    if (*rows53 == 0) *rows24 = *rows53 = kMaxForget;  // short lines: no start had the rows
}

// Division by a divisor known in advance: with zh = 1/d rounded down and zl
// = 1/d - zh rounded, RN(x zh + RN(x zl)) differs from x/d before the last
// rounding by less than 2^(2-2p) of it (p mantissa bits: 2^-2p from the
// rounding of zl, twice that from x zl).  It is the correctly rounded
// quotient unless x/d lies that close to the middle M of two neighbouring
// numbers.  With X and Y the p-bit integer mantissas of x and d, M = N /
// 2^K (N odd, p+1 bits; K = p for X >= Y, else p + 1) and R = 2^K X - N Y
// such an x has |R| < 16, so N = -R / Y modulo 2^K: every candidate is
// listed and tried.  (Brisebarre, Muller and Raina, IEEE Transactions on
// Computers 53(8), 2004.)
template <typename C>
bool known_divisor_impl(C d, int p, C* zh, C* zl) {
    if (!(d > static_cast<C>(0x1p-40) && d < static_cast<C>(0x1p40))) return false;
    C h = static_cast<C>(1) / d;
    C e = std::fma(-d, h, static_cast<C>(1));
    if (e < 0) {
        h = std::nextafter(h, static_cast<C>(0));
        e = std::fma(-d, h, static_cast<C>(1));
    }
    *zh = h;
    *zl = e / d;
    int exponent = 0;
    const uint64_t Y = static_cast<uint64_t>(std::ldexp(std::frexp(d, &exponent), p));
    int s = 0;
    while (((Y >> s) & 1) == 0) ++s;
    const uint64_t odd = Y >> s;
    uint64_t inv = odd;  // inverse modulo 2^64 by Newton's iteration
    for (int i = 0; i < 6; ++i) inv *= 2 - odd * inv;
    for (int K = p; K <= p + 1; ++K)
        for (int64_t R = -16; R <= 16; ++R) {
            if (R == 0 || (R & ((int64_t{1} << std::min(s, 40)) - 1)) != 0) continue;
            const uint64_t mod = uint64_t{1} << (K - s);
            const uint64_t first = (static_cast<uint64_t>(-(R >> s)) * inv) & (mod - 1);
            for (uint64_t N = first; N < (uint64_t{1} << (p + 1)); N += mod) {
                if (N < (uint64_t{1} << p) || (N & 1) == 0) continue;
                const __int128 num = static_cast<__int128>(N) * Y + R;
                const uint64_t X = static_cast<uint64_t>(num >> K);
                if (X < (uint64_t{1} << (p - 1)) || X >= (uint64_t{1} << p)) continue;
                const C x = static_cast<C>(X);
                const C low = x * *zl;
                if (std::fma(x, *zh, low) != x / d) return false;
            }
        }
    return true;
}

// Segment plan of one compute type from its factors, rows [equal_lo,
// equal_hi] of which are known to be equal.  The warm-up covers
// the decay of the starting state to a rounding (`base` rows) and
// then the rows two almost equal states take to round to the same bits,
// 4 decades of probability in about 10 r^2 + 2 rows, r = rows per factor e
// of decay (fitted to measured merges, orders 2 to 7); 2.2 times that
// leaves about one failed comparison in 10^10.
template <typename C>
SegmentPlan segment_plan(const LineFactors& f, const std::vector<C>& lower, const std::vector<C>& upper,
                         const std::vector<C>& diag, int base, int rows53, int64_t equal_lo, int64_t equal_hi) {
    SegmentPlan s;
    const int bw = f.p;
    const int64_t n = f.n;
    if (n >= (int64_t{1} << 30)) return s;
    auto same = [&](const std::vector<C>& v, int w, int64_t a, int64_t b) {
        return w == 0 || std::memcmp(&v[static_cast<size_t>(a * w)], &v[static_cast<size_t>(b * w)],
                                     static_cast<size_t>(w) * sizeof(C)) == 0;
    };
    // grown from the rows known to be equal
    if (equal_lo > equal_hi) equal_lo = equal_hi = n / 2;
    const int64_t mid = equal_lo;
    int64_t a = mid, e = equal_hi + 1;
    while (a > 0 && same(lower, bw, a - 1, mid)) --a;
    while (e < n && same(lower, bw, e, mid)) ++e;
    s.flo = static_cast<int>(a);
    s.fhi = static_cast<int>(e);
    a = mid;
    e = equal_hi + 1;
    while (a > 0 && same(upper, bw, a - 1, mid) && same(diag, 1, a - 1, mid)) --a;
    while (e < n && same(upper, bw, e, mid) && same(diag, 1, e, mid)) ++e;
    s.blo = static_cast<int>(a);
    s.bhi = static_cast<int>(e);
    for (int m = 0; m < bw; ++m) {
        s.eq_lower[m] = static_cast<double>(lower[static_cast<size_t>(s.flo * bw + m)]);
        s.eq_upper[m] = static_cast<double>(upper[static_cast<size_t>(s.blo * bw + m)]);
    }
    if (bw > 0) {
        if (base >= kMaxForget) return s;
        const double r = rows53 / 36.74;
        s.warm = (static_cast<int>(base + 2.2 * (10.0 * r * r + 2.0)) + 7) / 8 * 8;
        C zh = 0, zl = 0;
        s.fast_divide = known_divisor(diag[static_cast<size_t>(s.blo)], &zh, &zl);
        s.zh = static_cast<double>(zh);
        s.zl = static_cast<double>(zl);
        for (int q = 0; f.cyclic && q < bw; ++q)
            for (int64_t j = s.warm; j < n; ++j)
                s.strip_rest = std::max(s.strip_rest, std::fabs(f.bottom[static_cast<size_t>(q * n + j)]));
        // as a C, not below any rounded strip entry
        s.strip_rest = static_cast<double>(std::nextafter(static_cast<C>(s.strip_rest), static_cast<C>(1)));
    }
    return s;
}

// Span containing x among t[order .. last]: the unique mu with
// t[mu] <= x < t[mu+1], clamped to [order, last] (BSpline.hpp:146-156).
int64_t find_span(const std::vector<double>& t, int order, double x, int64_t last) {
    int64_t lo = order + 1, hi = last + 1;
    while (lo < hi) {
        const int64_t mid = lo + (hi - lo) / 2;
        if (x < t[static_cast<size_t>(mid)])
            hi = mid;
        else
            lo = mid + 1;
    }
    return lo - 1;
}

}  // namespace

void fill_reciprocals(int order, DimSetup& s) {
    const int64_t nt = static_cast<int64_t>(s.knots.size());
    const int T = order * (order + 1) / 2;
    s.recip.assign(static_cast<size_t>(nt * std::max(T, 1)), 0.0);
    const double* t = s.knots.data();
    for (int64_t mu = order; mu <= nt - order - 2; ++mu)
        for (int i = 1; i <= order; ++i)
            for (int a = 1; a <= i; ++a) {
                const double d = t[mu + a] - t[mu + a - i];
                s.recip[static_cast<size_t>(mu * T + i * (i - 1) / 2 + a - 1)] = d != 0.0 ? 1.0 / d : 0.0;
            }
}

namespace {

// Power-basis coefficients (in u = (x - t[mu]) / dx) of the order+1 B-splines
// non-zero on span mu: the Cox-de Boor recursion run on polynomials.
void span_polynomials(const std::vector<double>& t, int k, int64_t mu, double dx, double* out) {
    const int w = k + 1;
    std::vector<double> tau(static_cast<size_t>(2 * k + 2), 0.0);  // tau[i + k] = knot mu+i, i in [-k, k+1]
    for (int i = -k; i <= k + 1; ++i) {
        const int64_t idx = mu + i;
        if (idx >= 0 && idx < static_cast<int64_t>(t.size()))
            tau[static_cast<size_t>(i + k)] = (t[static_cast<size_t>(idx)] - t[static_cast<size_t>(mu)]) / dx;
    }
    auto T = [&](int i) { return tau[static_cast<size_t>(i + k)]; };
    std::vector<double> b(static_cast<size_t>(w * w), 0.0);  // b[j*w + p]
    b[static_cast<size_t>(k * w)] = 1.0;
    for (int i = 1; i <= k; ++i) {
        const int first = k - i;
        for (int j = 0; j <= i; ++j) {
            const int idx = first + j;
            std::vector<double> nb(static_cast<size_t>(w), 0.0);
            if (j != 0) {  // b[idx] * (u - tau_{j-i}) / (tau_j - tau_{j-i})
                const double lo = T(j - i), den = T(j) - T(j - i);
                for (int p = 0; p < w; ++p) {
                    const double c = b[static_cast<size_t>(idx * w + p)] / den;
                    if (p + 1 < w) nb[static_cast<size_t>(p + 1)] += c;
                    nb[static_cast<size_t>(p)] -= c * lo;
                }
            }
            if (idx != k) {  // b[idx+1] * (tau_{j+1} - u) / (tau_{j+1} - tau_{j+1-i})
                const double hi = T(j + 1), den = T(j + 1) - T(j + 1 - i);
                for (int p = 0; p < w; ++p) {
                    const double c = b[static_cast<size_t>((idx + 1) * w + p)] / den;
                    nb[static_cast<size_t>(p)] += c * hi;
                    if (p + 1 < w) nb[static_cast<size_t>(p + 1)] -= c;
                }
            }
            for (int p = 0; p < w; ++p) b[static_cast<size_t>(idx * w + p)] = nb[static_cast<size_t>(p)];
        }
    }
    for (int q = 0; q < w * w; ++q) out[q] = b[static_cast<size_t>(q)];
}

void fill_uniform_classes(int k, DimSetup& s, double xmin, double xmax) {
    const int64_t nt = static_cast<int64_t>(s.knots.size());
    const int64_t last = nt - k - 2;
    const int64_t nspan = last - k + 1;
    s.xmin = xmin;
    s.xmax = xmax;
    s.half = 0.5 * static_cast<double>(nt - (s.n + (s.periodic ? 1 : 0)));
    if (s.periodic) {
        s.nleft = s.nright = 0;
    } else {
        // span mu is interior when knots mu-k+1 .. mu+k all lie in [k+1, nt-k-2]
        s.nleft = static_cast<int>(std::min<int64_t>(nspan, k));
        s.nright = static_cast<int>(std::min<int64_t>(nspan - s.nleft, k));
    }
    s.nclass = 1 + s.nleft + s.nright;
    const int w = k + 1;
    s.poly.assign(static_cast<size_t>(s.nclass * w * w), 0.0);
    const int64_t interior = s.periodic ? k : k + s.nleft;
    if (interior <= last - s.nright) span_polynomials(s.knots, k, interior, s.dx, &s.poly[0]);
    for (int c = 0; c < s.nleft; ++c)
        span_polynomials(s.knots, k, k + c, s.dx, &s.poly[static_cast<size_t>((1 + c) * w * w)]);
    for (int c = 0; c < s.nright; ++c)
        span_polynomials(s.knots, k, last - c, s.dx, &s.poly[static_cast<size_t>((1 + s.nleft + c) * w * w)]);
}

void set_range(int order, DimSetup& s) {
    const size_t nt = s.knots.size();
    s.lo = s.knots[static_cast<size_t>(order)];
    s.hi = s.knots[nt - static_cast<size_t>(order) - (2 - static_cast<size_t>(order % 2))];
}

}  // namespace

bool known_divisor(double d, double* zh, double* zl) { return known_divisor_impl(d, 53, zh, zl); }
bool known_divisor(float d, float* zh, float* zl) { return known_divisor_impl(d, 24, zh, zl); }

int64_t knot_count(int order, bool periodic, int64_t n) {
    const int64_t np = n + (periodic ? 1 : 0);
    return np + (periodic ? 2 * order + (1 - order % 2) : order + 1);
}

void basis_values(const double* t, int64_t mu, double x, int order, int spline_order, double* b) {
    for (int i = 0; i <= order; ++i) b[i] = 0.0;
    b[order] = 1.0;
    for (int i = 1; i <= spline_order; ++i) {
        const int first = order - i;
        for (int j = 0; j <= i; ++j) {
            const int64_t l = mu - (i - j), r = mu + j + 1;
            const double left = j == 0 ? 0.0 : b[first + j] * (x - t[l]) / (t[r - 1] - t[l]);
            const double right = first + j == order ? 0.0 : b[first + j + 1] * (t[r] - x) / (t[r] - t[l + 1]);
            b[first + j] = left + right;
        }
    }
}

std::string setup_dimension(int order, bool periodic, int64_t n, double xmin, double xmax,
                            const double* nodes, DimSetup& s, bool refined) {
    const int k = order;
    if (n < std::max<int64_t>(2, k + 1)) return "too few values along a dimension for the spline order";
    const int bw = periodic ? k / 2 : (k == 0 ? 0 : k - 1);
    if (periodic && n < 2 * bw + 2) return "too few values along a periodic dimension for the spline order";
    s.periodic = periodic;
    s.n = n;
    const int64_t np = n + (periodic ? 1 : 0);
    const int64_t nt = knot_count(k, periodic, n);
    s.knots.assign(static_cast<size_t>(nt), 0.0);
    double* t = s.knots.data();
    if (!nodes) {
        // uniform knots: Interpolation.hpp:322-362
        if (!(xmax > xmin)) return "range maximum must exceed the minimum";
        s.uniform = true;
        s.dx = (xmax - xmin) / static_cast<double>(np - 1);
        const int64_t extra = nt - np;
        const double half = 0.5 * static_cast<double>(extra);
        for (int64_t i = 0; i < nt; ++i) t[i] = xmin;
        if (periodic) {
            for (int64_t i = 0; i < nt; ++i) t[i] = xmin + (static_cast<double>(i) - half) * s.dx;
        } else {
            for (int64_t i = k + 1; i < nt - k - 1; ++i) t[i] = xmin + (static_cast<double>(i) - half) * s.dx;
            for (int64_t i = nt - k - 1; i < nt; ++i) t[i] = xmax;
        }
        set_range(k, s);
        fill_uniform_classes(k, s, xmin, xmax);
    } else {
        // node-coordinate knots: Interpolation.hpp:365-447
        s.uniform = false;
        s.nodes.assign(nodes, nodes + np);
        for (int64_t i = 0; i + 1 < np; ++i)
            if (!(nodes[i + 1] > nodes[i])) return "Given coordinate is not monotonically increasing";
        if (periodic) {
            for (int64_t i = k + 1; i < k + np; ++i)
                t[i] = k % 2 == 0 ? 0.5 * (nodes[i - k - 1] + nodes[i - k]) : nodes[i - k];
            const double period = nodes[np - 1] - nodes[0];
            for (int64_t i = 0; i < k + 1; ++i) {
                t[i] = t[np + i - 1] - period;
                t[nt - i - 1] = t[nt - i - np] + period;
            }
        } else {
            if (k == 0) return "order 0 is not defined on a non-uniform dimension";
            for (int64_t i = 0; i <= k; ++i) t[i] = nodes[0];
            double window = 0.0;
            for (int64_t i = 1; i < k; ++i) window += nodes[i];
            for (int64_t i = k + 1; i < np; ++i) {
                window += nodes[i - 1];
                t[i] = window / static_cast<double>(k);
                window -= nodes[i - k];
            }
            for (int64_t i = np; i < np + k + 1; ++i) t[i] = nodes[np - 1];
        }
    }
    set_range(k, s);

    // collocation matrix: InterpolationTemplate.hpp:254-426
    PatternMatrix m(n, bw, bw, periodic);
    double bv[64];
    if (periodic && s.uniform)
        basis_values(t, k, t[k] + static_cast<double>(1 - k % 2) * s.dx * 0.5, k, k, bv);
    for (int64_t i = 0; i < n; ++i) {
        if (!periodic && (i == 0 || i == n - 1)) {
            m.at(i, i) = 1.0;
            continue;
        }
        int64_t mu;
        const bool internal = i > k / 2 && i < n - k / 2 - 1;
        if (s.uniform) {
            mu = periodic ? i + k : std::min<int64_t>(nt - k - 2, i > k / 2 ? i + (k + 1) / 2 : k);
            // clamped rows near the ends recompute the basis; interior rows
            // reuse the last one (the interior basis is translation
            // invariant on a uniform grid)
            if (!periodic && (mu <= 2 * k + 1 || mu >= nt - 2 * k - 2))
                basis_values(t, mu, s.lo + static_cast<double>(i) * s.dx, k, k, bv);
        } else {
            const double x = s.nodes[static_cast<size_t>(i)];
            if (periodic) {
                mu = i + k;
            } else {
                const int64_t last = std::min<int64_t>(nt - k - 1, i + k);
                const int64_t hint = i + 1;
                mu = (t[hint] <= x && t[hint + 1] > x) ? hint : find_span(s.knots, k, x, last);
            }
            basis_values(t, mu, x, k, k, bv);
        }
        const int64_t cnt = periodic ? (k | 1) : k == 1 ? 1 : (s.uniform && internal) ? (k | 1) : k + 1;
        const int64_t row0 = i + (periodic ? bw : 0), col0 = mu - k;
        if (row0 < n && col0 >= 0 && col0 + cnt <= n && m.in_band(row0, col0) && m.in_band(row0, col0 + cnt - 1)) {
            std::copy_n(bv, cnt, m.band_row(row0) + (col0 - row0 + bw));
            continue;
        }
        for (int64_t j = 0; j < cnt; ++j) {
            const int64_t row = row0 % n;
            const int64_t col = (col0 + j) % n;
            if (!m.stored(row, col)) return "collocation entry outside the band pattern";
            m.at(row, col) = bv[j];
        }
    }
    // the unfactored matrix, row-wise, for FP64 residuals
    s.colloc_w = bw;
    if (refined) m.rows(s.colloc);
    // equal rows: those that reuse the interior basis (their spans lie past
    // the recomputed ones), or all of a circulant but its wrapped ends
    if (!s.uniform)
        m.factor(n, 0);
    else if (periodic)
        m.factor(bw, n - 2 * bw - 2);
    else
        m.factor(2 * k + 2 - (k + 1) / 2, nt - 2 * k - 3 - (k + 1) / 2);
    m.export_factors(s.lu);
    auto round32 = [](const std::vector<double>& v, std::vector<float>& out) {
        out.resize(v.size());
        for (size_t i = 0; i < v.size(); ++i) out[i] = static_cast<float>(v[i]);
    };
    if (refined) {
        round32(s.lu.lower, s.lower32);
        round32(s.lu.upper, s.upper32);
        round32(s.lu.diag, s.diag32);
        round32(s.lu.bottom, s.bottom32);
        round32(s.lu.right, s.right32);
    }
    for (int64_t i = 0; i < n; ++i)
        if (!(std::fabs(s.lu.diag[static_cast<size_t>(i)]) > 0.0) || !std::isfinite(s.lu.diag[static_cast<size_t>(i)]))
            return "singular collocation matrix";
    if (n < kMinSegmentRows) return "";  // never cut: the segment plans stay empty
    int rows24 = 0, rows53 = 0;
    if (s.lu.p > 0) forget_rows(s.lu, s.uniform, &rows24, &rows53);
    s.lu.seg64 = segment_plan(s.lu, s.lu.lower, s.lu.upper, s.lu.diag, rows53, rows53, m.settled_lo(), m.settled_hi());
    if (refined)
        s.lu.seg32 = segment_plan(s.lu, s.lower32, s.upper32, s.diag32, rows24, rows53, m.settled_lo(), m.settled_hi());
    return "";
}

std::string setup_from_knots(int order, bool periodic, int64_t n, const double* knots, int64_t nknots,
                             DimSetup& s) {
    const int64_t want = n + order + 1 + (periodic ? order : 0);
    if (nknots != want) return "Inconsistency between knot number and control point number";
    if (n < order + 1) return "fewer control points than order + 1";
    for (int64_t i = 0; i + 1 < nknots; ++i)
        if (knots[i + 1] < knots[i]) return "knot vector must be non-decreasing";
    s.periodic = periodic;
    s.uniform = false;
    s.n = n;
    s.knots.assign(knots, knots + nknots);
    set_range(order, s);
    s.dx = 0.0;
    fill_reciprocals(order, s);
    return "";
}

}  // namespace intp_amd
