// The factors of setup_dimension(), which copies rows that have settled,
// against the elimination of every entry of the dense matrix, bit for bit.

#include <cstdio>
#include <cstring>
#include <vector>

#include "setup.hpp"

using intp_amd::DimSetup;

namespace {

bool check(int order, bool periodic, int64_t n, bool uniform) {
    std::vector<double> x(static_cast<size_t>(n + 1));
    for (int64_t i = 0; i <= n; ++i) x[static_cast<size_t>(i)] = 0.3 * i + 0.1 * ((i * 7) % 3);
    DimSetup s, plain;
    const double* nodes = uniform ? nullptr : x.data();
    if (!setup_dimension(order, periodic, n, -0.4, 1.7, nodes, s, true).empty()) return false;
    if (!setup_dimension(order, periodic, n, -0.4, 1.7, nodes, plain, false).empty()) return false;
    const int w = s.colloc_w;
    std::vector<double> a(static_cast<size_t>(n * n), 0.0);
    auto at = [&](int64_t i, int64_t j) -> double& { return a[static_cast<size_t>(i * n + j)]; };
    for (int64_t i = 0; i < n; ++i)
        for (int m = -w; m <= w; ++m) {
            const int64_t j = periodic ? (i + m + n) % n : i + m;
            if (j >= 0 && j < n) at(i, j) = s.colloc[static_cast<size_t>(i * (2 * w + 1) + m + w)];
        }
    for (int64_t k = 0; k + 1 < n; ++k)
        for (int64_t i = k + 1; i < n; ++i) {
            if (at(i, k) == 0.0) continue;
            at(i, k) /= at(k, k);
            for (int64_t j = k + 1; j < n; ++j)
                if (at(k, j) != 0.0) at(i, j) -= at(i, k) * at(k, j);
        }
    auto equal = [](double u, double v) { return u == v; };
    for (int64_t i = 0; i < n; ++i) {
        if (!equal(s.lu.diag[static_cast<size_t>(i)], at(i, i))) return false;
        for (int m = 1; m <= w; ++m) {
            if (i - m >= 0 && !equal(s.lu.lower[static_cast<size_t>(i * w + m - 1)], at(i, i - m))) return false;
            if (i + m < n && !equal(s.lu.upper[static_cast<size_t>(i * w + m - 1)], at(i, i + m))) return false;
        }
    }
    for (int q = 0; periodic && q < w; ++q)
        for (int64_t j = 0; j < n - w + q - w; ++j) {
            if (!equal(s.lu.bottom[static_cast<size_t>(q * n + j)], at(n - w + q, j))) return false;
            if (!equal(s.lu.right[static_cast<size_t>(q * n + j)], at(j, n - w + q))) return false;
        }
    // the tables of refined builds change nothing in the others
    return plain.lu.lower == s.lu.lower && plain.lu.upper == s.lu.upper && plain.lu.diag == s.lu.diag &&
           plain.lu.bottom == s.lu.bottom && plain.lu.right == s.lu.right && plain.colloc.empty();
}

}  // namespace

int main() {
    for (int order = 0; order <= 7; ++order)
        for (int periodic = 0; periodic < 2; ++periodic)
            for (int uniform = order == 0 && !periodic ? 1 : 0; uniform < 2; ++uniform)
                for (int64_t n : {8, 9, 12, 15, 16, 17, 23, 31, 40, 61, 64, 100, 161, 240})
                    if (!check(order, periodic != 0, n, uniform != 0)) {
                        std::printf("order %d periodic %d n %d uniform %d\n", order, periodic, static_cast<int>(n), uniform);
                        return 1;
                    }
    return 0;
}
