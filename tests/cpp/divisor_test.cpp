// known_divisor (setup.cpp): x zh + (x zl), product and sum rounded once
// each, against x / d.  FP32: every numerator mantissa of each accepted
// divisor.  FP64: random numerators, and the pivots every order's uniform
// collocation matrix repeats in its interior.
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <random>

#include "setup.hpp"

using namespace intp_amd;

int main() {
    std::mt19937_64 rng(20261202);
    int accepted32 = 0, rejected32 = 0;
    for (int t = 0; t < 24; ++t) {
        const float d = std::ldexp(1.0f + static_cast<float>(rng() & 0x7fffff) * 0x1p-23f, static_cast<int>(rng() % 5) - 3);
        float zh, zl;
        if (!known_divisor(d, &zh, &zl)) {
            ++rejected32;
            continue;
        }
        ++accepted32;
        for (uint32_t m = 0; m < (1u << 23); ++m) {
            const float x = 1.0f + static_cast<float>(m) * 0x1p-23f;
            const float low = x * zl;
            if (std::fma(x, zh, low) != x / d) {
                std::printf("FP32: %a / %a\n", x, d);
                return 1;
            }
        }
    }
    int accepted64 = 0;
    auto check64 = [&](double d) {
        double zh, zl;
        if (!known_divisor(d, &zh, &zl)) return true;
        ++accepted64;
        for (int r = 0; r < 20000; ++r) {
            const double x = std::ldexp(1.0 + static_cast<double>(rng() >> 12) * 0x1p-52, static_cast<int>(rng() % 1800) - 880) *
                             (r % 2 ? 1.0 : -1.0);
            const double low = x * zl;
            if (std::fma(x, zh, low) != x / d) {
                std::printf("FP64: %a / %a\n", x, d);
                return false;
            }
        }
        const double z = -0.0, low = z * zl;
        return std::signbit(std::fma(z, zh, low));
    };
    for (int t = 0; t < 200; ++t)
        if (!check64(std::ldexp(1.0 + static_cast<double>(rng() >> 12) * 0x1p-52, static_cast<int>(rng() % 5) - 3))) return 1;
    for (int order = 2; order <= 7; ++order)
        for (int periodic = 0; periodic < 2; ++periodic) {
            DimSetup s;
            if (!setup_dimension(order, periodic != 0, 300, 0.0, 1.0, nullptr, s).empty()) return 1;
            if (!check64(s.lu.diag[static_cast<size_t>(s.lu.seg64.blo)])) return 1;
            // the rows of equal factors really are equal, and the interior is long
            if (s.lu.seg64.warm % 8 != 0 || s.lu.seg64.bhi - s.lu.seg64.blo < 200) return 1;
        }
    std::printf("divisor test: %d FP32 divisors accepted, %d rejected; %d FP64\n", accepted32, rejected32, accepted64);
    return accepted32 > 0 && accepted64 > 100 ? 0 : 1;
}
