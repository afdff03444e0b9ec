// Test helper: compares quotient(x, d, RN(1/d)) (lbm_amd/csrc/quotient.hpp)
// with the division of the host for the divisors of the fp64 collision and
// for relaxation times: random numerators, and numerators next to rounding
// boundaries of the quotient. Prints the number compared and of mismatches.
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <random>

#include "quotient.hpp"

using namespace lbm_amd;

int main(int argc, char** argv) {
    const long n = argc > 1 ? std::atol(argv[1]) : 100000;
    std::mt19937_64 rng(7);
    std::uniform_real_distribution<double> uni(0.0, 1.0);
    const double cs = kCS;
    long done = 0, bad = 0;
    auto check = [&](double x, double d, double y) {
        const double a = quotient(x, d, y), b = x / d;
        ++done;
        bad += std::memcmp(&a, &b, sizeof(a)) != 0 && !(a == 0 && b == 0);
    };
    auto divisor = [&](double d) {
        if (!quotient_divisor_ok(d)) return;
        const double y = 1.0 / d;
        for (long i = 0; i < n; ++i) {
            const double x = (uni(rng) - 0.5) * std::exp2(std::floor(uni(rng) * 600) - 500);
            check(x, d, y);
            // x next to (quotient half way between two doubles) * d
            const double q = x / d, up = std::nextafter(q, INFINITY);
            const double mid = std::fma(q, d, 0.5 * (up - q) * d);
            check(mid, d, y);
            check(std::nextafter(mid, INFINITY), d, y);
            check(std::nextafter(mid, -INFINITY), d, y);
        }
        check(0.0, d, y);
    };
    divisor(cs * cs);
    divisor(2 * cs * cs * cs * cs);
    divisor(2 * cs * cs);
    for (double tau : {0.5024, 0.53, 0.55, 0.6, 0.7, 0.8, 0.9, 1.0, 1.5, 1.7, 1.9999, 2.0, 3.0, 7.3, 1000.0}) divisor(tau);
    for (int i = 0; i < 40; ++i) divisor(0.5 + 1.5 * uni(rng));
    std::printf("%ld %ld\n", done, bad);
    return 0;
}
