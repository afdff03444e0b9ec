// Correctly rounded fp64 quotients x / d for a divisor d whose reciprocal is
// known beforehand, y = RN(1/d): one product and one residual correction
//   q = RN(x y),  r = RN(x - q d),  x / d = RN(q + r y)
// (Brisebarre, Muller, Raina, "Accelerating correctly rounded floating-point
// division when the divisor is known in advance", IEEE Transactions on
// Computers 53(8), 2004). Three instructions where a general division takes
// about eleven, and the same bits wherever
//   - x, q and r are normal numbers (or x = 0), and
//   - the significand of d is not within quotient_divisor_ok of 2: then |q -
//     x/d| stays below 1.5 ulp by a margin, so that a quotient next to a
//     rounding boundary has |q - x/d| close to half an ulp, r is exact, and
//     the reciprocal's error cannot move q + r y over the boundary.
#pragma once

#include <cstdint>

#include "lbm_hip/lattice.hpp"

namespace lbm_amd {

LBM_HD inline double quotient(double x, double d, double y) {
    const double q = x * y;
    const double r = __builtin_fma(-q, d, x);
    return __builtin_fma(r, y, q);
}

// Significand of d below 2 - 2^-20 (its top 20 bits not all ones).
LBM_HD inline bool quotient_divisor_ok(double d) {
    uint64_t b;
    __builtin_memcpy(&b, &d, sizeof(b));
    return ((b >> 32) & 0xFFFFFu) != 0xFFFFFu;
}

}  // namespace lbm_amd
