// Reciprocals of the Newton matrix's pivots.
#pragma once
#include "bdf_core.h"

namespace ucg {

// 1/x from an estimate good to 24 bits (the hardware's, 4.3e-8) and two Newton steps, whose last
// rounding is the only one that counts: half a unit in the last place, as the quotient.  NaN where x
// is zero, infinite or NaN, or so small that 1/x is not finite; `bad` is raised then.  It asks the
// result, since a pivot that passed a test of its own could still be too small: 0x1p-1030 gave NaN.
BDF_HD double pivot_reciprocal(double x, double estimate, bool &bad)
{
    double r = estimate;
    r = __builtin_fma(r, __builtin_fma(-x, r, 1.0), r);
    r = __builtin_fma(r, __builtin_fma(-x, r, 1.0), r);
    bad |= !(r == r);
    return r;
}

}  // namespace ucg
