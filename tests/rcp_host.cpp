// Host build of the pivots' reciprocal (uclchem_amd/csrc/ucg_recip.h) with an estimate as coarse as
// the GPU's: 24 bits, subnormal results included.  Test infrastructure: built by
// tests/test_reciprocal_host.py with g++.
#include <cmath>
#include "../uclchem_amd/csrc/ucg_recip.h"

static double estimate(double x)
{
    const double r = 1.0 / x;
    if (r == 0.0 || !std::isfinite(r)) return r;
    int e;
    const double m = std::frexp(r, &e);
    return std::ldexp(std::floor(std::ldexp(m, 24)), e - 24);
}

extern "C" void pivot_reciprocals(int n, const double *x, double *r, int *bad)
{
    for (int i = 0; i < n; i++) {
        bool b = false;
        r[i] = ucg::pivot_reciprocal(x[i], estimate(x[i]), b);
        bad[i] = b;
    }
}
