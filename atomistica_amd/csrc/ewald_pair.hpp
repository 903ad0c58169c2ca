// Radial functions of the Ewald real-space pair sum, shared by ewald.hip and
// ewald_batch.hip: erfc(beta r) / r and
// (erfc(beta r) + 2 beta r / sqrt(pi) exp(-(beta r)^2)) / r^3
// (pme.f90:386-437).
#pragma once
#include <hip/hip_runtime.h>

namespace agpu {

// (1 + 2 x) exp(x^2) erfc(x) as a polynomial in t = (x - 3.75) / (x + 3.75),
// x >= 0: a Chebyshev series in t (the variable and the factor of Shepherd
// and Laframboise, Math. Comp. 36, 249 (1981)), coefficients from 50-digit
// arithmetic, written in powers of t.  Its error is below 5.2e-16 of the
// value for every x (1.2e-16 rms).
constexpr int EWP_DEG = 22;
__device__ constexpr double ewp_c[EWP_DEG + 1] = {
    1.23751263083782748e+00, -1.40240598585545245e-01, 3.58541548547902569e-03,
    8.22767384899950605e-02, -1.08803930142444619e-01, 9.23043211642812500e-02,
    -5.86933985766493402e-02, 2.83622773721111388e-02, -9.74657968326526208e-03,
    1.75562616519706364e-03, 2.93714378044955624e-04, -2.90155352460771292e-04,
    5.16465297417822530e-05, 2.23875657149000459e-05, -1.14380480333641408e-05,
    -9.79262570713956290e-07, 1.74198215864572570e-06, -5.08446538007496260e-08,
    -2.48571262499349461e-07, 1.87908232302200536e-08, 3.19792667255042236e-08,
    -1.95513588820174288e-09, -2.62310734887227245e-09};

// 1 / x for normal x > 0: the hardware's estimate and two Newton steps
__device__ __forceinline__ double ewp_rcp(double x)
{
    double y = __builtin_amdgcn_rcp(x);
    y = fma(y, fma(-x, y, 1.0), y);
    return fma(y, fma(-x, y, 1.0), y);
}

// e = erfc(beta r) / r, f = the force factor, from r^2.  Both share one
// exp(-(beta r)^2), so the FP64 form needs no erfc of its own: the pair costs
// about 75 FP64 operations (about 180 with erfc, exp, a square root and
// divisions, whose branches all run in a wavefront of mixed distances).
__device__ __forceinline__ void ewp_pair(double r2, double beta, double sap, double &e, double &f)
{
    // r = 0 and no NaN at r2 = 0: coincident charges give an infinite e, as
    // erfc(0) / 0 does
    const double ri = rsqrt(r2), r = fmax(r2 * ri, 0.0), x = beta * r;
    const double x1 = fma(2.0, x, 1.0), xk = x + 3.75;
    const double q = ewp_rcp(x1 * xk);
    const double t = (x - 3.75) * (q * x1);
    double p = ewp_c[EWP_DEG];
#pragma unroll
    for (int k = EWP_DEG - 1; k >= 0; --k) p = fma(p, t, ewp_c[k]);
    const double g = exp(-(beta * beta) * r2) * ri;
    const double w = p * (q * xk);                    // exp(x^2) erfc(x)
    e = g * w;
    f = g * (ri * ri) * fma(2.0 * sap, r, w);   // sap = beta / sqrt(pi)
}

__device__ __forceinline__ void ewp_pair(double r2, float beta, float sap, double &e, double &f)
{
    const float r = (float)sqrt(r2), ri = 1.0f / r;
    const float ec = erfcf(beta * r);
    e = (double)(ec * ri);
    f = (double)(ri * ri * ri * (ec + 2.0f * sap * r * expf(-(beta * beta) * (float)r2)));
}

}  // namespace agpu
