// sin and cos in double for the kernels that need one argument's pair per lane: fewer registers
// and instructions than the general routine, which also serves arguments up to 1e308.
#pragma once
#include <hip/hip_runtime.h>

// range of sincos_reduced: |x| below it keeps n = rint(2x/pi) an exact int
constexpr double kSincosLimit = 1e9;

// 1/k! with alternating signs, rounded to double: from 1/17! down to -1/3!, and from -1/18! down to -1/2!
#define SINCOS_COEFFICIENTS                                                                                              \
    {2.8114572543455206e-15, -7.647163731819816e-13, 1.6059043836821613e-10, -2.505210838544172e-08,                       \
     2.7557319223985893e-06, -0.0001984126984126984, 0.008333333333333333, -0.16666666666666666,                            \
     -1.5619206968586225e-16, 4.779477332387385e-14, -1.1470745597729725e-11, 2.08767569878681e-09,                       \
     -2.755731922398589e-07, 2.48015873015873e-05, -0.001388888888888889, 0.041666666666666664, -0.5}
constexpr double kSincosCoef[17] = SINCOS_COEFFICIENTS;

// sin and cos of y + n pi/2 for |y| a little over pi/4, n mod 4 = q: Taylor series of sin y (through
// y^17) and cos y (through y^18), whose first omitted terms are below 1e-19; k: kSincosCoef
template <typename K>
__device__ inline void sincos_quadrant(double y, int q, double *s, double *c, const K &k)
{
    const double z = y * y;
    double ps = k[0], pc = k[8];
#pragma unroll
    for (int i = 1; i < 8; i++) ps = fma(ps, z, k[i]);
#pragma unroll
    for (int i = 9; i < 17; i++) pc = fma(pc, z, k[i]);
    const double sy = fma(y * z, ps, y), cy = fma(z, pc, 1.0);
    const double sa = (q & 1) ? cy : sy, ca = (q & 1) ? sy : cy;
    *s = (q & 2) ? -sa : sa;
    *c = ((q + 1) & 2) ? -ca : ca;
}

// x - n pi/2 with pi/2 split into three doubles (c1 + c2 + c3; each product n * c_i exact inside an FMA)
__device__ inline double minus_quadrants(double x, double n)
{
    constexpr double c1 = 0x1.921fb54442d18p+0, c2 = 0x1.1a62633145c07p-54, c3 = -0x1.f1976b7ed8fbcp-110;
    return fma(-n, c3, fma(-n, c2, fma(-n, c1, x)));
}

constexpr double kTwoOverPi = 0x1.45f306dc9c883p-1;

// sin and cos of x for |x| < kSincosLimit: Cody-Waite reduction x = n pi/2 + y
__device__ inline void sincos_reduced(double x, double *s, double *c)
{
    const double n = rint(x * kTwoOverPi);
    sincos_quadrant(minus_quadrants(x, n), (int)n & 3, s, c, kSincosCoef);
}

// The same for every x, with no branch: n is rounded by adding 1.5 2^52, whose sum's low bits are n
// mod 4.  From 2^50 on, where neighbouring doubles lie 0.2 rad and more apart, x counts as 0 (a phase
// of modulus 1 like any other there); infinities and NaN give NaN.
template <typename K>
__device__ inline void sincos_wide(double x, double *s, double *c, const K &k)
{
    x = fabs(x) >= 0x1p50 ? x - x : x;
    const double t = fma(x, kTwoOverPi, 0x1.8p52), n = t - 0x1.8p52;
    sincos_quadrant(minus_quadrants(x, n), (int)__builtin_bit_cast(long long, t), s, c, k);
}
__device__ inline void sincos_wide(double x, double *s, double *c) { sincos_wide(x, s, c, kSincosCoef); }
