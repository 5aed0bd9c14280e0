// FP64 quotient and square root for the pair kernels.  The compiler's division
// and sqrt take about 60 SIMD cycles per wave64 each with their scaling and
// special cases; the pair kernels know their ranges, so these take Newton steps
// from the hardware's approximation.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace vx {

// g / a for a normal a > 0, correctly rounded as `/` gives it: the start's
// residual e is below 2^-24, so y is within 2^-48, and the quotient's residual,
// a remainder of a few dozen ulp without rounding error of note, takes w to
// 2^-43 ulp of the quotient before the last rounding.  2^30 random pairs: no
// difference from `/`.
__device__ __forceinline__ double div_pos_exact(double g, double a) {
    double y = __builtin_amdgcn_rcp(a);
    y = fma(y, fma(-a, y, 1.0), y);
    const double w = g * y;
    return fma(fma(-a, w, g), y, w);
}

// g / a for any a >= 0 that is no denormal number: infinities, zeros and NaN as
// `/` has them.
__device__ __forceinline__ double div_nonneg(double g, double a) {
    return __builtin_amdgcn_div_fixup(div_pos_exact(g, a), a, g);
}

// sqrt(a) for a normal a > 0, correctly rounded as sqrt() gives it, and g over
// it, correctly rounded, by the same steps (the start's e = (1 - a y^2) / 2 is
// below 2^-24; 2^30 random pairs: no difference from sqrt and `/`).
__device__ __forceinline__ double sqrt_pos_exact(double a, double g, double &q) {
    double y = __builtin_amdgcn_rsq(a);
    const double t = a * y;
    const double e = fma(-t, 0.5 * y, 0.5);
    const double s0 = fma(t, e, t);
    y = fma(y, e, y);
    const double s = fma(fma(-s0, s0, a), 0.5 * y, s0);
    const double w = g * y;
    q = fma(fma(-s, w, g), y, w);
    return s;
}

__device__ __forceinline__ void order2(double &a, double &b) {
    const double lo = fmin(a, b), hi = fmax(a, b);
    a = lo;
    b = hi;
}

// Four values at a time: they are sorted (5 exchanges), the pairwise minima
// with the kept ones in reverse are the four smallest of the eight, a bitonic
// run that 4 exchanges sort.  FP64 has no med3: 5.5 min/max a value against 13.
// The values must be no NaN (an exchange would double its neighbour).
__device__ __forceinline__ void keep4x4(double &m0, double &m1, double &m2, double &m3, double a, double b, double c,
                                        double d) {
    order2(a, b);
    order2(c, d);
    order2(a, c);
    order2(b, d);
    order2(b, c);
    m0 = fmin(m0, d);
    m1 = fmin(m1, c);
    m2 = fmin(m2, b);
    m3 = fmin(m3, a);
    order2(m0, m2);
    order2(m1, m3);
    order2(m0, m1);
    order2(m2, m3);
}

// Neither NaN nor an infinity nor above 2^500, so that squares of differences
// stay in range.  odd_bit's top bit is set for any other value; the bits of several
// values are or-ed.  Integer operations only: on wave-uniform values they run on
// the scalar unit (a maximum of several would go to the vector unit's max3).
__device__ __forceinline__ uint32_t odd_bit(double v) {
    return ((uint32_t)__double2hiint(v) & 0x7fffffffu) + (0x80000000u - 0x5f300000u);
}
__device__ __forceinline__ uint32_t odd_bit(float) { return 0; }  // FP32 takes every value through one path
template <typename T>
__device__ __forceinline__ bool ordinary(T v) { return (int32_t)odd_bit(v) >= 0; }

// A softening eps^2 that div_pos_exact divides by.
__device__ __forceinline__ bool ordinary_eps2(double v) { return v > 0x1p-1000 && v < 0x1p1000; }
__device__ __forceinline__ bool ordinary_eps2(float) { return true; }

}  // namespace vx
