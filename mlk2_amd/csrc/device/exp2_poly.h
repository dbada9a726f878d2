// 2^y in f64 by a polynomial, for the softmax kernels.
#pragma once

#include <hip/hip_runtime.h>

/// 2^f on |f| <= 1/2 by Chebyshev interpolation at 10 nodes: relative error
/// 1.9e-14.
constexpr double kExp2C10[10] = {1.0000000000000135,    0.6931471805599462,     0.2402265069564034,
                                 0.05550410866465166,   0.00961812919393429,    0.0013333558200796013,
                                 0.0001540343375126647, 1.5252672924257465e-05, 1.3259645241948732e-06,
                                 1.020590550210069e-07};

/// 2^y (times the coefficients' common factor) for y in [-1000, 1000]; NaN
/// stays NaN. y + 1.5 * 2^52 leaves rint(y) in the low word, from where it is
/// added into the exponent field.
template <int N>
__device__ __forceinline__ double exp2Poly(double y, const double (&c)[N]) {
    const double t = y + 0x1.8p52;
    const double f = y - (t - 0x1.8p52);
    double p = c[N - 1];
#pragma unroll
    for (int i = N - 2; i >= 0; --i) p = __builtin_fma(p, f, c[i]);
    return __hiloint2double(__double2hiint(p) + (__double2loint(t) << 20), __double2loint(p));
}
