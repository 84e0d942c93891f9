// Quotients by a divisor that many values share: one reciprocal, then a
// multiplication and one residual correction each (Markstein), which gives the
// correctly rounded quotient except in rare near-ties.
#pragma once

#include <hip/hip_runtime.h>

namespace rlg {

// 1 / d to an ulp or two from the hardware's estimate (Newton's iteration);
// 0 for an infinite d, NaN for a NaN.
__device__ __forceinline__ double recip(double d) {
    double y = __builtin_amdgcn_rcp(d);
#pragma unroll
    for (int i = 0; i < 2; ++i) y = fma(fma(-d, y, 1.0), y, y);
    return fabs(d) == __builtin_inf() ? 0.0 : y;
}
// a / d from r = 1 / d; the correction is left out where the residual is not
// finite.
template <class T> __device__ __forceinline__ T div_recip(T a, T d, T r) {
    const T q = a * r, e = fma(-q, d, a);
    return fabs(e) < T(__builtin_inf()) ? fma(e, r, q) : q;
}

}  // namespace rlg
