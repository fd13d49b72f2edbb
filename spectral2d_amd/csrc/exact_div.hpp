// exact_div.hpp -- correctly rounded divisions by a constant, without the
// division's instructions.
//
// With y = 1 / d rounded, q = x y is within one ulp of x / d, its remainder
// x - d q is exact under FMA, and one correction rounds to x / d (Markstein).
// The remainder of a zero is +0 whatever the zero's sign, so the result takes
// x's sign (d is positive).
#pragma once

#include <hip/hip_runtime.h>

namespace s2d {

// x / d with r = 1 / d rounded, d > 0. *odd is set where the remainder would
// underflow or is not a number: those take the division.
__host__ __device__ __forceinline__ double div_by(double x, double d, double r, bool *odd)
{
    const double q = x * r;
    const double a = __builtin_fabs(x);
    *odd |= !(a < 1.0e300) || (a < 1.0e-280 && a > 0.0);
    return __builtin_copysign(__builtin_fma(__builtin_fma(-d, q, x), r, q), x);
}

// x / 3, except that an infinity gives a NaN and a negative zero +0.
template <typename T>
__host__ __device__ __forceinline__ T div3(T x)
{
    constexpr T y = (T)(1.0L / 3.0L);
    const T q = x * y;
    if constexpr (sizeof(T) == 8) return __builtin_fma(__builtin_fma(-3.0, q, x), y, q);
    else return __builtin_fmaf(__builtin_fmaf(-3.0f, q, x), y, q);
}

// x / 3 for every x: infinities stay, zeros keep their sign.
template <typename T>
__host__ __device__ __forceinline__ T div3_any(T x)
{
    const T r = div3(x);
    if constexpr (sizeof(T) == 8) return x - x == 0.0 ? __builtin_copysign(r, x) : x;
    else return x - x == 0.0f ? __builtin_copysignf(r, x) : x;
}

} // namespace s2d
