// Correctly rounded FP64 division by a divisor that many quotients share.
//
// The reference-order kernels divide by metrics, time steps and constants
// that are the same for every point of a grid; the hardware's IEEE sequence
// (two scalings, a quarter-rate reciprocal, seven multiply-adds, a fix-up: 14
// issue slots) starts from nothing each time.  With y = RN(1/b) and the rest
// z = 1/b - y at hand, q0 = a y + a z is within an ulp of a / b, its remainder
// r = a - b q0 is exact, and RN(q0 + r y) is the correctly rounded quotient
// (P. Markstein, IBM J. Res. Dev. 34, 1990): 4 multiply-adds, and the
// hardware's fix-up for zeros (their sign), infinities and NaN.  The one
// condition is that nothing overflows or underflows on the way, so callers
// look at the numerators' exponents (ExpCheck) and take IEEE divisions for the
// waves that hold one out of range.
#pragma once

#include <cmath>

#include <hip/hip_runtime.h>

namespace ibt {

struct Den {
    double b, y, z;
};

// b > 0
__host__ __device__ inline Den make_den(double b)
{
    const double y = 1.0 / b;
    return Den{b, y, fma(-b, y, 1.0) * y};
}

__device__ __forceinline__ double quot(double a, const Den &d)
{
    const double q0 = __builtin_fma(a, d.y, a * d.z);
    const double q = __builtin_fma(__builtin_fma(-d.b, q0, a), d.y, q0);
    return __builtin_amdgcn_div_fixup(q, d.b, a);
}

// a[k] = a[k] / d, correctly rounded; ieee (uniform over the wave): by IEEE
// divisions
template <int N>
__device__ __forceinline__ void quots(double (&a)[N], const Den &d, bool ieee)
{
    if (__builtin_expect(ieee, 0)) {
#pragma unroll
        for (int k = 0; k < N; ++k) a[k] = a[k] / d.b;
    } else {
#pragma unroll
        for (int k = 0; k < N; ++k) a[k] = quot(a[k], d);
    }
}
// a[k] = a[k] / d / d
template <int N>
__device__ __forceinline__ void quots2(double (&a)[N], const Den &d, bool ieee)
{
    if (__builtin_expect(ieee, 0)) {
#pragma unroll
        for (int k = 0; k < N; ++k) a[k] = a[k] / d.b / d.b;
    } else {
#pragma unroll
        for (int k = 0; k < N; ++k) a[k] = quot(quot(a[k], d), d);
    }
}

// Whether numerators lie within 2^-500 .. 2^500 (zeros, infinities and NaN
// count as in range: the fix-up covers them), by the sum of their binary
// exponents' squares: divisors within 2^-120 .. 2^120 and sums of a few such
// numerators (which may cancel by 53 bits) then stay clear of the format's
// limits.  One operation each; a sum past the limit without a number past it
// only costs the wave its IEEE divisions.
struct ExpCheck {
    static constexpr int LIMIT = 500 * 500;
    int sum = 0;
    __device__ __forceinline__ void add(double x)
    {
        const int e = __builtin_amdgcn_frexp_exp(x);
        sum = __mul24(e, e) + sum;
    }
    __device__ __forceinline__ bool any(int limit) const { return __any(sum > limit); }
};

}  // namespace ibt
