// sk_math.h -- base-2 scalar helpers shared by the float32 Sinkhorn kernels.
#pragma once

#include <hip/hip_runtime.h>

namespace tmamd {

constexpr double kLog2eD = 1.4426950408889634074;
constexpr double kLn2D = 0.69314718055994530942;

// log2 of a float32 s > 0 in float64: s = m * 2^e with m in [sqrt(1/2),
// sqrt(2)), e exact and the native log on m only.  The native log is
// accurate near 1 but its error grows with |log2 s| (up to one float32 ulp
// of the result, biased low), and a bias common to every row or column is
// what the balanced potentials' neutral mode accumulates step after step.
// +inf, 0 and NaN go to the native log directly.
__device__ __forceinline__ double log2_split(float s) {
    if (!(s > 0.f) || !__builtin_isfinite(s))
        return (double)__builtin_amdgcn_logf(s);
    int e = __builtin_amdgcn_frexp_expf(s);
    float m = __builtin_amdgcn_frexp_mantf(s);  // [0.5, 1)
    if (m < 0.70710678f) {
        m *= 2.f;
        e -= 1;
    }
    return (double)e + (double)__builtin_amdgcn_logf(m);
}

// log2 of a float64 sum s > 0: log2_split of its float32 rounding plus the
// first-order term of the rounding (relative <= 2^-24, so the second-order
// term is below 2^-49).
__device__ __forceinline__ double log2_of_sum(double s) {
    const float h = (float)s;
    const float r = (float)(s - (double)h);  // exact: |r| <= ulp(h) / 2
    return log2_split(h) + (double)(r * __builtin_amdgcn_rcpf(h) * 1.4426950408889634f);
}

// 2^t of a float64 t as a float32, to about 1e-7 relative: 2^round(t)
// exactly (ldexp) times the native 2^f of the float32 fraction f, |f| <= 1/2,
// with f's own rounding r restored to first order (2^(f + r) = 2^f (1 + r ln 2)).
__device__ __forceinline__ float pow2_of(double t) {
    const double ti = fmin(fmax(rint(t), -300.0), 300.0);
    const double fd = t - ti;
    const float f = (float)fd;
    const float r = (float)(fd - (double)f);
    const float e = __builtin_amdgcn_exp2f(f);
    return ldexpf(fmaf(e, r * 0.6931471805599453f, e), (int)ti);
}

} // namespace tmamd
