// fp64_ops.h -- FP64 square root and division without the steps that only numbers
// at the ends of the exponent range need.
//
// The compiler's FP64 division and square root scale their operands, refine a
// hardware estimate (v_rcp_f64, v_rsq_f64) with fused multiply-adds, correct the
// result by its residual, and undo the scaling: 11 and about 18 instructions.  The
// forms here are the refinement alone (Newton's steps for 1/d, then q = n y
// corrected by (n - d q) y; Goldschmidt's steps for sqrt): the same operations on
// the same numbers wherever the scaling would have been by one, hence the same
// correctly rounded results.  Quotients with one denominator share its refined
// reciprocal, so each further one costs three instructions.
//
// Quotients hold for finite arguments with 2^-900 < |n|, |d|, |n/d| < 2^900, where all
// residuals are normal numbers, or n = 0 (whose sign is not kept); fp_div_any's n may
// also be infinite or a NaN.  Square roots hold for x = 0, 2^-900 < x < 2^900, +inf and
// NaN.  On the host they are the plain operations.
#pragma once
#include <hip/hip_runtime.h>
#include <math.h>

// refined 1/d for fp_quot
__host__ __device__ __forceinline__ double fp_recip(double d)
{
#ifdef __HIP_DEVICE_COMPILE__
    double y = __builtin_amdgcn_rcp(d);
    y = __builtin_fma(y, __builtin_fma(-d, y, 1.0), y);
    return __builtin_fma(y, __builtin_fma(-d, y, 1.0), y);
#else
    return 1.0 / d;
#endif
}

// n / d with y = fp_recip(d)
__host__ __device__ __forceinline__ double fp_quot(double n, double d, double y)
{
#ifdef __HIP_DEVICE_COMPILE__
    const double q = n * y;
    return __builtin_fma(__builtin_fma(-d, q, n), y, q);
#else
    (void)y;
    return n / d;
#endif
}

__host__ __device__ __forceinline__ double fp_div(double n, double d) { return fp_quot(n, d, fp_recip(d)); }

// n / d where n may be infinite or a NaN: the division's last step, one instruction,
// which replaces the quotient in these cases
__host__ __device__ __forceinline__ double fp_div_any(double n, double d)
{
#ifdef __HIP_DEVICE_COMPILE__
    return __builtin_amdgcn_div_fixup(fp_div(n, d), d, n);
#else
    return n / d;
#endif
}

// the smaller and the larger of two numbers, the other one where one is a NaN, by one
// instruction (fmin and fmax put canonicalising ones before it)
__host__ __device__ __forceinline__ double fp_min(double a, double b)
{
#ifdef __HIP_DEVICE_COMPILE__
    double r;
    asm("v_min_f64 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
#else
    return fmin(a, b);
#endif
}
__host__ __device__ __forceinline__ double fp_max(double a, double b)
{
#ifdef __HIP_DEVICE_COMPILE__
    double r;
    asm("v_max_f64 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
#else
    return fmax(a, b);
#endif
}

// sqrt(x), x >= 0
__host__ __device__ __forceinline__ double fp_sqrt(double x)
{
#ifdef __HIP_DEVICE_COMPILE__
    const double r = __builtin_amdgcn_rsq(x);
    double g = x * r, h = 0.5 * r;
    const double e = __builtin_fma(-h, g, 0.5);
    g = __builtin_fma(g, e, g);
    h = __builtin_fma(h, e, h);
    g = __builtin_fma(__builtin_fma(-g, g, x), h, g);
    g = __builtin_fma(__builtin_fma(-g, g, x), h, g);
    return __builtin_amdgcn_class(x, 0x260) ? x : g;   // +-0 and +inf, where x * rsq(x) is a NaN
#else
    return sqrt(x);
#endif
}
