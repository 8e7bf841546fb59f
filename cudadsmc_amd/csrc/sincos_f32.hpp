// sincos_f32.hpp -- sine and cosine of an FP32 angle, for the spin substeps
// of the FP32 form (the rotation angle of each substep).
//
// Cody and Waite's argument reduction (1980): x = k pi/2 + r with pi/2 split
// into three floats (hi + mid + lo, their sum pi/2 to about 1e-22) and the
// products taken with fma, so r is accurate for |k| up to thousands; then the
// Taylor series of sin and cos on |r| <= pi/4 (coefficients 1/n!, truncated
// after r^9 and r^10: remainders below 2e-9 and 2e-10, far under FP32
// rounding), and the quadrant k mod 4.  Beyond kSinCosReduceMax (and for NaN
// or infinity) it falls back to the library's sincosf.  Plain C++ so that the
// same code is tested on the host.
#pragma once

#include <cmath>
#include <cstdint>

#ifndef DSMC_HOST_DEVICE
#if defined(__HIPCC__)
#define DSMC_HOST_DEVICE __host__ __device__
#else
#define DSMC_HOST_DEVICE
#endif
#endif

namespace dsmc {

constexpr float kSinCosReduceMax = 8192.0f;

// For |x| <= kSinCosReduceMax.
DSMC_HOST_DEVICE inline void sincos_reduced(float x, float *sp, float *cp)
{
    // k = the multiple of pi/2 nearest to x: adding 3 2^22 rounds to a whole
    // number and leaves k in the sum's low bits, which saves the conversion
    const float big = x * 0.636619772f + 12582912.0f;
    const float kf = big - 12582912.0f;
    float r = fmaf(-kf, 1.57079637e+00f, x);              // pi/2 = hi
    r = fmaf(-kf, -4.37113883e-08f, r);                   //      + mid
    r = fmaf(-kf, -1.71512451e-15f, r);                   //      + lo
    const float r2 = r * r;
    // sin r = r - r^3/3! + r^5/5! - r^7/7! + r^9/9!
    const float ps = fmaf(r2, fmaf(r2, fmaf(r2, 2.75573192e-06f, -1.98412698e-04f), 8.33333333e-03f),
                          -1.66666667e-01f);
    const float s = fmaf(r * r2, ps, r);
    // cos r = 1 - r^2/2! + r^4/4! - r^6/6! + r^8/8! - r^10/10!
    const float pc = fmaf(r2, fmaf(r2, fmaf(r2, fmaf(r2, -2.75573192e-07f, 2.48015873e-05f), -1.38888889e-03f),
                                   4.16666667e-02f),
                          -0.5f);
    const float c = fmaf(r2, pc, 1.0f);
    // quadrant k mod 4: odd k swaps sine and cosine; the sine changes sign
    // for k = 2, 3 and the cosine for k = 1, 2 (mod 4): bit 1 of k and of
    // k + 1, moved to the sign bit
    const uint32_t q30 = __builtin_bit_cast(uint32_t, big) << 30;
    const uint32_t odd = (uint32_t)((int32_t)(q30 << 1) >> 31);
    const uint32_t us = __builtin_bit_cast(uint32_t, s), uc = __builtin_bit_cast(uint32_t, c);
    const uint32_t d = (us ^ uc) & odd, sv = us ^ d, cv = uc ^ d;
    *sp = __builtin_bit_cast(float, sv ^ (q30 & 0x80000000u));
    *cp = __builtin_bit_cast(float, cv ^ ((q30 + 0x40000000u) & 0x80000000u));
}

DSMC_HOST_DEVICE inline void sincos_f32(float x, float *sp, float *cp)
{
    if (fabsf(x) <= kSinCosReduceMax) sincos_reduced(x, sp, cp);
    else sincosf(x, sp, cp);
}

}  // namespace dsmc
