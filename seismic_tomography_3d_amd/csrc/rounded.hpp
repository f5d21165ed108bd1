// rounded.hpp -- correctly rounded quotients and square roots in their short
// forms, for the kernels whose results have to keep every bit.  No HIP header:
// the arithmetic also builds for the host, where a test runs it.
#pragma once

namespace st {

// RN(a / b) for b > 0 from y = RN(1 / b) without a division: q = a y, one
// fma residual correction makes q faithful, and Markstein's final step (the
// residual a - b q is exact by fma, q + r y rounded once) returns the
// correctly rounded quotient.  The residual has to be a normal number or 0,
// which holds for a = 0 and for |a| >= 2^-101 with |a / b| >= 2^-125; Accurate_FSM
// and Podvin see to it by the ranges of units they take their short forms for
// (fsm_fast; h s above 1e-9).  The ray tracer uses the integer part only, which
// is 0 below that range either way.  Equal to IEEE division in every bit on
// 1.2e9 quotients of 1,200 divisors from 2^-40 to 2^41 (sqrt 2, odd ones and ones
// next to powers of two among them) over that range, and on every float |a| in
// [2^-20, 2^20) for 16 spacings from 1e-3 to 9999.
__device__ __forceinline__ float div_rn(float a, float b, float y) {
    float q = a * y;
    float r = __builtin_fmaf(-q, b, a);
    q = __builtin_fmaf(r, y, q);
    r = __builtin_fmaf(-q, b, a);
    return __builtin_fmaf(r, y, q);
}

// Correctly rounded square root of x = 0 or x >= 2^-101 in six instructions:
// with r = rsq(x) to one ulp, x r is within 1.5 ulp of the root, its residual
// x - s^2 is exact by fma and half of r turns it into the correction, rounded
// once.  Equal to sqrtf in every bit for every such float (checked on all
// 2^31 of them; below 2^-102 the residual is no longer a normal number).  The
// 2^-126 keeps r finite at 0, is lost in rounding from 2^-101 on, and leaves a
// negative x negative: a NaN, as sqrtf gives (from -2^-125 down).
__device__ __forceinline__ float sqrt_rn(float x) {
    const float r = __builtin_amdgcn_rsqf(x + 1.17549435e-38f);
    const float s = x * r;
    return __builtin_fmaf(__builtin_fmaf(-s, s, x), 0.5f * r, s);
}

}  // namespace st
