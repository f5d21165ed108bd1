// rounded.hpp -- correctly rounded quotients and square roots in their short
// forms, for the kernels whose results have to keep every bit.  No HIP header:
// the arithmetic also builds for the host, where a test runs it.
#pragma once

namespace st {

// RN(a / b) for b > 0 from y = RN(1 / b) without a division: q = a y, one
// fma residual correction makes q faithful, and Markstein's final step (the
// residual a - b q is exact by fma, q + r y rounded once) returns the
// correctly rounded quotient.  Where intermediate results could leave the
// normal range (|a / b| < 2^-100), the quotient's integer part, the only use
// here, is 0 either way.  Checked against IEEE division on every float
// |a| in [2^-20, 2^20) for 16 spacings from 1e-3 to 9999: all bits equal.
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
