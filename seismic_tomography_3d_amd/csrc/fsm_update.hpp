// fsm_update.hpp -- the update of one cell of Accurate_FSM in its two forms:
// as the method's code has it, and the short form the sweeps run in ordinary
// ranges of units.  No HIP header: it also builds for the host, where a test
// compares the two over the whole range that the short form is admitted for.
//
// Both take -ffp-contract=off; min/max follow std::min/std::max operand order
// where a NaN could reach them.
#pragma once

#include <algorithm>

#include "rounded.hpp"

namespace st {

__device__ __forceinline__ float smin(float a, float b) { return (b < a) ? b : a; }
__device__ __forceinline__ float smax(float a, float b) { return (a < b) ? b : a; }

// Geometry and the constants eikonal_equation derives from the spacing
// (accurate_FSM.cpp:632-644), all computed on the host in FP32.
struct FsmGeo {
    int nxx, nyy, nzz;      // padded extent (model + 2)
    long long nB;           // nxx * nyy * nzz
    float dx, dy, dz;
    float dz2i, dx2i, dy2i, dz2dx2, dz2dy2, dx2dy2, dsum;
    float zx, zy, xy;       // dz2i + dx2i, dz2i + dy2i, dx2i + dy2i
    float rzx, rzy, rxy, rdsum;   // correctly rounded reciprocals of those and dsum
    float dmin;             // 0.99 of the least spacing
    float wv, we, wn, wev, wen, wnv;   // weights of the upwind times in the mean of the 3D arms
};

inline FsmGeo fsm_geometry(int nx, int ny, int nz, float dx, float dy, float dz) {
    FsmGeo g;
    g.nxx = nx + 2; g.nyy = ny + 2; g.nzz = nz + 2;
    g.nB = (long long)g.nxx * g.nyy * g.nzz;
    g.dx = dx; g.dy = dy; g.dz = dz;
    g.dz2i = 1.0f / (g.dz * g.dz);
    g.dx2i = 1.0f / (g.dx * g.dx);
    g.dy2i = 1.0f / (g.dy * g.dy);
    g.dz2dx2 = g.dz2i * g.dx2i;
    g.dz2dy2 = g.dz2i * g.dy2i;
    g.dx2dy2 = g.dx2i * g.dy2i;
    g.dsum = g.dz2i + g.dx2i + g.dy2i;
    g.zx = g.dz2i + g.dx2i;
    g.zy = g.dz2i + g.dy2i;
    g.xy = g.dx2i + g.dy2i;
    g.rzx = 1.0f / g.zx;
    g.rzy = 1.0f / g.zy;
    g.rxy = 1.0f / g.xy;
    g.rdsum = 1.0f / g.dsum;
    g.dmin = 0.99f * std::min({g.dx, g.dy, g.dz});
    const float z = g.dz2i / g.dsum, x = g.dx2i / g.dsum, y = g.dy2i / g.dsum;
    g.wv = z - 0.5f * (x + y);
    g.we = x - 0.5f * (z + y);
    g.wn = y - 0.5f * (z + x);
    g.wev = 0.5f * (x + z) - y;
    g.wen = 0.5f * (x + y) - z;
    g.wnv = 0.5f * (z + y) - x;
    return g;
}

// Whether the FAST update's ranges hold: spacings and their squares far from
// under- and overflow and within a factor of 1000 of each other (the slack of
// its 2D bound); root arguments 0 or of 2^-101 and more (an argument is (s / d)^2
// times at least 8 less another number, and where the two cancel, a multiple of
// 2^-25 of it); no time above the 1e6 of unreached cells, not even the seeds'.
inline bool fsm_fast(const FsmGeo &g, float slow_min, float slow_max) {
    const float lo = std::min({g.dx, g.dy, g.dz}), hi = std::max({g.dx, g.dy, g.dz});
    return lo > 1e-6f && hi < 1e6f && hi < 1000.0f * lo && slow_min > 1e-9f &&
           slow_min > 1e-11f * hi && slow_max < 1e4f && slow_max * hi < 1e5f;
}

// Upwind travel times of a cell (v along z, e along x, n along y and their
// combinations) and the slownesses of its operators: the least of the four
// voxels around each upwind edge (sv, se, sn), of the two voxels on each
// upwind face (sve, svn, sen) and the upwind voxel (s).
struct FsmIn {
    float tv, te, tn, tev, ten, tnv, tnve;
    float sv, se, sn, sve, svn, sen, s;
};

// Least of slownesses, which are never negative nor NaN: their bit patterns order
// as integers, and an integer minimum needs no quieting of its operands.
__device__ __forceinline__ float pmin(float a, float b) {
    return __int_as_float(min(__float_as_int(a), __float_as_int(b)));
}
// The same of times, which can be negative (beside a source the 3D operator gives
// such times where spacings and slownesses differ much).  A NaN is left out.  The
// instructions by name: the compiler would first quiet every time that was loaded.
__device__ __forceinline__ float tmin(float a, float b) {
#if defined(__AMDGCN__)
    float r;
    asm("v_min_f32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
#else
    return __builtin_fminf(a, b);
#endif
}
__device__ __forceinline__ float tmin3(float a, float b, float c) {
#if defined(__AMDGCN__)
    float r;
    asm("v_min3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
    return r;
#else
    return __builtin_fminf(a, __builtin_fminf(b, c));
#endif
}
__device__ __forceinline__ float tmax3(float a, float b, float c) {
#if defined(__AMDGCN__)
    float r;
    asm("v_max3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
    return r;
#else
    return __builtin_fmaxf(a, __builtin_fmaxf(b, c));
#endif
}
// the largest magnitude
__device__ __forceinline__ float tmag3(float a, float b, float c) {
#if defined(__AMDGCN__)
    float r;
    asm("v_max3_f32 %0, |%1|, |%2|, |%3|" : "=v"(r) : "v"(a), "v"(b), "v"(c));
    return r;
#else
    return tmax3(__builtin_fabsf(a), __builtin_fabsf(b), __builtin_fabsf(c));
#endif
}

// The arms of the 3D operator.  Products with 0.5 are exact, so the fused
// forms round as the separate ones do.
__device__ __forceinline__ void fsm_arms(const FsmIn &c, float &ta, float &tb, float &tc) {
    auto half = [](float a, float b) { return __builtin_fmaf(0.5f, a, b); };
    ta = half(c.tev, half(-c.tv, half(c.ten, half(-c.tn, c.te)))) - c.tnv + c.tnve;
    tb = half(c.tev, half(-c.te, half(c.tnv, half(-c.tn, c.tv)))) - c.ten + c.tnve;
    tc = half(c.tnv, half(-c.tv, half(c.ten, half(-c.te, c.tn)))) - c.tev + c.tnve;
}

// The update of one cell, accurate_FSM.cpp:159-265 (inner_sweep), as written
// there.
__device__ float fsm_update_any(float T, const FsmIn &c, const FsmGeo &g) {
    const float dx = g.dx, dy = g.dy, dz = g.dz;
    const float tv = c.tv, te = c.te, tn = c.tn;
    // 1D operators: upwind time plus spacing times the least slowness
    const float t1D = smin(tv + dz * c.sv, smin(te + dx * c.se, tn + dy * c.sn));
    // 2D four-point operators in the xz, yz and xy planes
    float t2D1 = 1e6f, t2D2 = 1e6f, t2D3 = 1e6f;
    if ((tv < te + dx * c.sve) && (te < tv + dz * c.sve)) {
        const float ta = c.tev + te - tv;
        const float tb = c.tev - te + tv;
        t2D1 = ((tb * g.dz2i + ta * g.dx2i) +
                sqrtf(4.0f * c.sve * c.sve * g.zx - g.dz2dx2 * (ta - tb) * (ta - tb))) / g.zx;
    }
    if ((tv < tn + dy * c.svn) && (tn < tv + dz * c.svn)) {
        const float ta = tv - tn + c.tnv;
        const float tb = tn - tv + c.tnv;
        t2D2 = ((ta * g.dz2i + tb * g.dy2i) +
                sqrtf(4.0f * c.svn * c.svn * g.zy - g.dz2dy2 * (ta - tb) * (ta - tb))) / g.zy;
    }
    if ((te < tn + dy * c.sen) && (tn < te + dx * c.sen)) {
        const float ta = te - tn + c.ten;
        const float tb = tn - te + c.ten;
        t2D3 = ((ta * g.dx2i + tb * g.dy2i) +
                sqrtf(4.0f * c.sen * c.sen * g.xy - g.dx2dy2 * (ta - tb) * (ta - tb))) / g.xy;
    }
    const float t2D = smin(t2D1, smin(t2D2, t2D3));
    // 3D operator on the upwind octant
    float t3D = 1e6f;
    if (smin(t1D, t2D) > smax(tv, smax(te, tn))) {
        float ta, tb, tc;
        fsm_arms(c, ta, tb, tc);
        const float t2 = 9.0f * c.s * c.s * g.dsum;
        const float t3 = g.dz2dx2 * (ta - tb) * (ta - tb) + g.dz2dy2 * (tb - tc) * (tb - tc) +
                         g.dx2dy2 * (ta - tc) * (ta - tc);
        if (t2 >= t3) {
            const float t1 = tb * g.dz2i + ta * g.dx2i + tc * g.dy2i;
            t3D = (t1 + sqrtf(t2 - t3)) / g.dsum;
        }
    }
    return smin(T, smin(t1D, smin(t2D, t3D)));
}

// The same update, bit for bit, in the ranges fsm_fast checks: square roots
// and quotients by the spacing constants in their short correctly rounded
// forms, and with PRUNE operators that cannot lower the cell left out.
//
// The root argument of a 2D operator can be negative: where its diagonal time
// is still 1e6, sums with it round to a sixteenth of a second, and a difference
// of axis times within the admitted range can come out several times as large
// (25 m cells at 1,500 m/s beside the source already); so can times far from
// the source across spacings that differ much.  The code's result is then a
// NaN, and std::min keeps its first argument if either is one: the operators
// are combined here in the code's order with the code's operands, so that a NaN
// takes the same others with it.  The 3D operator comes last: with a NaN before it
// it is dropped, and the 1e6 it stands at where it does not apply offers nothing.
//
// PRUNE, with lim the least of the cell's time and the 1D operators:
// * t3D is at least the weighted mean of its arms (its root is not negative
//   and rounding is monotone), a linear form of the seven upwind times; above
//   lim by more than rounding (2^-17 of lim and the times) it is ruled out;
// * a 2D operator is at least its diagonal time plus the slowness times the
//   lesser spacing (its root term is concave in the difference of the two
//   axis times, with the spacings' values at the ends of the admitted range);
//   with 1 % of that term and the same share for rounding, at or above lim it
//   is ruled out -- unless the 3D operator is in play, whose condition reads
//   the 2D times.
// A NaN left out offers nothing but may have kept others from lowering the
// cell, so with PRUNE cells the general form lowers are lowered, others may be.
// In the full sweeps a cell's front mostly does not come from the sweep's
// octant, and in their test the operators fall away for whole waves: branches
// are wave-uniform (any lane needs the operator), the lanes that do not are
// masked by selects.  A walk's lanes are cells that change, where some lane
// needs each operator at nearly every step: without the tests a lone shot's
// launch takes 16 us instead of 19, 64 shots 25.5 ms instead of 27.5.
// big, with PRUNE: at least the largest magnitude of the upwind times.
template <bool PRUNE>
__device__ __forceinline__ float fsm_update_fast(float T, const FsmIn &c, bool on,
                                                 const FsmGeo &g, float big = 0.0f) {
    const float dx = g.dx, dy = g.dy, dz = g.dz;
    const float tv = c.tv, te = c.te, tn = c.tn;
    const float t1D = tmin3(tv + dz * c.sv, te + dx * c.se, tn + dy * c.sn);
    const float latest = tmax3(tv, te, tn);
    const float lim = tmin(T, t1D);
    bool try3 = true, pxz = true, pyz = true, pxy = true;
    if (PRUNE) {
        float l3 = __builtin_fmaf(g.wv, tv, c.tnve);
        l3 = __builtin_fmaf(g.we, te, l3);
        l3 = __builtin_fmaf(g.wn, tn, l3);
        l3 = __builtin_fmaf(g.wev, c.tev, l3);
        l3 = __builtin_fmaf(g.wen, c.ten, l3);
        l3 = __builtin_fmaf(g.wnv, c.tnv, l3);
        const float far = __builtin_fmaf(big + __builtin_fabsf(lim), 7.6293945e-6f, lim);
        try3 = on & (t1D > latest) & (l3 < far);
        pxz = try3 | (on & (__builtin_fmaf(c.sve, g.dmin, c.tev) < far));
        pyz = try3 | (on & (__builtin_fmaf(c.svn, g.dmin, c.tnv) < far));
        pxy = try3 | (on & (__builtin_fmaf(c.sen, g.dmin, c.ten) < far));
    }
    float xz = 1e6f, yz = 1e6f, xy = 1e6f;
    if (!PRUNE || __any(pxz)) {
        const bool ok = pxz & (tv < te + dx * c.sve) & (te < tv + dz * c.sve);
        const float ta = c.tev + te - tv;
        const float tb = c.tev - te + tv;
        const float q = 4.0f * c.sve * c.sve * g.zx - g.dz2dx2 * (ta - tb) * (ta - tb);
        const float t = div_rn((tb * g.dz2i + ta * g.dx2i) + sqrt_rn(q), g.zx, g.rzx);
        xz = ok ? t : xz;
    }
    if (!PRUNE || __any(pyz)) {
        const bool ok = pyz & (tv < tn + dy * c.svn) & (tn < tv + dz * c.svn);
        const float ta = tv - tn + c.tnv;
        const float tb = tn - tv + c.tnv;
        const float q = 4.0f * c.svn * c.svn * g.zy - g.dz2dy2 * (ta - tb) * (ta - tb);
        const float t = div_rn((ta * g.dz2i + tb * g.dy2i) + sqrt_rn(q), g.zy, g.rzy);
        yz = ok ? t : yz;
    }
    if (!PRUNE || __any(pxy)) {
        const bool ok = pxy & (te < tn + dy * c.sen) & (tn < te + dx * c.sen);
        const float ta = te - tn + c.ten;
        const float tb = tn - te + c.ten;
        const float q = 4.0f * c.sen * c.sen * g.xy - g.dx2dy2 * (ta - tb) * (ta - tb);
        const float t = div_rn((ta * g.dx2i + tb * g.dy2i) + sqrt_rn(q), g.xy, g.rxy);
        xy = ok ? t : xy;
    }
    // (with PRUNE a NaN of the xz plane, with which the cell is not lowered, is
    // left out)
    const float t2D = PRUNE ? tmin(xz, smin(yz, xy)) : smin(xz, smin(yz, xy));
    const bool use3 = try3 & (t1D > latest) & (t2D > latest);   // not with a NaN
    const float res = PRUNE ? tmin(lim, t2D) : smin(lim, t2D);
    if (!PRUNE || __any(use3)) {
        float ta, tb, tc;
        fsm_arms(c, ta, tb, tc);
        const float t2 = 9.0f * c.s * c.s * g.dsum;
        const float t3 = g.dz2dx2 * (ta - tb) * (ta - tb) + g.dz2dy2 * (tb - tc) * (tb - tc) +
                         g.dx2dy2 * (ta - tc) * (ta - tc);
        const float t1 = tb * g.dz2i + ta * g.dx2i + tc * g.dy2i;
        const float t = div_rn(t1 + sqrt_rn(t2 - t3), g.dsum, g.rdsum);
        return (use3 & (t2 >= t3) & (t < res)) ? t : res;
    }
    return res;
}

}  // namespace st
