// The two forms of Accurate_FSM's cell update, built for the host: the short
// form against the form of the method's code.
//
//   fsm_update_host walk|test|roots <draws of units> <neighbourhoods per units> <seed>
//
// Units are drawn over the whole range that the short form is admitted for
// (with 0 draws: a list of ordinary ones).  For each set of units,
// neighbourhoods of the kinds the sweeps meet: partly unreached ones (1e6),
// passing fronts at a distance of up to 10^5 cells, times at the edges of the
// operators' ranges to the last bit, and arbitrary ones, negative among them.
// walk: the form of the blocks' walk must equal the general one in every bit;
// test: the form with operators left out must lower every cell the general one
// lowers; roots: as walk, with units of the least slowness to spacing and one
// time of each neighbourhood moved to where the argument of the 3D operator's
// root is a few units of its last place.  Prints what differs and the counts;
// fails if any does.
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <random>
#include <vector>

#define __device__
#define __forceinline__ inline
#define __any(x) (x)
// one lane's part of v_rsq_f32, correctly rounded; negative numbers give a NaN
static inline float host_rsq(float x) { return (float)(1.0 / std::sqrt((double)x)); }
#define __builtin_amdgcn_rsqf(x) host_rsq(x)
static inline int __float_as_int(float f) { int i; std::memcpy(&i, &f, 4); return i; }
static inline float __int_as_float(int i) { float f; std::memcpy(&f, &i, 4); return f; }
using std::max;
using std::min;
#include "fsm_update.hpp"

using namespace st;

namespace {

std::mt19937_64 rng;
double uni(double a, double b) { return std::uniform_real_distribution<double>(a, b)(rng); }
double logu(double a, double b) { return std::exp(uni(std::log(a), std::log(b))); }
int pick(int n) { return (int)(rng() % (unsigned)n); }
float ulps(float v, int n) {   // n units up or down
    for (; n > 0; n--) v = std::nextafterf(v, 1e30f);
    for (; n < 0; n++) v = std::nextafterf(v, 0.0f);
    return v;
}

struct Units {
    float dx, dy, dz, lo, hi;   // spacings, least and largest slowness
};

FsmIn neighbourhood(const Units &u, float &T) {
    FsmIn c;
    const float s = (float)logu(u.lo, u.hi), w = pick(3) ? s : (float)logu(u.lo, u.hi);
    c.s = s;
    c.sve = pick(3) ? s : std::min(s, w);
    c.svn = pick(3) ? s : std::min(s, w);
    c.sen = pick(3) ? s : std::min(s, w);
    c.sv = std::min({c.sve, c.svn, w});
    c.se = std::min({c.sve, c.sen, w});
    c.sn = std::min({c.svn, c.sen, w});
    // a front through the cell's upwind octant, at a distance
    double d[3] = {uni(-1, 1), uni(-1, 1), uni(-1, 1)};
    if (pick(4) == 0) d[pick(3)] = 0;
    if (pick(4) == 0) d[pick(3)] *= 1e-3;
    const double n = std::sqrt(d[0] * d[0] + d[1] * d[1] + d[2] * d[2]) + 1e-30;
    const double step = std::min({u.dx, u.dy, u.dz}) * s;
    const double far = pick(4) ? logu(1, 1e5) * step : uni(0, 4) * step;
    const double gz = -d[0] / n * s * u.dz, gx = -d[1] / n * s * u.dx, gy = -d[2] / n * s * u.dy;
    auto at = [&](int z, int x, int y) {
        return (float)std::max(0.0, far + z * gz + x * gx + y * gy);
    };
    c.tv = at(1, 0, 0);
    c.te = at(0, 1, 0);
    c.tn = at(0, 0, 1);
    c.tev = at(1, 1, 0);
    c.tnv = at(1, 0, 1);
    c.ten = at(0, 1, 1);
    c.tnve = at(1, 1, 1);
    T = at(0, 0, 0);
    float *t[7] = {&c.tv, &c.te, &c.tn, &c.tev, &c.tnv, &c.ten, &c.tnve};
    switch (pick(5)) {
    case 0:   // partly unreached
        for (float *p : t)
            if (pick(3) == 0) *p = 1e6f;
        break;
    case 1:   // the edges of the 2D operators' ranges
        c.te = pick(2) ? ulps(c.tv + u.dz * c.sve, pick(9) - 4) : c.te;
        c.tv = pick(2) ? ulps(c.te + u.dx * c.sve, pick(9) - 4) : c.tv;
        c.tn = pick(2) ? ulps(c.tv + u.dz * c.svn, pick(9) - 4)
                       : ulps(c.te + u.dx * c.sen, pick(9) - 4);
        break;
    case 2: {   // rough times, some negative
        const double least = pick(2) ? 0.0 : -1e30, by = logu(1e-4, 10);
        for (float *p : t) *p = (float)std::max(least, *p + uni(-1, 1) * step * by);
        if (pick(2)) T = (float)std::max(least, T + uni(-1, 1) * step * by);
        break;
    }
    case 3:   // as they come, a few units off
        for (float *p : t) *p = ulps(*p, pick(7) - 3);
        break;
    default: break;
    }
    switch (pick(4)) {   // the cell's own time: unreached, or near the arrival
    case 0: T = 1e6f; break;
    case 1: T = fsm_update_any(1e6f, c, fsm_geometry(2, 2, 2, u.dx, u.dy, u.dz));
            T = ulps(T, pick(7) - 3); break;
    case 2: T = (float)(T + uni(-1, 1) * step * logu(1e-5, 10)); break;
    default: break;
    }
    for (float *p : t) *p = std::min(*p, 1e6f);   // no time is above unreached ones
    T = std::min(T, 1e6f);
    return c;
}

float test_update(float T, const FsmIn &c, const FsmGeo &g) {
    const float big = tmag3(tmag3(c.tv, c.te, c.tn), tmag3(c.tev, c.ten, c.tnv), c.tnve);
    return fsm_update_fast<true>(T, c, true, g, big);
}

// t2 - t3 of the 3D operator, as the update has them
float root_argument(const FsmIn &c, const FsmGeo &g) {
    float ta, tb, tc;
    fsm_arms(c, ta, tb, tc);
    const float t2 = 9.0f * c.s * c.s * g.dsum;
    const float t3 = g.dz2dx2 * (ta - tb) * (ta - tb) + g.dz2dy2 * (tb - tc) * (tb - tc) +
                     g.dx2dy2 * (ta - tc) * (ta - tc);
    return t2 - t3;
}

// Moves tnv, which two arms hold with different signs, until the argument
// passes zero, and leaves it within three units of there.
void cancel_root(FsmIn &c, const FsmGeo &g) {
    if (!(root_argument(c, g) > 0)) return;
    FsmIn out = c;
    const float step = c.s * std::min({g.dx, g.dy, g.dz});
    for (int k = 0; k < 8 && root_argument(out, g) >= 0; k++) out.tnv += step;
    if (root_argument(out, g) >= 0) return;
    int a = __float_as_int(c.tnv), b = __float_as_int(out.tnv);
    while (b - a > 1) {
        out.tnv = __int_as_float(a + (b - a) / 2);
        (root_argument(out, g) >= 0 ? a : b) = a + (b - a) / 2;
    }
    c.tnv = __int_as_float(std::max(0, a - pick(4)));
}

}  // namespace

int main(int argc, char **argv) {
    if (argc != 5) return 2;
    const bool roots = !std::strcmp(argv[1], "roots"), walk = roots || !std::strcmp(argv[1], "walk");
    const int draws = std::atoi(argv[2]), per = std::atoi(argv[3]);
    rng.seed((unsigned)std::atoi(argv[4]));
    std::vector<Units> units;
    if (draws == 0)
        for (float h : {5.0f, 12.5f, 25.0f, 50.0f, 100.0f, 130.0f, 200.0f, 250.0f, 500.0f, 1000.0f, 0.1f})
            for (float v : {1500.0f, 3000.0f, 6000.0f, 12500.0f, 20000.0f, 5.0f}) {
                units.push_back({h, h, h, 1 / v, 1 / v});
                units.push_back({h, 0.8f * h, 0.5f * h, 0.25f / v, 1 / v});
            }
    while ((int)units.size() < draws) {
        Units u;
        const double mid = logu(roots ? 1e3 : 1e-6, 1e6), ratio = logu(1, roots ? 2 : 1000);
        float *d[3] = {&u.dx, &u.dy, &u.dz};
        for (float *p : d) *p = (float)(mid * std::pow(ratio, uni(0, 1)));
        u.lo = (float)logu(1e-9, 1e4);
        if (roots) u.lo = (float)(mid * logu(1e-15, 1e-10));
        u.hi = roots || pick(2) ? u.lo : (float)logu(u.lo, 1e4);
        if (fsm_fast(fsm_geometry(2, 2, 2, u.dx, u.dy, u.dz), u.lo, u.hi)) units.push_back(u);
    }
    long all = 0, bad = 0;
    for (const Units &u : units) {
        const FsmGeo g = fsm_geometry(2, 2, 2, u.dx, u.dy, u.dz);
        for (int k = 0; k < per; k++) {
            float T;
            FsmIn c = neighbourhood(u, T);
            if (roots) cancel_root(c, g);
            const float a = fsm_update_any(T, c, g), b = walk ? fsm_update_fast<false>(T, c, true, g)
                                                             : test_update(T, c, g);
            all++;
            if (walk ? std::memcmp(&a, &b, 4) == 0 : a == T || b != T) continue;
            if (bad++ < 20)
                std::printf("d %g %g %g s %g %g %g %g: T %.9g general %.9g short %.9g, times %.9g %.9g "
                            "%.9g %.9g %.9g %.9g %.9g\n", u.dx, u.dy, u.dz, c.s, c.sve, c.svn, c.sen, T,
                            a, b, c.tv, c.te, c.tn, c.tev, c.ten, c.tnv, c.tnve);
        }
    }
    std::printf("%zu sets of units, %ld updates, %ld wrong\n", units.size(), all, bad);
    return bad ? 1 : 0;
}
