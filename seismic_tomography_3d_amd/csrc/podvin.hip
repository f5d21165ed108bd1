// podvin.hip -- Podvin & Lecomte (1991) first arrivals on the device
// (src/eikonal/classic/classic.cpp, the reference's eikonal_type 0),
// bit-identical to the reference's CPU code.
//
// The reference iterates a Jacobi step nItEikonal times (classic.cpp:284-
// 1833): every active cell takes the lowest of its old time and the arrivals
// of the 1D head-wave, edge and corner diffraction, 2D and 3D Huygens
// operators computed from the old times; a cell that did not improve turns
// inactive, and the 26 neighbours of every cell that did become the next
// active set.
//
// Here a step is one launch over the 8^3 tiles that hold an active cell, for
// all shots of the batch.  A workgroup stages a tile with its halo in LDS,
// finds the active cells, evaluates them 64 to a wave and writes the tile to
// the other of two time volumes (a step reads one, writes the other).  A
// stored time carries "changed in this step" in its sign (times are not
// negative), so the next step sees both in one load: a cell is active when
// one of its 26 neighbours has the sign set.  A tile that changed, or still
// holds signs, is listed for the next step, with the neighbours its changed
// cells touch; a tile that is not listed is the same, without signs, in both
// volumes.  Nothing is read back to the host between steps.
//
// Exactness: a step reads only old times, so cells and operators may be taken
// in any order, and operators that cannot lower the cell are left out:
// * one none of whose times changed in the last step gave the same arrival
//   when they last changed (the cell was active then), and the cell has kept
//   the minimum (from the start on, where unreached times offer nothing: no
//   time is above them but that of a source that starts no front);
// * arrivals of the form X + root are not below X, rounding being monotone;
//   N + P - M + root with M <= N, P is not below max(N, P) but for rounding.
// The arithmetic of the others is the CPU code's, in FP32 (this file is built
// with -ffp-contract=off; products with 2 are exact, so fma(2, a, b) rounds as
// 2 a + b does), so the times are the same bit for bit.
//
// The 3D operators are evaluated by (cell, face of an octant) and the 2D ones
// by (cell, quarter plane): a cell's lane tests which of its 24 faces and 12
// quarter planes could lower it (few: their times have to lie in the order the
// operator is for, before the cell's), lists those in LDS, and the lanes of the
// workgroup take the listed ones.  Evaluating all operators per cell cost 2.4
// times the instructions, half the lanes masked.
//
// What bounds it: vector issue (21 of 37 ms for 8 shots of 201 x 201 x 101) with
// the barriers between a tile's phases; for a lone shot the latency of a step,
// 12 to 18 us.  Measured: 8 shots of 201 x 201 x 101 175 -> 37 ms, one of 101 x
// 101 x 51 6.7 -> 2.05 ms, against a list of cells selected from stamps of all
// cells every step.
//
// Layout: per shot two padded volumes, z fastest, whose extents are a multiple
// of 8 plus a cell on each side; cells outside the model stay at 1e6.
#include <cmath>

#include "st_common.hpp"

namespace st {

void launch_picks_padvol(hipStream_t st, const float *T, long long vol, int nxx, int nzz,
                         int nshot, const float *rcv, int nr, float *out, int nx, int ny, int nz,
                         float dx, float dy, float dz);

namespace {

constexpr int kTile = 8;
constexpr int kSeg = 16;          // append segments of the tile lists
constexpr int kCntStride = 32;    // one 128-byte line per segment counter

// Padded extents and tiles of a model.
struct PodGeo {
    int nx, ny, nz;
    int px, py, pz;        // volume extents: 8 tiles + 2
    int ntx, nty, ntz;
    int nt;                // tiles per shot
    long long vol;         // cells per volume
};

PodGeo pod_geo(const st_ctx *ctx) {
    PodGeo g;
    g.nx = ctx->nx; g.ny = ctx->ny; g.nz = ctx->nz;
    g.ntx = (g.nx + kTile - 1) / kTile;
    g.nty = (g.ny + kTile - 1) / kTile;
    g.ntz = (g.nz + kTile - 1) / kTile;
    g.px = g.ntx * kTile + 2; g.py = g.nty * kTile + 2; g.pz = g.ntz * kTile + 2;
    g.nt = g.ntx * g.nty * g.ntz;
    g.vol = (long long)g.px * g.py * g.pz;
    return g;
}

struct PodArgs {
    const float *S;        // slowness, model extent, z fastest
    float *T;              // [shot][2][vol]
    int *stamp;            // [shot][nt]: last step a tile was listed for
    int *list0, *list1;    // tile lists by step parity, kSeg segments of cap
    long long cap;
    int *cnt;              // segment lengths, three rotating slots
    const int *nit;        // steps per shot
    PodGeo g;
    float h, hh, hr2, hr3;       // h, h h, h sqrt(2), h sqrt(3)
    float sqrt2, rsqrt2;         // sqrt(2) and its correctly rounded reciprocal
};

__device__ __forceinline__ float smin(float a, float b) { return b < a ? b : a; }   // std::min

template <bool FAST> __device__ __forceinline__ float pod_sqrt(float x) {
    return FAST ? sqrt_rn(x) : sqrtf(x);
}

// LDS tile of the times (10^3, halo included) and of the voxels (9^3: the
// voxel before each cell first), z fastest
constexpr int kTX = 11, kTY = 113, kTN = 10 * kTY;
constexpr int kSX = 9, kSY = 83, kSN = 9 * kSY;
// cell e = z + 8 x + 64 y of a tile in the time tile
__device__ __forceinline__ int tile_at(int e) {
    return ((e >> 6) + 1) * kTY + (((e >> 3) & 7) + 1) * kTX + (e & 7) + 1;
}

__device__ __forceinline__ float pmin(float p, float q) {   // floats that are not negative
    return __int_as_float(min(__float_as_int(p), __float_as_int(q)));
}

// The simple operators of one cell (classic.cpp:301-429) and which of the
// others are in play: bit 3 o + f of faces for face f (along z, x, y) of octant
// o (4 z + 2 x + y, 1 for the side after the cell), bit 4 plane + 2 p + q of
// quads for the quarter planes (planes xy, xz, yz with the sides of their two
// axes).  t points at the cell in the time tile, s at the voxel after it on
// every axis.  Times are compared as the integers of their bits, truth values
// are signs: a - b < 0 says a < b.
__device__ __forceinline__ float pod_simple(const int *t, const float *s, const PodArgs &a,
                                            unsigned &faces, unsigned &quads) {
    // times without their marks by (y, x, z) side; the marks as bits 9 y + 3 x + z
    int A[3][3][3];
    unsigned marks = 0;
#pragma unroll
    for (int k = 26; k >= 0; k--) {
        const int y = k / 9, x = k / 3 % 3, z = k % 3;
        const int v = t[(y - 1) * kTY + (x - 1) * kTX + (z - 1)];
        marks = __builtin_amdgcn_alignbit(marks, (unsigned)v, 31);   // marks << 1 | sign
        A[y][x][z] = v & 0x7FFFFFFF;
    }
    float low = __int_as_float(A[1][1][1]);
    {
        float V[2][2][2];
#pragma unroll
        for (int y = 0; y < 2; y++)
#pragma unroll
            for (int x = 0; x < 2; x++)
#pragma unroll
                for (int z = 0; z < 2; z++)
                    V[y][x][z] = s[(y - 1) * kSY + (x - 1) * kSX + (z - 1)];
        auto offer = [&](int tt, float c, float v) { low = pmin(low, __int_as_float(tt) + c * v); };
        // edges along z, x, y: [y][x], [y][z], [x][z]
        float Ez[2][2], Ex[2][2], Ey[2][2];
#pragma unroll
        for (int p = 0; p < 2; p++)
#pragma unroll
            for (int q = 0; q < 2; q++) {
                Ez[p][q] = pmin(V[p][q][0], V[p][q][1]);
                Ex[p][q] = pmin(V[p][0][q], V[p][1][q]);
                Ey[p][q] = pmin(V[0][p][q], V[1][p][q]);
            }
#pragma unroll
        for (int p = 0; p < 2; p++) {
            // head waves: the four voxels around the edge
            offer(A[1][2 * p][1], a.h, pmin(Ez[0][p], Ez[1][p]));
            offer(A[2 * p][1][1], a.h, pmin(Ez[p][0], Ez[p][1]));
            offer(A[1][1][2 * p], a.h, pmin(Ex[0][p], Ex[1][p]));
            // edge diffractions (two voxels), corner diffractions (one)
#pragma unroll
            for (int q = 0; q < 2; q++) {
                offer(A[2 * p][2 * q][1], a.hr2, Ez[p][q]);
                offer(A[2 * p][1][2 * q], a.hr2, Ex[p][q]);
                offer(A[1][2 * p][2 * q], a.hr2, Ey[p][q]);
#pragma unroll
                for (int r = 0; r < 2; r++) offer(A[2 * p][2 * q][2 * r], a.hr3, V[p][q][r]);
            }
        }
    }
    auto bit = [](int y, int x, int z) { return 1u << (9 * y + 3 * x + z); };
    const int ilow = __float_as_int(low), ilim = __float_as_int(low * 1.0000153f);
    // an operator's arrival is not below the latest time it reads (the first
    // 3D one: but for rounding), and needs its times in the order it is for
    faces = 0;
#pragma unroll
    for (int o = 7; o >= 0; o--) {
        const int z = o & 4 ? 2 : 0, x = o & 2 ? 2 : 0, y = o & 1 ? 2 : 0;
        const int M = A[y][x][z], zx = A[1][x][z], zy = A[y][1][z], xy = A[y][x][1];
        const int mzx = zx - M, mzy = zy - M, mxy = xy - M;   // < 0: after its diagonal
        const unsigned bM = bit(y, x, z), bzx = bit(1, x, z), bzy = bit(y, 1, z), bxy = bit(y, x, 1);
        auto face = [&](int N, int P, int mn, int mp, int Q, unsigned from) {
            const int qn = Q - N, qp = Q - P;
            const int none = (qn | qp) & (mn | qn) & (mp | qp);
            const int k234 = ~none & (Q - ilow);
            const int k1 = ~(mn | mp) & (max(N, P) - ilim);
            const int k = (k234 | k1) & -(int)(marks & from);
            faces = __builtin_amdgcn_alignbit(faces, (unsigned)k, 31);   // faces << 1 | sign
        };
        face(xy, zy, mxy, mzy, A[y][1][1], bM | bxy | bzy | bit(y, 1, 1));
        face(zx, xy, mzx, mxy, A[1][x][1], bM | bzx | bxy | bit(1, x, 1));
        face(zx, zy, mzx, mzy, A[1][1][z], bM | bzx | bzy | bit(1, 1, z));
    }
    quads = 0;
#pragma unroll
    for (int k = 11; k >= 0; k--) {
        const int p = k & 2 ? 2 : 0, q = k & 1 ? 2 : 0;
        int ta, tb, td;
        unsigned from;
        if (k < 4) {
            ta = A[1][p][1]; tb = A[q][1][1]; td = A[q][p][1];
            from = bit(1, p, 1) | bit(q, 1, 1) | bit(q, p, 1);
        } else if (k < 8) {
            ta = A[1][p][1]; tb = A[1][1][q]; td = A[1][p][q];
            from = bit(1, p, 1) | bit(1, 1, q) | bit(1, p, q);
        } else {
            ta = A[p][1][1]; tb = A[1][1][q]; td = A[p][1][q];
            from = bit(p, 1, 1) | bit(1, 1, q) | bit(p, 1, q);
        }
        // an axis time after the diagonal's and before the cell's
        const int w = (((td - ta) & (ta - ilow)) | ((td - tb) & (tb - ilow))) & -(int)(marks & from);
        quads = __builtin_amdgcn_alignbit(quads, (unsigned)w, 31);
    }
    return low;
}

// The two 2D operators of one quarter plane (classic.cpp:431-765): axis times
// ta, tb, the diagonal's t2, the lesser voxel; low: what has to be beaten.
template <bool FAST>
__device__ __forceinline__ float pod_quad(float ta, float tb, float t2, float sref, float low,
                                          const PodArgs &a) {
    const float da = ta - t2, db = tb - t2;
    const float lim = FAST ? div_rn(a.h * sref, a.sqrt2, a.rsqrt2) : a.h * sref / a.sqrt2;
    const float hs2 = a.hh * sref * sref;
    const bool ka = (da > 0.0f) & (da < lim), kb = (db > 0.0f) & (db < lim);
    const float va = ta + pod_sqrt<FAST>(ka ? hs2 - da * da : hs2);
    const float vb = tb + pod_sqrt<FAST>(kb ? hs2 - db * db : hs2);
    low = ka ? pmin(low, va) : low;
    return kb ? pmin(low, vb) : low;
}

// The four 3D operators of one face of an octant (classic.cpp:767-1773).
// Every arrival here is compared as the reference compares it; an argument
// of a root that rounds below zero (a NaN there) offers nothing.
template <bool FAST>
__device__ __forceinline__ float pod_face(float M, float N, float P, float Q, float hs2,
                                          float low) {
    const float u = N - M, w = P - M, c = Q - N, d = Q - P;
    const float uu = u * u, ww = w * w, cc = c * c, dd = d * d;
    const float hs05 = 0.5f * hs2;
    // N + P - M + root
    const float a1 = hs2 - uu - ww;
    const bool k1 = (u >= 0.0f) & (w >= 0.0f) & (__builtin_fmaf(2.0f, ww, uu) <= hs2) &
                    (__builtin_fmaf(2.0f, uu, ww) <= hs2) & (uu + ww + u * w >= hs05) &
                    (a1 >= 0.0f);
    if (__any(k1)) {
        const float v = N + P - M + pod_sqrt<FAST>(k1 ? a1 : hs2);
        low = k1 & (v < low) ? v : low;
    }
    // Q + root: the least of the three arguments that apply gives the least
    // arrival (root and sum are monotone)
    const float a2 = hs2 - cc - dd, a3 = hs2 - cc - uu, a4 = hs2 - dd - ww;
    const bool k2 = (c >= 0.0f) & (d >= 0.0f) & (cc + dd + c * d <= hs05) & (a2 >= 0.0f);
    const bool k3 = (u >= 0.0f) & (u <= c) & (__builtin_fmaf(2.0f, cc, uu) <= hs2) & (a3 >= 0.0f);
    const bool k4 = (w >= 0.0f) & (w <= d) & (__builtin_fmaf(2.0f, dd, ww) <= hs2) & (a4 >= 0.0f);
    const bool k = (Q < low) & (k2 | k3 | k4);
    if (__any(k)) {
        float arg = k2 ? a2 : hs2;   // hs2 is above every argument
        arg = k3 ? fminf(arg, a3) : arg;
        arg = k4 ? fminf(arg, a4) : arg;
        const float v = Q + pod_sqrt<FAST>(arg);
        low = k & (v < low) ? v : low;
    }
    return low;
}

// Which of a face's two diagonal times is N and which P matters only for the
// order in which their squares are subtracted; per octant (three bits each,
// octant 0 lowest) the reference's choice: bit 0, N is the zx diagonal of the
// face along z (else zy), bit 1, zx along x (else xy), bit 2, xy along y (else
// zy).
constexpr unsigned kPodN = 07u | (06u << 3) | (02u << 6) | (01u << 9) | (06u << 12) | (01u << 15) |
                           (01u << 18) | (06u << 21);

// T = 1e6 everywhere, tiles never listed, counters zero (classic.cpp:198-219)
__global__ void pod_fill(float *__restrict__ T, long long n, int *__restrict__ stamp, int nstamp,
                         int *__restrict__ cnt) {
    const long long q0 = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    const long long step = (long long)gridDim.x * blockDim.x;
    for (long long q = q0; q < n; q += step) T[q] = 1e6f;
    for (long long q = q0; q < nstamp; q += step) stamp[q] = -1;
    if (q0 < 3 * kSeg * kCntStride) cnt[q0] = 0;
}

// the source node, marked changed in the volume step 0 reads, and the tiles of
// its 26 neighbours listed for step 0 (classic.cpp:186-246); one thread per
// shot
__global__ void pod_seed(PodArgs a, const float *__restrict__ src, int nshot, float dx, float dy,
                         float dz) {
    const int s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= nshot) return;
    const PodGeo g = a.g;
    const float sx = src[3 * s], sy = src[3 * s + 1], sz = src[3 * s + 2];
    const int ix = (int)(sx / dx), iy = (int)(sy / dy), iz = (int)(sz / dz);   // model node
    const float gx = floorf(sx / dx) * dx, gy = floorf(sy / dy) * dy, gz = floorf(sz / dz) * dz;
    const float ex = sx - gx, ey = sy - gy, ez = sz - gz;
    const float dist = sqrtf(ex * ex + ey * ey + ez * ez);
    const float t0 = dist * a.S[iz + (long long)ix * g.nz + (long long)iy * g.nx * g.nz];
    float *Ts = a.T + (long long)s * 2 * g.vol;
    const long long c = (iz + 1) + (long long)(ix + 1) * g.pz + (long long)(iy + 1) * g.px * g.pz;
    // a source later than unreached times lowers no cell, and is not one of the
    // cells that step 0 may lower: no front
    const bool front = t0 < 1e6f;
    Ts[c] = front ? -t0 : t0;
    Ts[g.vol + c] = t0;
    if (!front || a.nit[s] <= 0) return;
    const int seg = s % kSeg;
    for (int dy1 = -1; dy1 <= 1; dy1++)
        for (int dx1 = -1; dx1 <= 1; dx1++)
            for (int dz1 = -1; dz1 <= 1; dz1++) {
                const int z = iz + dz1, x = ix + dx1, y = iy + dy1;
                if (z < 0 || z >= g.nz || x < 0 || x >= g.nx || y < 0 || y >= g.ny) continue;
                const int tile = z / kTile + g.ntz * (x / kTile + g.ntx * (y / kTile));
                const int id = s * g.nt + tile;
                if (a.stamp[id] == 0) continue;
                a.stamp[id] = 0;
                a.list0[seg * a.cap + atomicAdd(&a.cnt[seg * kCntStride], 1)] = id;
            }
}

// One Jacobi step over the listed tiles, NT threads to a tile.  Workgroup b takes
// items of segment b % kSeg.
template <bool FAST, int NT>
__global__ __launch_bounds__(NT, 4) void pod_step(PodArgs a, int step) {
    __shared__ int tT[kTN];                    // float bits, sign = changed
    __shared__ float tS[kSN];
    __shared__ int tLow[512];                  // least arrival so far (float bits)
    __shared__ unsigned short cells[512];
    __shared__ unsigned short faces[24 * NT]; // cell | face << 9
    __shared__ unsigned short quads[12 * NT]; // cell | quarter plane << 9
    __shared__ int4 ftab[24];                  // per face: N, P, M offsets, Q and voxel offsets
    __shared__ int4 qtab[12];                  // per quarter plane: ta, tb, two voxel offsets
    __shared__ int ncell, touched, signs, nface, nquad;
    const PodGeo &g = a.g;
    const int tid = threadIdx.x, lane = tid & 63;
    const int seg = blockIdx.x % kSeg, first = blockIdx.x / kSeg, stride = gridDim.x / kSeg;
    const int n = a.cnt[((step % 3) * kSeg + seg) * kCntStride];
    if (blockIdx.x == 0 && tid < kSeg) a.cnt[(((step + 2) % 3) * kSeg + tid) * kCntStride] = 0;
    const int *cur = ((step & 1) ? a.list1 : a.list0) + seg * a.cap;
    int *next = (step & 1) ? a.list0 : a.list1;
    int *next_cnt = &a.cnt[((step + 1) % 3) * kSeg * kCntStride];
    const long long PXZ = (long long)g.px * g.pz;
    if (tid < 24) {
        const int o = tid / 3, f = tid % 3, oz = o >> 2, ox = (o >> 1) & 1, oy = o & 1;
        const int dz = 2 * oz - 1, dx = (2 * ox - 1) * kTX, dy = (2 * oy - 1) * kTY;
        // the face's axis, and the axes of its first and second diagonal (zx
        // and zy, zx and xy, xy and zy)
        const int d0 = f == 0 ? dz : (f == 1 ? dx : dy);
        const int d1 = f == 1 ? dz : dx, d2 = f == 2 ? dz : dy;
        const bool n1 = (kPodN >> (3 * o + f)) & 1;
        ftab[tid] = make_int4(d0 + (n1 ? d1 : d2), d0 + (n1 ? d2 : d1), dx + dy + dz,
                              ((oy - 1) * kSY + (ox - 1) * kSX + oz - 1) * 65536 + (d0 & 0xFFFF));
    } else if (tid >= 64 && tid < 76) {
        const int k = tid - 64, plane = k >> 2, p = (k >> 1) & 1, q = k & 1;
        const int s1 = plane == 2 ? kSY : kSX, s2 = plane == 0 ? kSY : 1;
        const int s3 = plane == 0 ? 1 : (plane == 1 ? kSY : kSX);
        const int v = (p - 1) * s1 + (q - 1) * s2;
        qtab[k] = make_int4((2 * p - 1) * (plane == 2 ? kTY : kTX),
                            (2 * q - 1) * (plane == 0 ? kTY : 1), v - s3, v);
    }
    // the next item's id travels with this item's work (the first one with the
    // count; every index is inside the list)
    int ahead = cur[first];
    for (int item = first; item < n; item += stride) {
        const int id = ahead;
        if (item + stride < n) ahead = cur[item + stride];
        const int shot = id / g.nt, tile = id - shot * g.nt;
        const int tz = tile % g.ntz, tr = tile / g.ntz, tx = tr % g.ntx, ty = tr / g.ntx;
        const float *src = a.T + ((long long)shot * 2 + (step & 1)) * g.vol;
        float *dst = a.T + ((long long)shot * 2 + ((step + 1) & 1)) * g.vol;
        const long long org = tz * kTile + (long long)tx * kTile * g.pz + ty * kTile * PXZ;
        // stage the times (volume coordinates: the halo starts at org) and
        // the voxels (clamped into the model: the reference's padding)
        constexpr int UT = (1000 + NT - 1) / NT, US = (729 + NT - 1) / NT, UC = 512 / NT;
        float vt[UT], vs[US];
#pragma unroll
        for (int u = 0; u < UT; u++) {
            const int e = min(tid + NT * u, 999), z = e % 10, r = e / 10, x = r % 10, y = r / 10;
            vt[u] = src[org + z + (long long)x * g.pz + y * PXZ];
        }
#pragma unroll
        for (int u = 0; u < US; u++) {
            const int e = min(tid + NT * u, 728), z = e % 9, r = e / 9, x = r % 9, y = r / 9;
            const int iz = min(max(tz * kTile + z - 1, 0), g.nz - 1);
            const int ix = min(max(tx * kTile + x - 1, 0), g.nx - 1);
            const int iy = min(max(ty * kTile + y - 1, 0), g.ny - 1);
            vs[u] = a.S[iz + (long long)ix * g.nz + (long long)iy * g.nx * g.nz];
        }
        if (tid == 0) touched = signs = ncell = 0;
#pragma unroll
        for (int u = 0; u < UT; u++) {
            const int e = min(tid + NT * u, 999), z = e % 10, r = e / 10, x = r % 10, y = r / 10;
            tT[y * kTY + x * kTX + z] = __float_as_int(vt[u]);
        }
#pragma unroll
        for (int u = 0; u < US; u++) {
            const int e = min(tid + NT * u, 728), z = e % 9, r = e / 9, x = r % 9, y = r / 9;
            tS[y * kSY + x * kSX + z] = vs[u];
        }
        __syncthreads();
        // Cells to evaluate: one of the 27 times around changed and is below
        // the cell's (an arrival is not below the times it is made of).  As
        // signed integers the changed times order below all others and among
        // themselves, so the least of the 27 words decides.  A thread takes
        // two cells along z.
        if (tid < 256) {
            const int z = 2 * (tid & 3), x = (tid >> 2) & 7, y = tid >> 5, e = z + 8 * x + 64 * y;
            int lv[4];
#pragma unroll
            for (int u = 0; u < 4; u++) {
                int m = 0x7FFFFFFF;
#pragma unroll
                for (int q = 0; q < 9; q++)
                    m = min(m, tT[(y + q / 3) * kTY + (x + q % 3) * kTX + z + u]);
                lv[u] = m;
            }
            const bool col = tx * kTile + x < g.nx && ty * kTile + y < g.ny;
            bool want[2];
            int own[2];
#pragma unroll
            for (int u = 0; u < 2; u++) {
                own[u] = tT[tile_at(e + u)];
                const int tc = own[u] & 0x7FFFFFFF;
                tLow[e + u] = tc;
                const int m = min(lv[u], min(lv[u + 1], lv[u + 2]));
                const float lim = __int_as_float(tc) * 1.0000153f;
                want[u] = m < 0 && col && tz * kTile + z + u < g.nz &&
                          __int_as_float(m & 0x7FFFFFFF) < lim;
            }
            if (__any((own[0] | own[1]) < 0) && lane == 0) signs = 1;
            const unsigned long long b0 = __ballot(want[0]), b1 = __ballot(want[1]);
            const unsigned long long below = (1ull << lane) - 1ull;
            int base = 0;
            if (lane == 0) base = atomicAdd(&ncell, __popcll(b0) + __popcll(b1));
            base = __builtin_amdgcn_readfirstlane(base) + __popcll(b0 & below) + __popcll(b1 & below);
            if (want[0]) cells[base] = (unsigned short)e;
            if (want[1]) cells[base + (want[0] ? 1 : 0)] = (unsigned short)(e + 1);
        }
        __syncthreads();
        // NT of them at a time: their simple operators, then the faces and
        // quarter planes in play, listed for the whole workgroup
        const int nc = ncell;
        for (int i0 = 0; i0 < nc; i0 += NT) {
            if (tid == 0) nface = nquad = 0;
            __syncthreads();
            if (i0 + (tid & ~63) < nc) {
                const bool in = i0 + tid < nc;
                const int e = cells[in ? i0 + tid : nc - 1];
                const int z = e & 7, x = (e >> 3) & 7, y = e >> 6;
                unsigned wf, wq;
                const float low = pod_simple(tT + tile_at(e),
                                             tS + (y + 1) * kSY + (x + 1) * kSX + z + 1, a, wf, wq);
                if (in) tLow[e] = __float_as_int(low);
                else wf = wq = 0;
                const int k = __popc(wf) | (__popc(wq) << 16);
                int at = k;
#pragma unroll
                for (int o = 1; o < 64; o <<= 1) {
                    const int v = __shfl_up(at, o);
                    if (lane >= o) at += v;
                }
                const int total = __builtin_amdgcn_readlane(at, 63);
                int bf = 0, bq = 0;
                if (lane == 0) {
                    bf = atomicAdd(&nface, total & 0xFFFF);
                    bq = atomicAdd(&nquad, total >> 16);
                }
                at -= k;
                int af = (at & 0xFFFF) + __builtin_amdgcn_readfirstlane(bf);
                int aq = (at >> 16) + __builtin_amdgcn_readfirstlane(bq);
                while (wf) {
                    faces[af++] = (unsigned short)(e | (__builtin_ctz(wf) << 9));
                    wf &= wf - 1;
                }
                while (wq) {
                    quads[aq++] = (unsigned short)(e | (__builtin_ctz(wq) << 9));
                    wq &= wq - 1;
                }
            }
            __syncthreads();
            const int nf = nface, nq = nquad;
            auto time = [&](int at) { return __int_as_float(tT[at] & 0x7FFFFFFF); };
            for (int j0 = tid & ~63; j0 < nf; j0 += NT) {
                const int it = faces[min(j0 + lane, nf - 1)], e = it & 511;
                const int4 f = ftab[it >> 9];
                const int at = tile_at(e);
                const float v = tS[((e >> 6) + 1) * kSY + (((e >> 3) & 7) + 1) * kSX + (e & 7) + 1 +
                                   (f.w >> 16)];
                const float low0 = __int_as_float(tLow[e]);
                const float low = pod_face<FAST>(time(at + f.z), time(at + f.x), time(at + f.y),
                                                 time(at + (short)(f.w & 0xFFFF)), a.hh * v * v,
                                                 low0);
                if (low < low0) atomicMin(&tLow[e], __float_as_int(low));
            }
            // the quarter planes from the last wave down, which the faces
            // load least
            for (int j0 = NT - 64 - (tid & ~63); j0 < nq; j0 += NT) {
                const int it = quads[min(j0 + lane, nq - 1)], e = it & 511;
                const int4 f = qtab[it >> 9];
                const int at = tile_at(e);
                const float *sv = tS + ((e >> 6) + 1) * kSY + (((e >> 3) & 7) + 1) * kSX + (e & 7) + 1;
                const float low0 = __int_as_float(tLow[e]);
                const float low = pod_quad<FAST>(time(at + f.x), time(at + f.y),
                                                 time(at + f.x + f.y), pmin(sv[f.z], sv[f.w]), low0,
                                                 a);
                if (low < low0) atomicMin(&tLow[e], __float_as_int(low));
            }
            __syncthreads();
        }
        // the tile to the other volume, changed cells marked
        int touch = 0;
#pragma unroll
        for (int u = 0; u < UC; u++) {
            const int e = tid + NT * u, z = e & 7, x = (e >> 3) & 7, y = e >> 6;
            const int low = tLow[e];
            const bool chg = low < (tT[tile_at(e)] & 0x7FFFFFFF);
            dst[org + (z + 1) + (long long)(x + 1) * g.pz + (y + 1) * PXZ] =
                __int_as_float(chg ? low | (int)0x80000000 : low);
            if (chg)
                touch |= 1 | (z == 0 ? 2 : 0) | (z == 7 ? 4 : 0) | (x == 0 ? 8 : 0) |
                         (x == 7 ? 16 : 0) | (y == 0 ? 32 : 0) | (y == 7 ? 64 : 0);
        }
        if (__any(touch)) {
            int all = 0;
#pragma unroll
            for (int b = 0; b < 7; b++) all |= __any(touch & (1 << b)) ? 1 << b : 0;
            if (lane == 0) atomicOr(&touched, all);
        }
        __syncthreads();
        // the tile and the neighbours that changed cells touch
        if (tid < 64 && step + 1 < a.nit[shot]) {
            const int tc = touched;
            bool want = false;
            int target = 0;
            if (lane < 27) {
                const int ez = lane % 3 - 1, ex = (lane / 3) % 3 - 1, ey = lane / 9 - 1;
                const int need = 1 | (ez < 0 ? 2 : ez > 0 ? 4 : 0) | (ex < 0 ? 8 : ex > 0 ? 16 : 0) |
                                 (ey < 0 ? 32 : ey > 0 ? 64 : 0);
                const int nz1 = tz + ez, nx1 = tx + ex, ny1 = ty + ey;
                want = ((tc & need) == need || (lane == 13 && signs)) && nz1 >= 0 && nz1 < g.ntz &&
                       nx1 >= 0 && nx1 < g.ntx && ny1 >= 0 && ny1 < g.nty;
                target = shot * g.nt + nz1 + g.ntz * (nx1 + g.ntx * ny1);
            }
            if (want) want = atomicMax(&a.stamp[target], step + 1) < step + 1;
            const unsigned long long m = __ballot(want);
            if (m) {
                int base = 0;
                const int to = (item + seg) % kSeg;   // spreads a segment's items over all
                if (lane == 0) base = atomicAdd(&next_cnt[to * kCntStride], __popcll(m));
                base = __builtin_amdgcn_readfirstlane(base);
                if (want) next[to * a.cap + base + __popcll(m & ((1ull << lane) - 1ull))] = target;
            }
        }
        __syncthreads();
    }
}

// the times without their marks in the first volume of each shot, which holds
// the last step's (an even number of steps) or takes it from the second
__global__ void pod_finish(float *__restrict__ T, long long vol, int nshot,
                           const int *__restrict__ nit) {
    const long long n = vol * nshot;
    for (long long q = (long long)blockIdx.x * blockDim.x + threadIdx.x; q < n;
         q += (long long)gridDim.x * blockDim.x) {
        const long long s = q / vol, c = q - s * vol;
        float *Ts = T + s * 2 * vol;
        Ts[c] = fabsf(Ts[(nit[s] & 1 ? vol : 0) + c]);
    }
}

// first volumes -> cropped (nz, nx, ny) volumes (reduce_model,
// classic.cpp:62-72)
__global__ void pod_crop(const float *__restrict__ T, float *__restrict__ out, PodGeo g,
                         int nshot) {
    const long long per = (long long)g.nx * g.ny * g.nz, n = per * nshot;
    for (long long q = (long long)blockIdx.x * blockDim.x + threadIdx.x; q < n;
         q += (long long)gridDim.x * blockDim.x) {
        const long long s = q / per, r = q - s * per;
        const int z = (int)(r % g.nz);
        const long long r2 = r / g.nz;
        const int x = (int)(r2 % g.nx), y = (int)(r2 / g.nx);
        out[q] = T[s * 2 * g.vol + (z + 1) + (long long)(x + 1) * g.pz +
                   (long long)(y + 1) * g.px * g.pz];
    }
}

int grid_for(long long n) { return (int)std::min<long long>((n + 255) / 256, 65536); }

}  // namespace

// nItEikonal of classic.cpp:248-273: the largest source-to-corner distance in
// padded nodes (powf(x, 2.0f) is the square the reference's optimised build
// computes)
int podvin_iterations(int sidx, int sidy, int sidz, int nxx, int nyy, int nzz) {
    const float fx = (float)sidx, fy = (float)sidy, fz = (float)sidz;
    const float gx = (float)(nxx - sidx), gy = (float)(nyy - sidy), gz = (float)(nzz - sidz);
    const float c[8][3] = {{fx, fy, fz}, {gx, fy, fz}, {fx, gy, fz}, {fx, fy, gz},
                           {fx, gy, gz}, {gx, fy, gz}, {gx, gy, fz}, {gx, gy, gz}};
    int n = 0;
    for (int q = 0; q < 8; q++) {
        const int aux = (int)sqrtf(c[q][0] * c[q][0] + c[q][1] * c[q][1] + c[q][2] * c[q][2]);
        if (aux > n) n = aux;
    }
    return n;
}

// Device memory of a batch: bytes per shot, and the layout the forward pass
// traces rays on (cells per shot stride, extents along x and z).
size_t podvin_bytes_per_shot(const st_ctx *ctx) {
    const PodGeo g = pod_geo(ctx);
    return sizeof(float) * 2 * (size_t)g.vol + sizeof(int) * (size_t)g.nt * (1 + 2 * kSeg);
}
void podvin_layout(const st_ctx *ctx, long long &stride, int &nxx, int &nzz) {
    const PodGeo g = pod_geo(ctx);
    stride = 2 * g.vol;
    nxx = g.px;
    nzz = g.pz;
}
// largest batch the lists' 32-bit tile ids allow
long long podvin_max_batch(const st_ctx *ctx) { return ((1LL << 31) - 1) / pod_geo(ctx).nt; }
void podvin_reserve(st_ctx *ctx, int batch) {
    const PodGeo g = pod_geo(ctx);
    ctx->pod_T.reserve(sizeof(float) * 2 * g.vol * batch);
    ctx->pod_stamp.reserve(sizeof(int) * (size_t)g.nt * batch);
    ctx->pod_list.reserve(sizeof(int) * 2 * kSeg * (size_t)g.nt * batch);
    ctx->pod_counts.reserve(sizeof(int) * 3 * kSeg * kCntStride);
    ctx->pod_nit.reserve(sizeof(int) * batch);
}

// Solves nshot shots (device sources dsrc, host copies hsrc) into ctx->pod_T;
// returns the device time in ms.
double podvin_batch(st_ctx *ctx, const float *dsrc, const float *hsrc, int nshot) {
    PodArgs a{};
    const PodGeo g = a.g = pod_geo(ctx);
    a.S = ctx->slow_zxy.as<float>();
    a.T = ctx->pod_T.as<float>();
    a.stamp = ctx->pod_stamp.as<int>();
    a.cap = (long long)g.nt * nshot;
    a.list0 = ctx->pod_list.as<int>();
    a.list1 = a.list0 + kSeg * a.cap;
    a.cnt = ctx->pod_counts.as<int>();
    a.nit = ctx->pod_nit.as<int>();
    a.h = ctx->dx;
    a.sqrt2 = sqrtf(2.0f);
    a.rsqrt2 = 1.0f / a.sqrt2;
    a.hh = a.h * a.h;
    a.hr2 = a.h * a.sqrt2;
    a.hr3 = a.h * sqrtf(3.0f);
    std::vector<int> nit(nshot);
    int maxit = 0;
    for (int s = 0; s < nshot; s++) {
        const int sidx = (int)(hsrc[3 * s] / ctx->dx) + 1, sidy = (int)(hsrc[3 * s + 1] / ctx->dy) + 1,
                  sidz = (int)(hsrc[3 * s + 2] / ctx->dz) + 1;
        nit[s] = podvin_iterations(sidx, sidy, sidz, g.nx + 2, g.ny + 2, g.nz + 2);
        maxit = std::max(maxit, nit[s]);
    }
    ST_HIP(hipMemcpyAsync(ctx->pod_nit.ptr, nit.data(), sizeof(int) * nshot, hipMemcpyHostToDevice,
                          ctx->stream));
    ST_HIP(hipEventRecord(ctx->ev[2], ctx->stream));
    const long long total = 2 * g.vol * nshot;
    hipLaunchKernelGGL(pod_fill, dim3(grid_for(total)), dim3(256), 0, ctx->stream, a.T, total,
                       a.stamp, g.nt * nshot, a.cnt);
    hipLaunchKernelGGL(pod_seed, dim3((nshot + 63) / 64), dim3(64), 0, ctx->stream, a, dsrc, nshot,
                       ctx->dx, ctx->dy, ctx->dz);
    ST_HIP(hipGetLastError());
    // short roots and quotients where h S and its square are of ordinary size
    const bool fast = a.h * ctx->smin > 1e-9f && a.h * ctx->smax < 1e9f;
    // A front of 8^3 tiles per shot is about nt^(2/3) of them, and a step visits
    // one to two fronts.  Up to half the chip's 512-thread workgroups (two per
    // CU), a step lasts as long as its fullest tile and eight waves to a tile
    // shorten that (a shot of 101 x 101 x 51: 2.04 ms against 2.26); beyond, four
    // waves leave fewer idle at the barriers (8 shots of 201 x 201 x 101: 37.0 ms
    // against 43.6).
    const bool wide = nshot * std::cbrt((double)g.nt) * std::cbrt((double)g.nt) <= 256.0;
    auto kernel = wide ? (fast ? pod_step<true, 512> : pod_step<false, 512>)
                       : (fast ? pod_step<true, 256> : pod_step<false, 256>);
    const dim3 block(wide ? 512 : 256);
    // enough workgroups for the tiles of the fronts, eight per CU at most
    const int grid = kSeg * (int)std::max(1LL, std::min(a.cap / kSeg, 2048LL / kSeg));
    for (int step = 0; step < maxit; step++)
        hipLaunchKernelGGL(kernel, dim3(grid), block, 0, ctx->stream, a, step);
    hipLaunchKernelGGL(pod_finish, dim3(grid_for(g.vol * nshot)), dim3(256), 0, ctx->stream, a.T,
                       g.vol, nshot, a.nit);
    ST_HIP(hipGetLastError());
    ST_HIP(hipEventRecord(ctx->ev[3], ctx->stream));
    ST_HIP(hipEventSynchronize(ctx->ev[3]));
    float ms = 0.f;
    ST_HIP(hipEventElapsedTime(&ms, ctx->ev[2], ctx->ev[3]));
    return ms;
}

void podvin_picks(st_ctx *ctx, int nshot, const float *drcv, int nrcv, float *dpicks) {
    const PodGeo g = pod_geo(ctx);
    launch_picks_padvol(ctx->stream, ctx->pod_T.as<float>(), 2 * g.vol, g.px, g.pz, nshot, drcv,
                        nrcv, dpicks, ctx->nx, ctx->ny, ctx->nz, ctx->dx, ctx->dy, ctx->dz);
}

void podvin_crop_volumes(st_ctx *ctx, float *dout, int nshot) {
    const PodGeo g = pod_geo(ctx);
    const long long n = (long long)g.nx * g.ny * g.nz * nshot;
    hipLaunchKernelGGL(pod_crop, dim3(grid_for(n)), dim3(256), 0, ctx->stream,
                       ctx->pod_T.as<float>(), dout, g, nshot);
    ST_HIP(hipGetLastError());
}

}  // namespace st
