// fsm.hip -- the reference's CPU eikonal, Accurate_FSM (Noble, Gesret and
// Belayouni 2014 operators; src/eikonal/accurate_FSM/accurate_FSM.cpp), on
// the GPU for a batch of shots, bit-identical to the CPU code.
//
// Why a parallel schedule can reproduce the sequential sweeps exactly: the
// update of cell (i, j, k) in a sweep with directions (sz, sx, sy) reads T
// only at offsets (-sz or 0, -sx or 0, -sy or 0) -- its own value and seven
// upwind neighbours (accurate_FSM.cpp:168-175).  Number the cells of a
// sweep's box by p = a + b + c, their distances from the box's start corner
// along z, x, y.  Every upwind neighbour has a smaller p, and the loop nest
// (k outer, j, i inner) also visits every cell after all cells of smaller p
// that it reads.  So any schedule that updates a cell after its upwind
// neighbours gives each update the same inputs, and with the same arithmetic
// the same result.
//
// Schedule: a sweep's box is cut into blocks of 8 x 8 columns (x, y) by a
// chunk of z, and the blocks with equal A + B + C (block distances from the
// start corner) are one launch; a block's upwind neighbours lie in blocks of
// earlier launches or in itself.  One wave updates one block of one shot: lane
// (x, y) walks its column and is x + y steps behind lane (0, 0), so that at
// each step the wave updates a diagonal plane of the block and every lane's
// upwind neighbours were updated in earlier steps.  The block and its upwind
// halo sit in LDS while the wave works on it (travel times and slowness read
// once per block, in rows along z), the values along z stay in registers.
// Each shot's source-bounded sweeps cover that shot's own boxes only.
//
// The full sweeps change few blocks (14 % of 64 shots of 201 x 201 x 101 in a
// gradient, 12 to 65 % a sweep of other cases): each begins with a test of all
// cells at once (fsm_test) against the times as they stand, which marks the
// blocks with a cell that would be lowered.  The first cell of a sweep's order
// to change in a block either was marked or reads a changed cell of an upwind
// block, so a launch walks the marked blocks and those behind a face that has
// changed, and every other block keeps the values the sweep would give it.
// The blocks to walk are lists per diagonal, so that the waves of a launch are
// its first workgroups and spread evenly; without lists the working blocks
// fall unevenly on the SIMDs (33 us for a launch of 870 of them, 22 with).
//
// What bounds it: a step of the walk is about 210 vector instructions of one
// wave, some 1,000 cycles, so a launch takes 16 us for a lone shot (4 of them
// the launch itself) and there are (blocks along the longest diagonal) of
// them per sweep; a batch adds the vector issue of the busiest SIMD.
// Measured: one shot of 121 x 97 x 61 cells 21.1 ms with a launch per plane of
// cells, 6.5 with all blocks walked, 4.4 to 5.2 now (by the model); 64 shots of
// 201 x 201 x 101 77.5, 39.2, 25.9 ms (walks 19.5, tests 5.7).  Blocks of 9 / 11 /
// 14 / 15 / 22 cells of z, before the update followed negative roots and times
// (25.5 ms): 26.7 / 25.9 / 25.5 / 25.5 / 26.9 ms for the 64 shots, 4.8 / 4.9 / 5.0
// / 5.0 / 5.4 for the lone one.
//
// Layout: one padded volume per shot, z fastest.
//
// Compiled with -ffp-contract=off and HIP's correctly rounded square root;
// divisions by the spacing constants are correctly rounded without a divide
// (div_rn); min/max follow std::min/std::max operand order where a NaN could
// reach them.  The seeds' powf(x, 2.0f) are computed as x*x, the form the
// reference's compiler emits for them (exact squares; the oracle's CPU build
// agrees bit for bit).
#include "st_common.hpp"

#include "fsm_update.hpp"

namespace st {

void launch_picks_padvol(hipStream_t st, const float *T, long long vol, int nxx, int nzz,
                         int nshot, const float *rcv, int nr, float *out, int nx, int ny, int nz,
                         float dx, float dy, float dz);

// One sweep: directions (1 forward, -1 backward) for z (i), x (j), y (k),
// and whether it is one of the eight source-bounded sweeps of init_sweep.
struct FsmSweep {
    int tz, tx, ty;
    int init;
};

// Start and extent of a sweep along one axis (n = padded length, sid = the
// source's padded index): init_sweep (accurate_FSM.cpp:267-388) starts the
// forward loops at max(1, sid) and the backward loops at sid + 1;
// full_sweep (:390-511) runs 1 .. n-1 forward and n-2 .. 0 backward.  For a
// source on the last node the reference's backward start sid + 1 = n - 1
// reads one cell past the array; the start is clamped to n - 2 there (the
// CPU oracle does the same).
__host__ __device__ inline void sweep_axis(int t, int init, int n, int sid, int &start, int &len) {
    if (t > 0) {
        start = init ? (sid > 1 ? sid : 1) : 1;
        len = n - start;
    } else {
        const int s = init ? (sid < n - 3 ? sid : n - 3) + 1 : n - 2;
        start = s;
        len = s + 1;
    }
}

// Slowness padded by one cell, edge replicated: expand_model
// (accurate_FSM.cpp:8-60) copies the boundary plane outward along z, then
// x, then y, which is the model value at the clamped index.
__global__ void fsm_pad_model(const float *__restrict__ s, float *__restrict__ S, int nx, int ny,
                              int nz) {
    const int nzz = nz + 2, nxx = nx + 2, nyy = ny + 2;
    const long long n = (long long)nzz * nxx * nyy;
    for (long long q = (long long)blockIdx.x * blockDim.x + threadIdx.x; q < n;
         q += (long long)gridDim.x * blockDim.x) {
        const int z = (int)(q % nzz);
        const long long r = q / nzz;
        const int x = (int)(r % nxx), y = (int)(r / nxx);
        const int zs = min(max(z - 1, 0), nz - 1), xs = min(max(x - 1, 0), nx - 1),
                  ys = min(max(y - 1, 0), ny - 1);
        S[q] = s[zs + (long long)xs * nz + (long long)ys * nx * nz];
    }
}

// T = 1e6 everywhere (accurate_FSM.cpp:591-592), four cells per thread plus
// the n % 4 tail
__global__ void fsm_fill(float *__restrict__ T, long long n) {
    const long long n4 = n / 4;
    float4 *T4 = reinterpret_cast<float4 *>(T);
    for (long long q = (long long)blockIdx.x * blockDim.x + threadIdx.x; q < n4;
         q += (long long)gridDim.x * blockDim.x)
        T4[q] = make_float4(1e6f, 1e6f, 1e6f, 1e6f);
    if (blockIdx.x == 0 && threadIdx.x < (unsigned)(n - 4 * n4)) T[4 * n4 + threadIdx.x] = 1e6f;
}

// The 27 analytic seeds around the source node (accurate_FSM.cpp:596-630):
// entry e writes the node at index offset (iz, ix, iy) with S[source] times
// the distance of the node at offset (dz, dx, dy).  The two xz diagonals of
// lines 608-609 pair an index offset with the mirrored node's distance; the
// table keeps that pairing so the results match.
__constant__ signed char kSeed[27][6] = {
    {0, 0, 0, 0, 0, 0},
    {1, 0, 0, 1, 0, 0},     {-1, 0, 0, -1, 0, 0},
    {0, 1, 0, 0, 1, 0},     {0, -1, 0, 0, -1, 0},
    {0, 0, 1, 0, 0, 1},     {0, 0, -1, 0, 0, -1},
    {1, 1, 0, 1, 1, 0},     {1, -1, 0, -1, 1, 0},
    {-1, 1, 0, 1, -1, 0},   {-1, -1, 0, -1, -1, 0},
    {1, 0, 1, 1, 0, 1},     {1, 0, -1, 1, 0, -1},
    {-1, 0, 1, -1, 0, 1},   {-1, 0, -1, -1, 0, -1},
    {0, 1, 1, 0, 1, 1},     {0, 1, -1, 0, 1, -1},
    {0, -1, 1, 0, -1, 1},   {0, -1, -1, 0, -1, -1},
    {1, 1, 1, 1, 1, 1},     {1, -1, 1, 1, -1, 1},
    {1, 1, -1, 1, 1, -1},   {1, -1, -1, 1, -1, -1},
    {-1, 1, 1, -1, 1, 1},   {-1, -1, 1, -1, -1, 1},
    {-1, 1, -1, -1, 1, -1}, {-1, -1, -1, -1, -1, -1},
};

// One thread per shot, the entries in table order (entries that name the
// same node are written in the reference's order: the last wins).
__global__ void fsm_seed(float *__restrict__ T, const float *__restrict__ S,
                         const float *__restrict__ src, const int *__restrict__ sid, int nshot,
                         FsmGeo g) {
    const int s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= nshot) return;
    const int nb = 1;
    const float sx = src[3 * s], sy = src[3 * s + 1], sz = src[3 * s + 2];
    const int sidz = sid[3 * s], sidx = sid[3 * s + 1], sidy = sid[3 * s + 2];
    const long long NZ = g.nzz, NXZ = (long long)g.nxx * g.nzz;
    const long long sId = sidz + sidx * NZ + sidy * NXZ;
    float *Ts = T + s * g.nB;
    const float S0 = S[sId];
    for (int e = 0; e < 27; e++) {
        const int iz = kSeed[e][0], ix = kSeed[e][1], iy = kSeed[e][2];
        const int oz = kSeed[e][3], ox = kSeed[e][4], oy = kSeed[e][5];
        const float ex = ((sidx - nb) + ox) * g.dx - sx;
        const float ey = ((sidy - nb) + oy) * g.dy - sy;
        const float ez = ((sidz - nb) + oz) * g.dz - sz;
        Ts[sId + iz + ix * NZ + iy * NXZ] = S0 * sqrtf(ex * ex + ey * ey + ez * ez);
    }
}

// One diagonal D of one sweep's blocks, for all shots.  Blocks are (A, B, C)
// = distances from the start corner of the shot's box in units of zc cells
// along z and eight along x and y; workgroup q walks entry q / 8 of the list
// of residue q % 8, and leaves at once where the list is shorter.
//
// The LDS tiles hold planes 0 (the upwind halo) .. 8 along x and y and 0 ..
// zc along z, in sweep order.  P even and Q = 9 mod 16 put the 64 lanes of a
// step, whose z differ by x + y, on 64 different banks.  Slowness is stored
// as the voxel on the downwind side of each cell, so a cell's eight voxels
// are the tile's entries at offsets 0 and -1 per axis: padded voxel i for a
// forward sweep and i - 1 for a backward one.  The reference's index clamps
// (max(i - 1, 1), min(i, n - 1)) only choose between a padding voxel and the
// edge voxel it copies, so clamping at 0 gives the same value.
constexpr int kFsmZ = 14;   // most z cells of a block
template <int LZ> struct FsmTile {
    static constexpr int P = (LZ + 2) & ~1;
    static constexpr int Q = ((9 * P - 9 + 15) / 16) * 16 + 9;
    static constexpr int N = 9 * Q;
};

// The blocks a sweep has to walk, in a list per diagonal D = A + B + C and per
// residue of shot + B (workgroups of one residue run on one XCD).  A block is
// its number ((shot nC + C) nB + B) nA + A.
struct FsmQueue {
    unsigned *list;         // [D][8][cap]
    unsigned *count;        // [D][8] of this sweep
    unsigned *flag;         // per block, the full sweep it was last marked in
    unsigned cap;
    int sweep;              // 1 .. 8
    int nA, nB, nC;
    __device__ unsigned number(int shot, int A, int B, int C) const {
        return ((unsigned)(shot * nC + C) * nB + B) * nA + A;
    }
    __device__ void put(int shot, int A, int B, int C) const {
        const int e = (A + B + C) * 8 + ((shot + B) & 7);
        list[(long long)e * cap + atomicAdd(count + e, 1u)] = number(shot, A, B, C);
    }
    // the same for a block that several may list
    __device__ void put_once(int shot, int A, int B, int C) const {
        unsigned *f = flag + number(shot, A, B, C);
        if (__builtin_nontemporal_load(f) != (unsigned)sweep &&
            atomicExch(f, (unsigned)sweep) != (unsigned)sweep)
            put(shot, A, B, C);
    }
};

// The blocks a sweep starts with: all blocks of the shots' boxes if it is
// source-bounded, the marked ones if not; one thread per block of the largest
// box.
__global__ __launch_bounds__(256) void fsm_list(const int *__restrict__ sid, int nshot, FsmGeo g,
                                                FsmSweep w, int zc, FsmQueue q) {
    const long long id = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    const int shot = (int)(id / ((long long)q.nA * q.nB * q.nC));
    if (shot >= nshot || (!w.init && q.flag[id] != (unsigned)q.sweep)) return;
    const int r = (int)(id - (long long)shot * q.nA * q.nB * q.nC);
    const int A = r % q.nA, B = r / q.nA % q.nB, C = r / (q.nA * q.nB);
    int s0, zl, xl, yl;
    sweep_axis(w.tz, w.init, g.nzz, sid[3 * shot], s0, zl);
    sweep_axis(w.tx, w.init, g.nxx, sid[3 * shot + 1], s0, xl);
    sweep_axis(w.ty, w.init, g.nyy, sid[3 * shot + 2], s0, yl);
    if (zc * A < zl && 8 * B < xl && 8 * C < yl) q.put(shot, A, B, C);
}

// Whether a cell of a full sweep would be lowered by the times as they stand,
// for all cells at once: marks the blocks that hold one.  Lanes run over the
// (z, x) cells of the box in memory order, each walks the eight y planes of a
// block, the times and voxels of one plane serving as the next one's upwind
// ones.  w.init = 0: all shots sweep the same box.
template <bool FAST>
__global__ __launch_bounds__(256) void fsm_test(const float *__restrict__ T,
                                                const float *__restrict__ S, FsmGeo g, FsmSweep w,
                                                int zc, FsmQueue queue) {
    int zs, zl, xs, xl, ys, yl;
    sweep_axis(w.tz, 0, g.nzz, 0, zs, zl);
    sweep_axis(w.tx, 0, g.nxx, 0, xs, xl);
    sweep_axis(w.ty, 0, g.nyy, 0, ys, yl);
    const int q = blockIdx.x * blockDim.x + threadIdx.x;
    const bool on = q < zl * xl;
    const int b = on ? q / zl : 0, a = on ? q - b * zl : 0;
    const int C = blockIdx.y, shot = blockIdx.z;
    const int i = zs + w.tz * a, j = xs + w.tx * b;
    const int bz = w.tz < 0, bx = w.tx < 0, by = w.ty < 0;
    // a cell and its upwind neighbours, a voxel and its upwind neighbours
    const int t00 = i + g.nzz * j, t10 = t00 - w.tz, t01 = t00 - w.tx * g.nzz, t11 = t01 - w.tz;
    const int iu = i - w.tz - bz, id = max(i - bz, 0);
    const int ju = j - w.tx - bx, jd = max(j - bx, 0);
    const int s00 = id + g.nzz * jd, s10 = iu + g.nzz * jd, s01 = id + g.nzz * ju,
              s11 = iu + g.nzz * ju;
    const long long plane = (long long)g.nxx * g.nzz;
    const float *Ts = T + shot * g.nB;
    const int y1 = ys + w.ty * (8 * C), nc = min(8, yl - 8 * C);
    const float *Tk = Ts + plane * (y1 - w.ty), *Sk = S + plane * (y1 - w.ty - by);
    float u00 = Tk[t00], u10 = Tk[t10], u01 = Tk[t01], u11 = Tk[t11];
    float v00 = Sk[s00], v10 = Sk[s10], v01 = Sk[s01], v11 = Sk[s11];
    float ubig = tmag3(tmag3(u00, u10, u01), u11, u11);
    bool hit = false;
    for (int c = 0; c < nc; c++) {
        const int k = y1 + w.ty * c;
        Tk = Ts + plane * k;
        Sk = S + plane * max(k - by, 0);
        const float n00 = Tk[t00], n10 = Tk[t10], n01 = Tk[t01], n11 = Tk[t11];
        const float m00 = Sk[s00], m10 = Sk[s10], m01 = Sk[s01], m11 = Sk[s11];
        FsmIn f;
        f.tv = n10;
        f.te = n01;
        f.tev = n11;
        f.tn = u00;
        f.tnv = u10;
        f.ten = u01;
        f.tnve = u11;
        f.sve = pmin(m11, v11);
        f.svn = pmin(v11, v10);
        f.sen = pmin(v11, v01);
        f.sv = pmin(f.sve, pmin(m10, v10));
        f.se = pmin(f.sve, pmin(m01, v01));
        f.sn = pmin(f.svn, pmin(v01, v00));
        f.s = v11;
        const float nbig = tmag3(n10, n01, n11);
        const float res = FAST ? fsm_update_fast<true>(n00, f, on, g, tmag3(nbig, ubig, ubig))
                               : fsm_update_any(n00, f, g);
        hit |= !(res == n00);
        ubig = tmag3(nbig, n00, n00);
        u00 = n00;
        u10 = n10;
        u01 = n01;
        u11 = n11;
        v00 = m00;
        v10 = m10;
        v01 = m01;
        v11 = m11;
    }
    if (hit & on) queue.flag[queue.number(shot, a / zc, b / 8, C)] = queue.sweep;
}

template <int LZ, bool FAST, bool FULL>
__global__ __launch_bounds__(64) void fsm_block(float *__restrict__ T,
                                                const float *__restrict__ S,
                                                const int *__restrict__ sid, FsmGeo g,
                                                FsmSweep w, int zc, int D, FsmQueue queue) {
    using Tile = FsmTile<LZ>;
    constexpr int P = Tile::P, Q = Tile::Q;
    __shared__ float tt[Tile::N + 1];
    __shared__ float ts[Tile::N];
    const unsigned pos = blockIdx.x >> 3, e = D * 8 + (blockIdx.x & 7);
    if (pos >= queue.count[e]) return;
    const unsigned id = queue.list[(long long)e * queue.cap + pos];
    const unsigned ab = id / queue.nA, cb = ab / queue.nB;
    const int A = id - ab * queue.nA, B = ab - cb * queue.nB;
    const int shot = cb / queue.nC, C = cb - shot * queue.nC;
    int zs, zl, xs, xl, ys, yl;
    sweep_axis(w.tz, w.init, g.nzz, sid[3 * shot], zs, zl);
    sweep_axis(w.tx, w.init, g.nxx, sid[3 * shot + 1], xs, xl);
    sweep_axis(w.ty, w.init, g.nyy, sid[3 * shot + 2], ys, yl);
    const int lane = threadIdx.x;
    float *Ts = T + shot * g.nB;
    const int len = min(zc, zl - zc * A);      // z cells of this block
    const int nb = min(8, xl - 8 * B), nc = min(8, yl - 8 * C);
    const int z1 = zs + w.tz * (zc * A), x1 = xs + w.tx * (8 * B), y1 = ys + w.ty * (8 * C);
    const int bz = w.tz < 0, bx = w.tx < 0, by = w.ty < 0;

    // stage: RPW rows along z per load, a plane of y at a time; indices are
    // clamped into the volume, entries past the box are not used
    constexpr int RZ = LZ < 16 ? 16 : (LZ < 32 ? 32 : 64), RPW = 64 / RZ;
    constexpr int NB = (9 + RPW - 1) / RPW;   // loads per plane
    const int rz = lane & (RZ - 1), row0 = lane / RZ;
    {
        const int i = min(max(z1 + w.tz * (rz - 1), 0), g.nzz - 1);
        const int iv = max(i - bz, 0);
        int ot[NB], os[NB];
#pragma unroll
        for (int u = 0; u < NB; u++) {
            const int j = min(max(x1 + w.tx * (row0 + u * RPW - 1), 0), g.nxx - 1);
            ot[u] = i + g.nzz * j;
            os[u] = iv + g.nzz * max(j - bx, 0);
        }
        float *t0 = tt + row0 * P + rz, *s0 = ts + row0 * P + rz;
        float vt[9 * NB], vs[9 * NB];
#pragma unroll
        for (int c = 0; c < 9; c++) {
            const int k = min(max(y1 + w.ty * (c - 1), 0), g.nyy - 1);
            const float *Tk = Ts + (long long)k * g.nxx * g.nzz;
            const float *Sk = S + (long long)max(k - by, 0) * g.nxx * g.nzz;
#pragma unroll
            for (int u = 0; u < NB; u++) {
                vt[c * NB + u] = Tk[ot[u]];
                vs[c * NB + u] = Sk[os[u]];
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        if (rz <= LZ) {
#pragma unroll
            for (int c = 0; c < 9; c++)
#pragma unroll
                for (int u = 0; u < NB; u++)
                    if (u * RPW + RPW <= 9 || row0 < 9 - u * RPW) {
                        t0[c * Q + u * RPW * P] = vt[c * NB + u];
                        s0[c * Q + u * RPW * P] = vs[c * NB + u];
                    }
        }
    }
    wave_sync();

    // the walk: lane (x, y) is at z cell a = s - x - y; a = -1 reads the
    // halo plane into the registers that carry the values along z
    const int x = lane & 7, y = lane >> 3;
    int at = (y + 1) * Q + (x + 1) * P - x - y;   // tile index of a, at s = -1
    // a = at - lo, in [0, len) for the cells of the block
    const int lo = x < nb && y < nc ? (y + 1) * Q + (x + 1) * P + 1 : 1 << 24;
    float tv = 0, tev = 0, tnv = 0, tnve = 0;
    float suu = 0, sxu = 0, syu = 0, s4 = 0;      // upwind voxels: (x, y) up, x up, y up, all four
    // own time and voxels of the step, read one step ahead (no other lane
    // writes them)
    float own = tt[at], vdd = ts[at], vud = ts[at - P], vdu = ts[at - Q], vuu = ts[at - P - Q];
    bool changed = false;
#pragma unroll 2
    for (int s = -1; s < len + 14; s++, at++) {
        FsmIn c;
        c.te = tt[at - P];
        c.tn = tt[at - Q];
        c.ten = tt[at - P - Q];
        const float own1 = tt[at + 1], vdd1 = ts[at + 1], vud1 = ts[at + 1 - P],
                    vdu1 = ts[at + 1 - Q], vuu1 = ts[at + 1 - P - Q];
        c.tv = tv;
        c.tev = tev;
        c.tnv = tnv;
        c.tnve = tnve;
        const float nxu = pmin(vuu, vud), nyu = pmin(vuu, vdu);
        c.sv = s4;
        c.se = pmin(sxu, nxu);
        c.sn = pmin(syu, nyu);
        c.sve = sxu;
        c.svn = syu;
        c.sen = pmin(suu, vuu);
        c.s = suu;
        const bool on = (unsigned)(at - lo) < (unsigned)len;
        float res = FAST ? fsm_update_fast<false>(own, c, on, g) : fsm_update_any(own, c, g);
        res = on ? res : own;
        if (FULL) changed |= on & !(res == own);
        tt[on ? at : Tile::N] = res;   // the last word takes what is not a cell
        tv = res;
        tev = c.te;
        tnv = c.tn;
        tnve = c.ten;
        suu = vuu;
        sxu = nxu;
        syu = nyu;
        s4 = pmin(nxu, pmin(vdu, vdd));
        own = own1;
        vdd = vdd1;
        vud = vud1;
        vdu = vdu1;
        vuu = vuu1;
        wave_sync();
    }

    if (FULL) {
        if (!__any(changed)) return;
        const bool cx = __any(changed & (x == nb - 1)), cy = __any(changed & (y == nc - 1));
        // lanes 1 .. 7: the downwind neighbours that read a changed plane
        const int dA = lane & 1, dB = (lane >> 1) & 1, dC = lane >> 2;
        if (lane > 0 && lane < 8 && (!dB | cx) && (!dC | cy) && A + dA < queue.nA &&
            B + dB < queue.nB && C + dC < queue.nC)
            queue.put_once(shot, A + dA, B + dB, C + dC);
    }

    // the block back to memory
    if (rz >= 1 && rz <= len) {
        const int i = z1 + w.tz * (rz - 1);
        constexpr int NS = 8 / RPW;
        int o[NS];
#pragma unroll
        for (int u = 0; u < NS; u++) o[u] = i + g.nzz * (x1 + w.tx * (row0 + u * RPW));
        const float *t0 = tt + Q + (row0 + 1) * P + rz;
#pragma unroll
        for (int c = 0; c < 8; c++) {
            if (c >= nc) break;
            float *Tk = Ts + (long long)(y1 + w.ty * c) * g.nxx * g.nzz;
#pragma unroll
            for (int u = 0; u < NS; u++)
                if (row0 + u * RPW < nb) Tk[o[u]] = t0[c * Q + u * RPW * P];
        }
    }
}

// reduce_model (accurate_FSM.cpp:62-72): padded -> model extent, z fastest
__global__ void fsm_crop(const float *__restrict__ T, float *__restrict__ out, int nx, int ny,
                         int nz, long long nB, int nshot) {
    const long long npts = (long long)nx * ny * nz;
    const long long n = npts * nshot;
    const int nzz = nz + 2, nxx = nx + 2;
    for (long long q = (long long)blockIdx.x * blockDim.x + threadIdx.x; q < n;
         q += (long long)gridDim.x * blockDim.x) {
        const long long s = q / npts, r = q - s * npts;
        const int z = (int)(r % nz);
        const long long r2 = r / nz;
        const int x = (int)(r2 % nx), y = (int)(r2 / nx);
        out[q] = T[s * nB + (z + 1) + (long long)(x + 1) * nzz + (long long)(y + 1) * nxx * nzz];
    }
}

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------
static unsigned grid_for(long long n) {
    return (unsigned)std::min<long long>(std::max<long long>((n + 255) / 256, 1), 1 << 20);
}

static FsmGeo fsm_geo(const st_ctx *ctx) {
    return fsm_geometry(ctx->nx, ctx->ny, ctx->nz, ctx->dx, ctx->dy, ctx->dz);
}

// The 16 sweeps of eikonal_equation: init_sweep then full_sweep, each in the
// reference's direction order (accurate_FSM.cpp:270-388, 393-511).
static const int kDirs[8][3] = {{1, 1, 1},  {-1, 1, 1},  {1, 1, -1},  {-1, 1, -1},
                                {1, -1, 1}, {-1, -1, 1}, {1, -1, -1}, {-1, -1, -1}};

// Blocks along the axes and most blocks of one residue of shot + B on the
// diagonals of a box of nA x nB x nC blocks, for all shots together.
static void fsm_diagonals(int nA, int nB, int nC, int nshot, std::vector<unsigned> &most) {
    most.assign(nA + nB + nC - 2, 0);
    for (int D = 0; D < (int)most.size(); D++) {
        long long on[8] = {};   // blocks per residue of B
        for (int B = std::max(0, D - (nA - 1) - (nC - 1)); B <= std::min(D, nB - 1); B++) {
            const int r = D - B;
            on[B & 7] += std::min(r, nA - 1) - std::max(0, r - (nC - 1)) + 1;
        }
        for (int e = 0; e < 8; e++) {
            long long n = 0;
            for (int t = 0; t < 8; t++) n += on[t] * ((nshot + 7 - ((e - t) & 7)) / 8);
            most[D] = (unsigned)std::max<long long>(most[D], n);
        }
    }
}

// The sixteen sweeps of nshot shots (padded volumes T, source nodes dsid on
// the device and hsid on the host) on one stream.  A launch per diagonal has
// as many workgroups as its lists could hold.
template <int LZ>
static void fsm_sweeps(hipStream_t st, bool fast, float *T, const float *S, const int *dsid,
                       const int *hsid, int nshot, const FsmGeo &g, DevBuf &lists) {
    FsmQueue q{};
    std::vector<unsigned> most;
    const int mA = (g.nzz - 1 + LZ - 1) / LZ, mB = (g.nxx + 6) / 8, mC = (g.nyy + 6) / 8;
    const size_t nD = mA + mB + mC - 2, blocks = (size_t)mA * mB * mC * nshot;
    ST_REQUIRE(blocks < (1ull << 31), ST_ERR_ARG, "too many blocks for one batch of the sweeps");
    fsm_diagonals(mA, mB, mC, nshot, most);
    q.cap = *std::max_element(most.begin(), most.end());
    const size_t nz = blocks + 16 * nD * 8;   // flags and counts, zero at first
    lists.reserve(sizeof(unsigned) * (nz + nD * 8 * q.cap));
    q.flag = lists.as<unsigned>();
    q.count = q.flag + blocks;
    q.list = q.flag + nz;
    ST_HIP(hipMemsetAsync(lists.ptr, 0, sizeof(unsigned) * nz, st));
    for (int pass = 0; pass < 2; pass++) {
        for (int d = 0; d < 8; d++) {
            const FsmSweep w{kDirs[d][0], kDirs[d][1], kDirs[d][2], pass == 0 ? 1 : 0};
            // the longest box along each axis
            int len[3];
            const int dir[3] = {w.tz, w.tx, w.ty}, n[3] = {g.nzz, g.nxx, g.nyy};
            for (int ax = 0; ax < 3; ax++) {
                len[ax] = 0;
                for (int s = 0; s < (w.init ? nshot : 1); s++) {
                    int st0, l;
                    sweep_axis(dir[ax], w.init, n[ax], hsid[3 * s + ax], st0, l);
                    len[ax] = std::max(len[ax], l);
                }
            }
            const int nA0 = (len[0] + LZ - 1) / LZ;
            const int zc = (len[0] + nA0 - 1) / nA0;   // chunks of equal length
            q.nA = (len[0] + zc - 1) / zc;
            q.nB = (len[1] + 7) / 8;
            q.nC = (len[2] + 7) / 8;
            q.sweep = d + 1;
            if (!w.init) {
                const dim3 grid((unsigned)(((long long)len[0] * len[1] + 255) / 256),
                                (unsigned)q.nC, (unsigned)nshot);
                hipLaunchKernelGGL(fast ? fsm_test<true> : fsm_test<false>, grid, dim3(256), 0, st,
                                   T, S, g, w, zc, q);
            }
            const long long nb = (long long)q.nA * q.nB * q.nC * nshot;
            hipLaunchKernelGGL(fsm_list, dim3((unsigned)((nb + 255) / 256)), dim3(256), 0, st, dsid,
                               nshot, g, w, zc, q);
            fsm_diagonals(q.nA, q.nB, q.nC, nshot, most);
            const auto walk = fast ? (w.init ? fsm_block<LZ, true, false> : fsm_block<LZ, true, true>)
                                   : (w.init ? fsm_block<LZ, false, false> : fsm_block<LZ, false, true>);
            for (int D = 0; D < (int)most.size(); D++)
                hipLaunchKernelGGL(walk, dim3(most[D] * 8), dim3(64), 0, st, T, S, dsid, g, w, zc, D,
                                   q);
            ST_HIP(hipGetLastError());
            q.count += nD * 8;
        }
    }
}

// Solves nshot shots (device sources dsrc, host copies hsrc) into ctx->T
// (one padded volume per shot); returns the device time in ms.
double fsm_batch(st_ctx *ctx, const float *dsrc, const float *hsrc, int nshot, const float *S) {
    const FsmGeo g = fsm_geo(ctx);
    std::vector<int> hsid(3 * nshot);
    for (int s = 0; s < nshot; s++) {
        hsid[3 * s] = (int)(hsrc[3 * s + 2] / ctx->dz) + 1;      // z
        hsid[3 * s + 1] = (int)(hsrc[3 * s] / ctx->dx) + 1;      // x
        hsid[3 * s + 2] = (int)(hsrc[3 * s + 1] / ctx->dy) + 1;  // y
    }
    ctx->fsm_sid.reserve(sizeof(int) * 3 * std::max(nshot, 1));
    int *dsid = ctx->fsm_sid.as<int>();
    ST_HIP(hipMemcpyAsync(dsid, hsid.data(), sizeof(int) * 3 * nshot, hipMemcpyHostToDevice,
                          ctx->stream));
    ST_HIP(hipEventRecord(ctx->ev[2], ctx->stream));
    const long long nT = (long long)nshot * g.nB;
    float *T = ctx->T.as<float>();
    ST_REQUIRE(ctx->T.bytes >= sizeof(float) * (size_t)nT, ST_ERR_STATE, "travel-time buffer too small");
    hipLaunchKernelGGL(fsm_fill, dim3(grid_for(nT / 4)), dim3(256), 0, ctx->stream, T, nT);
    hipLaunchKernelGGL(fsm_seed, dim3((nshot + 63) / 64), dim3(64), 0, ctx->stream, T, S, dsrc,
                       dsid, nshot, g);
    ST_HIP(hipGetLastError());
    const bool fast = fsm_fast(g, ctx->smin, ctx->smax);
    fsm_sweeps<kFsmZ>(ctx->stream, fast, T, S, dsid, hsid.data(), nshot, g,
                      ctx->fsm_lists);
    ST_HIP(hipEventRecord(ctx->ev[3], ctx->stream));
    ST_HIP(hipEventSynchronize(ctx->ev[3]));
    float ms = 0.f;
    ST_HIP(hipEventElapsedTime(&ms, ctx->ev[2], ctx->ev[3]));
    return ms;
}

void fsm_pad(st_ctx *ctx, float *S) {
    const long long n = (long long)(ctx->nx + 2) * (ctx->ny + 2) * (ctx->nz + 2);
    hipLaunchKernelGGL(fsm_pad_model, dim3(grid_for(n)), dim3(256), 0, ctx->stream,
                       ctx->slow_zxy.as<float>(), S, ctx->nx, ctx->ny, ctx->nz);
    ST_HIP(hipGetLastError());
}

void fsm_picks(st_ctx *ctx, int nshot, const float *drcv, int nrcv, float *dpicks) {
    const FsmGeo g = fsm_geo(ctx);
    launch_picks_padvol(ctx->stream, ctx->T.as<float>(), g.nB, g.nxx, g.nzz, nshot, drcv, nrcv,
                        dpicks, ctx->nx, ctx->ny, ctx->nz, ctx->dx, ctx->dy, ctx->dz);
}

void fsm_crop_volumes(st_ctx *ctx, float *dout, int nshot) {
    const long long n = (long long)ctx->nx * ctx->ny * ctx->nz * nshot;
    hipLaunchKernelGGL(fsm_crop, dim3(grid_for(n)), dim3(256), 0, ctx->stream, ctx->T.as<float>(),
                       dout, ctx->nx, ctx->ny, ctx->nz, fsm_geo(ctx).nB, nshot);
    ST_HIP(hipGetLastError());
}

}  // namespace st
