// eikonal3d.hip -- 3-D first-arrival traveltimes on gfx950.
//
// Replaces the SFMM solve inside fastMarching3D (fastmarching/fastMarching.cpp
// :26-129, fmm/fmm.hpp:92-158).  Instead of a serial heap, the grid is cut into
// 4x4x4 tiles, one wave64 per tile, one node per lane.  A round processes every
// active tile of every problem (problem = chain x wave type x source): the wave
// stages its tile and a 2-deep face halo in LDS, relaxes the local upwind
// update to convergence (a wave ballot ends the loop), writes back, and
// activates the face neighbours whose halo it changed.  Rounds repeat until no
// tile is active (block fast-iterative method).
//
// The local update is the reference's: solveEikonal (eikonalsolver.hpp:50-79)
// for order 0, highAccuracySolveEikonal (:83-145) for order 1, with the cell's
// current value as the filter and a new value kept only when it improves
// (fmm.hpp:141-150).  For order 0 the FMM answer is the unique fixed point of
// that update, so the tiles converge to it; arithmetic is FP32 with each
// quadratic written relative to its smallest neighbour time, which removes the
// cancellation of the reference's b^2-4ac form.
#include "mct_internal.h"
#include <float.h>
#include <stdlib.h>

#pragma clang fp contract(fast)

#define EIK_INF __builtin_huge_valf()
template <class TT> __device__ __forceinline__ TT tinf();
template <> __device__ __forceinline__ float tinf<float>() { return __builtin_huge_valf(); }
template <> __device__ __forceinline__ double tinf<double>() { return __builtin_huge_val(); }
// LDS box: the 4^3 tile at offset 2 inside an 8^3 box (2-deep face halo).
#define BX(x, y, z) ((((z) + 2) << 6) | (((y) + 2) << 3) | ((x) + 2))

// The local solves below run in R = float (velocities and increments in FP32)
// or R = double (the FP64 mode: the reference's own precision).
__device__ __forceinline__ float lsqrt(float x) { return sqrtf(x); }
__device__ __forceinline__ double lsqrt(double x) { return sqrt(x); }

// Compare-and-swap of (time, 1/h^2, h) triples by time; the swap keeps the
// earlier dimension first on equal times (std::sort on <= 16 elements is an
// insertion sort, which is stable).
template <class R>
__device__ __forceinline__ void cas3(R &t0, R &a0, R &h0, R &t1, R &a1, R &h1)
{
    bool sw = t1 < t0;
    R tt = sw ? t1 : t0, aa = sw ? a1 : a0, hh = sw ? h1 : h0;
    t1 = sw ? t0 : t1; a1 = sw ? a0 : a1; h1 = sw ? h0 : h1;
    t0 = tt; a0 = aa; h0 = hh;
}

template <class R>
__device__ __forceinline__ void cas4(R &t0, R &u0, R &a0, R &h0, R &t1, R &u1, R &a1, R &h1)
{
    bool sw = t1 < t0;
    R tt = sw ? t1 : t0, uu = sw ? u1 : u0, aa = sw ? a1 : a0, hh = sw ? h1 : h0;
    t1 = sw ? t0 : t1; u1 = sw ? u0 : u1; a1 = sw ? a0 : a1; h1 = sw ? h0 : h1;
    t0 = tt; u0 = uu; a0 = aa; h0 = hh;
}

// root of sum_i al_i (tau - dl_i)^2 = s2 (larger root), INF if none
template <class R>
__device__ __forceinline__ R root2(R a0, R d0, R a1, R d1, R s2)
{
    R A = a0 + a1, B = a0 * d0 + a1 * d1, C = a0 * d0 * d0 + a1 * d1 * d1 - s2;
    R disc = B * B - A * C;
    return disc < R(0) ? tinf<R>() : (B + lsqrt(disc)) / A;
}

template <class R>
__device__ __forceinline__ R root3(R a0, R d0, R a1, R d1, R a2, R d2, R s2)
{
    R A = a0 + a1 + a2, B = a0 * d0 + a1 * d1 + a2 * d2;
    R C = a0 * d0 * d0 + a1 * d1 * d1 + a2 * d2 * d2 - s2;
    R disc = B * B - A * C;
    return disc < R(0) ? tinf<R>() : (B + lsqrt(disc)) / A;
}

// v_min / v_max without the compiler's extra canonicalising instructions (no
// arrival time is a NaN)
__device__ __forceinline__ double tmin(double a, double b)
{
    double r;
    asm("v_min_f64 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}
__device__ __forceinline__ double tmax(double a, double b)
{
    double r;
    asm("v_max_f64 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}
__device__ __forceinline__ float tmin(float a, float b) { return fminf(a, b); }
__device__ __forceinline__ float tmax(float a, float b) { return fmaxf(a, b); }

// sqrt of a discriminant: values are far from the ends of the exponent range (a
// time squared, or a slowness over a spacing squared), so the library's scaling
// steps go; two Goldschmidt steps and a residual correction from v_rsq_f64 leave
// the rounding they leave there.  Negative (rounding around 0) counts as 0.
__device__ __forceinline__ double dsqrt(double x)
{
    x = tmax(x, 1e-200);
    const double r = __builtin_amdgcn_rsq(x);
    double g = x * r, h = 0.5 * r;
    const double e = __builtin_fma(-h, g, 0.5);
    g = __builtin_fma(g, e, g);
    h = __builtin_fma(h, e, h);
    g = __builtin_fma(__builtin_fma(-g, g, x), h, g);
    return __builtin_fma(__builtin_fma(-g, g, x), h, g);
}
__device__ __forceinline__ float dsqrt(float x) { return sqrtf(fmaxf(x, 0.f)); }

// solveEikonal (first order), eikonalsolver.hpp:50-79: the dimensions' smaller
// neighbour times in ascending order, one more taken while it lies below the
// solution.  The reference leaves out neighbours at or above the cell's own
// time; such a neighbour cannot lower it, so the caller's comparison does the
// same.  All times are relative to the smallest one.

// The same spacing h in all dimensions, s = h / v: d1 <= d2 the other two times.
template <class R>
__device__ __forceinline__ R update_iso(R d1, R d2, R s)
{
    R u = s;
    if (s > d1) {
        u = R(0.5) * (d1 + dsqrt(R(2) * s * s - d1 * d1));
        if (u > d2) {
            const R q = d1 + d2;
            u = (q + dsqrt(q * q - R(3) * (d1 * d1 + d2 * d2 - s * s))) * R(1.0 / 3.0);
        }
    }
    return u;
}

// Different spacings: n the times, t0 the smallest, d1 <= d2 the other two
// relative to it; al = 1/h^2, ra = 1 / (sum of the al but one) and 1 / (all).
// On equal times the earlier dimension comes first (std::sort on <= 16
// elements is an insertion sort, which is stable).
template <class TT, class R>
__device__ __forceinline__ R update_aniso(const TT n[3], TT t0, R d1, R d2, const R h[3], const R al[3], const R ra[4],
                                          R inv_v, R s2)
{
    const R hm = n[0] == t0 ? h[0] : (n[1] == t0 ? h[1] : h[2]);
    R u = hm * inv_v;
    if (u > d1) {
        // without the largest: the last dimension among equals
        const bool ez = n[2] >= n[0] && n[2] >= n[1], ey = !ez && n[1] >= n[0];
        const bool ex = !ez && !ey;
        const R dx = ex ? R(0) : (R)(n[0] - t0), dy = ey ? R(0) : (R)(n[1] - t0), dz = ez ? R(0) : (R)(n[2] - t0);
        const R ax = ex ? R(0) : al[0], ay = ey ? R(0) : al[1], az = ez ? R(0) : al[2];
        const R A = ax + ay + az, B = ax * dx + ay * dy + az * dz;
        const R C = ax * dx * dx + ay * dy * dy + az * dz * dz - s2;
        u = (B + dsqrt(B * B - A * C)) * (ex ? ra[0] : (ey ? ra[1] : ra[2]));
        if (u > d2) {
            const R am = ex ? al[0] : (ey ? al[1] : al[2]);
            const R A3 = al[0] + al[1] + al[2], B3 = B + am * d2, C3 = C + am * d2 * d2;
            u = (B3 + dsqrt(B3 * B3 - A3 * C3)) * ra[3];
        }
    }
    return u;
}

// highAccuracySolveEikonal: per dimension the smaller one-away time t and, when
// the two-away time on that side is upwind (<= t), the second-order value
// (4t - t2)/3 with weight 9/4; try all included dimensions first and drop the
// largest while the root does not exceed that dimension's time.
template <class R>
__device__ __forceinline__ R update_order1(const R m1[3], const R m2[3], R tself, const R h[3], const R ih2[3],
                                           R inv_v, R s2)
{
    const R INF = tinf<R>();
    R t[3], u[3], al[3], hh[3];
    for (int d = 0; d < 3; d++) {
        bool inc = m1[d] < tself;
        bool two = m2[d] < INF;
        t[d] = inc ? m1[d] : INF;
        u[d] = two ? m2[d] : INF;
        al[d] = two ? R(2.25) * ih2[d] : ih2[d];
        hh[d] = h[d];
    }
    cas4(t[0], u[0], al[0], hh[0], t[1], u[1], al[1], hh[1]);
    cas4(t[1], u[1], al[1], hh[1], t[2], u[2], al[2], hh[2]);
    cas4(t[0], u[0], al[0], hh[0], t[1], u[1], al[1], hh[1]);
    if (t[0] == INF) return tself;
    const R t0 = t[0];
    R dl[3];
    for (int d = 0; d < 3; d++)
        dl[d] = u[d] < INF ? (R(4) * (t[d] - t0) - (u[d] - t0)) * (R(1) / R(3)) : t[d] - t0;
    if (t[2] < INF) {
        R tau = root3(al[0], dl[0], al[1], dl[1], al[2], dl[2], s2);
        if (tau < INF && tau > t[2] - t0) return t0 + tau;
    }
    if (t[1] < INF) {
        R tau = root2(al[0], dl[0], al[1], dl[1], s2);
        if (tau < INF && tau > t[1] - t0) return t0 + tau;
    }
    return t0 + hh[0] * inv_v;
}

// ---- initial points --------------------------------------------------------------
// One thread per (problem, corner): Solver::setInitialPoints (solver.hpp:72-92)
// with getVel / getNeighbors(point) (ndgridmap.hpp:158-191,433-460).
__device__ __forceinline__ void pt_coord(const mct_geom &G, const double p[3], const double leaf[3],
                                         int c[3])
{
    int dims[3] = {G.nx, G.ny, G.nz};
    for (int d = 0; d < 3; d++) {
        // int(p/h) truncates toward zero, then clamps (getPointCoord);
        // done in double so out-of-range inputs never reach the conversion
        double qd = p[d] / leaf[d];
        int ci = !(qd >= 1.0) ? 0 : (qd >= (double)dims[d] ? dims[d] - 1 : (int)qd);
        c[d] = ci;
    }
}

__device__ __forceinline__ long tl_index(const mct_geom &G, int x, int y, int z)
{
    int tile = ((z >> 2) * G.nty + (y >> 2)) * G.ntx + (x >> 2);
    int lane = ((z & 3) << 4) | ((y & 3) << 2) | (x & 3);
    return ((long)tile << 6) | lane;
}

template <class TT>
__global__ void k_eik_clear(TT *T, long n)
{
    for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x)
        T[i] = tinf<TT>();
}

template <class TT>
__global__ void k_eik_init(mct_eik_problem_set P, const double *src_pts, int src_stride,
                           long src_chain_stride, double xmin, double ymin, double zmin, double lx,
                           double ly, double lz)
{
    int prob = blockIdx.x * blockDim.x + threadIdx.x;
    if (prob >= P.nprob) return;
    const mct_geom &G = P.G;
    int s = prob % P.nsrc_eff, cw = prob / P.nsrc_eff;          // cw = chain*nwave + wave
    int c = cw / P.nwave;
    const double *sp0 = src_pts + (long)c * src_chain_stride + (long)s * src_stride;
    double p[3] = {sp0[0] - xmin, sp0[1] - ymin, sp0[2] - zmin};
    double leaf[3] = {lx, ly, lz};
    int dims[3] = {G.nx, G.ny, G.nz};
    int pc[3];
    pt_coord(G, p, leaf, pc);
    const float *V = P.vel ? P.vel + (long)cw * G.ntiles * MCT_TILE_N : nullptr;
    const double *V64 = P.vel64 ? P.vel64 + (long)cw * G.ntiles * MCT_TILE_N : nullptr;
    TT *T = (TT *)P.T + (long)prob * G.ntiles * MCT_TILE_N;
    int cx[8], cy[8], cz[8];
    double vn[8];
    for (int v = 0; v < 8; v++) {
        int vc[3];
        for (int d = 0; d < 3; d++) {
            vc[d] = pc[d] + ((v >> (2 - d)) & 1);
            if (vc[d] >= dims[d]) vc[d] = dims[d] - 1;
        }
        cx[v] = vc[0]; cy[v] = vc[1]; cz[v] = vc[2];
        const long q = tl_index(G, vc[0], vc[1], vc[2]);
        vn[v] = V64 ? V64[q] : (double)V[q];
    }
    // getVel: trilinear weights with clamped corners
    double vs = 0.0;
    for (int v = 0; v < 8; v++) {
        int cc[3] = {cx[v], cy[v], cz[v]};
        double w = 1.0;
        for (int d = 0; d < 3; d++) {
            double sd = p[d] - leaf[d] * pc[d];
            double wj = fabs((double)(cc[d] - pc[d]) * leaf[d] - leaf[d] + sd);
            w = w * wj / leaf[d];
        }
        vs = vs + w * vn[v];
    }
    for (int v = 0; v < 8; v++) {
        double q[3] = {cx[v] * leaf[0], cy[v] * leaf[1], cz[v] * leaf[2]};
        double dist = 0.0;
        for (int d = 0; d < 3; d++) dist = dist + (q[d] - p[d]) * (q[d] - p[d]);
        dist = sqrt(dist);
        T[tl_index(G, cx[v], cy[v], cz[v])] = (TT)(dist * 2 / (vs + vn[v]));
    }
    // seed: the 3x3x3 block of tiles around each corner's tile
    P.any[0] = 1u;
    for (int v = 0; v < 8; v++) {
        int tx = cx[v] >> 2, ty = cy[v] >> 2, tz = cz[v] >> 2;
        for (int dz = -1; dz <= 1; dz++)
            for (int dy = -1; dy <= 1; dy++)
                for (int dx = -1; dx <= 1; dx++) {
                    int ax = tx + dx, ay = ty + dy, az = tz + dz;
                    if (ax < 0 || ay < 0 || az < 0 || ax >= G.ntx || ay >= G.nty || az >= G.ntz) continue;
                    long key = (long)prob * G.ntiles + (long)((az * G.nty + ay) * G.ntx + ax);
                    P.flags[0][key] = 1;
                    P.key[0][key] = 0u;
                }
    }
}

// ---- one relaxation round ----------------------------------------------------------
__device__ __forceinline__ float wave_min(float v)
{
    for (int o = 32; o > 0; o >>= 1) v = fminf(v, __shfl_xor(v, o, 64));
    return v;
}

__device__ __forceinline__ uint32_t fbits(float f) { return __float_as_uint(f); }


// Minimum over the wave by DPP moves (row_shr 1, 2, 4, 8, then the two row
// broadcasts): lane 63 ends with it.
__device__ __forceinline__ uint32_t wave_min_u(uint32_t v)
{
#define EIK_DPP(ctrl, rm)                                                                                              \
    {                                                                                                                  \
        const uint32_t o = (uint32_t)__builtin_amdgcn_update_dpp(-1, (int)v, ctrl, rm, 0xf, false);                    \
        v = o < v ? o : v;                                                                                             \
    }
    EIK_DPP(0x111, 0xf) EIK_DPP(0x112, 0xf) EIK_DPP(0x114, 0xf) EIK_DPP(0x118, 0xf) EIK_DPP(0x142, 0xa) EIK_DPP(0x143, 0xc)
#undef EIK_DPP
    return (uint32_t)__builtin_amdgcn_readlane((int)v, 63);
}

// One relaxation round of the first-order update.  Active tiles are byte flags
// (no lists, no counters); each carries a key, the smallest arrival time that
// activated it.  A tile is relaxed only once the round's band time tau has
// passed its key, so the front is swept roughly in arrival order (a tile sees
// its upwind halo nearly final); tiles not yet due are carried to the next round.
//
// What bounds it: many chains move 4.25 TB/s of tiles and halos past L2 (a large copy:
// 4.9; 42 % L2 hits) with the VALUs 49 % busy, so a visit saved counts on both
// sides; one chain (34 % busy, 1.4 TB/s, 9.5 waves per CU) waits, in the rounds with
// many tiles.  A visit relaxes its 64 nodes about six times, whatever few of them
// change: ISO (one spacing) needs no sort, no division and two short square roots
// (60 instructions instead of 150).  A neighbour tile is activated only by a face node whose new time lies
// below the neighbour's node across the face: any other cannot lower it.  The
// halo may be older than the neighbour's times, never lower, so no activation is
// missed.  That drops the 42% of the visits that changed nothing, most of them to
// the tiles the front came from.
//
// TT is the storage type of arrival times, CT that of the local solve, which
// runs on times relative to the smallest upwind neighbour t0 (an increment of
// about h/v) and is added to t0 in TT: with TT = double and CT = float the
// rounding of each step is that of the small increment.
template <int ISO, class TT, class CT>
__global__ __launch_bounds__(64) void k_eik_round0(mct_eik_problem_set P, int round, double hxd, double hyd,
                                                   double hzd)
{
    // the 4^3 tile at offset 1 inside a 6^3 box
    __shared__ TT box[216];
    __shared__ uint32_t fkey[6];
    const mct_geom &G = P.G;
    const TT TINF = tinf<TT>();
    const CT CINF = tinf<CT>();
    const int cur = round & 1, nxt = cur ^ 1;
    const int lane = threadIdx.x;
    const int lx = lane & 3, ly = (lane >> 2) & 3, lz = lane >> 4;
    const CT h[3] = {(CT)hxd, (CT)hyd, (CT)hzd};
    const CT al[3] = {CT(1) / (h[0] * h[0]), CT(1) / (h[1] * h[1]), CT(1) / (h[2] * h[2])};
    const CT ra[4] = {CT(1) / (al[1] + al[2]), CT(1) / (al[0] + al[2]), CT(1) / (al[0] + al[1]),
                      CT(1) / (al[0] + al[1] + al[2])};
    if (blockIdx.x == 0 && lane == 0) P.any[(round + 2) % 3] = 0u;   // flag of round r+2
    const uint32_t ntiles = (uint32_t)G.ntiles;
    const uint32_t nkeys = (uint32_t)P.nprob * ntiles;
    const uint32_t stride = gridDim.x;
    uint8_t *fcur = P.flags[cur], *fnxt = P.flags[nxt];
    uint32_t *kcur = P.key[cur], *knxt = P.key[nxt];
    unsigned int *any_next = &P.any[(round + 1) % 3];
    const bool banded = round < P.band_rounds;
    // Relative change that counts.  In the FP64 mode every decrease counts, so
    // the rounds end only at the update's fixed point, whatever order the tiles
    // ran in (a batch gives each chain the times its own call gives); with FP32
    // increments a change is at least an FP32 step of the increment anyway.
    const TT thr = sizeof(CT) == 8 ? (TT)0 : sizeof(TT) == 8 ? (TT)1e-9 : (TT)1e-7;
    TT *Tall = (TT *)P.T;
    // face halo: 6 faces x 16 nodes (-x, +x, -y, +y, -z, +z), up to 2 per lane: the
    // neighbour tile's offset, the node's place in it and in the box
    const int toff[6] = {-1, 1, -G.ntx, G.ntx, -G.ntx * G.nty, G.ntx * G.nty};
    int hface[2], hidx[2], hbox[2];
    for (int r = 0; r < 2; r++) {
        const int q = lane + 64 * r, f = q >> 4, a = q & 3, b = (q >> 2) & 3;
        const int in = (f & 1) ? 0 : 3, out = (f & 1) ? 5 : 0;
        hface[r] = f < 6 ? f : 0;
        hidx[r] = f < 2 ? (b << 4) | (a << 2) | in : f < 4 ? (b << 4) | (in << 2) | a : (in << 4) | (b << 2) | a;
        hbox[r] = f < 2 ? (b + 1) * 36 + (a + 1) * 6 + out
                        : f < 4 ? (b + 1) * 36 + out * 6 + a + 1 : out * 36 + (b + 1) * 6 + a + 1;
    }
    const int ho0 = toff[hface[0]], ho1 = toff[hface[1]];
    const int me = (lz + 1) * 36 + (ly + 1) * 6 + lx + 1;

    // Keys are visited lane-strided: block b, pass i covers keys
    // b + stride*(64*i + lane), so every key has exactly one owner.
    for (uint32_t base = blockIdx.x; base < nkeys; base += stride * 64u) {
        const uint32_t mykey = base + stride * (uint32_t)lane;
        uint8_t f = mykey < nkeys ? fcur[mykey] : 0;
        bool due = false;
        if (f) {
            fcur[mykey] = 0;                       // consumed
            uint32_t kc = kcur[mykey];
            kcur[mykey] = 0xffffffffu;
            const uint32_t prob = mykey / ntiles;
            const float tau = banded ? (float)(round + 1) * P.band_h / P.vmax[prob / (uint32_t)P.nsrc_eff]
                                     : __builtin_huge_valf();
            if (__uint_as_float(kc) <= tau || kc == 0xffffffffu) {
                due = true;
            } else {                               // not yet: carry to the next round
                fnxt[mykey] = 1;
                atomicMin(&knxt[mykey], kc);
                *any_next = 1u;
            }
        }
        uint64_t todo = __ballot(due);
        while (todo) {
            const int src_lane = __ffsll((unsigned long long)todo) - 1;
            todo &= todo - 1;
            const uint32_t key = base + stride * (uint32_t)src_lane;
            const uint32_t prob = key / ntiles;
            const uint32_t tile = key - prob * ntiles;
            const int tx = (int)(tile % (uint32_t)G.ntx);
            const int tyz = (int)(tile / (uint32_t)G.ntx);
            const int ty = tyz % G.nty, tz = tyz / G.nty;
            // the faces with a tile behind them
            const int nbr = (tx > 0) | (tx < G.ntx - 1) << 1 | (ty > 0) << 2 | (ty < G.nty - 1) << 3 | (tz > 0) << 4 |
                            (tz < G.ntz - 1) << 5;
            const bool inside = tx * 4 + lx < G.nx && ty * 4 + ly < G.ny && tz * 4 + lz < G.nz;
            TT *T = Tall + (size_t)prob * ((size_t)ntiles << 6);
            const uint32_t cw = prob / (uint32_t)P.nsrc_eff;
            const size_t vi = (size_t)cw * ((size_t)ntiles << 6) + ((size_t)tile << 6) + lane;
            const CT v = sizeof(CT) == 8 ? (CT)P.vel64[vi] : (CT)P.vel[vi];
            // nodes of a tile beyond the grid hold +inf, as absent tiles do
            const bool ok0 = (nbr >> hface[0]) & 1, ok1 = lane < 32 && ((nbr >> hface[1]) & 1);
            TT t = T[((size_t)tile << 6) + lane];
            const TT g0 = T[((size_t)(ok0 ? (int)tile + ho0 : (int)tile) << 6) + hidx[0]];
            const TT g1 = T[((size_t)(ok1 ? (int)tile + ho1 : (int)tile) << 6) + hidx[1]];
            const TT t_in = t;
            box[me] = t;
            box[hbox[0]] = ok0 ? g0 : TINF;
            if (lane < 32) box[hbox[1]] = ok1 ? g1 : TINF;
            if (lane < 6) fkey[lane] = 0xffffffffu;
            __syncthreads();
            const CT inv_v = CT(1) / v;
            const CT s = h[0] * inv_v, s2 = inv_v * inv_v;
            const bool solve = inside && v >= CT(2.220446e-11);   // isOccupied(): velocity < COMP_MARGIN
            bool capped = true;
            for (int it = 0; it < 48; it++) {
                TT n[3];
                n[0] = tmin(box[me - 1], box[me + 1]);
                n[1] = tmin(box[me - 6], box[me + 6]);
                n[2] = tmin(box[me - 36], box[me + 36]);
                const TT lo = tmin(n[0], n[1]), hi = tmax(n[0], n[1]);
                const TT t0 = tmin(lo, n[2]);
                TT u = TINF;
                if (solve && t0 < t) {
                    const TT t1 = tmax(lo, tmin(hi, n[2])), t2 = tmax(hi, n[2]);
                    // times relative to t0 in CT; absent neighbours stay INF
                    const CT d1 = (CT)(t1 - t0), d2 = (CT)(t2 - t0);
                    const CT du = ISO ? update_iso<CT>(d1, d2, s)
                                      : update_aniso<TT, CT>(n, t0, d1, d2, h, al, ra, inv_v, s2);
                    u = t0 + (TT)du;
                }
                const bool better = u < t;
                const bool sig = better && (u < t - thr * t || t == TINF);
                if (better) t = u;
                __syncthreads();
                box[me] = t;
                __syncthreads();
                if (__ballot(sig) == 0ull) { capped = false; break; }
            }
            const bool changed = t < t_in && (t < t_in - thr * t_in || t_in == TINF);
            if (inside && t < t_in) T[((size_t)tile << 6) + lane] = t;
            if (__ballot(changed) || capped) {
                // key of a tile this visit activates: the smallest time that does
                if (changed) {
                    const uint32_t kb = fbits((float)t);
                    if (lx == 0 && t < box[me - 1]) atomicMin(&fkey[0], kb);
                    if (lx == 3 && t < box[me + 1]) atomicMin(&fkey[1], kb);
                    if (ly == 0 && t < box[me - 6]) atomicMin(&fkey[2], kb);
                    if (ly == 3 && t < box[me + 6]) atomicMin(&fkey[3], kb);
                    if (lz == 0 && t < box[me - 36]) atomicMin(&fkey[4], kb);
                    if (lz == 3 && t < box[me + 36]) atomicMin(&fkey[5], kb);
                }
                __syncthreads();
                bool act = false;
                uint32_t nkey = 0, kbits = 0xffffffffu;
                if (lane < 6) {
                    kbits = fkey[lane];
                    act = kbits != 0xffffffffu && ((nbr >> lane) & 1);
                    nkey = (uint32_t)((int)key + toff[lane]);
                }
                if (capped) {
                    const uint32_t own = wave_min_u(inside ? fbits((float)t) : 0xffffffffu);
                    if (lane == 6) { nkey = key; act = true; kbits = own; }
                }
                if (act) {
                    fnxt[nkey] = 1;
                    atomicMin(&knxt[nkey], kbits);
                }
                if (__ballot(act) != 0ull && lane == 0) *any_next = 1u;
            }
            __syncthreads();
        }
    }
}

// The mixed-order update's parallel fixed point (mct_body_set_order1 "parallel"),
// on the same tiles and schedule; a tile's neighbours read two of its layers.
template <class TT, class CT>
__global__ __launch_bounds__(64) void k_eik_round1(mct_eik_problem_set P, int round, double hxd, double hyd,
                                                  double hzd)
{
    __shared__ TT box[512];
    const mct_geom &G = P.G;
    const TT TINF = tinf<TT>();
    const CT CINF = tinf<CT>();
    const int cur = round & 1, nxt = cur ^ 1;
    const int lane = threadIdx.x;
    const int lx = lane & 3, ly = (lane >> 2) & 3, lz = lane >> 4;
    const CT h[3] = {(CT)hxd, (CT)hyd, (CT)hzd};
    const CT ih2[3] = {CT(1) / (h[0] * h[0]), CT(1) / (h[1] * h[1]), CT(1) / (h[2] * h[2])};
    if (blockIdx.x == 0 && lane == 0) P.any[(round + 2) % 3] = 0u;   // flag of round r+2
    const uint32_t ntiles = (uint32_t)G.ntiles;
    const uint32_t nkeys = (uint32_t)P.nprob * ntiles;
    const uint32_t stride = gridDim.x;
    uint8_t *fcur = P.flags[cur], *fnxt = P.flags[nxt];
    uint32_t *kcur = P.key[cur], *knxt = P.key[nxt];
    unsigned int *any_next = &P.any[(round + 1) % 3];
    const bool banded = round < P.band_rounds;
    // Relative change that counts.  In the FP64 mode every decrease counts, so
    // the rounds end only at the update's fixed point, whatever order the tiles
    // ran in (a batch gives each chain the times its own call gives); with FP32
    // increments a change is at least an FP32 step of the increment anyway.
    const TT thr = sizeof(CT) == 8 ? (TT)0 : sizeof(TT) == 8 ? (TT)1e-9 : (TT)1e-7;
    TT *Tall = (TT *)P.T;
    // face lane masks (bit l = lane l): the layers a neighbour reads as halo
    const int deep = 1;
    uint64_t fm_mine = 0;
    for (int l = 0; l < 64; l++) {
        int ax = l & 3, ay = (l >> 2) & 3, az = l >> 4, f = lane;
        bool in = (f == 0 && ax <= deep) || (f == 1 && ax >= 3 - deep) || (f == 2 && ay <= deep) ||
                  (f == 3 && ay >= 3 - deep) || (f == 4 && az <= deep) || (f == 5 && az >= 3 - deep);
        if (in) fm_mine |= 1ull << l;
    }

    // Keys are visited lane-strided: block b, pass i covers keys
    // b + stride*(64*i + lane), so every key has exactly one owner.
    for (uint32_t base = blockIdx.x; base < nkeys; base += stride * 64u) {
        const uint32_t mykey = base + stride * (uint32_t)lane;
        uint8_t f = mykey < nkeys ? fcur[mykey] : 0;
        bool due = false;
        if (f) {
            fcur[mykey] = 0;                       // consumed
            uint32_t kc = kcur[mykey];
            kcur[mykey] = 0xffffffffu;
            const uint32_t prob = mykey / ntiles;
            const float tau = banded ? (float)(round + 1) * P.band_h / P.vmax[prob / (uint32_t)P.nsrc_eff]
                                     : __builtin_huge_valf();
            if (__uint_as_float(kc) <= tau || kc == 0xffffffffu) {
                due = true;
            } else {                               // not yet: carry to the next round
                fnxt[mykey] = 1;
                atomicMin(&knxt[mykey], kc);
                *any_next = 1u;
            }
        }
        uint64_t todo = __ballot(due);
        while (todo) {
            const int src_lane = __ffsll((unsigned long long)todo) - 1;
            todo &= todo - 1;
            const uint32_t key = base + stride * (uint32_t)src_lane;
            const uint32_t prob = key / ntiles;
            const uint32_t tile = key - prob * ntiles;
            const int tx = (int)(tile % (uint32_t)G.ntx);
            const int tyz = (int)(tile / (uint32_t)G.ntx);
            const int ty = tyz % G.nty, tz = tyz / G.nty;
            const int gx = tx * 4 + lx, gy = ty * 4 + ly, gz = tz * 4 + lz;
            const bool inside = gx < G.nx && gy < G.ny && gz < G.nz;
            TT *T = Tall + (size_t)prob * ((size_t)ntiles << 6);
            const uint32_t cw = prob / (uint32_t)P.nsrc_eff;
            const size_t vi = (size_t)cw * ((size_t)ntiles << 6) + ((size_t)tile << 6) + lane;
            const CT v = sizeof(CT) == 8 ? (CT)P.vel64[vi] : (CT)P.vel[vi];
            TT t = inside ? T[((size_t)tile << 6) + lane] : TINF;
            const TT t_in = t;
            box[BX(lx, ly, lz)] = t;
            // face halo: 6 faces x 2 layers x 16 nodes = 192 values, 3 per lane
            for (int r = 0; r < 3; r++) {
                int q = lane + 64 * r;
                int face = q >> 5, layer = (q >> 4) & 1, a = q & 3, b = (q >> 2) & 3;
                int ox, oy, oz;
                int dep = -1 - layer;
                switch (face) {
                    case 0: ox = dep; oy = a; oz = b; break;          // -x
                    case 1: ox = 3 - dep; oy = a; oz = b; break;      // +x
                    case 2: ox = a; oy = dep; oz = b; break;          // -y
                    case 3: ox = a; oy = 3 - dep; oz = b; break;      // +y
                    case 4: ox = a; oy = b; oz = dep; break;          // -z
                    default: ox = a; oy = b; oz = 3 - dep; break;     // +z
                }
                int nxg = tx * 4 + ox, nyg = ty * 4 + oy, nzg = tz * 4 + oz;
                TT hv = TINF;
                if (nxg >= 0 && nyg >= 0 && nzg >= 0 && nxg < G.nx &&
                    nyg < G.ny && nzg < G.nz)
                    hv = T[tl_index(G, nxg, nyg, nzg)];
                box[BX(ox, oy, oz)] = hv;
            }
            __syncthreads();
            const CT inv_v = CT(1) / v;
            const CT s2 = inv_v * inv_v;
            const bool solve = inside && v >= CT(2.220446e-11);   // isOccupied(): velocity < COMP_MARGIN
            const int me = BX(lx, ly, lz);
            const int st[3] = {1, 8, 64};
            bool capped = true;
            for (int it = 0; it < 48; it++) {
                TT n1[3], n2[3];
                TT t0 = TINF;
                for (int d = 0; d < 3; d++) {
                    TT a1 = box[me - st[d]], b1 = box[me + st[d]];
                    bool useb = b1 < a1;
                    n1[d] = useb ? b1 : a1;
                    TT two = useb ? box[me + 2 * st[d]] : box[me - 2 * st[d]];
                    n2[d] = (n1[d] < TINF && two <= n1[d]) ? two : TINF;
                    t0 = n1[d] < t0 ? n1[d] : t0;
                }
                TT u = TINF;
                if (solve && t0 < t) {
                    // times relative to t0 in CT; excluded/absent neighbours stay INF
                    CT m1[3], m2[3];
                    const CT fself = t < TINF ? (CT)(t - t0) : CINF;
                    for (int d = 0; d < 3; d++) {
                        m1[d] = n1[d] < TINF ? (CT)(n1[d] - t0) : CINF;
                        m2[d] = n2[d] < TINF ? (CT)(n2[d] - t0) : CINF;
                    }
                    CT du = update_order1<CT>(m1, m2, fself, h, ih2, inv_v, s2);
                    if (du < CINF) u = t0 + (TT)du;
                }
                bool better = u < t;
                bool sig = better && (u < t - thr * t || t == TINF);
                if (better) t = u;
                __syncthreads();
                box[me] = t;
                __syncthreads();
                if (__ballot(sig) == 0ull) { capped = false; break; }
            }
            const bool changed = t < t_in && (t < t_in - thr * t_in || t_in == TINF);
            if (inside && t < t_in) T[((size_t)tile << 6) + lane] = t;
            const uint64_t bal = __ballot(changed);
            if (bal || capped) {
                // key of the tiles this visit activates: the smallest changed time
                const float kmin = wave_min(changed ? (float)t : __builtin_huge_valf());
                const float kown = wave_min(inside ? (float)t : __builtin_huge_valf());
                bool act = false;
                uint32_t nkey = 0;
                uint32_t kbits = fbits(kmin);
                if (lane < 6 && (bal & fm_mine)) {
                    int ax = tx + (lane == 0 ? -1 : lane == 1 ? 1 : 0);
                    int ay = ty + (lane == 2 ? -1 : lane == 3 ? 1 : 0);
                    int az = tz + (lane == 4 ? -1 : lane == 5 ? 1 : 0);
                    if (ax >= 0 && ay >= 0 && az >= 0 && ax < G.ntx && ay < G.nty && az < G.ntz) {
                        nkey = prob * ntiles + (uint32_t)((az * G.nty + ay) * G.ntx + ax);
                        act = true;
                    }
                }
                if (lane == 6 && capped) { nkey = key; act = true; kbits = fbits(kown); }
                if (act) {
                    fnxt[nkey] = 1;
                    atomicMin(&knxt[nkey], kbits);
                }
                if (__ballot(act) != 0ull && lane == 0) *any_next = 1u;
            }
            __syncthreads();
        }
    }
}

int mct_launch_eik_init(const mct_eik_problem_set &P, const double *src_pts, int src_stride,
                        long src_chain_stride, double xmin, double ymin, double zmin,
                        double lx, double ly, double lz, hipStream_t s)
{
    long n = (long)P.nprob * P.G.ntiles * MCT_TILE_N;
    long nf = (long)P.nprob * P.G.ntiles;
    if (P.t64) hipLaunchKernelGGL(k_eik_clear<double>, dim3(4096), dim3(256), 0, s, (double *)P.T, n);
    else hipLaunchKernelGGL(k_eik_clear<float>, dim3(4096), dim3(256), 0, s, (float *)P.T, n);
    MCT_CHECK(hipGetLastError());
    MCT_CHECK(hipMemsetAsync(P.flags[0], 0, (size_t)((nf + 3) & ~3L), s));
    MCT_CHECK(hipMemsetAsync(P.flags[1], 0, (size_t)((nf + 3) & ~3L), s));
    MCT_CHECK(hipMemsetAsync(P.any, 0, 3 * sizeof(uint32_t), s));
    MCT_CHECK(hipMemsetAsync(P.key[0], 0xff, sizeof(uint32_t) * nf, s));
    MCT_CHECK(hipMemsetAsync(P.key[1], 0xff, sizeof(uint32_t) * nf, s));
    if (P.t64)
        hipLaunchKernelGGL(k_eik_init<double>, dim3((P.nprob + 63) / 64), dim3(64), 0, s, P, src_pts,
                           src_stride, src_chain_stride, xmin, ymin, zmin, lx, ly, lz);
    else
        hipLaunchKernelGGL(k_eik_init<float>, dim3((P.nprob + 63) / 64), dim3(64), 0, s, P, src_pts,
                           src_stride, src_chain_stride, xmin, ymin, zmin, lx, ly, lz);
    MCT_CHECK(hipGetLastError());
    return MCT_OK;
}

int mct_launch_eik_round(const mct_eik_problem_set &P, int round, double hx, double hy, double hz,
                         int grid_blocks, hipStream_t s)
{
    dim3 g(grid_blocks), b(64);
    const bool iso = hx == hy && hx == hz;
#define EIK_LAUNCH(TT, CT)                                                                                             \
    do {                                                                                                               \
        if (P.order == 1) hipLaunchKernelGGL((k_eik_round1<TT, CT>), g, b, 0, s, P, round, hx, hy, hz);                \
        else if (iso) hipLaunchKernelGGL((k_eik_round0<1, TT, CT>), g, b, 0, s, P, round, hx, hy, hz);                 \
        else hipLaunchKernelGGL((k_eik_round0<0, TT, CT>), g, b, 0, s, P, round, hx, hy, hz);                          \
    } while (0)
    if (P.vel64) {   // FP64 velocities and local solves (arrival times FP64 too)
        if (!P.t64) return MCT_ERR_ARG;
        EIK_LAUNCH(double, double);
    } else if (P.t64) {
        EIK_LAUNCH(double, float);
    } else {
        EIK_LAUNCH(float, float);
    }
#undef EIK_LAUNCH
    MCT_CHECK(hipGetLastError());
    return MCT_OK;
}

// Largest velocity per (chain, wave), for the band schedule: the front needs
// band_h / vmax to cross the tiles a round advances by.  Positive floats order as
// their bits; the blocks of one grid meet in an atomic maximum (a single block
// took 1.0 ms at 101^3, 64 take 0.02).
template <class VT>
__global__ __launch_bounds__(256) void k_vmax(const VT *vel, long tsz, uint32_t *vmax)
{
    __shared__ float sm[4];
    const int cw = blockIdx.x;
    const VT *V = vel + (long)cw * tsz;
    float m = 0.f;
    for (long i = (long)blockIdx.y * 256 + threadIdx.x; i < tsz; i += (long)gridDim.y * 256) m = fmaxf(m, (float)V[i]);
    for (int o = 32; o > 0; o >>= 1) m = fmaxf(m, __shfl_xor(m, o, 64));
    if ((threadIdx.x & 63) == 0) sm[threadIdx.x >> 6] = m;
    __syncthreads();
    if (threadIdx.x == 0) atomicMax(&vmax[cw], fbits(fmaxf(fmaxf(sm[0], sm[1]), fmaxf(sm[2], sm[3]))));
}

int mct_launch_vmax(const float *vel, const double *vel64, long tsz, int ncw, float *vmax, hipStream_t s)
{
    int rc = mct_fill_i32((int32_t *)vmax, ncw, 0, s);
    if (rc) return rc;
    const long per = (tsz + 256 * 16 - 1) / (256 * 16);       // 16 values a thread
    const dim3 g((unsigned)ncw, (unsigned)(per < 64 ? per : 64));
    if (vel64) hipLaunchKernelGGL(k_vmax<double>, g, dim3(256), 0, s, vel64, tsz, (uint32_t *)vmax);
    else hipLaunchKernelGGL(k_vmax<float>, g, dim3(256), 0, s, vel, tsz, (uint32_t *)vmax);
    MCT_CHECK(hipGetLastError());
    return MCT_OK;
}

float mct_band_tiles(float set, int order, long tiles)
{
    if (set > 0.f) return set;
    const char *e = getenv("MCT_BAND_TILES");
    const float v = e ? (float)atof(e) : 0.f;
    if (v > 0.f) return v;
    // A narrow band visits a tile less often, a wide one needs fewer rounds.  A
    // round costs about 10 us however little it holds, a visit 2 ns of the full
    // card, and the visits per tile grow by about 3.2 times the band's width, so
    // the sum is smallest near sqrt(8e4 / tiles).  Measured at 101^3, 16 chains
    // (14 M tiles): 78 ms at 0.25, 103 at 0.5, 171 at 0.75; one chain (0.88 M):
    // 9.9 ms at 0.35, 10.7 at 0.5; one source at 83 x 71 x 61 (6 k): 1.13 ms at
    // 0.5, 1.05 at 0.75.  (The mixed-order fixed point keeps its 0.5.)
    if (order == 1) return 0.5f;
    const float w = sqrtf(8e4f / (float)(tiles > 1 ? tiles : 1));
    return w < 0.25f ? 0.25f : (w > 0.75f ? 0.75f : w);
}

int mct_default_f64()
{
    const char *e = getenv("MCT_EIK_F64");
    return e ? (atoi(e) != 0) : 1;
}

int mct_default_t64()
{
    const char *e = getenv("MCT_EIK_F32");
    return (e && atoi(e) == 1) ? 0 : 1;
}
