// sfmm.hip -- exact 3-D first-arrival traveltimes: the SFMM heap loop of
// fastMarching3D replayed step for step, one wave per problem.
//
// fastMarching3D (fastmarching/fastMarching.cpp:26-129) runs
// FMM::computeInternal (fmm/fmm.hpp:92-158) over SFMM's queue (fmm/sfmm.hpp
// :44-52, fmm/fmdata/fmpriorityqueue.hpp:27-86): a binary heap of cells whose
// keys are read live from the cells (FMCompare, fmm/fmdata/fmcompare.hpp
// :29-32); a cell is pushed again on every improvement and its older entries
// stay in the heap.  With the mixed-order update (highAccuracySolveEikonal,
// fmm/eikonalsolver.hpp:83-145) a cell's time depends on the values its
// neighbours held when each of them was popped, so the times are a function
// of the pop order, not of the field alone.  The only way to reproduce them is
// to replay the heap: the same pushes, the same sift steps (GCC libstdc++
// push_heap / pop_heap: the hole is moved down to a leaf, then val sifts up),
// and the same local solves in FP64 in the reference's operation order
// (contraction off).
//
// One wave runs one problem: the replay stays sequential, the lanes carry the
// memory traffic.  A pop reads the five-level subtree under the hole (62
// entries, then their live keys) in two round trips and walks it with lane
// reads; the val sift-up that ends a pop needs no loads (its comparisons are
// against the entries just walked).  A push reads every ancestor of its slot
// at once.  The six neighbours of a popped cell are solved by six lanes; only
// the plus neighbour of a dimension reads a value the minus neighbour may
// have just changed (its two-away cell), so the plus lanes solve again after
// the minus lanes' updates.  Frozen cells keep their time with the sign bit
// set (times are never negative): a neighbour's state and value arrive in one
// load, the keys are |t|, and a last pass clears the bit.
#include "mct_internal.h"
#include <float.h>
#include <stdlib.h>
#include <string.h>

#pragma clang fp contract(off)

#define SF_MARGIN (DBL_EPSILON * 1e5)     // utils::COMP_MARGIN (utils/utils.h:27)
#define SF_LEVELS 5                       // subtree levels read per sift-down block

enum { SF_ERR_HEAP = 1u, SF_ERR_POPS = 2u, SF_ERR_OPEN_INF = 4u };

namespace {

__device__ __forceinline__ double sf_inf() { return __builtin_huge_val(); }

__device__ __forceinline__ double rl_d(double v, int l)
{
    const unsigned long long b = (unsigned long long)__double_as_longlong(v);
    const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)(b & 0xffffffffull), l);
    const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)(b >> 32), l);
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

__device__ __forceinline__ uint32_t rl_u(uint32_t v, int l)
{
    return (uint32_t)__builtin_amdgcn_readlane((int)v, l);
}

__device__ __forceinline__ uint32_t first_u(uint32_t v) { return (uint32_t)__builtin_amdgcn_readfirstlane((int)v); }

__device__ __forceinline__ double first_d(double v) { return rl_d(v, 0); }

// Lanes of one wave read what other lanes of it wrote: order the accesses.
__device__ __forceinline__ void wave_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

__device__ __forceinline__ long sf_index(const mct_geom &G, int x, int y, int z)
{
    const int tile = ((z >> 2) * G.nty + (y >> 2)) * G.ntx + (x >> 2);
    const int ln = ((z & 3) << 4) | ((y & 3) << 2) | (x & 3);
    return ((long)tile << 6) | ln;
}

// The cell, its velocity and, per dimension, the times one and two cells away
// on the minus and plus sides (|t|; `h*` says the cell exists).
struct sf_stencil {
    double tself, vel;
    double m1[3], m2[3], p1[3], p2[3];
    bool hm1[3], hm2[3], hp1[3], hp2[3];
};

// Stable sort of three (t1, t2, h) triples by t1 (std::sort on <= 16
// elements is an insertion sort: equal keys keep their order).  Absent
// dimensions carry t1 = +inf and end up last.
__device__ __forceinline__ void sf_cas(double &a1, double &a2, double &ah, double &b1, double &b2, double &bh)
{
    const bool sw = b1 < a1;
    const double x1 = sw ? b1 : a1, x2 = sw ? b2 : a2, xh = sw ? bh : ah;
    b1 = sw ? a1 : b1; b2 = sw ? a2 : b2; bh = sw ? ah : bh;
    a1 = x1; a2 = x2; ah = xh;
}

__device__ __forceinline__ void sf_sort3(double t1[3], double t2[3], double hh[3])
{
    sf_cas(t1[0], t2[0], hh[0], t1[1], t2[1], hh[1]);
    sf_cas(t1[1], t2[1], hh[1], t1[2], t2[2], hh[2]);
    sf_cas(t1[0], t2[0], hh[0], t1[1], t2[1], hh[1]);
}

// solveEikonalNDims (eikonalsolver.hpp:292-322) over the first `dims` entries
__device__ __forceinline__ double sf_nd1(const double t1[3], const double hh[3], int dims, double vel)
{
    if (dims == 1) return t1[0] + hh[0] / vel;
    double a = 0.0, b = 0.0, c = -1.0 / (vel * vel);
#pragma unroll
    for (int i = 0; i < 3; i++) {
        if (i < dims) {
            const double alpha = 1.0 / (hh[i] * hh[i]);
            c += t1[i] * t1[i] * alpha;
            b += -2.0 * t1[i] * alpha;
            a += alpha;
        }
    }
    const double q = b * b - 4 * a * c;
    if (q < 0) return sf_inf();
    return (-b + sqrt(q)) / (2 * a);
}

// highAccuracySolveEikonalNDims (eikonalsolver.hpp:326-368)
__device__ __forceinline__ double sf_nd2(const double t1[3], const double t2[3], const double hh[3], int dims,
                                         double vel)
{
    if (dims == 1) return t1[0] + hh[0] / vel;
    double a = 0.0, b = 0.0, c = -1.0 / (vel * vel);
#pragma unroll
    for (int i = 0; i < 3; i++) {
        if (i < dims) {
            if (!__builtin_isinf(t2[i])) {
                const double alpha = 9.0 / 4.0 / (hh[i] * hh[i]);
                const double t = (4.0 * t1[i] - t2[i]) / 3.0;
                c += t * t * alpha;
                b += -2.0 * t * alpha;
                a += alpha;
            } else if (t1[i] < DBL_MAX) {
                const double alpha = 1.0 / (hh[i] * hh[i]);
                c += t1[i] * t1[i] * alpha;
                b += -2.0 * t1[i] * alpha;
                a += alpha;
            }
        }
    }
    const double q = b * b - 4 * a * c;
    if (q < 0) return sf_inf();
    return (-b + sqrt(q)) / (2 * a);
}

// solveEikonal (eikonalsolver.hpp:50-79): per dimension the smaller of the
// two neighbours, kept when finite and below the cell's own time; dimensions
// are added in time order until one more would not lower the result.
__device__ __forceinline__ double sf_solve1(const sf_stencil &S, const double leaf[3])
{
    double t1[3], t2[3], hh[3];
    int a = 0;
#pragma unroll
    for (int d = 0; d < 3; d++) {
        const double m = (S.hm1[d] && S.hp1[d]) ? (S.m1[d] < S.p1[d] ? S.m1[d] : S.p1[d])
                                                : (S.hm1[d] ? S.m1[d] : S.p1[d]);
        const bool in = !__builtin_isinf(m) && m < S.tself;
        t1[d] = in ? m : sf_inf();
        t2[d] = sf_inf();
        hh[d] = leaf[d];
        a += in ? 1 : 0;
    }
    if (a == 0) return sf_inf();
    sf_sort3(t1, t2, hh);
    double up = sf_inf();
#pragma unroll
    for (int i = 1; i <= 3; i++) {
        if (i <= a) {
            up = sf_nd1(t1, hh, i, S.vel);
            if (i == a || (up - t1[i < 3 ? i : 2]) < SF_MARGIN) break;
        }
    }
    return up;
}

// highAccuracySolveEikonal (eikonalsolver.hpp:83-145): per dimension the
// smaller one-away time, with the two-away time behind it when that is
// finite and not larger; the widest stencil whose root lies above its
// largest neighbour time (by COMP_MARGIN) wins.
__device__ __forceinline__ double sf_solve2(const sf_stencil &S, const double leaf[3])
{
    double t1[3], t2[3], hh[3];
    int a = 0;
#pragma unroll
    for (int d = 0; d < 3; d++) {
        double minT = DBL_MAX, minT2 = DBL_MAX;
        if (S.hm1[d]) {
            const double tv = S.m1[d];
            if (!__builtin_isinf(tv) && tv < minT) {
                minT = tv;
                minT2 = DBL_MAX;
                if (S.hm2[d]) {
                    const double tv2 = S.m2[d];
                    if (!__builtin_isinf(tv2) && tv2 <= tv) minT2 = tv2;
                }
            }
        }
        if (S.hp1[d]) {
            const double tv = S.p1[d];
            if (!__builtin_isinf(tv) && tv < minT) {
                minT = tv;
                minT2 = DBL_MAX;
                if (S.hp2[d]) {
                    const double tv2 = S.p2[d];
                    if (!__builtin_isinf(tv2) && tv2 <= tv) minT2 = tv2;
                }
            }
        }
        const bool in = minT < DBL_MAX && minT < S.tself;
        t1[d] = in ? minT : sf_inf();
        t2[d] = (in && minT2 < DBL_MAX) ? minT2 : sf_inf();
        hh[d] = leaf[d];
        a += in ? 1 : 0;
    }
    if (a == 0) return S.tself;
    sf_sort3(t1, t2, hh);
#pragma unroll
    for (int i = 3; i >= 1; i--) {
        if (i <= a) {
            const double cur = sf_nd2(t1, t2, hh, i, S.vel);
            if (!__builtin_isinf(cur) && (cur - t1[i - 1]) > SF_MARGIN) return cur;
        }
    }
    return sf_inf();
}

// the replay of one problem by a wave, its heap in global memory
template <int HIGH>
__device__ __forceinline__ void sf_replay(const mct_sfmm_args &A, int prob)
{
    const int lane = threadIdx.x;
    const mct_geom G = A.G;
    const long tsz = (long)G.ntiles * MCT_TILE_N;
    const int si = prob % A.nsrc_eff, cw = prob / A.nsrc_eff, ch = cw / A.nwave;
    double *T = A.T + (long)prob * tsz;
    const double *V = A.V + (long)cw * tsz;
    uint32_t *H = A.heap + (long)prob * A.hcap;
    const double leaf[3] = {A.lx, A.ly, A.lz};
    const int dims[3] = {G.nx, G.ny, G.nz};
    uint32_t err = 0;

    // ---- Solver::setInitialPoints (fmm/solver.hpp:72-92): the eight corner
    // cells of the source's grid cell get dist * 2 / (v_source + v_corner),
    // v_source trilinear with clamped corners (ndgridmap.hpp:158-191,433-489),
    // and are pushed in corner order.
    const double *sp0 = A.src + (long)ch * A.src_chain_stride + (long)si * A.src_stride;
    const double p[3] = {sp0[0] - A.xmin, sp0[1] - A.ymin, sp0[2] - A.zmin};
    int pc[3];
#pragma unroll
    for (int d = 0; d < 3; d++) {
        const double qd = p[d] / leaf[d];
        pc[d] = !(qd >= 1.0) ? 0 : (qd >= (double)dims[d] ? dims[d] - 1 : (int)qd);
    }
    uint32_t cq[8];
    double vn[8];
    int cc[8][3];
#pragma unroll
    for (int v = 0; v < 8; v++) {
#pragma unroll
        for (int d = 0; d < 3; d++) {
            int c = pc[d] + ((v >> (2 - d)) & 1);
            cc[v][d] = c >= dims[d] ? dims[d] - 1 : c;
        }
        cq[v] = (uint32_t)sf_index(G, cc[v][0], cc[v][1], cc[v][2]);
        vn[v] = V[cq[v]];
    }
    double vs = 0.0;
#pragma unroll
    for (int v = 0; v < 8; v++) {
        double w = 1.0;
#pragma unroll
        for (int d = 0; d < 3; d++) {
            const double sd = p[d] - leaf[d] * pc[d];
            const double wj = fabs((double)(cc[v][d] - pc[d]) * leaf[d] - leaf[d] + sd);
            w = w * wj / leaf[d];
        }
        vs = vs + w * vn[v];
    }
    if (lane == 0) {
#pragma unroll
        for (int v = 0; v < 8; v++) {
            double dist = 0.0;
#pragma unroll
            for (int d = 0; d < 3; d++) {
                const double xi = (cc[v][d] * leaf[d] - p[d]) * (cc[v][d] * leaf[d] - p[d]);
                dist = dist + xi;
            }
            dist = sqrt(dist);
            T[cq[v]] = dist * 2 / (vs + vn[v]);
        }
    }
    wave_sync();

    long hs = 0;
    // push_heap: the new entry sifts up from slot hs.  Lane l (1..m) holds the
    // ancestor l levels up and its live key; the entry stops below the first
    // ancestor whose key is not larger than its own.  Loads are unconditional
    // (inactive lanes read slot 0 and cell 0) so they issue together.
    auto push = [&](uint32_t cell, double kc) -> bool {
        if (hs >= A.hcap) return false;
        const unsigned long long k1 = (unsigned long long)hs + 1ull;
        hs = hs + 1;
        const int m = 63 - __builtin_clzll(k1);
        const bool act = lane >= 1 && lane <= m;
        const unsigned long long slot = act ? (k1 >> lane) - 1ull : 0ull;
        const uint32_t e = act ? H[slot] : 0u;
        const double ke = fabs(T[e]);
        const unsigned long long stop = __ballot(act && !(ke > kc));
        const int ls = stop ? __builtin_ctzll(stop) : m + 1;
        if (lane >= 1 && lane < ls) H[(k1 >> (lane - 1)) - 1] = e;
        if (lane == 0) H[(k1 >> (ls - 1)) - 1] = cell;
        wave_sync();
        return true;
    };

    for (int v = 0; v < 8 && !err; v++) {
        const double kc = first_d(fabs(T[cq[v]]));
        if (!push(cq[v], kc)) err |= SF_ERR_HEAP;
    }

    // lanes 0..61 of a sift-down block: level lv (1..5) and offset under the hole
    const int lv = 31 - __builtin_clz((unsigned)lane + 2u);
    const int off = lane + 2 - (1 << lv);
    // lanes 0..5: neighbour s = 2*dim + side of a popped cell (fmm.hpp:117-120,
    // ndgridmap.hpp:158-191: x-, x+, y-, y+, z-, z+)
    const int ndim = lane >> 1;
    const int nstep = (lane & 1) ? 1 : -1;

    const long max_pops = 64L * (long)G.nx * G.ny * G.nz + 64;
    long pops = 0;
    while (hs > 0 && !err) {
        if (++pops > max_pops) { err |= SF_ERR_POPS; break; }
        // ---- pop_heap (libstdc++ __pop_heap / __adjust_heap).  First round
        // trip: the root, the last entry and the subtree block under the root.
        const long n = hs - 1;
        hs = n;
        long idx = (1L << lv) - 1 + off;
        bool ok = lane < 62 && idx < n;
        const uint32_t h0 = H[0];
        const uint32_t hn = H[n];
        uint32_t e = H[ok ? idx : 0];
        __builtin_amdgcn_sched_barrier(0);
        const uint32_t top = first_u(h0);
        const uint32_t val = first_u(hn);
        // Second round trip: the block's live keys, the popped cell, val's key
        // and the neighbours' stencils (cells off the grid read the cell itself),
        // issued in that order so that the walk waits for the keys alone.
        const double k0 = T[e];
        const double ttop_v = T[top];
        const double kval_v = T[val];
        __builtin_amdgcn_sched_barrier(0);
        const int tile = (int)(top >> 6), tl = (int)(top & 63u);
        const int tx = tile % G.ntx, tyz = tile / G.ntx;
        const int ty = tyz % G.nty, tz = tyz / G.nty;
        const int cx = tx * 4 + (tl & 3), cy = ty * 4 + ((tl >> 2) & 3), cz = tz * 4 + (tl >> 4);
        int jc[3] = {cx, cy, cz};
#pragma unroll
        for (int d = 0; d < 3; d++) jc[d] += (d == ndim) ? nstep : 0;
        const int jn = ndim == 0 ? jc[0] : (ndim == 1 ? jc[1] : jc[2]);
        const int dn = ndim == 0 ? dims[0] : (ndim == 1 ? dims[1] : dims[2]);
        const bool nvalid = lane < 6 && jn >= 0 && jn < dn;
        if (!nvalid) { jc[0] = cx; jc[1] = cy; jc[2] = cz; }
        sf_stencil S;
        const uint32_t jq = (uint32_t)sf_index(G, jc[0], jc[1], jc[2]);
        const double traw = T[jq];
        S.vel = V[jq];
#pragma unroll
        for (int d = 0; d < 3; d++) {
            S.hm1[d] = jc[d] >= 1; S.hm2[d] = jc[d] >= 2;
            S.hp1[d] = jc[d] <= dims[d] - 2; S.hp2[d] = jc[d] <= dims[d] - 3;
            int c[3] = {jc[0], jc[1], jc[2]};
            c[d] = S.hm1[d] ? jc[d] - 1 : jc[d]; S.m1[d] = T[sf_index(G, c[0], c[1], c[2])];
            c[d] = S.hm2[d] ? jc[d] - 2 : jc[d]; S.m2[d] = T[sf_index(G, c[0], c[1], c[2])];
            c[d] = S.hp1[d] ? jc[d] + 1 : jc[d]; S.p1[d] = T[sf_index(G, c[0], c[1], c[2])];
            c[d] = S.hp2[d] ? jc[d] + 2 : jc[d]; S.p2[d] = T[sf_index(G, c[0], c[1], c[2])];
        }
        __builtin_amdgcn_sched_barrier(0);
        {
            // (with n = 0 the walk is empty and val, the popped entry, is
            // written back to the dead slot 0)
            const double kval = first_d(fabs(kval_v));
            double k = fabs(k0);
            const long lim = n > 0 ? (n - 1) / 2 : 0;
            long hole = 0;
            int m = 0;                         // path levels walked
            uint32_t pe = 0;                   // lane l: entry moved up from level l
            double pk = 0.0;                   //          its key
            long pp = 0;                       //          its position
            while (hole < lim) {
                if (!ok) k = 0.0;
                int r = 1;                     // subtree node (root 1, children 2r and 2r+1)
                for (int st = 0; st < SF_LEVELS && hole < lim; st++) {
                    const double kr = rl_d(k, 2 * r - 1), kl = rl_d(k, 2 * r - 2);
                    const bool left = kr > kl;
                    const int pick = left ? 2 * r - 2 : 2 * r - 1;
                    const uint32_t ec = rl_u(e, pick);
                    const long child = 2 * (hole + 1) - (left ? 1 : 0);
                    m++;
                    if (lane == m) { pe = ec; pk = left ? kl : kr; pp = child; }
                    hole = child;
                    r = pick + 2;
                }
                if (hole < lim) {              // the next block, under the new hole
                    idx = ((hole + 1) << lv) - 1 + off;
                    ok = lane < 62 && idx < n;
                    e = H[ok ? idx : 0];
                    k = fabs(T[e]);
                }
            }
            if ((n & 1) == 0 && hole == (n - 2) / 2) {
                const long child = 2 * (hole + 1);
                const uint32_t ec = first_u(H[child - 1]);
                const double kc = first_d(fabs(T[ec]));
                m++;
                if (lane == m) { pe = ec; pk = kc; pp = child - 1; }
                hole = child - 1;
            }
            // __push_heap of val from the leaf hole: it climbs past the path
            // entries whose keys are larger and stops below the first that is
            // not; the entries above that point stay one level up.
            const unsigned long long keep = __ballot(lane >= 1 && lane <= m && !(pk > kval));
            const int js = keep ? 63 - __builtin_clzll(keep) : 0;
            const uint32_t pe_below = (uint32_t)__shfl_down((int)pe, 1, 64);
            if (lane < js) H[pp] = pe_below;
            if (lane == js) H[pp] = val;
        }
        // the popped cell is frozen (fmm.hpp:123)
        if (lane == 0) T[top] = -fabs(ttop_v);
        wave_sync();
        // the stencil values are |t| (frozen cells carry the sign bit)
        S.tself = fabs(traw);
#pragma unroll
        for (int d = 0; d < 3; d++) {
            S.m1[d] = fabs(S.m1[d]); S.m2[d] = fabs(S.m2[d]);
            S.p1[d] = fabs(S.p1[d]); S.p2[d] = fabs(S.p2[d]);
        }

        // ---- neighbour updates (fmm.hpp:124-154)
        const bool live = nvalid && !signbit(traw) && !(S.vel < SF_MARGIN);
        double nt = 0.0;
        bool upd = false;
        if (live) {
            nt = HIGH ? sf_solve2(S, leaf) : sf_solve1(S, leaf);
            upd = nt + SF_MARGIN < S.tself;
        }
        if (HIGH) {
            // the plus neighbour's two-away cell on its minus side is the
            // minus neighbour: solve again with its value after the update
            // (only when that neighbour was updated: otherwise the value the
            // plus lane loaded is already the one the reference reads)
            const double after = upd ? nt : S.tself;
            const double from_minus = __shfl(after, lane - 1 < 0 ? 0 : lane - 1, 64);
            const bool minus_upd = __shfl(upd ? 1 : 0, lane - 1 < 0 ? 0 : lane - 1, 64) != 0;
            const bool hm2n = ndim == 0 ? S.hm2[0] : (ndim == 1 ? S.hm2[1] : S.hm2[2]);
            if (live && (lane & 1) && hm2n && minus_upd) {
#pragma unroll
                for (int d = 0; d < 3; d++)
                    if (d == ndim) S.m2[d] = from_minus;
                nt = sf_solve2(S, leaf);
                upd = nt + SF_MARGIN < S.tself;
            }
        }
        if (__ballot(live && __builtin_isinf(S.tself) && __builtin_isinf(nt))) err |= SF_ERR_OPEN_INF;
        unsigned long long todo = __ballot(upd);
        while (todo && !err) {
            const int s = __builtin_ctzll(todo);
            todo &= todo - 1;
            const uint32_t cell = rl_u(jq, s);
            const double tn = rl_d(nt, s);
            if (lane == 0) T[cell] = tn;
            wave_sync();
            if (!push(cell, tn)) err |= SF_ERR_HEAP;
        }
    }
    err = first_u(err);
    if (A.pops && lane == 0) A.pops[prob] = (uint32_t)(pops > 0xffffffffL ? 0xffffffffL : pops);
    if (err && lane == 0) atomicOr(A.err, err);
}

template <int HIGH>
__global__ __launch_bounds__(64) void k_sfmm(mct_sfmm_args A)
{
    if (A.done && A.done[blockIdx.x]) return;        // solved by k_sfmm_lds
    sf_replay<HIGH>(A, blockIdx.x);
}

// ---- the replay with the heap in LDS ----------------------------------------------
// The same loop for grids whose narrow band fits a compute unit's LDS.  A band cell
// gets a slot; a heap entry is a slot (16 bits), and a table of the slots' live
// keys stands beside the heap, so a comparison is two LDS reads (an entry, its
// key) instead of two trips to L2, and an improvement writes one key that every
// entry of the cell sees.  A slot is kept while entries name it (a count) and then
// returned to a list linked through the free keys.
//
// What bounds it: one wave runs a problem.  At the four cycles that it needs per
// instruction the 690 of a pop are 57 % of its 4,800 cycles, the rest waits for LDS
// and L2 (99.5 % hits).  The grid is laid out
// with its border (two cells of -inf: frozen, and no value to a stencil), x
// fastest, so a neighbour or a stencil cell is a constant away per lane and no
// lane tests coordinates.  Lanes 4n + i take dimension i of neighbour n's stencil and
// the solution over its i + 1 smallest dimensions, so the reference's three
// successive quadratics run side by side.  The path of a pop comes from a ballot
// against each lane's ancestors (five levels a block), not from a walk.
// Measured with 14 problems of 47 x 57 x 41 (122,000 pops each): 2.0 us per pop
// instead of 4.3, 377 VALU and 278 scalar instructions instead of about 980 and 500.
// Cells between the grid's rows and slabs, and slabs before and after it: a border
// neighbour's stencil is read too (and ignored), three slabs from the grid.
#define SFL_PAD 2
#define SFL_SLABS 3

struct sfl_grid {
    int sy, sz;               // strides of y and z (x: 1)
    uint32_t base, n;         // index of cell (0,0,0), cells of a padded grid
};

__host__ __device__ __forceinline__ sfl_grid sfl_layout(const mct_geom &G)
{
    sfl_grid L;
    L.sy = G.nx + SFL_PAD;
    L.sz = L.sy * (G.ny + SFL_PAD);
    L.base = (uint32_t)(SFL_SLABS * (L.sz + L.sy + 1));
    L.n = L.base + (uint32_t)((G.nz + SFL_SLABS) * L.sz);
    return L;
}

// the interior cell of padded index i, if it is one
__device__ __forceinline__ bool sfl_cell(const mct_geom &G, const sfl_grid &L, uint32_t i, int &x, int &y, int &z)
{
    if (i < L.base) return false;
    const uint32_t r = i - L.base;
    z = (int)(r / (uint32_t)L.sz);
    const uint32_t q = r - (uint32_t)z * (uint32_t)L.sz;
    y = (int)(q / (uint32_t)L.sy);
    x = (int)(q - (uint32_t)y * (uint32_t)L.sy);
    return x < G.nx && y < G.ny && z < G.nz;
}

// padded times (+inf inside, -inf on the border) and velocities
__global__ __launch_bounds__(256) void k_sfl_fill(mct_geom G, sfl_grid L, double *T, long nprob)
{
    const uint32_t i = blockIdx.x * 256u + threadIdx.x;
    if (i >= L.n) return;
    int x, y, z;
    const double v = sfl_cell(G, L, i, x, y, z) ? sf_inf() : -sf_inf();
    for (long p = blockIdx.y; p < nprob; p += gridDim.y) T[p * (long)L.n + i] = v;
}

__global__ __launch_bounds__(256) void k_sfl_vel(mct_geom G, sfl_grid L, const double *V, double *VL, long ncw)
{
    const uint32_t i = blockIdx.x * 256u + threadIdx.x;
    if (i >= L.n) return;
    int x, y, z;
    const bool in = sfl_cell(G, L, i, x, y, z);
    const long q = in ? sf_index(G, x, y, z) : 0;
    for (long c = blockIdx.y; c < ncw; c += gridDim.y)
        VL[c * (long)L.n + i] = in ? V[c * (long)G.ntiles * MCT_TILE_N + q] : 0.0;
}

// solved problems' times into the tiles
__global__ __launch_bounds__(256) void k_sfl_tiles(mct_geom G, sfl_grid L, const double *TL, double *T,
                                                   const uint32_t *done, long nprob)
{
    const uint32_t i = blockIdx.x * 256u + threadIdx.x;
    int x, y, z;
    if (i >= L.n || !sfl_cell(G, L, i, x, y, z)) return;
    const long q = sf_index(G, x, y, z);
    for (long p = blockIdx.y; p < nprob; p += gridDim.y)
        if (done[p] == 1u) T[p * (long)G.ntiles * MCT_TILE_N + q] = fabs(TL[p * (long)L.n + i]);
}

// Band cells of a homogeneous medium with the source in cell p when the front has
// radius r / 24 of the way to the farthest corner: per axis, the grid lines that cross
// the front where that axis has the largest share of its normal.  h: spacings (their
// ratios count); the lines are dealt to `lanes` lanes.
#define SFL_RADII 24
__host__ __device__ static int sfl_front(const int n[3], const float h[3], const int p[3], int r, int lane, int lanes)
{
    float far2 = 0.f;
    for (int d = 0; d < 3; d++) {
        const float x = (p[d] > n[d] - 1 - p[d] ? p[d] : n[d] - 1 - p[d]) * h[d];
        far2 += x * x;
    }
    const float t2 = far2 * (float)(r * r) / (float)(SFL_RADII * SFL_RADII);
    int c = 0;
#pragma unroll
    for (int x = 0; x < 3; x++) {
        const int a = x == 0 ? 1 : 0, b = x == 2 ? 1 : 2;
        for (int j = 0; j < n[b]; j++) {
            const float xb = (j - p[b]) * h[b];
            for (int i = lane; i < n[a]; i += lanes) {
                const float xa = (i - p[a]) * h[a], w2 = t2 - xa * xa - xb * xb;
                const float w = sqrtf(w2 > 0.f ? w2 : 0.f), off = w / h[x];
                const bool on = w2 > 0.f && w * h[x] >= fabsf(xa) * h[a] && w * h[x] >= fabsf(xb) * h[b];
                c += on ? (p[x] + off <= n[x] - 1) + (p[x] - off >= 0.f) : 0;
            }
        }
    }
    return c;
}

struct sfl_args {
    mct_sfmm_args A;
    sfl_grid L;
    double *T;                // (nprob, L.n) padded times
    const double *V;          // (chains * waves, L.n) padded velocities
    uint16_t *slot;           // (nprob, L.n) a narrow cell's slot
    uint32_t *done;           // (nprob) 1 when solved with the heap in LDS, 2 in global memory
    int ns, ne;               // slots and heap entries in LDS
    int most;                 // where a wider band is expected (err[2]) all problems are left at once
    int here;                 // problems left later go on in this kernel (all of its problems run at once)
};

// lane i of the quad to all four of its lanes
template <int I>
__device__ __forceinline__ double quad_d(double v)
{
    constexpr int ctrl = I | I << 2 | I << 4 | I << 6;
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_update_dpp((int)b, (int)b, ctrl, 0xf, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp((int)(b >> 32), (int)(b >> 32), ctrl, 0xf, 0xf, false);
    return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}

// the sibling's value: the lane whose index differs in bit 0
__device__ __forceinline__ double swap_d(double v)
{
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_update_dpp((int)b, (int)b, 0xb1, 0xf, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp((int)(b >> 32), (int)(b >> 32), 0xb1, 0xf, 0xf, false);
    return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}

__device__ __forceinline__ double ld_d(const double *p, uint32_t byte) { return *(const double *)((const char *)p + byte); }

// a ballot straight from the comparison's mask (__ballot takes an int: two more
// instructions)
__device__ __forceinline__ unsigned long long ballot(bool p) { return __builtin_amdgcn_ballot_w64(p); }

// Compare-and-swap by t, the earlier one first on equal keys.
__device__ __forceinline__ void sfl_cas(double &t0, double &u0, double &a0, double &t1, double &u1, double &a1)
{
    const bool sw = t1 < t0;
    const double t = sw ? t1 : t0, u = sw ? u1 : u0, a = sw ? a1 : a0;
    t1 = sw ? t0 : t1; u1 = sw ? u0 : u1; a1 = sw ? a0 : a1;
    t0 = t; u0 = u; a0 = a;
}

// highAccuracySolveEikonal (eikonalsolver.hpp:83-145) on the lanes 4n + i of a
// neighbour: m1, m2, p1, p2 the times one and two cells away in dimension i, al1 and
// al2 that dimension's weights of the first- and second-order stencil.  Every lane
// of the quad returns the new time (tself when no dimension counts, +inf when no
// quadratic is accepted).
__device__ __forceinline__ double sfl_solve(int i, double m1, double m2, double p1, double p2, double tself, double vel,
                                            double hx, double hy, double hz, double al1, double al2)
{
    const bool plus = p1 < m1;
    const double one = plus ? p1 : m1, two = plus ? p2 : m2;
    const bool in = one < tself;                      // finite, and below the cell's own
    const bool second = in & (two <= one);
    const double t = in ? one : sf_inf();
    const double u = second ? (4.0 * one - two) / 3.0 : t;
    const double al = second ? al2 : al1;
    double t0 = quad_d<0>(t), t1 = quad_d<1>(t), t2 = quad_d<2>(t);
    double u0 = quad_d<0>(u), u1 = quad_d<1>(u), u2 = quad_d<2>(u);
    double a0 = quad_d<0>(al), a1 = quad_d<1>(al), a2 = quad_d<2>(al);
    // the spacing of the smallest time's dimension
    const double hm = (t0 <= t1) & (t0 <= t2) ? hx : (t1 <= t2 ? hy : hz);
    sfl_cas(t0, u0, a0, t1, u1, a1);
    sfl_cas(t1, u1, a1, t2, u2, a2);
    sfl_cas(t0, u0, a0, t1, u1, a1);
    // highAccuracySolveEikonalNDims (:326-368) over the first i + 1 entries
    double c = -1.0 / (vel * vel), b = 0.0, a = 0.0;
    c += u0 * u0 * a0; b += -2.0 * u0 * a0; a += a0;
    c += u1 * u1 * a1; b += -2.0 * u1 * a1; a += a1;
    const double c3 = c + u2 * u2 * a2, b3 = b + -2.0 * u2 * a2, a3 = a + a2;
    const bool three = i == 2;
    c = three ? c3 : c; b = three ? b3 : b; a = three ? a3 : a;
    const double q = b * b - 4 * a * c;
    const double root = (-b + sqrt(q)) / (2 * a);     // q < 0: a NaN, which no test below accepts
    const double cand = i == 0 ? t0 + hm / vel : root;
    const double last = i == 0 ? t0 : (i == 1 ? t1 : t2);
    // counted (its last dimension is in), finite, and above its last time
    const bool ok = (last < sf_inf()) & (cand < sf_inf()) & ((cand - last) > SF_MARGIN);
    const double r = ok ? cand : sf_inf();
    const double r0 = quad_d<0>(r), r1 = quad_d<1>(r), r2 = quad_d<2>(r);
    const double best = r2 < sf_inf() ? r2 : (r1 < sf_inf() ? r1 : r0);
    return t0 < sf_inf() ? best : tself;
}

// The widest band that is expected of the problems (sfl_front) to err[2].
__global__ __launch_bounds__(64) void k_sfl_band(sfl_args S)
{
    const mct_sfmm_args &A = S.A;
    const int lane = threadIdx.x, prob = blockIdx.x;
    const int si = prob % A.nsrc_eff, ch = prob / A.nsrc_eff / A.nwave;
    const double *s0 = A.src + (long)ch * A.src_chain_stride + (long)si * A.src_stride;
    const double p[3] = {s0[0] - A.xmin, s0[1] - A.ymin, s0[2] - A.zmin}, leaf[3] = {A.lx, A.ly, A.lz};
    const int dims[3] = {A.G.nx, A.G.ny, A.G.nz};
    const float h[3] = {1.f, (float)(leaf[1] / leaf[0]), (float)(leaf[2] / leaf[0])};
    int pc[3];
#pragma unroll
    for (int d = 0; d < 3; d++) {
        const double qd = p[d] / leaf[d];
        pc[d] = !(qd >= 1.0) ? 0 : (qd >= (double)dims[d] ? dims[d] - 1 : (int)qd);
    }
    int widest = 0;
    for (int r = 1; r <= SFL_RADII; r++) {
        int c = sfl_front(dims, h, pc, r, lane, 64);
        for (int o = 32; o > 0; o >>= 1) c += __shfl_xor(c, o, 64);
        widest = c > widest ? c : widest;
    }
    if (lane == 0) atomicMax(A.err + 2, (uint32_t)widest);
}

__global__ __launch_bounds__(64) void k_sfmm_lds(sfl_args S)
{
    extern __shared__ double sfl_lds[];
    const mct_sfmm_args &A = S.A;
    const mct_geom &G = A.G;
    const int lane = threadIdx.x;
    const int prob = blockIdx.x;
    if (S.most > 0 && A.err[2] > (uint32_t)S.most) {
        if (lane == 0) {
            S.done[prob] = 0u;
            atomicAdd(A.err + 1, 1u);
        }
        return;
    }
    const int si = prob % A.nsrc_eff, cw = prob / A.nsrc_eff, ch = cw / A.nwave;
    double *T = S.T + (long)prob * S.L.n;
    const double *V = S.V + (long)cw * S.L.n;
    uint16_t *SL = S.slot + (long)prob * S.L.n;
    double *K = sfl_lds;                              // keys; a free slot's word links to the next
    uint32_t *C = (uint32_t *)(K + S.ns);             // cells
    uint16_t *H = (uint16_t *)(C + S.ns);             // the heap
    uint8_t *N = (uint8_t *)(H + S.ne);               // entries per slot
    const double leaf[3] = {A.lx, A.ly, A.lz};
    const int dims[3] = {G.nx, G.ny, G.nz};
    uint32_t err = 0;
    bool full = false;

    // ---- Solver::setInitialPoints, as in k_sfmm above
    const double *sp0 = A.src + (long)ch * A.src_chain_stride + (long)si * A.src_stride;
    const double p[3] = {sp0[0] - A.xmin, sp0[1] - A.ymin, sp0[2] - A.zmin};
    int pc[3];
#pragma unroll
    for (int d = 0; d < 3; d++) {
        const double qd = p[d] / leaf[d];
        pc[d] = !(qd >= 1.0) ? 0 : (qd >= (double)dims[d] ? dims[d] - 1 : (int)qd);
    }
    uint32_t cq[8];
    double vn[8], tc[8];
    int cc[8][3];
#pragma unroll
    for (int v = 0; v < 8; v++) {
#pragma unroll
        for (int d = 0; d < 3; d++) {
            int c = pc[d] + ((v >> (2 - d)) & 1);
            cc[v][d] = c >= dims[d] ? dims[d] - 1 : c;
        }
        cq[v] = first_u(S.L.base + (uint32_t)(cc[v][0] + cc[v][1] * S.L.sy + cc[v][2] * S.L.sz));
        vn[v] = V[cq[v]];
    }
    double vs = 0.0;
#pragma unroll
    for (int v = 0; v < 8; v++) {
        double w = 1.0;
#pragma unroll
        for (int d = 0; d < 3; d++) {
            const double sd = p[d] - leaf[d] * pc[d];
            const double wj = fabs((double)(cc[v][d] - pc[d]) * leaf[d] - leaf[d] + sd);
            w = w * wj / leaf[d];
        }
        vs = vs + w * vn[v];
    }
#pragma unroll
    for (int v = 0; v < 8; v++) {
        double dist = 0.0;
#pragma unroll
        for (int d = 0; d < 3; d++) {
            const double xi = (cc[v][d] * leaf[d] - p[d]) * (cc[v][d] * leaf[d] - p[d]);
            dist = dist + xi;
        }
        dist = sqrt(dist);
        tc[v] = dist * 2 / (vs + vn[v]);
        if (lane == 0) T[cq[v]] = tc[v];
    }

    int hs = 0;                                       // heap entries
    int nb = 0;                                       // slots ever used
    int fh = -1;                                      // head of the free list
    // push_heap (as in k_sfmm): lane j - 1 holds the ancestor j levels up.  The other
    // lanes read entry 0 and its key too, so entry 0 names a slot before the first push.
    if (lane == 0) H[0] = 0;
    wave_sync();
    auto push = [&](int slot, double kc) {
        const int k1 = (int)first_u((uint32_t)hs) + 1;
        hs = k1;
        const int m = 31 - __builtin_clz(k1);
        const int e = H[lane < m ? (k1 >> (lane + 1)) - 1 : 0];
        const double ke = K[e];
        const unsigned long long stop = ~ballot(ke > kc) & ((1ull << m) - 1ull);
        const int n = stop ? __builtin_ctzll(stop) : m;
        if (lane <= n) H[(k1 >> lane) - 1] = (uint16_t)(lane == n ? slot : e);
        wave_sync();
    };
    // the corners are pushed in order; clamped corners repeat a cell, which then has
    // one slot and as many entries
    int cs[8];
#pragma unroll
    for (int v = 0; v < 8; v++) {
        int slot = nb, cnt = 1;
#pragma unroll
        for (int w = 0; w < v; w++)
            if (cq[w] == cq[v]) { slot = cs[w]; cnt++; }
        cs[v] = slot = (int)first_u((uint32_t)slot);
        nb += slot == nb ? 1 : 0;
        if (lane == 0) {
            C[slot] = cq[v];
            SL[cq[v]] = (uint16_t)slot;
            K[slot] = tc[v];
            N[slot] = (uint8_t)cnt;
        }
        wave_sync();
        push(slot, tc[v]);
        // A source on a node of velocity 0 has a NaN among its corners' times.  The
        // ballots below compare a path's entries all at once, which puts NaN keys
        // elsewhere than the loop does: such a problem is left to k_sfmm too.
        full |= !(tc[v] < sf_inf());
    }

    // a lane's place in a block of five levels under the hole, and its ancestors there
    const int lv = 31 - __builtin_clz((unsigned)lane + 2u);
    const int off = lane + 2 - (1 << lv);
    unsigned long long anc = 0;
    for (int j = lane + 2; j >= 2; j >>= 1) anc |= 1ull << (j - 2);
    // lanes 4n + i: neighbour n (x-, x+, y-, y+, z-, z+: fmm.hpp:117-120), dimension i
    const int nn = lane >> 2, i = lane & 3;
    const int ndim = nn >> 1;
    const int nstride = ndim == 0 ? 1 : (ndim == 1 ? S.L.sy : S.L.sz);
    const int noff = lane < 24 ? ((nn & 1) ? nstride : -nstride) : 0;
    const int st8 = 8 * (i == 0 ? 1 : (i == 1 ? S.L.sy : (i == 2 ? S.L.sz : 0)));
    const double hi = i == 0 ? leaf[0] : (i == 1 ? leaf[1] : leaf[2]);
    const double al1 = 1.0 / (hi * hi), al2 = 9.0 / 4.0 / (hi * hi);

    const long max_pops = 64L * (long)G.nx * G.ny * G.nz + 64;
    long pops = 0;
    while (hs > 0 && !err && !full) {
        if (++pops > max_pops) { err |= SF_ERR_POPS; break; }
        // ---- pop_heap: the root, the last entry and the block under the root, then
        // their keys and the popped cell
        const int n = (int)first_u((uint32_t)hs) - 1;
        hs = n;
        const int idx = (1 << lv) - 1 + off;
        const int h0 = first_u(H[0]);
        const int hn = first_u(H[n]);
        int e0 = H[((lane < 62) & (idx < n)) ? idx : 0];
        double k0 = K[e0];
        const uint32_t cell = first_u(C[h0]);
        const double ttop = K[h0];
        const int left = (int)first_u(N[h0]);
        const double kval = K[hn];
        // the neighbours' stencils, in flight while the heap moves
        const uint32_t nb8 = (cell + (uint32_t)noff) * 8u;
        const double traw = ld_d(T, nb8);
        double m1 = ld_d(T, nb8 - (uint32_t)st8), p1 = ld_d(T, nb8 + (uint32_t)st8);
        double m2 = ld_d(T, nb8 - 2u * (uint32_t)st8), p2 = ld_d(T, nb8 + 2u * (uint32_t)st8);
        const double vel = ld_d(V, nb8);
        const int nslot = *(const uint16_t *)((const char *)SL + (nb8 >> 2));
        __builtin_amdgcn_sched_barrier(0);
        {
            // The hole goes down to a leaf, to the right child unless its key is
            // larger; then val climbs back past the path entries with larger keys.
            // So the path's entries down to the last one not larger move up one
            // place each, and val takes that one's.
            constexpr unsigned long long EVEN = 0x5555555555555555ull;
            unsigned long long path[3] = {0, 0, 0};
            int c[3] = {1, 1, 1}, en[3] = {0, 0, 0};
            int hole = 1;                              // 1-based
            int js = 1, jb = 0;                        // where val goes, and the block it lies in
            unsigned long long jm = 0;                 // that block's entries that move
            bool more = n > 0;
#pragma unroll
            for (int b = 0; b < 3; b++) {
                if (!more) break;
                c[b] = (hole << lv) + off;             // 1-based
                const bool ok = (lane < 62) & (c[b] <= n);
                if (b > 0) {
                    e0 = H[ok ? c[b] - 1 : 0];
                    k0 = K[e0];
                }
                en[b] = e0;
                const double k = ok ? k0 : sf_inf();
                const double ks = swap_d(k);
                // left (even lane): the right one is larger; right: it is not
                const unsigned long long M = ((ballot(ks > k) & EVEN) | (~ballot(k > ks) & ~EVEN)) & ballot(ok);
                path[b] = ballot((M & anc) == anc);
                const unsigned long long keep = path[b] & ~ballot(k > kval);
                more = false;
                if (path[b]) {
                    if (keep) {
                        const int jl = 63 - __builtin_clzll(keep), l = 31 - __builtin_clz(jl + 2);
                        js = (hole << l) + jl + 2 - (1 << l);
                        jb = b;
                        jm = path[b] & ((2ull << jl) - 1ull);
                    }
                    const int j = 63 - __builtin_clzll(path[b]) + 2, l = 31 - __builtin_clz(j);
                    hole = (hole << l) + j - (1 << l);
                    more = l == 5 && 2 * hole <= n;
                }
            }
#pragma unroll
            for (int b = 0; b < 3; b++) {
                const unsigned long long mv = b < jb ? path[b] : (b == jb ? jm : 0ull);
                if (mv && ((mv >> lane) & 1ull)) H[(c[b] >> 1) - 1] = (uint16_t)en[b];
            }
            if (lane == 0) {
                H[js - 1] = (uint16_t)hn;
                N[h0] = (uint8_t)(left - 1);
            }
        }
        // the entry leaves its slot (free when it was the last)
        if (left == 1) {
            if (lane == 0) *(int *)&K[h0] = fh;
            fh = h0;
        }
        wave_sync();
        // ---- neighbour updates (fmm.hpp:124-154); frozen cells carry the sign bit
        const double tself = fabs(traw);
        m1 = fabs(m1); m2 = fabs(m2); p1 = fabs(p1); p2 = fabs(p2);
        const bool live = (lane < 24) & (__double_as_longlong(traw) >= 0) & !(vel < SF_MARGIN);
        const unsigned long long LV = ballot(live);
        double nt = sfl_solve(i, m1, m2, p1, p2, tself, vel, leaf[0], leaf[1], leaf[2], al1, al2);
        // the plus neighbour's two-away cell on its minus side is the minus
        // neighbour: solved again with its value after the update
        unsigned long long U = LV & ballot(nt + SF_MARGIN < tself);
        if (((U & 0x10101ull) << 4) & LV) {
            const double from_minus = __shfl(nt, lane >= 4 ? (lane & ~3) - 4 : lane, 64);
            const bool again = (nn & 1) && ((U >> ((lane & ~3) - 4)) & 1);
            const double nt2 = sfl_solve(i, m1, (again && i == ndim) ? from_minus : m2, p1, p2, tself, vel,
                                         leaf[0], leaf[1], leaf[2], al1, al2);
            if (again) nt = nt2;
            U = LV & ballot(nt + SF_MARGIN < tself);
        }
        if (LV & ballot(tself == sf_inf()) & ballot(nt == sf_inf())) err |= SF_ERR_OPEN_INF;
        // the popped cell is frozen (fmm.hpp:123); stored after the loads have landed
        // (a wait for a load also waits for the stores before it)
        if (lane == 0) T[cell] = -ttop;
        unsigned long long todo = U & 0x111111ull;
        while (todo && !full) {
            const int s = __builtin_ctzll(todo);
            todo &= todo - 1;
            const uint32_t c8 = rl_u(nb8, s);
            const double tn = rl_d(nt, s);
            const bool narrow = !__builtin_isinf(rl_d(tself, s));
            int slot, cnt = 0;
            if (narrow) {
                slot = (int)rl_u((uint32_t)nslot, s);
                cnt = (int)first_u(N[slot]);
            } else if (fh >= 0) {
                slot = fh;
                fh = (int)first_u(*(const uint32_t *)&K[slot]);
            } else {
                slot = nb++;
            }
            if (nb > S.ns || hs >= S.ne || cnt >= 255) { full = true; break; }
            if (lane == 0) {
                *(double *)((char *)T + c8) = tn;
                K[slot] = tn;
                N[slot] = (uint8_t)(cnt + 1);
                if (!narrow) {
                    C[slot] = c8 >> 3;
                    *(uint16_t *)((char *)SL + (c8 >> 2)) = (uint16_t)slot;
                }
            }
            wave_sync();
            push(slot, tn);
        }
    }
    // a band that outgrew the tables, or was expected to, or had a key that is no number:
    // the replay with the heap in global memory, here or by k_sfmm
    if (lane == 0) {
        S.done[prob] = !full ? 1u : (S.here ? 2u : 0u);
        if (full) atomicAdd(A.err + 1, 1u);
    }
    if (full) {
        if (S.here) sf_replay<1>(A, prob);
        return;
    }
    if (A.pops && lane == 0) A.pops[prob] = (uint32_t)(pops > 0xffffffffL ? 0xffffffffL : pops);
    if (err && lane == 0) atomicOr(A.err, err);
}

// Frozen cells carry the sign bit: clear it (cells never reached keep +inf).
__global__ void k_sfmm_thaw(double *T, long n)
{
    for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x)
        T[i] = fabs(T[i]);
}

} // namespace

long mct_sfmm_heap_cap(const mct_geom &G)
{
    const long cells = (long)G.nx * G.ny * G.nz;
    long cap = cells / 8;
    if (cap < 65536) cap = 65536;
    return cap;
}

// How the replay in LDS would run: slots and heap entries per problem, or 0 slots
// where it does not pay.
struct sfl_plan { int ns, ne, most, here; size_t lds; };

static sfl_plan sfl_make_plan(const mct_geom &G, long nprob)
{
    sfl_plan P = {0, 0, 0, 0, 0};
    int dev = 0, max_lds = 0, cus = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&max_lds, hipDeviceAttributeMaxSharedMemoryPerBlock, dev) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus < 1)
        return P;
    const sfl_grid L = sfl_layout(G);
    // 32-bit byte offsets into a padded grid
    if ((double)(G.nz + 2 * SFL_SLABS) * (G.ny + SFL_PAD + 1) * (G.nx + SFL_PAD + 1) * 8.0 > 2e9) return P;
    // The band holds 0.2 to 0.97 cells per cell of the grid's three faces (1,080 problems:
    // media of one cell to 1,000 and a gradient, spacings 1:1 to 1:2; sources at a corner
    // to 0.5, in the middle 0.6 to 0.97), and about 1.06 entries a cell.  15.3 bytes a
    // slot.
    const double area = (double)G.nx * G.ny + (double)G.ny * G.nz + (double)G.nx * G.nz;
    const double room = (max_lds - 256) / 15.3;
    if (0.55 * area > room) return P;
    int per_cu = (int)(room / (0.75 * area + 64.0));
    per_cu = per_cu < 1 ? 1 : (per_cu > 16 ? 16 : per_cu);
    // The units take turns of per_cu problems each; with heaps in global memory all
    // problems run at once.  Measured, this against that: 57^3 (one a unit) 414 / 876
    // ms for 128 problems, 833 / 1032 for 512, 2488 / 1423 for 1,536; 41^3 (two a
    // unit) 151 / 307 for 128, 313 / 452 for 1,024.
    if (nprob > 2L * per_cu * cus) return P;
    // In two turns the problems that are left run after the others (33^3, one of 1,300 left
    // 351 ms, all in global memory 241): only where every band fits.  Run at once, they
    // go on in place.
    P.here = nprob <= (long)per_cu * cus;
    if (!P.here && room / per_cu < area) return P;
    // no more problems to a unit than it takes to run all at once: wider tables
    while (per_cu > 1 && nprob <= (long)(per_cu - 1) * cus) per_cu--;
    P.ns = (int)(room / per_cu) & ~7;
    if (P.ns > 65528) P.ns = 65528;
    // MCT_SFMM_SLOTS: at most this many, so that wider bands are handed over when they
    // are that wide
    const char *e = getenv("MCT_SFMM_SLOTS");
    const int most = e ? atoi(e) & ~7 : 0;
    if (most > 0 && P.ns > most) P.ns = most < 64 ? 64 : most;
    P.ne = P.ns + P.ns / 8 + 64;
    P.lds = 12 * (size_t)P.ns + 2 * (size_t)P.ne + (size_t)P.ns;
    while (P.lds * per_cu > (size_t)max_lds && P.ns > 64) {
        P.ns -= 8;
        P.ne = P.ns + P.ns / 8 + 64;
        P.lds = 12 * (size_t)P.ns + 2 * (size_t)P.ne + (size_t)P.ns;
    }
    // A band that outgrows the tables has its problem begun twice: a source in the
    // middle of a 74^3 grid 2.25 s with the tables first, 1.88 at once in global memory,
    // one at its corner 0.90 in LDS.  Where the tables may be too small, the widest band
    // of a homogeneous medium tells (the 1,080 problems' was 1.08 times that in the
    // median, 0.98 to 1.26 for 80 % of them).  Leaving a band that fits costs more than
    // trying one that does not, so the line lies where about half outgrow the tables.
    // A launch takes as long as its slowest problem, so one that is left takes the others
    // along (72^3, 5 of 200 left, some of them late: 2.24 s, all in global memory 1.93).
    if (!(most > 0) && area > P.ns) P.most = (int)(0.95 * P.ns);
    return P;
}

size_t mct_sfmm_lin_bytes(const mct_geom &G, long nprob, long ncw)
{
    if (sfl_make_plan(G, nprob).ns == 0) return 0;
    const sfl_grid L = sfl_layout(G);
    return 8 * (size_t)L.n * (size_t)(nprob + ncw) + 2 * (size_t)L.n * (size_t)nprob + 4 * (size_t)nprob + 64;
}

int mct_launch_sfmm(const mct_sfmm_args &a0, hipStream_t s)
{
    mct_sfmm_args a = a0;
    if (a.nprob < 1 || !a.T || !a.V || !a.src || !a.heap || !a.err || a.hcap < 16 ||
        a.nsrc_eff < 1 || a.nwave < 1)
        return MCT_ERR_ARG;
    if ((long)a.G.ntiles * MCT_TILE_N > 0xffffffffL) return MCT_ERR_ARG;
    MCT_CHECK(hipMemsetAsync(a.err, 0, 3 * sizeof(uint32_t), s));
    a.done = nullptr;
    const long ncw = (a.nprob + a.nsrc_eff - 1) / a.nsrc_eff;
    const sfl_plan P = a.order == 1 && a.lin ? sfl_make_plan(a.G, a.nprob) : sfl_plan{0, 0, 0, 0, 0};
    if (P.ns > 0) {
        sfl_args S;
        S.L = sfl_layout(a.G);
        S.T = (double *)a.lin;
        S.V = S.T + (size_t)S.L.n * a.nprob;
        S.done = (uint32_t *)(S.V + (size_t)S.L.n * ncw);
        S.slot = (uint16_t *)(S.done + a.nprob);
        S.ns = P.ns;
        S.ne = P.ne;
        S.most = P.most;
        S.here = P.here;
        a.done = S.done;
        S.A = a;
        const unsigned gx = (S.L.n + 255) / 256;
        const unsigned gy = a.nprob < 1024 ? (unsigned)a.nprob : 1024u, gc = ncw < 1024 ? (unsigned)ncw : 1024u;
        hipLaunchKernelGGL(k_sfl_fill, dim3(gx, gy), dim3(256), 0, s, a.G, S.L, S.T, (long)a.nprob);
        hipLaunchKernelGGL(k_sfl_vel, dim3(gx, gc), dim3(256), 0, s, a.G, S.L, a.V, (double *)S.V, ncw);
        if (P.lds > 64 * 1024)
            MCT_CHECK(hipFuncSetAttribute((const void *)k_sfmm_lds, hipFuncAttributeMaxDynamicSharedMemorySize, (int)P.lds));
        if (P.most > 0) hipLaunchKernelGGL(k_sfl_band, dim3((unsigned)a.nprob), dim3(64), 0, s, S);
        hipLaunchKernelGGL(k_sfmm_lds, dim3((unsigned)a.nprob), dim3(64), P.lds, s, S);
        hipLaunchKernelGGL(k_sfl_tiles, dim3(gx, gy), dim3(256), 0, s, a.G, S.L, S.T, a.T, S.done, (long)a.nprob);
        MCT_CHECK(hipGetLastError());
    }
    if (a.order == 1)
        hipLaunchKernelGGL(k_sfmm<1>, dim3((unsigned)a.nprob), dim3(64), 0, s, a);
    else
        hipLaunchKernelGGL(k_sfmm<0>, dim3((unsigned)a.nprob), dim3(64), 0, s, a);
    MCT_CHECK(hipGetLastError());
    const long n = (long)a.nprob * a.G.ntiles * MCT_TILE_N;
    hipLaunchKernelGGL(k_sfmm_thaw, dim3(4096), dim3(256), 0, s, a.T, n);
    MCT_CHECK(hipGetLastError());
    return MCT_OK;
}

// problems that the calling thread's last replay in LDS left to k_sfmm
static thread_local long long g_sfmm_handover = 0;

extern "C" int mct_sfmm_last_handover(long long *n)
{
    if (!n) return MCT_ERR_ARG;
    *n = g_sfmm_handover;
    return MCT_OK;
}

int mct_sfmm_status(const uint32_t *err)
{
    const uint32_t err_bits = err[0];
    g_sfmm_handover = err[1];
    if (!err_bits) return MCT_OK;
    return (err_bits & SF_ERR_HEAP) ? MCT_ERR_NOMEM : MCT_ERR_NOCONV;
}

int mct_default_heap_order1()
{
    const char *e = getenv("MCT_EIK_ORDER1");
    return !(e && strcmp(e, "parallel") == 0);
}
