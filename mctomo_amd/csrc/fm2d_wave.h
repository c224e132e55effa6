// fm2d_wave.h -- parts of the 2-D heap loops that a wave (or a part of one) runs
// together: k_fm2d_wave's and k_fm2d_near's.
#pragma once
#include <hip/hip_runtime.h>
#include "fp64_ops.h"

#pragma clang fp contract(off)

namespace {

// Lanes of one wave read what others of it wrote: keep the accesses in order.
__device__ __forceinline__ void w_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

__device__ __forceinline__ int w_level(int p) { return 31 - __clz(p); }

// the value of the lane whose index differs in bit 0 (0xb1) or bit 1 (0x4e)
template <int CTRL>
__device__ __forceinline__ double w_quad_d(double v)
{
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_update_dpp((int)b, (int)b, CTRL, 0xf, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp((int)(b >> 32), (int)(b >> 32), CTRL, 0xf, 0xf, false);
    return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}

// One quadrant of fouds1 (fm2d_ttime.f90:248-332) or fouds2 (:342-518): tj, tk the
// x and z neighbours' times, tj2, tk2 the ones behind them, a* whether alive.
// Returns a NaN when neither neighbour is alive: the minimum over the quadrants leaves
// it out.  A node next to a popped one always has a quadrant with a time.  Where
// the velocity is 0 the slowness, and with it the time, is infinite.
template <int FOM>
__device__ __forceinline__ double w_quadrant(bool aj, bool aj2, bool ak, bool ak2, double tj, double tj2, double tk,
                                             double tk2, double slown, double dnx, double dnz)
{
    const bool J = FOM != 0 && aj && aj2 && tj > tj2, K = FOM != 0 && ak && ak2 && tk > tk2;
    const double ss = slown * slown, xx = dnx * dnx, zz = dnz * dnz;
    double a = 1.0, b = 0.0, c, tref, tdiv = 1.0;
    if (aj && ak) {
        double uu, vv, em;
        if (J && K) {
            uu = 4.0 * xx; vv = 4.0 * zz;
            tref = 4.0 * tj - tj2;
            em = tref - 4.0 * tk;
            em = em + tk2;
            a = vv + uu;
            b = 2.0 * em * uu;
            tdiv = 3.0;
        } else if (J) {
            uu = zz; vv = 4.0 * xx;
            em = 3.0 * tk - 4.0 * tj + tj2;
            a = vv + 9.0 * uu;
            b = 6.0 * em * uu;
            tref = tk;
        } else if (K) {
            uu = xx; vv = 4.0 * zz;
            em = 3.0 * tj - 4.0 * tk + tk2;
            a = vv + 9.0 * uu;
            b = 6.0 * em * uu;
            tref = tj;
        } else {
            uu = xx; vv = zz;
            em = tk - tj;
            a = uu + vv;
            b = -(2.0 * uu * em);
            tref = tj;
        }
        c = uu * (em * em - vv * ss);
    } else if (aj) {
        c = -((J ? 4.0 * xx : xx) * ss);
        tref = J ? 4.0 * tj - tj2 : tj;
        tdiv = J ? 3.0 : 1.0;
    } else if (ak) {
        // fouds1 squares slown * dnz as one product, fouds2 the squares of each
        const double sz = slown * dnz;
        c = FOM == 0 ? -(sz * sz) : -((K ? 4.0 * zz : zz) * ss);
        tref = K ? 4.0 * tk - tk2 : tk;
        tdiv = K ? 3.0 : 1.0;
    } else {
        return __builtin_nan("");
    }
    double rd1 = b * b - 4.0 * a * c;
    if (rd1 < 0.0) rd1 = 0.0;
    const double tdsh = fp_div_any(-b + fp_sqrt(rd1), 2.0 * a);
    const double trav = tref + tdsh;
    if (FOM == 0 || tdiv == 1.0) return trav;
    return fp_div_any(trav, 3.0);
}

} // namespace
