// Host-side check of the range in which the period equations take the short
// quotients and square roots: built with a fp64_ops.h that counts operands outside
// 2^+-900 (tests/test_dispersion_range.py writes it beside copies of the sources),
// it evaluates random layer models from all over dsp_in_range and from earth
// models in km and in m.
#include "dispersion.hip"
#include <cstdio>
#include <cstdlib>
#include <random>

long fp_bad = 0;

int mct_fill_i32(int32_t *, long, int32_t, hipStream_t) { return 0; }

int main(int argc, char **argv)
{
    const long n = argc > 1 ? atol(argv[1]) : 100000;
    std::mt19937_64 rng(20261205);
    std::uniform_real_distribution<double> U(0.0, 1.0);
    long bad = 0, slow_earth = 0, taken = 0, earth_n = 0;
    for (long it = 0; it < n; it++) {
        float d[16], a[16], b[16], rho[16];
        const bool earth = it % 4 == 0;
        const double unit = earth && it % 8 == 0 ? 1000.0 : 1.0;
        int lim = 0;                        // the exponent range that dsp_in_range takes
        while (dsp_in_range(ldexp(1.0, lim + 1))) lim++;
        auto any = [&]() {                  // often at its ends
            const double u = rng() % 4 == 0 ? (rng() % 2 ? 1.0 : -1.0) : 2.0 * U(rng) - 1.0;
            return (float)exp2(lim * u);
        };
        dsp_model_t<1> M;
        M.mmax = 2 + (int)(rng() % 14);
        M.llw = rng() % 4 == 0 ? 2 : 1;
        for (int i = 0; i < M.mmax; i++) {
            if (earth) {
                const double vs = 0.3 + 4.5 * U(rng), vp = 1.4 * vs + 1.5 * U(rng);
                b[i] = (float)(unit * vs); a[i] = (float)(unit * vp);
                rho[i] = (float)((unit > 1.0 ? 1000.0 : 1.0) * (1.5 + 2.0 * U(rng)));
                d[i] = (float)(unit * (rng() % 8 ? exp2(10.0 * U(rng) - 5.0) : 0.0));
            } else {
                b[i] = any(); a[i] = any(); rho[i] = any();
                d[i] = rng() % 8 ? any() : 0.0f;
            }
        }
        if (M.llw == 2) b[0] = 0.0f;
        d[M.mmax - 1] = 0.0f;
        M.d = d; M.a = a; M.b = b; M.rho = rho;
        const double omega = earth ? exp2(10.0 * U(rng) - 6.0) : (double)any();
        const double c = earth ? unit * (0.25 + 4.5 * U(rng)) : (double)any();
        for (int ifunc = 1; ifunc <= 2; ifunc++) {
            if (ifunc == 1 && M.llw == 2) continue;
            fp_bad = 0;
            bool ok = true;
            volatile double r = d_dltar<true>(omega / c, omega, ifunc, M, ok);
            (void)r;
            earth_n += earth;
            taken += ok;
            if (earth && !ok) slow_earth++;
            if (ok && fp_bad) {
                if (bad < 5) printf("out of range: ifunc %d omega %g c %g layers %d (%ld operands)\n", ifunc, omega, c,
                                    M.mmax, fp_bad);
                bad++;
            }
        }
    }
    printf("evaluations taken %ld out of range %ld earth %ld refused %ld\n", taken, bad, earth_n, slow_earth);
    return bad != 0 || slow_earth != 0;
}
