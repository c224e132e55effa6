// Host-side check of sfl_front (sfmm.hip), the band of a homogeneous medium from which
// the order-1 3-D replay tells whether its tables in LDS suffice: against the cells
// that lie beyond the front and next to a cell within it, counted one by one.  Built
// with hipcc and run on the CPU by tests/test_sfmm_band.py.
#include "../../mctomo_amd/csrc/sfmm.hip"
#include <cstdio>
#include <random>
#include <vector>

int main()
{
    std::mt19937_64 rng(7);
    double lo = 1e9, hi = 0.0;
    long bad = 0;
    const float hs[] = {0.5f, 1.0f, 2.0f};
    for (int it = 0; it < 120; it++) {
        int n[3], p[3];
        float h[3] = {1.0f, hs[rng() % 3], hs[rng() % 3]};
        for (int d = 0; d < 3; d++) {
            n[d] = 9 + (int)(rng() % 32);
            const int k = (int)(rng() % 4);
            p[d] = k == 0 ? 0 : k == 1 ? n[d] / 2 : (int)(rng() % (unsigned)n[d]);
        }
        int est = 0;
        for (int r = 1; r <= SFL_RADII; r++) {
            const int c = sfl_front(n, h, p, r, 0, 1);
            int parts = 0;
            for (int l = 0; l < 64; l++) parts += sfl_front(n, h, p, r, l, 64);
            bad += parts != c;
            est = c > est ? c : est;
        }
        auto t2 = [&](int x, int y, int z) {
            const double a = (x - p[0]) * h[0], b = (y - p[1]) * h[1], c = (z - p[2]) * h[2];
            return a * a + b * b + c * c;
        };
        double far2 = 0.0;
        for (int c = 0; c < 8; c++) far2 = fmax(far2, t2(c & 1 ? n[0] - 1 : 0, c & 2 ? n[1] - 1 : 0, c & 4 ? n[2] - 1 : 0));
        int band = 0;
        for (int r = 1; r <= 2 * SFL_RADII; r++) {
            const double R = far2 * r * r / (4.0 * SFL_RADII * SFL_RADII);
            int c = 0;
            for (int x = 0; x < n[0]; x++)
                for (int y = 0; y < n[1]; y++)
                    for (int z = 0; z < n[2]; z++) {
                        if (t2(x, y, z) <= R) continue;
                        c += (x > 0 && t2(x - 1, y, z) <= R) || (x + 1 < n[0] && t2(x + 1, y, z) <= R) ||
                             (y > 0 && t2(x, y - 1, z) <= R) || (y + 1 < n[1] && t2(x, y + 1, z) <= R) ||
                             (z > 0 && t2(x, y, z - 1) <= R) || (z + 1 < n[2] && t2(x, y, z + 1) <= R);
                    }
            band = c > band ? c : band;
        }
        const double q = (double)band / est;
        lo = fmin(lo, q);
        hi = fmax(hi, q);
    }
    printf("band / estimate %.3f to %.3f, lanes differ %ld\n", lo, hi, bad);
    return bad != 0 || lo < 0.95 || hi > 1.2;
}
