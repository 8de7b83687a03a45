// Row ranges found by bisection against a test of every pixel, and the
// nearest-pixel index against a scan, over grids of many periods, among them
// ones whose limits fall on a pixel.
#include "../../ms-stem-fem_amd/csrc/msf_host.hpp"

#include <cmath>
#include <cstdio>
#include <random>

using namespace msf;

template <typename Pred> static long differ(const RowRanges& r, int nx, int ny, Pred keep)
{
    long n = 0;
    for (int i = 0; i < nx; ++i)
        for (int j = 0; j < ny; ++j)
            n += keep(i, j) != (j < r.ab[2 * i] || j >= ny - r.ab[2 * i + 1]);
    return n;
}

int main()
{
    std::mt19937 gen(7);
    std::uniform_real_distribution<double> U(0.0, 1.0);
    const int lengths[] = {16, 32, 64, 96, 128, 192, 256};
    long bad = 0, cols = 0, idx = 0, whole = 0;
    for (int t = 0; t < 400; ++t) {
        const int nx = lengths[gen() % 7], ny = lengths[gen() % 7];
        double lx = std::round((4.0 + 20.0 * U(gen)) * 100) / 100;
        double ly = (t % 3) ? lx * ny / nx : std::round((4.0 + 20.0 * U(gen)) * 100) / 100;
        const Domain d = make_domain(nx, ny, lx, ly, U(gen) - 0.5, 0.0, 200e3);
        const std::vector<double> kx2 = pow2_all(d.kx), ky2 = pow2_all(d.ky);
        const double c_bw = ref_pow2(d.bw_t), c_pr = d.bw_t * d.bw_t, c2 = d.bw_pap * d.bw_pap;
        const RowRanges keep = slice_keep_ranges(d);
        bad += differ(keep, nx, ny, [&](int i, int j) {
            const double k2 = kx2[i] + ky2[j];
            return !(k2 >= c_bw) && (k2 < c_pr);
        });
        bad += differ(bwlimit_keep_ranges(d), nx, ny,
                      [&](int i, int j) { return !(kx2[i] + ky2[j] >= c_bw); });
        bad += differ(template_keep_ranges(d), nx, ny,
                      [&](int i, int j) { return kx2[i] + ky2[j] < c2; });
        const double a = 0.001 + 0.3 * U(gen) * U(gen), l2 = d.lambda * d.lambda, a2 = a * a;
        const RowRanges ap = aperture_keep_ranges(d, a);
        bad += differ(ap, nx, ny, [&](int i, int j) {
            const double ksqr = d.kx[i] * d.kx[i] + d.ky[j] * d.ky[j];
            return l2 * ksqr < a2;
        });
        whole += ap.amax == ny;
        const int nc = keep.amax + keep.bmax, ncp = (nc + 15) / 16 * 16;
        const RowRanges ck = column_keep_ranges(keep, nx, ny, ncp);
        for (int jc = 0; jc < ncp; ++jc)
            for (int i = 0; i < nx; ++i) {
                const int j = jc < keep.amax ? jc : jc - nc + ny;
                const bool k = jc < nc && (j < keep.ab[2 * i] || j >= ny - keep.ab[2 * i + 1]);
                cols += k != (i < ck.ab[2 * jc] || i >= nx - ck.ab[2 * jc + 1]);
            }
        for (int n = 0; n < 200; ++n) {
            const double step = d.xx[1] - d.xx[0];
            double q = d.xx[0] + (1.4 * U(gen) - 0.2) * lx;
            if (n % 4 == 0) q = d.xx[gen() % nx] + 0.5 * step * (double)((int)(gen() % 3) - 1);
            if (n == 1) q = 1e300;
            if (n == 2) q = -1e300;
            if (n == 3) q = std::nan("");
            int64_t want = 77;
            for (int i = 0; i < nx; ++i)
                if (d.xx[i] - q >= 0.5 * step) {
                    want = i - 1;
                    break;
                }
            idx += shift_index(d.xx, q, 77) != want;
        }
    }
    std::printf("ranges %ld columns %ld indices %ld whole rows %d\n", bad, cols, idx, whole > 0);
    return 0;
}
