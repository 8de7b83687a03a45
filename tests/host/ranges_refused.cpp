// Sets that are not a disk in FFT order are reported, not cut to one: spatial
// frequencies out of order along y make every row range invalid, along x the
// columns of the kept set; frequencies in order, for every compiled length,
// are accepted, sets of whole rows and empty sets among them.
#include "../../ms-stem-fem_amd/csrc/msf_host.hpp"

#include <algorithm>
#include <cmath>
#include <cstdio>

using namespace msf;

static RowRanges columns(const Domain& d, const RowRanges& keep)
{
    return column_keep_ranges(keep, d.nx, d.ny, (keep.amax + keep.bmax + 15) / 16 * 16);
}

int main()
{
    const int lengths[] = {16, 32, 64, 96, 128, 192, 256, 384, 512, 768, 1024};
    long refused = 0, accepted = 0;
    for (int nx : lengths)
        for (int ny : lengths) {
            const Domain d = make_domain(nx, ny, nx * 0.07, ny * 0.09, 0.3, 0.0, 300e3);
            const RowRanges keep = slice_keep_ranges(d);
            refused += !keep.ok + !columns(d, keep).ok + !bwlimit_keep_ranges(d).ok +
                       !template_keep_ranges(d).ok;
            for (double a : {0.0, 0.003, 0.02, 0.4}) refused += !aperture_keep_ranges(d, a).ok;
            // a kept frequency moved among the ones left out, and NaN
            Domain y = d, n = d, x = d;
            std::swap(y.ky[1], y.ky[(size_t)ny / 2 - 1]);
            n.ky[(size_t)ny / 4] = std::nan("");
            std::swap(x.kx[1], x.kx[(size_t)nx / 2 - 1]);
            for (const Domain* b : {&y, &n})
                accepted += slice_keep_ranges(*b).ok + bwlimit_keep_ranges(*b).ok +
                            template_keep_ranges(*b).ok + aperture_keep_ranges(*b, 0.02).ok;
            const RowRanges kx = slice_keep_ranges(x);
            // the rows of x are disks, each on its own
            refused += !kx.ok;
            accepted += columns(x, kx).ok;
        }
    std::printf("refused %ld accepted %ld\n", refused, accepted);
    return 0;
}
