// msf_host.hpp -- host-side FP64 rules of the multislice path.
//
// Everything here is O(N) or O(N^2) bookkeeping that decides *which* pixel
// or atom goes where: grids, band-limit membership, the nearest-pixel shift
// rule, the auto-slicer, propagator tables, detector and FEM bin pixel
// lists.  These decisions are taken on the host in IEEE FP64 with the same
// expressions and comparison operators as the reference, so the device
// kernels only ever consume integer index data and never decide membership
// in FP32.
#pragma once
#include <array>
#include <cstdint>
#include <functional>
#include <string>
#include <vector>

namespace msf {

constexpr double kRefPi = 3.14159265369; // the reference's PI macro (slice.cpp:41 and others)

// libm pow(x, 2.0), as the reference's -O0 build calls it (build/Makefile:37-45);
// compilers fold a literal pow(x, 2) into x*x, which rounds differently.
double ref_pow2(double x);
// ref_pow2 of every element
std::vector<double> pow2_all(const std::vector<double>& k);

struct Domain {
    int nx = 0, ny = 0;
    double lambda = 0, gamma = 0;
    double bw_pap = 0, bw_t = 0;    // tem.cpp:683-695
    double sqrt_nxny = 0;           // adfstem.cpp:210-212
    double nxny = 0;                // tem.cpp:405
    std::vector<double> kx, ky, xx, yy;
};

// tem.cpp:424-438
void wavelength(double voltage, double& lambda, double& gamma);
// tem.cpp:683-695, :756-883, func.cpp:92-106, :147-167
Domain make_domain(int nx, int ny, double xperiod, double yperiod, double xmin, double ymin,
                   double voltage);

// Row-wise membership of a disk-like pixel set in FFT order: for row i the
// kept columns are [0, a_i) U [ny - b_i, ny); ok == false if a set is not
// known to be of that form (the ranges then are not used).
struct RowRanges {
    std::vector<int32_t> ab; // 2*nx: a_i, b_i
    int amax = 0, bmax = 0;  // union over rows
    bool ok = true;
};
// keep(i, j) holds from j = 0 up to some j and from some j on to ny - 1 when
// it tests a rounded sum that grows with |k_y|: k_y rises over [0, ny/2) and
// -k_y falls over [ny/2, ny), and IEEE rounding is monotone.  A bisection of
// each half then finds the same ranges as a test of every pixel.  `ordered`
// says that this holds (a bisection cannot tell).
template <typename Pred> RowRanges row_ranges(int nx, int ny, bool ordered, Pred keep)
{
    RowRanges r;
    r.ok = ordered;
    r.ab.assign(2 * (size_t)nx, 0);
    const int h = ny / 2;
    for (int i = 0; i < nx; ++i) {
        int a = 0, end = h; // first j of the low half that is not kept
        while (a < end) {
            const int m = a + (end - a) / 2;
            if (keep(i, m)) a = m + 1;
            else end = m;
        }
        int lo = h, hi = ny; // first j of the high half that is kept
        while (lo < hi) {
            const int m = lo + (hi - lo) / 2;
            if (keep(i, m)) hi = m;
            else lo = m + 1;
        }
        int b = ny - lo;
        if (a == h && lo == h) { // the whole row
            a = ny;
            b = 0;
        }
        r.ab[2 * i] = a;
        r.ab[2 * i + 1] = b;
        if (a > r.amax) r.amax = a;
        if (b > r.bmax) r.bmax = b;
    }
    return r;
}

// bw_limit.cpp:30-47 together with slice::propagate's test (slice.cpp:1388-1389):
// the pixels a slice step keeps.
RowRanges slice_keep_ranges(const Domain& d);
// The same kept set by column of the compact plane [nx][ncp] (compact
// column jc holds full column j = jc < ka ? jc : jc - (ka + kb) + ny): the
// kept rows of column jc are [0, c) U [nx - d, nx), returned as (c, d) pairs
// (2*ncp entries; padding columns keep nothing).  ok == false unless the rows'
// ranges shrink over i < nx/2 and grow from there on, which makes every column
// of that form.
RowRanges column_keep_ranges(const RowRanges& rows, int nx, int ny, int ncp);

// bw_limit.cpp:30-47 alone (transmission band limit, slice.cpp:1731-1737)
RowRanges bwlimit_keep_ranges(const Domain& d);
// scatterer_pap.hpp:108-109: template support |k|^2 < bwcutoff_pap^2
RowRanges template_keep_ranges(const Domain& d);
// probe_wavefunction.cpp:107-111: aperture lambda^2 k^2 < alpha_max^2
RowRanges aperture_keep_ranges(const Domain& d, double alpha_max);

// Nearest-pixel rule, slice.cpp:1554-1572 and adfstem.cpp:1590-1606: first i
// with grid[i] - q >= half spacing, minus one; `previous` if none.  Returns
// -1 where the reference's size_t index would underflow (q below the domain).
int64_t shift_index(const std::vector<double>& grid, double q, int64_t previous);

// slice.cpp:469-740 (assign_atoms_to_slices_z_auto)
struct Slices {
    std::vector<double> lower, thick;
    std::vector<std::vector<int32_t>> atoms; // per slice, in z-sorted order
};
Slices autoslice(const double* q, uint32_t n, double zmin, double zperiod, double min_thickness);

// slice.cpp:1293-1363 (update_propagator), one axis, FP64 (re, im) pairs
void propagator(double lambda, double thickness, const std::vector<double>& k, double bw_t,
                std::vector<double>& p);

// adfstem.cpp:947-972
int fem_bin_count(const Domain& d, double dr, double& delta_k);

// Pixel groups for the reductions: group 0 = ADF ring (func.cpp:2630-2637),
// groups 1..nbins = FEM rings (variance.cpp:160-228 membership,
// adfstem.cpp:1043-1062 sort key).  Offsets are into the compact exit-wave
// plane [nx][ncp], only pixels that can be non-zero after the slice step.
struct Groups {
    std::vector<int32_t> offsets; // G+1
    std::vector<int32_t> pixels;  // compact plane offsets
    std::vector<int32_t> kind;    // 0: sum |psi|^2, 1: sum |psi|
    std::vector<int32_t> counts;  // FEM: full-grid bin counts (k_bin_counts)
    std::vector<uint8_t> zeroed;  // FEM: direct-beam bins (adfstem.cpp:2518-2522)
    std::vector<double> edges;    // FEM: lower edges ii*delta_k
    int nbins = 0;
    int fem_abs = -1;             // first group of the FEM |psi| rings (-1: none)
    int fem_sqr = -1;             // first group of the FEM |psi|^2 rings (-1: none)
    int corr = -1;                // first correlograph sector group, [ii * nphi + jj] (-1: none)
    int nphi = 0;                 // correlograph phi sectors per ring
    // every pixel of every FEM bin in the bins' sorted order (bin ii owns
    // [bin_off[ii], bin_off[ii+1])): full-grid index i*ny + j and compact
    // offset, -1 where the slice step's band limit leaves the pixel zero
    std::vector<int32_t> bin_off, bin_full, bin_compact;
};
// group 0: the ADF ring; then, with fem, nbins |psi| rings and, with
// fem_sqr, nbins |psi|^2 rings over the same pixels
Groups build_groups(const Domain& d, const RowRanges& keep, int ncp, bool adf, double k1,
                    double k2, bool fem, double dr, double alpha_max, bool fem_sqr = false,
                    bool correlograph = false);
// adfstem.cpp:969-985: the correlograph's phi sector count for nbins rings of width delta_k
int correlograph_nphi(double delta_k, int nbins);

// The detector MTF sampled on the grid, real [nx][ny] (adfstem.cpp:300-376;
// the squared domain (0.5 rate d)^2 of tem.cpp:276-285 formed from the
// file's Nyquist units).  n >= 1.
std::vector<double> mtf_table_2d(const Domain& d, double xperiod, double yperiod,
                                 const double* mtf, const double* domain, int n, double rate);
// adfstem.cpp:2279-2290: 1 where lambda^2 k^2 > alpha_max^2 (kept as |psi|), else 0
std::vector<uint8_t> outside_aperture(const Domain& d, double alpha_max);

// Groups cut into segments of at most `seg` pixels, 64 segments per wavefront
// tile, pixel offsets interleaved [tile][k][lane] (-1 pads short segments) so
// that a wavefront's index loads are coalesced.  Segments of one group are
// consecutive; group g owns segments [seg_of_group[g], seg_of_group[g+1]).
struct SegmentTiles {
    std::vector<int32_t> pix;         // interleaved pixel offsets
    std::vector<int32_t> tile_off;    // n_tiles + 1, into pix (units of 64 entries)
    std::vector<int32_t> seg_kind;    // per segment: 0 |psi|^2, 1 |psi|
    std::vector<int32_t> seg_of_group;
    int n_segments = 0, n_tiles = 0;
};
SegmentTiles build_segments(const Groups& g, int seg);

// A run's positions in n batches of at most `depth`, in raster order: batch k
// holds positions [begin(k), begin(k + 1)).  unit 0: batches of `depth`, what
// is left in the last; else whole units of that many positions, shared so
// that batches differ by one unit (the last unit may be a partial one).
struct BatchSplit {
    int64_t P = 0, depth = 1, n = 1, unit = 0;
    int64_t begin(int64_t k) const
    {
        if (unit == 0) return k * depth < P ? k * depth : P;
        const int64_t units = (P + unit - 1) / unit, q = units / n, r = units % n;
        const int64_t b = unit * (k * q + (k < r ? k : r));
        return b < P ? b : P;
    }
};
// batches of `depth` positions
BatchSplit batches_of(int64_t P, int64_t depth);
// The rule, for waves of `plane` stored values on a grid of `pixels`: the
// fewest batches whose waves stay within 96 MiB, spread evenly; with pairs
// (two chains of batches) an even number of three or more, in units of the
// positions that a row-pass workgroup holds.
BatchSplit batch_rule(int64_t P, int64_t plane, int64_t pixels, bool pairs, int unit);
// Pixels of a launch from which two chains of batches are the rule.
constexpr int64_t kTwoChainPixels = 4ll << 20;

// Launch shapes of the autotuner: batch, column tile, chains, radix plans
// (vx + 2 vy).
using TunedShape = std::array<int, 4>;
struct TuneSpace {
    int64_t P = 0, B = 0;       // positions; batch depth by the rule
    int64_t plane = 0;          // stored values of a wave
    std::vector<int> plans;     // the rule's first
    std::function<int(int64_t b, int plans, bool beside)> tile; // the automatic tile of a batch
    // a batch takes the one-launch slice loop (null: none does), alone or
    // beside a second chain (null: as alone)
    std::function<bool(int64_t b, int plans)> loop, loop_beside;
    std::function<bool(int tile, int plans)> fused;  // chains 3 fuse their passes
};
// the shape a run of the rules takes
TunedShape tune_rule(const TuneSpace& t);
// The shapes to time: the rule's batch depth, half and twice it; column tiles
// 4, 8 and 16, or where the slice loop runs in one launch, which has no tiles,
// the automatic one; one chain, two chains, or fused batch pairs; and the
// rule's own shape.
std::vector<TunedShape> tune_candidates(const TuneSpace& t);

} // namespace msf
