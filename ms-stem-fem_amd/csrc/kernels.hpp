// kernels.hpp -- host-callable launchers of the device kernels.
//
// Wave layout of the hot path (FP32 complex), for a batch of B probe
// positions on an nx x ny grid whose slice step keeps the columns
// [0, ka) U [ny - kb, ny) (the 2/3 band limit; every other column of the
// (x, ky) representation is identically zero after the first slice):
//   psi[b][i][jc], jc < ncp, ncp >= ka + kb rounded up to the column tile.
// Between the two passes of a slice the wave is held with x along i and k
// along j.  A slice step is
//   row pass    : [IFFT_j] -> transmit -> FFT_j              (one pass over psi)
//   column pass : FFT_i -> mask * P_x * P_y / s -> [IFFT_i]  (one pass over psi)
// Only the scattered part phi = psi - psi0 of the wave is propagated in FP32;
// the vacuum wave psi0 (t = 1) of every slice is computed once per run in FP64.
// The reference's slice operator is linear over the reals (also with its
// in-place transmission update), so phi obeys
//   phi' = M P F[ T(F^-1 phi) + T(u0) - T_vac(u0) ],   u0 = s * shifted psi0(x),
// and FP32 round-off scales with |phi| instead of |psi|.  The first row pass
// has phi = 0; the last column pass adds the shifted vacuum exit wave back.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>
#include <vector>

namespace msf {

// Pair layout of the rows the row pass reads beside the wave (ny even): a
// lane holding elements j and j + ny/2 of a row fetches both with one 16-byte
// read.  Transmission rows store element j at pair_pos(j, ny); u0 rows hold,
// for every shift r in [0, ny), the pair (r, (r + ny/2) mod ny).
__host__ __device__ inline int pair_pos(int j, int n)
{
    return j < n / 2 ? 2 * j : 2 * (j - n / 2) + 1;
}

struct RowPassArgs {
    float2* psi;            // [B][nx][ncp] scattered wave phi
    const float2* t;        // [nx][ny] t - 1 of this slice, rows in the pair layout
    const float2* u0;       // [nx][ny][2] vacuum wave entering this slice, s * real space,
                            // rows as shift pairs (pair_pos)

    const int2* shift;      // [B] probe shifts of the batch
    const float2* tw;       // stage twiddle table of length ny (stage_twiddles)
    float inv_s;            // 1/sqrtNxNy
    int nx, ncp, ka, kb, batch;
    int prune;              // 1: columns [3ny/8, 5ny/8) are outside the kept band
    int plan;               // radix plan of length ny: 0 primary, 1 alternate (has_alt_plan)
    uint32_t div;           // set by the launch: div_mul of the workgroups per row
};

struct ColPassArgs {
    float2* psi;            // [B][nx][ncp]
    const float2* px;       // [nx] propagator along x of this slice
    const float2* py;       // [ny] propagator along y of this slice, scaled by 1/(nx ny)
    const int2* colkeep;    // [ncp] (c, d): kept rows [0, c) U [nx - d, nx) of compact column jc
    const float2* tw;       // stage twiddle table of length nx (stage_twiddles)
    const float2* psi0;     // [ny][nx] vacuum exit wave in k-space, column-major (last pass only)
    const int2* shift;      // [B] probe shifts (last pass only)
    const float2* twx_nat;  // [nx] roots W_nx^e (last pass only)
    const float2* twy;      // [ny] roots W_ny^e (last pass only)
    int ny, ncp, ka, kb, batch;
    int tile;               // columns per workgroup (4, 8 or 16; 0 = default)
    int prune;              // 1: rows [3nx/8, 5nx/8) are masked for every column
    int plan;               // radix plan of length nx: 0 primary, 1 alternate (has_alt_plan)
    int beside;             // 1: another chain of batches runs beside this one (col_tile_auto)
    uint32_t div;           // set by the launch: div_mul of the tiles per position
};
// multiplier for a kernel's division by d (1 <= d < 2^31)
inline uint32_t div_mul(uint32_t d) { return 0xffffffffu / d; }

// One launch with the row pass of one batch (ra) and the column pass of
// another (ca), same transform length n = nx = ny: the rows' FIRST and the
// columns' LAST flags as for the separate passes.  hipErrorNotSupported when
// fused_supported() is false for these arguments.
hipError_t launch_fused_pass(int n, bool first, bool last, int tmode, const RowPassArgs& ra,
                             const ColPassArgs& ca, hipStream_t s);
bool fused_supported(int n, const RowPassArgs& ra, const ColPassArgs& ca);
// true when length n has fused pass pairs for row plan vr, column plan vc and
// column tile `tile` (0: the plan's default)
bool fused_shape_ok(int n, int vr, int vc, int tile);

// The whole slice loop of a batch in one launch, one workgroup per position
// (kernels_loop.hip): both passes' arguments at slice 0, `slices` of them.
// Results equal the passes' bit for bit.
struct LoopArgs {
    RowPassArgs row;
    ColPassArgs col;
    int slices;
};
// true when the grid has such a launch for these arguments and it is the
// faster way for their batch; together: the positions of all batches where
// two chains of them run, else 0
bool loop_supported(int nx, int ny, const RowPassArgs& r, const ColPassArgs& c, int slices,
                    int64_t together);
hipError_t launch_slice_loop(int nx, int ny, int tmode, const LoopArgs& a, hipStream_t s);

// Grouped launches: one launch runs the same pass over the batches of up to
// kGroupMax runs of one transform length (each its own specimen, vacuum
// waves, kept columns and buffers).  Entry k owns launch blocks
// [off[k], off[k+1]), its first block a multiple of 8 (XCD banding within
// the entry); blocks past an entry's own count return at once.
constexpr int kGroupMax = 16;
struct RowGroupArgs {
    int n;
    int off[kGroupMax + 1];
    RowPassArgs a[kGroupMax];
};
struct ColGroupArgs {
    int n;
    int off[kGroupMax + 1];
    ColPassArgs a[kGroupMax];
};
// blocks of one entry (before the padding to a multiple of 8)
int row_group_blocks(int ny, const RowPassArgs& a);
int col_group_blocks(int nx, const ColPassArgs& a);
// Every entry: same length, plan, prune flag and (column pass) tile; the
// rows' FIRST and the columns' LAST flags shared by the launch.
hipError_t launch_row_group(int ny, bool first, int tmode, const RowGroupArgs& g, hipStream_t s);
hipError_t launch_col_group(int nx, bool last, const ColGroupArgs& g, hipStream_t s);
// the column tile a grouped column pass uses with a configured tile `tile`
// (0: the plan's default)
int col_group_tile(int nx, int v, int tile);

bool slice_lengths_ok(int n);
// concatenated per-stage twiddle tables of plan v (0 primary, 1 alternate) of
// length n, (re, im) FP64
bool stage_twiddles(int n, std::vector<double>& re_im, int v = 0);
// What a forward and an inverse FP32 transform of length n together multiply
// the mean amplitude by, against the exact n: 1 but for the rounding of
// sin 60 degrees in the radix-3 step of lengths with a factor 3.  The scale of
// one slice is rounded the same way at every pixel and every slice, so it
// would add up: 4.8e-8 of the intensity per slice.
double fp32_gain(int n);
// true when length n has an alternate radix plan for the slice passes
bool has_alt_plan(int n);
// positions that a row-pass workgroup of length ny and plan v holds
int row_positions(int ny, int v);
// the column count of the compact wave is padded to a multiple of this
int col_tile(int nx);
// the column-pass tile width used when none is configured, for plan v, alone
// or beside another chain of batches
int col_tile_default(int nx, int v = 0, bool beside = false);
// the tile used when none is configured: the default, or one column per
// workgroup when the launch would not give every CU a workgroup
int col_tile_auto(int nx, int v, int batch, int ncp, bool beside);
// true when the kept set leaves [3n/8, 5n/8) empty along the row (ka, kb) and
// every row i in [3nx/8, 5nx/8) fully masked (keep ranges)
bool row_prunable(int ny, int ka, int kb);
bool col_prunable(int nx, const int32_t* keep_ab);

// ev0/ev1 (optional): events the dispatch itself records at the kernel's
// start and end, for profiling without marker overhead
hipError_t launch_row_pass(int ny, bool first, int transmit_mode, const RowPassArgs& a,
                           hipStream_t s, hipEvent_t ev0 = nullptr, hipEvent_t ev1 = nullptr);
hipError_t launch_col_pass(int nx, bool last, const ColPassArgs& a, hipStream_t s,
                           hipEvent_t ev0 = nullptr, hipEvent_t ev1 = nullptr);

// per (position, segment) FP64 sums over interleaved pixel tiles:
// kind 0 -> |psi|^2, 1 -> |psi|; then per (position, group) the fixed-order
// sum of the group's segments
hipError_t launch_reduce_segments(const float2* psi, int64_t plane, const int32_t* pix,
                                  const int32_t* tile_off, const int32_t* seg_kind, int n_tiles,
                                  int batch, double* seg_out, hipStream_t s);
// (small: the groups of at most 64 segments, one lane each; large: the rest,
// one wavefront each; combine_split forms both lists from seg_of_group);
// adf (may be null) gets group 0 of every position
hipError_t launch_combine_segments(const double* seg_in, int n_seg_stride,
                                   const int32_t* seg_of_group, const int32_t* small, int n_small,
                                   const int32_t* large, int n_large, int groups, int batch,
                                   double* out, double* adf, hipStream_t s);
void combine_split(const std::vector<int32_t>& seg_of_group, std::vector<int32_t>& small,
                   std::vector<int32_t>& large);
// FEM statistics of a batch in raster order, from the ring sums at off_abs
// (|psi|) and off_sqr (|psi|^2): d1, the Welford state[3*nbins] = (n, mean,
// M2) and V_omega of the positions so far in v; d2, the Vbar_r sums in vsum
hipError_t launch_fem_stats(const double* partial, int groups, int batch, int nbins, bool d1,
                            bool d2, int off_abs, int off_sqr, const int32_t* counts,
                            const uint8_t* zeroed, double* state, double* v, double* vsum,
                            hipStream_t s);
// FP64 sums over pixel groups of count full-grid FP64 waves: out[count][groups]
hipError_t launch_group_sums_f64(const double2* psi, int64_t plane, const int32_t* offsets,
                                 const int32_t* pixels, const int32_t* kind, int groups,
                                 int count, double* out, hipStream_t s);
// |psi| outside the aperture of full FP64 planes in place; a /= d
hipError_t launch_mtf_magnitude_f64(double2* a, int64_t m, int count, const uint8_t* outside,
                                    hipStream_t s);
hipError_t launch_div_f64(double2* a, int64_t n, double d, hipStream_t s);
// correlograph sums of c and c^2 per (ring, phi sector) over a batch; with
// `each`, also c of every position of the batch ([b][ii + jj * nbins])
hipError_t launch_fem_correlograph(const double* partial, int groups, int batch, int nbins,
                                   int nphi, int off_abs, int off_corr, const int32_t* counts,
                                   const uint8_t* zeroed, double* csum, double* csqr,
                                   double* each, hipStream_t s);
// per-pixel FP64 sums of |psi| and |psi|^2 over the positions of a batch
hipError_t launch_pixel_moments(const float2* psi, int64_t plane, int batch, double* s1,
                                double* s2, hipStream_t s);
// ---------------------------------------------------------------- FP64 set-up
bool setup_lengths_ok(int n);
// in-place 2-D FFT of `count` planes of nx x ny complex doubles (twx, twy:
// stage twiddle tables)
hipError_t fft2d_f64(double2* data, int nx, int ny, int count, bool inverse, const double2* twx,
                     const double2* twy, hipStream_t s);
struct ProbeOptics {
    int corrected;
    double cs3, cs5, defocus, lambda, x0, y0;
};
// probe H(k) of probe_wavefunction.cpp:37-239 inside the aperture ranges
hipError_t launch_probe_k(double2* h, const double* kx, const double* ky, int nx, int ny,
                          const int2* aperture, const ProbeOptics& o, hipStream_t s);
// sum |a|^2 over n values (one workgroup, fixed order)
hipError_t launch_norm2(const double2* a, int64_t n, double* out, hipStream_t s);
// out[0, n16) = in[0, n16), 16-byte vectors; n16 a multiple of 1024
hipError_t launch_stream_copy(const float4* in, float4* out, int64_t n16, hipStream_t s);
// Transmission functions of a chunk of slices [s0, s0 + k).
struct BuildArgs {
    int nx, ny, nsp, k, s0;
    bool half;               // spectra on ky >= 0 only (sb == 0), the rest by conjugation
    int sa, sb, lds;         // columns of the template support [0, sa) U [ny - sb, ny), stride
    int ba, bb, ldb;         // columns of the band limit, stride
    double2* spec;           // [k][nsp][nx][lds]
    double2* band;           // [k][nx][ldb]
    uint32_t* maps;          // [k][nsp][nx][ny] atom counts, zeroed by the caller
    double* tmpl;            // [nsp][nx][lds] f_e lambda gamma / (a b), 0 outside the support
    const int4* atoms;       // (slice, species, sx, sy) of the chunk
    int n_atoms;
    const int2 *support, *bw; // per row
    const double *kx, *ky, *params /* nsp * 12 */;
    double xmin, ymin, lgab, s /* sqrt(nx ny) */, nxny;
    double2* t64;            // [k][nx][ny] t
    float2* t32;             // [k][nx][ny] t - 1, rows in the pair layout
};
// tmpl for every species (projected_atomic_potential.cpp:169-225)
hipError_t launch_templates(const BuildArgs& a, hipStream_t s);
// t64 and t32 of the chunk
hipError_t launch_build(const BuildArgs& a, const double2* twx, const double2* twy, hipStream_t s);
// zero outside the kept ranges
hipError_t launch_apply_keep(double2* a, int nx, int ny, int count, const int2* keep,
                             hipStream_t s);
// one vacuum slice step in k-space: a *= keep ? P_x[i] P_y[j] * scale : 0
hipError_t launch_vacuum_step(double2* a, int nx, int ny, const double2* px, const double2* py,
                              const int2* keep, double scale, hipStream_t s);
// FP64 transmission update of `count` real-space waves by one slice's t
hipError_t launch_transmit_f64(double2* a, const double2* t, int64_t m, int count, int mode,
                               double s, hipStream_t st);
// The detector MTF on a batch of compact FP32 exit waves in place
// (adfstem.cpp:2272-2385).
struct MtfArgs {
    float2* psi;             // [batch][nx][ncp]
    double2* work;           // [batch][nx][ld], ld = col_stride64(ka + kb, ny)
    const double2* mtf;      // [nx][ny] 2-D MTF
    const uint8_t* outside;  // [nx][ny] 1 outside the aperture
    const int2* keep;        // band limit per row
    int nx, ny, ncp, ka, kb, ld, batch;
    double s;                // sqrt(nx ny)
};
hipError_t launch_mtf(const MtfArgs& a, const double2* twx, const double2* twy, hipStream_t s);
// row stride of an FP64 array of nc <= ny columns: an odd number of 128-byte
// lines where that fits in ny columns (fft64_passes.hpp)
int col_stride64(int nc, int ny);
// Vacuum waves entering slices [n0, n1) of S, and with n1 == S the exit wave.
// The aperture's bounding box: rows [0, ra) U [nx - rb, nx), columns [0, ca)
// U [ny - cb, ny).
struct VacuumArgs {
    double2* w;              // work: [n1 - n0][nx][ld], ld = col_stride64(ca + cb, ny)
    float2* psi0;            // [ny][nx] k-space exit wave; pixels off the box are not written
    const double *kx, *ky;
    const int2 *ap, *keep;   // aperture and slice-step ranges per row
    const double2 *px, *py;  // [S][nx], [S][ny]
    ProbeOptics o;
    double norm;             // of H(k): s over the norm of its inverse transform
    int nx, ny, ld, ra, rb, ca, cb, n0, n1, S;
};
// u0: the waves of slices n0, n0 + 1, ... in real space as rows of FP32 shift
// pairs [nx][ny][2] (pair r of a row holds elements r and (r + ny/2) mod ny)
hipError_t launch_vacuum(const VacuumArgs& a, float2* u0, const double2* twx, const double2* twy,
                         hipStream_t s);

} // namespace msf
