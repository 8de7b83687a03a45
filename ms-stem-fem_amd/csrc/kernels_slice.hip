// kernels_slice.hip -- launches of the slice-step passes (slice_passes.hpp)
// one batch at a time, fused pass pairs, and the FP64 detector reductions.
//
// Reference behaviour restated (paths relative to the reference root):
//   reductions  = sum_detected_intensity (func.cpp:2593-2641) and
//                 integrate_out_phi_fftw (variance.cpp:64-300), FP64.
#include <algorithm>
#include <cmath>
#include <vector>

#include <hip/hip_ext.h>

#include "slice_passes.hpp"

namespace msf {

// ------------------------------------------------------- fused pass pair
// One launch runs a row pass of one batch and a column pass of another
// (independent buffers), so that the row workgroups, which compute more, and the
// memory-bound column workgroups share the CUs instead of following each
// other.  Both passes need workgroups of the same size (RT = W * T).  Launch
// blocks alternate in groups of eight, eight of each pass per sixteen, so
// that a pass's logical block k runs on XCD k % 8 as its XCD banding
// assumes (the row pass's block count, groups * nx, is a multiple of 8).
__device__ __forceinline__ bool fused_decode(int b, int nr, int nc, int& id)
{
    const int m8 = (nr < nc ? nr : nc) & ~7;
    if (b < 2 * m8) {
        const int g = b >> 4, k = b & 15;
        id = g * 8 + (k & 7);
        return k < 8;
    }
    const int r = b - 2 * m8;
    if (r < nr - m8) {
        id = m8 + r;
        return true;
    }
    id = m8 + (r - (nr - m8));
    return false;
}

template <int N, int VR, int VC, bool FIRST, bool LAST, int TMODE, bool PR, bool PC, int W, int RT>
__global__ void __launch_bounds__(RT) fused_pass_kernel(RowPassArgs ra, ColPassArgs ca, int nr, int nc)
{
    constexpr int LR = row_smem_len<N, VR, RT>(), LC = col_smem_len<N, VC, LAST, W>();
    __shared__ __align__(16) float2 smem[LR > LC ? LR : LC];
    int id = 0;
    if (fused_decode((int)blockIdx.x, nr, nc, id))
        row_body<N, VR, FIRST, TMODE, PR, RT>(ra, id, smem);
    else
        col_body<N, VC, LAST, W, PC>(ca, id, nc, smem);
}

// ---------------------------------------------------------------- dispatch
bool slice_lengths_ok(int n)
{
    switch (n) {
    case 16: case 32: case 64: case 96: case 128: case 192: case 256: case 384: case 512:
    case 768: case 1024:
        return true;
    default:
        return false;
    }
}

template <typename P> static void stage_table(std::vector<double>& out)
{
    out.clear();
    int ns = 1;
    for (int s = 0; s < P::kStages; ++s) {
        const int r = P::kRadix[s];
        if (ns > 1)
            for (int q = 1; q < r; ++q)
                for (int k = 0; k < ns; ++k) {
                    const long m = (long)ns * r;
                    const double a = 2.0 * M_PI * (double)(((long)q * k) % m) / (double)m;
                    out.push_back(std::cos(a));
                    out.push_back(-std::sin(a));
                }
        ns *= r;
    }
}

template <int N> static bool stage_table_v(int v, std::vector<double>& out)
{
    if (v == 0) {
        stage_table<Plan<N>>(out);
        return (int)out.size() == 2 * plan_tw_len<Plan<N>>();
    }
    if constexpr (AltPlan<N>::exists) {
        stage_table<AltPlan<N>>(out);
        return (int)out.size() == 2 * plan_tw_len<AltPlan<N>>();
    }
    return false;
}

bool stage_twiddles(int n, std::vector<double>& re_im, int v)
{
    switch (n) {
#define MSF_CASE(N) case N: return stage_table_v<N>(v, re_im);
        MSF_CASE(16) MSF_CASE(32) MSF_CASE(64) MSF_CASE(96) MSF_CASE(128) MSF_CASE(192)
        MSF_CASE(256) MSF_CASE(384) MSF_CASE(512) MSF_CASE(768) MSF_CASE(1024)
#undef MSF_CASE
    default:
        return false;
    }
}

bool has_alt_plan(int n)
{
    switch (n) {
#define MSF_CASE(N) case N: return AltPlan<N>::exists;
        MSF_CASE(16) MSF_CASE(32) MSF_CASE(64) MSF_CASE(96) MSF_CASE(128) MSF_CASE(192)
        MSF_CASE(256) MSF_CASE(384) MSF_CASE(512) MSF_CASE(768) MSF_CASE(1024)
#undef MSF_CASE
    default:
        return false;
    }
}

bool row_prunable(int ny, int ka, int kb)
{
    const int lo = (3 * ny + 7) / 8, hi = (5 * ny) / 8;
    return ka <= lo && ny - kb >= hi && ka >= ny / 4 && kb >= ny / 4;
}

bool col_prunable(int nx, const int32_t* ab)
{
    const int lo = (3 * nx + 7) / 8, hi = (5 * nx) / 8;
    for (int i = lo; i < hi; ++i)
        if (ab[2 * i] != 0 || ab[2 * i + 1] != 0) return false;
    return true;
}

int row_positions(int ny, int v)
{
    switch (ny) {
#define MSF_CASE(N)                                                                                \
    case N: {                                                                                      \
        constexpr int A = AltPlan<N>::exists ? 1 : 0;                                              \
        return v ? row_threads<N, A>() / PlanV<N, A>::T : row_threads<N, 0>() / PlanV<N, 0>::T;    \
    }
        MSF_CASE(16) MSF_CASE(32) MSF_CASE(64) MSF_CASE(96) MSF_CASE(128) MSF_CASE(192)
        MSF_CASE(256) MSF_CASE(384) MSF_CASE(512) MSF_CASE(768) MSF_CASE(1024)
#undef MSF_CASE
    default:
        return 1;
    }
}

int col_tile(int nx)
{
    switch (nx) {
#define MSF_CASE(N) case N: return ColTile<N>::WMAX;
        MSF_CASE(16) MSF_CASE(32) MSF_CASE(64) MSF_CASE(96) MSF_CASE(128) MSF_CASE(192)
        MSF_CASE(256) MSF_CASE(384) MSF_CASE(512) MSF_CASE(768) MSF_CASE(1024)
#undef MSF_CASE
    default:
        return 0;
    }
}

// 16-column tiles of a length that a CU holds at once; 0 for lengths of which
// 8 columns do not fill a wavefront (16 and 32): their tiles of 8 leave half
// or more of its lanes idle (12 slices, per column pass: 400 positions of 16 x 64
// 4.4 us with tiles of 16, 5.6 with 8; 900 of 16 x 256 14.0 and 20.2; 900 of
// 32 x 256 15.0 and 20.0; 900 of 64 x 32 10.3 and 9.3)
static int col_places16(int nx, int v)
{
    switch (nx) {
#define MSF_CASE(N) case N: return v ? col_per_cu<N, AltPlan<N>::exists ? 1 : 0, 16>(true) : col_per_cu<N, 0, 16>(true);
        MSF_CASE(64) MSF_CASE(96) MSF_CASE(128) MSF_CASE(192) MSF_CASE(256)
#undef MSF_CASE
    default:
        return 0;
    }
}

// Launches of so few positions that the default tiles would leave CUs idle
// (one position at 512^2: 44 workgroups of 8 columns for 256 CUs) take one
// column per workgroup instead.
// Launches of less than two rounds of 16-column tiles, with the GPU to
// themselves, take tiles of 8, whose last round leaves fewer CUs idle: column pass of 99 positions of 256^2
// (1,089 tiles of 16 for 1,024 places) 16.8 -> 16.0 us, of 192 26.8 -> 26.3,
// of 91 positions of 192 x 96 10.2 -> 9.5; 256 positions (2.75 rounds) 32.5
// against 33.0 with tiles of 8.  Beside a second chain its passes fill those
// CUs, and tiles of 16 stay: two batches on two chains, 12 slices, tiles of 8
// against 16: 256^2 96 positions a batch (1.03 rounds) 775 -> 732 us, 144 983 ->
// 947, 176 1155 -> 1120; 256 x 512 48 809 -> 770, 88 1270 -> 1211; 192^2 176 814 ->
// 750, 272 1063 -> 1056, 296 (1.85 rounds) 1153 -> 1171; 256 x 384 and 256 x 128
// within 2 % either way.  Row workgroups halved by the same rule: 3 % faster at
// 192 x 96, 1 to 2 % slower at 256^2, not kept.
int col_tile_auto(int nx, int v, int batch, int ncp, bool beside)
{
    const int w = col_tile_default(nx, v, beside);
    constexpr int64_t kCUs = 256;
    const int64_t tiles = (int64_t)batch * (ncp / std::max(w, 1));
    if (tiles < kCUs) return 1;
    return w == 16 && !beside && tiles < 2 * kCUs * col_places16(nx, v) ? 8 : w;
}

// The difference of two of a 3-point step's inputs carries a third of the
// energy and is the part scaled by sin 60 (squared amplitude 1 + 2 err); twice,
// for the forward and the inverse step.
double fp32_gain(int n)
{
    constexpr double s60 = 0.86602540378443864676;
    return n % 3 == 0 ? 1.0 + 2.0 * ((double)(float)s60 / s60 - 1.0) / 3.0 : 1.0;
}

// The alternate 1024 plan takes 4 columns where its launches have the GPU to
// themselves (64 positions of 1024 x 1024, 20 slices, one chain: 7.66 ms
// against 7.81 with 8) and 8 beside the row passes of a second chain: those
// hide what the larger tile loses in residency, and its 64-byte segments
// leave them more of the memory (two chains: 1024 x 1024, 50 slices, 256
// positions 72.7 -> 69.9 ms; 1024 x 512 13.4 -> 12.7, 1024 x 768 11.6 -> 11.0;
// 1024 x 128 and 1024 x 256 within 2 % either way).
int col_tile_default(int nx, int v, bool beside)
{
    if (nx == 1024 && v == 1 && beside) return 8;
    switch (nx) {
#define MSF_CASE(N) case N: return v ? ColTile<N, 1>::W : ColTile<N>::W;
        MSF_CASE(16) MSF_CASE(32) MSF_CASE(64) MSF_CASE(96) MSF_CASE(128) MSF_CASE(192)
        MSF_CASE(256) MSF_CASE(384) MSF_CASE(512) MSF_CASE(768) MSF_CASE(1024)
#undef MSF_CASE
    default:
        return 0;
    }
}

// With ev0/ev1 the dispatch packet itself stamps the kernel's start and end
// (hipExtLaunchKernelGGL), so profiled durations carry no marker overhead.
template <int NY, int V, int RT>
static hipError_t row_pass_rt(bool first, int tmode, RowPassArgs a, hipStream_t s,
                              hipEvent_t ev0, hipEvent_t ev1)
{
    constexpr int RPW = RT / PlanV<NY, V>::T;
    const int64_t groups = (a.batch + RPW - 1) / RPW;
    a.div = div_mul((uint32_t)groups);
    const dim3 grid((unsigned)(groups * a.nx));
    const dim3 block(RT);
#define MSF_ROW(F, M, PR)                                                                          \
    do {                                                                                           \
        if (ev0) hipExtLaunchKernelGGL((row_pass_kernel<NY, V, F, M, PR, RT>), grid, block, 0, s,  \
                                       ev0, ev1, 0, a);                                            \
        else hipLaunchKernelGGL((row_pass_kernel<NY, V, F, M, PR, RT>), grid, block, 0, s, a);    \
    } while (0)
    if (a.prune) {
        if (first) { if (tmode == 0) MSF_ROW(true, 0, true); else MSF_ROW(true, 1, true); }
        else { if (tmode == 0) MSF_ROW(false, 0, true); else MSF_ROW(false, 1, true); }
    } else {
        if (first) { if (tmode == 0) MSF_ROW(true, 0, false); else MSF_ROW(true, 1, false); }
        else { if (tmode == 0) MSF_ROW(false, 0, false); else MSF_ROW(false, 1, false); }
    }
#undef MSF_ROW
    return hipGetLastError();
}

// rows per workgroup follow the batch: a batch smaller than a full
// workgroup's rows launches one row per workgroup
template <int NY, int V>
static hipError_t row_pass_nv(bool first, int tmode, const RowPassArgs& a, hipStream_t s,
                              hipEvent_t ev0, hipEvent_t ev1)
{
    constexpr int RT = row_threads<NY, V>(), T = PlanV<NY, V>::T;
    if constexpr (RT > T) {
        if (a.batch < RT / T) return row_pass_rt<NY, V, T>(first, tmode, a, s, ev0, ev1);
    }
    return row_pass_rt<NY, V, RT>(first, tmode, a, s, ev0, ev1);
}

template <int NY>
static hipError_t row_pass_n(bool first, int tmode, const RowPassArgs& a, hipStream_t s,
                             hipEvent_t ev0, hipEvent_t ev1)
{
    if (a.plan == 0) return row_pass_nv<NY, 0>(first, tmode, a, s, ev0, ev1);
    if constexpr (AltPlan<NY>::exists) {
        if (a.plan == 1) return row_pass_nv<NY, 1>(first, tmode, a, s, ev0, ev1);
    }
    return hipErrorInvalidValue;
}

hipError_t launch_row_pass(int ny, bool first, int tmode, const RowPassArgs& a, hipStream_t s,
                           hipEvent_t ev0, hipEvent_t ev1)
{
    switch (ny) {
#define MSF_CASE(N) case N: return row_pass_n<N>(first, tmode, a, s, ev0, ev1);
        MSF_CASE(16) MSF_CASE(32) MSF_CASE(64) MSF_CASE(96) MSF_CASE(128) MSF_CASE(192)
        MSF_CASE(256) MSF_CASE(384) MSF_CASE(512) MSF_CASE(768) MSF_CASE(1024)
#undef MSF_CASE
    default:
        return hipErrorInvalidValue;
    }
}

template <int NX, int V, int W>
static hipError_t col_pass_w(bool last, ColPassArgs a, hipStream_t s, hipEvent_t ev0,
                             hipEvent_t ev1)
{
    if (a.ncp % W || a.ka + a.kb <= 0) return hipErrorInvalidValue;
    a.div = div_mul((uint32_t)((a.ka + a.kb + W - 1) / W));
    const dim3 grid((unsigned)((int64_t)a.batch * ((a.ka + a.kb + W - 1) / W)));
    const dim3 block(W * PlanV<NX, V>::T);
#define MSF_COL(L, PR)                                                                             \
    do {                                                                                           \
        if (ev0) hipExtLaunchKernelGGL((col_pass_kernel<NX, V, L, W, PR>), grid, block, 0, s,      \
                                       ev0, ev1, 0, a);                                            \
        else hipLaunchKernelGGL((col_pass_kernel<NX, V, L, W, PR>), grid, block, 0, s, a);        \
    } while (0)
    if (a.prune) {
        if (last) MSF_COL(true, true);
        else MSF_COL(false, true);
    } else {
        if (last) MSF_COL(true, false);
        else MSF_COL(false, false);
    }
#undef MSF_COL
    return hipGetLastError();
}

template <int NX, int V>
static hipError_t col_pass_nv(bool last, const ColPassArgs& a, hipStream_t s, hipEvent_t ev0,
                              hipEvent_t ev1)
{
    int w = col_tile_auto(NX, V, a.batch, a.ncp, a.beside != 0);
    if (a.tile == 4 || a.tile == 8 || a.tile == 16) w = a.tile;
    if (w == 1) return col_pass_w<NX, V, 1>(last, a, s, ev0, ev1);
    if constexpr (col_fits<NX, V, 16>()) {
        if (w == 16) return col_pass_w<NX, V, 16>(last, a, s, ev0, ev1);
    }
    if (w == 4) return col_pass_w<NX, V, 4>(last, a, s, ev0, ev1);
    return col_pass_w<NX, V, 8>(last, a, s, ev0, ev1);
}

template <int NX>
static hipError_t col_pass_n(bool last, const ColPassArgs& a, hipStream_t s, hipEvent_t ev0,
                             hipEvent_t ev1)
{
    if (a.plan == 0) return col_pass_nv<NX, 0>(last, a, s, ev0, ev1);
    if constexpr (AltPlan<NX>::exists) {
        if (a.plan == 1) return col_pass_nv<NX, 1>(last, a, s, ev0, ev1);
    }
    return hipErrorInvalidValue;
}

hipError_t launch_col_pass(int nx, bool last, const ColPassArgs& a, hipStream_t s,
                           hipEvent_t ev0, hipEvent_t ev1)
{
    switch (nx) {
#define MSF_CASE(N) case N: return col_pass_n<N>(last, a, s, ev0, ev1);
        MSF_CASE(16) MSF_CASE(32) MSF_CASE(64) MSF_CASE(96) MSF_CASE(128) MSF_CASE(192)
        MSF_CASE(256) MSF_CASE(384) MSF_CASE(512) MSF_CASE(768) MSF_CASE(1024)
#undef MSF_CASE
    default:
        return hipErrorInvalidValue;
    }
}

// Fused pass pairs exist for the lengths whose default row and column
// workgroups have the same size: 256 (alternate plans: 16 rows x 16 lanes,
// 16 columns x 16 lanes), 384 (8 x 32, 8 x 32) and 512 (8 x 64, 8 x 64),
// with both passes pruned.
template <int N> struct FusedShape { static constexpr bool exists = false; };
template <> struct FusedShape<256> { static constexpr bool exists = true; static constexpr int VR = 1, VC = 1; };
template <> struct FusedShape<384> { static constexpr bool exists = true; static constexpr int VR = 0, VC = 0; };
template <> struct FusedShape<512> { static constexpr bool exists = true; static constexpr int VR = 0, VC = 0; };

template <int N> static bool fused_ok(const RowPassArgs& ra, const ColPassArgs& ca)
{
    if constexpr (!FusedShape<N>::exists) {
        return false;
    } else {
        constexpr int VR = FusedShape<N>::VR, VC = FusedShape<N>::VC;
        constexpr int RT = row_threads<N, VR>(), W = ColTile<N, VC>::W;
        static_assert(RT == W * PlanV<N, VC>::T, "fused workgroups must match");
        const int w = (ca.tile == 4 || ca.tile == 8 || ca.tile == 16) ? ca.tile : W;
        return ra.plan == VR && ca.plan == VC && w == W && ra.prune && ca.prune &&
               ra.batch >= RT / PlanV<N, VR>::T && ca.ncp % W == 0 && ra.nx == N && ca.ny == N;
    }
}

template <int N> static bool fused_shape_n(int vr, int vc, int tile)
{
    if constexpr (!FusedShape<N>::exists) {
        return false;
    } else {
        constexpr int W = ColTile<N, FusedShape<N>::VC>::W;
        return vr == FusedShape<N>::VR && vc == FusedShape<N>::VC && (tile == 0 || tile == W);
    }
}

bool fused_shape_ok(int n, int vr, int vc, int tile)
{
    switch (n) {
    case 256: return fused_shape_n<256>(vr, vc, tile);
    case 384: return fused_shape_n<384>(vr, vc, tile);
    case 512: return fused_shape_n<512>(vr, vc, tile);
    default: return false;
    }
}

bool fused_supported(int n, const RowPassArgs& ra, const ColPassArgs& ca)
{
    switch (n) {
    case 256: return fused_ok<256>(ra, ca);
    case 384: return fused_ok<384>(ra, ca);
    case 512: return fused_ok<512>(ra, ca);
    default: return false;
    }
}

template <int N>
static hipError_t fused_n(bool first, bool last, int tmode, RowPassArgs ra, ColPassArgs ca,
                          hipStream_t s)
{
    if constexpr (!FusedShape<N>::exists) {
        return hipErrorNotSupported;
    } else {
        if (!fused_ok<N>(ra, ca)) return hipErrorNotSupported;
        constexpr int VR = FusedShape<N>::VR, VC = FusedShape<N>::VC;
        constexpr int RT = row_threads<N, VR>(), W = ColTile<N, VC>::W;
        constexpr int RPW = RT / PlanV<N, VR>::T;
        const int nr = ((ra.batch + RPW - 1) / RPW) * ra.nx;
        const int nc = ca.batch * ((ca.ka + ca.kb + W - 1) / W);
        ra.div = div_mul((uint32_t)((ra.batch + RPW - 1) / RPW));
        ca.div = div_mul((uint32_t)((ca.ka + ca.kb + W - 1) / W));
        const dim3 grid((unsigned)(nr + nc)), block(RT);
#define MSF_FUSED(F, L, M)                                                                         \
    hipLaunchKernelGGL((fused_pass_kernel<N, VR, VC, F, L, M, true, true, W, RT>), grid, block, 0,  \
                       s, ra, ca, nr, nc)
        if (first) {
            if (last) { if (tmode == 0) MSF_FUSED(true, true, 0); else MSF_FUSED(true, true, 1); }
            else { if (tmode == 0) MSF_FUSED(true, false, 0); else MSF_FUSED(true, false, 1); }
        } else {
            if (last) { if (tmode == 0) MSF_FUSED(false, true, 0); else MSF_FUSED(false, true, 1); }
            else { if (tmode == 0) MSF_FUSED(false, false, 0); else MSF_FUSED(false, false, 1); }
        }
#undef MSF_FUSED
        return hipGetLastError();
    }
}

hipError_t launch_fused_pass(int n, bool first, bool last, int tmode, const RowPassArgs& ra,
                             const ColPassArgs& ca, hipStream_t s)
{
    switch (n) {
    case 256: return fused_n<256>(first, last, tmode, ra, ca, s);
    case 384: return fused_n<384>(first, last, tmode, ra, ca, s);
    case 512: return fused_n<512>(first, last, tmode, ra, ca, s);
    default: return hipErrorNotSupported;
    }
}

// ------------------------------------------------------------- reductions
// Each lane sums one segment of a ring's pixel list in FP64, in a fixed order;
// the segments of a ring are then added in segment order.  Neither depends on
// the batch composition.
__global__ void __launch_bounds__(256) reduce_segments_kernel(const float2* psi, int64_t plane,
                                                               const int32_t* pix,
                                                               const int32_t* tile_off,
                                                               const int32_t* seg_kind,
                                                               int n_tiles, double* seg_out)
{
    const int lane = threadIdx.x & 63;
    // Tiles follow the groups in ring order, and neighbouring rings read the
    // same cache lines (a FEM ring is narrower than a pixel): give each XCD a
    // contiguous range of (position, tile group) so those reads meet in one L2
    const int gx = (int)gridDim.x;
    const int lin = xcd_band((int)(blockIdx.y * gridDim.x + blockIdx.x), gx * (int)gridDim.y);
    const int b = lin / gx;
    const int w = (lin - b * gx) * 4 + (threadIdx.x >> 6);
    if (w >= n_tiles) return;
    const float2* wave = psi + (int64_t)b * plane;
    const int k0 = tile_off[w], k1 = tile_off[w + 1];
    const bool amp = seg_kind[w * 64 + lane] != 0;
    double acc = 0.0;
    // chunks of 8 pixels: the index loads, then the wave loads (empty slots
    // read element 0), are issued back to back so their latencies overlap;
    // the sum runs over the pixels in the same order as one at a time
    constexpr int C = 8;
    for (int k = k0; k < k1; k += C) {
        int o[C];
#pragma unroll
        for (int j = 0; j < C; ++j) o[j] = (k + j < k1) ? pix[(int64_t)(k + j) * 64 + lane] : -1;
        float2 v[C];
#pragma unroll
        for (int j = 0; j < C; ++j) v[j] = wave[o[j] >= 0 ? o[j] : 0];
#pragma unroll
        for (int j = 0; j < C; ++j) {
            if (o[j] >= 0) {
                const double re = v[j].x, im = v[j].y;
                const double i2 = re * re + im * im;
                acc += amp ? sqrt(i2) : i2;
            }
        }
    }
    seg_out[(int64_t)b * n_tiles * 64 + w * 64 + lane] = acc;
}

hipError_t launch_reduce_segments(const float2* psi, int64_t plane, const int32_t* pix,
                                  const int32_t* tile_off, const int32_t* seg_kind, int n_tiles,
                                  int batch, double* seg_out, hipStream_t s)
{
    if (n_tiles <= 0 || batch <= 0) return hipSuccess;
    const dim3 grid((unsigned)((n_tiles + 3) / 4), (unsigned)batch);
    hipLaunchKernelGGL(reduce_segments_kernel, grid, dim3(256), 0, s, psi, plane, pix, tile_off,
                       seg_kind, n_tiles, seg_out);
    return hipGetLastError();
}

// Group sums from the segment sums, per (group, position), in an order that
// depends on the group only.  Groups of at most kWaveGroup segments: one lane
// adds them in segment order.  Larger groups (the ADF annulus at 1024^2:
// ~5,500 segments): one wavefront, lane l adding segments l, l + 64, ... in
// order, the lanes' sums meeting in a fixed butterfly.
// One launch forms both kinds (blocks below small_blocks: the small groups,
// the rest: one wavefront per large group) and writes group 0, the ADF ring,
// to adf as well, where there were three launches of ~4.5 us each.
constexpr int kWaveGroup = 64;

constexpr int kCombinePos = 4; // positions per workgroup: a small group's index loads serve them all

__global__ void __launch_bounds__(256) combine_segments_kernel(
    const double* seg_in, int n_seg_stride, const int32_t* seg_of_group, const int32_t* small,
    int n_small, int small_blocks, const int32_t* large, int groups, int batch, double* out,
    double* adf)
{
    if ((int)blockIdx.x < small_blocks) {
        const int id = (int)blockIdx.x * 256 + (int)threadIdx.x;
        if (id >= n_small) return;
        const int g = small[id];
        const int s0 = seg_of_group[g], s1 = seg_of_group[g + 1];
        const int b0 = (int)blockIdx.y * kCombinePos;
        const double* in[kCombinePos]; // positions past the batch repeat its last and store nothing
        double acc[kCombinePos] = {};
#pragma unroll
        for (int j = 0; j < kCombinePos; ++j)
            in[j] = seg_in + (int64_t)min(b0 + j, batch - 1) * n_seg_stride;
        for (int k = s0; k < s1; ++k)
#pragma unroll
            for (int j = 0; j < kCombinePos; ++j) acc[j] += in[j][k];
#pragma unroll
        for (int j = 0; j < kCombinePos; ++j)
            if (b0 + j < batch) {
                out[(int64_t)(b0 + j) * groups + g] = acc[j];
                if (adf && g == 0) adf[b0 + j] = acc[j];
            }
        return;
    }
    // one large group per workgroup, one position per wavefront
    const int b = (int)blockIdx.y * kCombinePos + (int)(threadIdx.x >> 6);
    if (b >= batch) return; // whole wavefronts
    const int lane = threadIdx.x & 63;
    const int g = large[(int)blockIdx.x - small_blocks];
    const int s1 = seg_of_group[g + 1];
    const double* in = seg_in + (int64_t)b * n_seg_stride;
    double acc = 0.0;
#pragma unroll 8
    for (int k = seg_of_group[g] + lane; k < s1; k += 64) acc += in[k];
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) acc += __shfl_xor(acc, off);
    if (lane == 0) {
        out[(int64_t)b * groups + g] = acc;
        if (adf && g == 0) adf[b] = acc;
    }
}

void combine_split(const std::vector<int32_t>& seg_of_group, std::vector<int32_t>& small,
                   std::vector<int32_t>& large)
{
    small.clear();
    large.clear();
    for (size_t g = 0; g + 1 < seg_of_group.size(); ++g)
        (seg_of_group[g + 1] - seg_of_group[g] > kWaveGroup ? large : small).push_back((int32_t)g);
}

hipError_t launch_combine_segments(const double* seg_in, int n_seg_stride,
                                   const int32_t* seg_of_group, const int32_t* small, int n_small,
                                   const int32_t* large, int n_large, int groups, int batch,
                                   double* out, double* adf, hipStream_t s)
{
    if (batch <= 0 || n_small + n_large <= 0) return hipSuccess;
    const int sb = (n_small + 255) / 256;
    hipLaunchKernelGGL(combine_segments_kernel, dim3((unsigned)(sb + n_large), (unsigned)((batch + kCombinePos - 1) / kCombinePos)),
                       dim3(256), 0, s, seg_in, n_seg_stride, seg_of_group, small, n_small, sb,
                       large, groups, batch, out, adf);
    return hipGetLastError();
}

// Per-bin FEM statistics over a batch in raster order.
//   which 0 (d1): r = radial sum / count (adfstem.cpp:2591-2599), direct-beam
//     bins zeroed first (:2518-2522), Welford (n, mean, M2) in state, and
//     V = Npos sum r^2 / (sum r)^2 - 1 = M2 / (n mean^2), 0 when sum r == 0
//     (:2837-2856), of the positions so far in v;
//   which 1 (d2, Vbar_r, :2688-2750): the sum over positions of
//     ((r2 / c) / ((r1 r1) / (c c))) - 1, r1 and r2 the ring sums of |psi| and
//     |psi|^2 (zero on the direct beam), c*c an integer product.
// Bound by latency: a bin's positions are a serial chain.  A workgroup takes
// 64 bins; its four wavefronts read and divide kStatChunk positions at a time
// into LDS (all loads of a chunk in flight, the next chunk's issued before
// this one's chain), the first wavefront runs the chain, whose steps are two
// dependent FP64 operations (1/n formed beside the loads, so mean += d / n is
// one fma).  One lane per bin that loaded, divided and chained one position
// after another took 34 us for 853 bins x 64 positions and 76 us for
// 42 x 256, and d2 and the final V a launch each; this form 12 and 15 us.
constexpr int kStatBins = 64, kStatChunk = 32;

__global__ void __launch_bounds__(256) fem_stats_kernel(
    const double* partial, int groups, int batch, int nbins, int which0, int off_abs, int off_sqr,
    const int32_t* counts, const uint8_t* zeroed, double* state, double* v, double* vsum)
{
    constexpr int PW = kStatChunk / 4; // positions per wavefront and chunk
    __shared__ double s_x[2][kStatChunk][kStatBins];
    __shared__ double s_inv[2][kStatChunk];
    const bool d1 = which0 + (int)blockIdx.y == 0;
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int k = blockIdx.x * kStatBins + lane;
    const int kc = min(k, nbins - 1); // lanes past the last bin repeat it and store nothing
    const int c = counts[kc];
    const double cd = (double)c, cc = (double)(c * c);
    const bool z = zeroed[kc] != 0;
    // positions before this batch: equal in every bin (own bin: another workgroup's may be updated already)
    const double n0 = d1 ? state[3 * kc] : 0.0;
    double r1[PW], r2[PW];
    auto load = [&](int b0) {
#pragma unroll
        for (int j = 0; j < PW; ++j) {
            const double* p = partial + (int64_t)min(b0 + wv * PW + j, batch - 1) * groups + kc;
            r1[j] = p[off_abs];
            r2[j] = d1 ? 0.0 : p[off_sqr];
        }
    };
    auto put = [&](int b0, int buf) {
#pragma unroll
        for (int j = 0; j < PW; ++j) {
            const double a = z ? 0.0 : r1[j], q = z ? 0.0 : r2[j];
            s_x[buf][wv * PW + j][lane] = d1 ? a / cd : ((q / cd) / ((a * a) / cc)) - 1.0;
        }
        if (threadIdx.x < kStatChunk) s_inv[buf][threadIdx.x] = 1.0 / (n0 + b0 + (threadIdx.x + 1.0));
    };
    double mean = 0.0, m2 = 0.0, acc = 0.0;
    if (wv == 0) {
        if (d1) {
            mean = state[3 * kc + 1];
            m2 = state[3 * kc + 2];
        } else {
            acc = vsum[kc];
        }
    }
    load(0);
    put(0, 0);
    __syncthreads();
    for (int b0 = 0, buf = 0; b0 < batch; b0 += kStatChunk, buf ^= 1) {
        const bool more = b0 + kStatChunk < batch;
        if (more) load(b0 + kStatChunk);
        if (wv == 0) {
            const int n = min(kStatChunk, batch - b0);
            if (d1) {
                for (int j = 0; j < n; ++j) {
                    const double x = s_x[buf][j][lane], d = x - mean;
                    mean = fma(d, s_inv[buf][j], mean);
                    m2 = fma(d, x - mean, m2);
                }
            } else {
                for (int j = 0; j < n; ++j) acc += s_x[buf][j][lane];
            }
        }
        if (more) put(b0 + kStatChunk, buf ^ 1);
        __syncthreads();
    }
    if (wv != 0 || k >= nbins) return;
    if (d1) {
        const double n = n0 + batch;
        state[3 * k] = n;
        state[3 * k + 1] = mean;
        state[3 * k + 2] = m2;
        v[k] = (mean == 0.0) ? 0.0 : m2 / (n * mean * mean);
    } else {
        vsum[k] = acc;
    }
}

hipError_t launch_fem_stats(const double* partial, int groups, int batch, int nbins, bool d1,
                            bool d2, int off_abs, int off_sqr, const int32_t* counts,
                            const uint8_t* zeroed, double* state, double* v, double* vsum,
                            hipStream_t s)
{
    if (nbins <= 0 || batch <= 0 || !(d1 || d2)) return hipSuccess;
    hipLaunchKernelGGL(fem_stats_kernel,
                       dim3((unsigned)((nbins + kStatBins - 1) / kStatBins), d1 && d2 ? 2u : 1u),
                       dim3(256), 0, s, partial, groups, batch, nbins, d1 ? 0 : 1, off_abs, off_sqr,
                       counts, zeroed, state, v, vsum);
    return hipGetLastError();
}

// Correlograph (adfstem.cpp:2603-2650): per position, ring ii and phi sector
// jj, c = count_ii * I_ii,jj / r_ii - 1 when that ratio is >= 1 and count,
// I and r are all non-zero, else 0; I and r are the sector and ring sums of
// |psi| (zero on direct-beam rings).  Sums of c and c^2 over positions in
// raster order, stored [ii + jj * nbins].  The sums of 8 positions are read
// ahead of their products: one at a time the pass waited for each position's
// loads (61 -> 41 us for 853 rings x 159 sectors x 64 positions, 69 MB).
__global__ void __launch_bounds__(256) fem_correlograph_kernel(
    const double* partial, int groups, int batch, int nbins, int nphi, int off_abs, int off_corr,
    const int32_t* counts, const uint8_t* zeroed, double* csum, double* csqr, double* each)
{
    const int k = blockIdx.x * blockDim.x + threadIdx.x; // ii * nphi + jj
    if (k >= nbins * nphi) return;
    const int ii = k / nphi, jj = k - ii * nphi;
    const int64_t o = (int64_t)ii + (int64_t)jj * nbins;
    const int c = counts[ii];
    const bool z = zeroed[ii] != 0;
    double a = csum[o], q = csqr[o];
    auto add = [&](int b, double r, double I) {
        if (z) r = I = 0.0;
        const double t = (c * I / r);
        double v = 0.0;
        if ((t >= 1) && (c != 0) && (I != 0) && (r != 0)) v = t - 1;
        a += v;
        q += v * v;
        if (each) each[(int64_t)b * nbins * nphi + o] = v; // per position (optional)
    };
    constexpr int C = 8;
    const double* w = partial;
    int b = 0;
    for (; b + C <= batch; b += C, w += (int64_t)C * groups) {
        double r[C], I[C];
#pragma unroll
        for (int j = 0; j < C; ++j) {
            r[j] = w[(int64_t)j * groups + off_abs + ii];
            I[j] = w[(int64_t)j * groups + off_corr + k];
        }
#pragma unroll
        for (int j = 0; j < C; ++j) add(b + j, r[j], I[j]);
    }
    for (; b < batch; ++b, w += groups) add(b, w[off_abs + ii], w[off_corr + k]);
    csum[o] = a;
    csqr[o] = q;
}

hipError_t launch_fem_correlograph(const double* partial, int groups, int batch, int nbins,
                                   int nphi, int off_abs, int off_corr, const int32_t* counts,
                                   const uint8_t* zeroed, double* csum, double* csqr,
                                   double* each, hipStream_t s)
{
    if (nbins <= 0 || nphi <= 0 || batch <= 0) return hipSuccess;
    const int n = nbins * nphi;
    hipLaunchKernelGGL(fem_correlograph_kernel, dim3((n + 255) / 256), dim3(256), 0, s, partial,
                       groups, batch, nbins, nphi, off_abs, off_corr, counts, zeroed, csum, csqr,
                       each);
    return hipGetLastError();
}

// FP64 group sums on full-grid FP64 waves (parity entry points): one
// workgroup per (group, wave), strided pixel loop and a fixed-order tree, so
// results do not depend on scheduling.  kind 0 sums |psi|^2, kind 1 |psi|.
__global__ void __launch_bounds__(256) group_sums_f64_kernel(const double2* psi, int64_t plane,
                                                             const int32_t* offsets,
                                                             const int32_t* pixels,
                                                             const int32_t* kind, int groups,
                                                             double* out)
{
    __shared__ double red[256];
    const int g = blockIdx.x, b = blockIdx.y, t = threadIdx.x;
    const double2* w = psi + (int64_t)b * plane;
    const bool amp = kind[g] == 1;
    double acc = 0.0;
    for (int k = offsets[g] + t; k < offsets[g + 1]; k += 256) {
        const double2 v = w[pixels[k]];
        const double i2 = v.x * v.x + v.y * v.y;
        acc += amp ? sqrt(i2) : i2;
    }
    red[t] = acc;
    __syncthreads();
    for (int h = 128; h > 0; h >>= 1) {
        if (t < h) red[t] += red[t + h];
        __syncthreads();
    }
    if (t == 0) out[(int64_t)b * groups + g] = red[0];
}

hipError_t launch_group_sums_f64(const double2* psi, int64_t plane, const int32_t* offsets,
                                 const int32_t* pixels, const int32_t* kind, int groups,
                                 int count, double* out, hipStream_t s)
{
    if (groups <= 0 || count <= 0) return hipSuccess;
    if (groups > 65535 || count > 65535) return hipErrorInvalidValue;
    hipLaunchKernelGGL(group_sums_f64_kernel, dim3((unsigned)groups, (unsigned)count), dim3(256),
                       0, s, psi, plane, offsets, pixels, kind, groups, out);
    return hipGetLastError();
}

// Detector MTF, first step (adfstem.cpp:2279-2292), on full-grid FP64 waves
// in place: |psi| outside the aperture (outside[i*ny+j] != 0), else 0.
__global__ void mtf_magnitude_f64_kernel(double2* a, int64_t m, int64_t total,
                                         const uint8_t* outside)
{
    const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= total) return;
    const double2 w = a[idx];
    const double v = outside[idx % m] ? sqrt((w.x * w.x) + (w.y * w.y)) : 0.0;
    a[idx] = double2{v, 0.0};
}

hipError_t launch_mtf_magnitude_f64(double2* a, int64_t m, int count, const uint8_t* outside,
                                    hipStream_t s)
{
    const int64_t n = m * count;
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(mtf_magnitude_f64_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0,
                       s, a, m, n, outside);
    return hipGetLastError();
}

// a /= d on both parts (the reference divides, it does not scale by 1/d)
__global__ void div_f64_kernel(double2* a, int64_t n, double d)
{
    const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= n) return;
    const double2 w = a[idx];
    a[idx] = double2{w.x / d, w.y / d};
}

hipError_t launch_div_f64(double2* a, int64_t n, double d, hipStream_t s)
{
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(div_f64_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, a, n, d);
    return hipGetLastError();
}

// Per-pixel sums over positions of |psi| and |psi|^2 in raster order, FP64
// (adfstem.cpp:2753-2781), on the compact plane of the exit waves.  8
// positions' waves are read ahead of their sums (56 -> 32 us for 512 x 352
// pixels x 64 positions, 92 MB).
__global__ void __launch_bounds__(256) pixel_moments_kernel(const float2* psi, int64_t plane,
                                                            int batch, double* s1, double* s2)
{
    const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= plane) return;
    double a = s1[p], q = s2[p];
    auto add = [&](float2 v) {
        const double re = v.x, im = v.y;
        const double m2 = re * re + im * im;
        a += sqrt(m2);
        q += m2;
    };
    constexpr int C = 8;
    const float2* w = psi + p;
    int b = 0;
    for (; b + C <= batch; b += C, w += C * plane) {
        float2 v[C];
#pragma unroll
        for (int j = 0; j < C; ++j) v[j] = w[j * plane];
#pragma unroll
        for (int j = 0; j < C; ++j) add(v[j]);
    }
    for (; b < batch; ++b, w += plane) add(*w);
    s1[p] = a;
    s2[p] = q;
}

hipError_t launch_pixel_moments(const float2* psi, int64_t plane, int batch, double* s1,
                                double* s2, hipStream_t s)
{
    if (plane <= 0 || batch <= 0) return hipSuccess;
    hipLaunchKernelGGL(pixel_moments_kernel, dim3((unsigned)((plane + 255) / 256)), dim3(256), 0,
                       s, psi, plane, batch, s1, s2);
    return hipGetLastError();
}

} // namespace msf
