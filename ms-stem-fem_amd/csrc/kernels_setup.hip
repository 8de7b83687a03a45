// kernels_setup.hip -- FP64 specimen and probe set-up on the device.
//
// Transmission functions (slice.cpp:1451-1757).  The reference sums, for every
// atom of a slice, its species template circularly shifted to the atom's
// nearest pixel (slice.cpp:1594-1648): sigma_v = sum_sp tmpl_sp (*) c_sp with
// c_sp the per-pixel atom count map of species sp.  With tmpl_sp =
// IFFT(T_sp)/sqrt(NxNy) (scatterer_pap.hpp:104-174) the same sum is
//     sigma_v = IFFT( sum_sp T_sp(k) * FFT(c_sp)(k) ) / sqrt(NxNy),
// which costs O(N^2 log N) per slice instead of O(atoms * N^2).  The rest
// follows the reference: t = exp(-Im v)(cos Re v, sin Re v), FORWARD FFT,
// bw_limit, BACKWARD FFT, / NxNy.  Everything here is FP64.
//
// Probe (adfstem.cpp:586-817): H(k) inside the aperture, BACKWARD FFT, norm.
#include <algorithm>

#include "fft64_passes.hpp"

namespace msf {

// ------------------------------------------------------------ 2-D FFT, FP64
template <int NY, bool INV>
__global__ void __launch_bounds__(256) fft64_rows_kernel(double2* data, int64_t rows,
                                                         const double2* tw)
{
    using P = Plan<NY>;
    constexpr int E = P::E, T = P::T;
    constexpr int RPW = 256 / T;
    constexpr int LEN = lds_len(NY);
    __shared__ double2 s_tw[stage_tw_len<NY>()];
    __shared__ double2 s_buf[RPW * LEN];
    for (int e = threadIdx.x; e < stage_tw_len<NY>(); e += blockDim.x) s_tw[e] = tw[e];
    __syncthreads();
    const int lr = threadIdx.x / T, t = threadIdx.x % T;
    const int64_t r = (int64_t)blockIdx.x * RPW + lr;
    const bool active = r < rows;
    double2* row = data + (active ? r : 0) * NY;
    double2 x[E];
#pragma unroll
    for (int p = 0; p < E; ++p) x[p] = active ? row[t + T * p] : double2{0.0, 0.0};
    P::template run<INV>(x, s_buf + lr * LEN, s_tw, t);
    if (active) {
#pragma unroll
        for (int p = 0; p < E; ++p) row[t + T * p] = x[p];
    }
}

template <int NX, bool INV>
__global__ void __launch_bounds__(256) fft64_cols_kernel(double2* data, int ny, int count,
                                                         const double2* tw)
{
    using P = Plan<NX>;
    constexpr int E = P::E, T = P::T;
    constexpr int W = (256 / T) < 4 ? (256 / T) : 4;
    constexpr int LEN = lds_len(NX);
    __shared__ double2 s_tw[stage_tw_len<NX>()];
    __shared__ double2 s_buf[W * LEN];
    for (int e = threadIdx.x; e < stage_tw_len<NX>(); e += blockDim.x) s_tw[e] = tw[e];
    __syncthreads();
    const int c = threadIdx.x % W, t = threadIdx.x / W;
    const int ntiles = ny / W;
    const int plane = blockIdx.x / ntiles;
    const int j = (blockIdx.x % ntiles) * W + c;
    const bool active = plane < count;
    double2* col = data + (int64_t)(active ? plane : 0) * NX * ny + j;
    double2 x[E];
#pragma unroll
    for (int p = 0; p < E; ++p) x[p] = active ? col[(int64_t)(t + T * p) * ny] : double2{0.0, 0.0};
    P::template run<INV>(x, s_buf + c * LEN, s_tw, t);
    if (active) {
#pragma unroll
        for (int p = 0; p < E; ++p) col[(int64_t)(t + T * p) * ny] = x[p];
    }
}

template <int N> static constexpr int col_w64() { return (256 / Plan<N>::T) < 4 ? (256 / Plan<N>::T) : 4; }

template <int NY>
static hipError_t rows64(double2* d, int64_t rows, bool inv, const double2* tw, hipStream_t s)
{
    constexpr int RPW = 256 / Plan<NY>::T;
    const dim3 grid((unsigned)((rows + RPW - 1) / RPW)), block(RPW * Plan<NY>::T);
    if (inv) hipLaunchKernelGGL((fft64_rows_kernel<NY, true>), grid, block, 0, s, d, rows, tw);
    else hipLaunchKernelGGL((fft64_rows_kernel<NY, false>), grid, block, 0, s, d, rows, tw);
    return hipGetLastError();
}

template <int NX>
static hipError_t cols64(double2* d, int ny, int count, bool inv, const double2* tw, hipStream_t s)
{
    constexpr int W = col_w64<NX>();
    if (ny % W) return hipErrorInvalidValue;
    const dim3 grid((unsigned)((int64_t)count * (ny / W))), block(W * Plan<NX>::T);
    if (inv) hipLaunchKernelGGL((fft64_cols_kernel<NX, true>), grid, block, 0, s, d, ny, count, tw);
    else hipLaunchKernelGGL((fft64_cols_kernel<NX, false>), grid, block, 0, s, d, ny, count, tw);
    return hipGetLastError();
}

bool setup_lengths_ok(int n) { return slice_lengths_ok(n); }

hipError_t fft2d_f64(double2* data, int nx, int ny, int count, bool inverse, const double2* twx,
                     const double2* twy, hipStream_t s)
{
    hipError_t e = hipErrorInvalidValue;
    const int64_t rows = (int64_t)count * nx;
    switch (ny) {
#define MSF_CASE(N) case N: e = rows64<N>(data, rows, inverse, twy, s); break;
        MSF_CASE(16) MSF_CASE(32) MSF_CASE(64) MSF_CASE(96) MSF_CASE(128) MSF_CASE(192)
        MSF_CASE(256) MSF_CASE(384) MSF_CASE(512) MSF_CASE(768) MSF_CASE(1024)
#undef MSF_CASE
    default:
        return hipErrorInvalidValue;
    }
    if (e != hipSuccess) return e;
    switch (nx) {
#define MSF_CASE(N) case N: return cols64<N>(data, ny, count, inverse, twx, s);
        MSF_CASE(16) MSF_CASE(32) MSF_CASE(64) MSF_CASE(96) MSF_CASE(128) MSF_CASE(192)
        MSF_CASE(256) MSF_CASE(384) MSF_CASE(512) MSF_CASE(768) MSF_CASE(1024)
#undef MSF_CASE
    default:
        return hipErrorInvalidValue;
    }
}

// ------------------------------------------------------------ probe
constexpr double kPi = 3.14159265369; // the reference's PI

// probe_wavefunction.cpp:37-137 / :139-239 with lenses.cpp:249-290
__device__ __forceinline__ double2 probe_h(double kx, double ky, const ProbeOptics& o)
{
    const double lsq = o.lambda * o.lambda;
    const double ksqr = kx * kx + ky * ky;
    double chi;
    if (o.corrected) {
        const double kl = ksqr * lsq;
        chi = kPi * o.lambda * ksqr * (-o.defocus + 0.5 * o.cs3 * kl + (1.0 / 3.0) * o.cs5 * (kl * kl));
    } else {
        chi = kPi * o.lambda * ksqr * (0.5 * o.cs3 * lsq * ksqr - o.defocus);
    }
    const double trig = chi + 2 * kPi * ((kx * o.x0) + (ky * o.y0));
    double sn, cs;
    sincos(trig, &sn, &cs);
    return double2{cs, -1.0 * sn};
}

__global__ void probe_k_kernel(double2* h, const double* kx, const double* ky, int nx, int ny,
                               const int2* ap, ProbeOptics o)
{
    const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= (int64_t)nx * ny) return;
    const int i = (int)(idx / ny), j = (int)(idx % ny);
    const int2 r = ap[i];
    double2 v{0.0, 0.0};
    if (j < r.x || j >= ny - r.y) v = probe_h(kx[i], ky[j], o);
    h[idx] = v;
}

hipError_t launch_probe_k(double2* h, const double* kx, const double* ky, int nx, int ny,
                          const int2* aperture, const ProbeOptics& o, hipStream_t s)
{
    const int64_t n = (int64_t)nx * ny;
    hipLaunchKernelGGL(probe_k_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, h, kx,
                       ky, nx, ny, aperture, o);
    return hipGetLastError();
}

// single workgroup, fixed thread count and tree: deterministic
__global__ void __launch_bounds__(1024) norm2_kernel(const double2* a, int64_t n, double* out)
{
    __shared__ double s[1024];
    double acc = 0.0;
    for (int64_t k = threadIdx.x; k < n; k += 1024) acc += a[k].x * a[k].x + a[k].y * a[k].y;
    s[threadIdx.x] = acc;
    __syncthreads();
    for (int w = 512; w >= 1; w >>= 1) {
        if ((int)threadIdx.x < w) s[threadIdx.x] += s[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0) *out = s[0];
}

hipError_t launch_norm2(const double2* a, int64_t n, double* out, hipStream_t s)
{
    hipLaunchKernelGGL(norm2_kernel, dim3(1), dim3(1024), 0, s, a, n, out);
    return hipGetLastError();
}

// ------------------------------------------------------------ measurement
// A streaming copy at the rate HBM sustains for a plain read + write: each
// lane moves four 16-byte vectors, the four loads issued before the stores.
// n16 is a multiple of 4 * 256 (the caller sizes the buffers so).
__global__ void __launch_bounds__(256) stream_copy_kernel(const float4* __restrict__ in,
                                                           float4* __restrict__ out)
{
    const int64_t base = (int64_t)blockIdx.x * (4 * 256) + threadIdx.x;
    float4 v[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) v[k] = in[base + k * 256];
#pragma unroll
    for (int k = 0; k < 4; ++k) out[base + k * 256] = v[k];
}

hipError_t launch_stream_copy(const float4* in, float4* out, int64_t n16, hipStream_t s)
{
    if (n16 <= 0 || n16 % (4 * 256)) return hipErrorInvalidValue;
    hipLaunchKernelGGL(stream_copy_kernel, dim3((unsigned)(n16 / (4 * 256))), dim3(256), 0, s, in,
                       out);
    return hipGetLastError();
}

// ------------------------------------------------------------ transmission
// Passes of one chunk of slices (columns of `spec` and `band` only):
//   scatter  atoms -> count maps (small integers, so the atomic sums are exact
//            and order-independent)
//   rows     FFT_y of the maps                              -> spec
//   columns  sum_sp T_sp(k) FFT_x(spec), IFFT_x             -> spec
//   rows     IFFT_y, t = exp(-Im v)(cos Re v, sin Re v), FFT_y -> band
//   columns  FFT_x, bw_limit, IFFT_x                        -> band (in place)
//   rows     IFFT_y, / NxNy                                 -> t64, t32
// Each transform pair shares a pass with the element-wise work between and
// around it, and only columns that carry data are stored (half the spectrum
// of a real map, 2/3 of a band-limited plane): 25 slices of 1024^2 with one
// species move 2.8 GB instead of 7.5 GB in eleven passes over full planes,
// whose column passes also lost half of each 128-byte line to another XCD;
// the kernels of that build went from 3.6 to 1.2 ms.
__global__ void scatter_atoms_kernel(BuildArgs a)
{
    const int n = blockIdx.x * blockDim.x + threadIdx.x;
    if (n >= a.n_atoms) return;
    const int4 at = a.atoms[n];
    atomicAdd(&a.maps[(((int64_t)(at.x - a.s0) * a.nsp + at.y) * a.nx + at.z) * a.ny + at.w], 1u);
}

// projected_atomic_potential.cpp:169-225: lambda*gamma/(ab) * f_e(|k|^2)
// inside the template support
__global__ void __launch_bounds__(256) template_kernel(BuildArgs a)
{
    const int nc = a.sa + a.sb;
    const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (idx >= (int64_t)a.nsp * a.nx * nc) return;
    const int c = (int)(idx % nc);
    const int64_t r = idx / nc;
    const int i = (int)(r % a.nx), sp = (int)(r / a.nx);
    const int j = c < a.sa ? c : c + a.ny - nc;
    const int2 k = a.support[i];
    double t = 0.0;
    if (j < k.x || j >= a.ny - k.y) {
        const double ksq = (a.kx[i] * a.kx[i]) + (a.ky[j] * a.ky[j]);
        const double* p = a.params + 12 * sp;
        t = a.lgab * (p[0] / (ksq + p[3]) + p[1] / (ksq + p[4]) + p[2] / (ksq + p[5])
                      + p[6] * exp(-p[9] * ksq) + p[7] * exp(-p[10] * ksq)
                      + p[8] * exp(-p[11] * ksq));
    }
    a.tmpl[r * a.lds + c] = t;
}

hipError_t launch_templates(const BuildArgs& a, hipStream_t s)
{
    const int64_t n = (int64_t)a.nsp * a.nx * (a.sa + a.sb);
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(template_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, a);
    return hipGetLastError();
}

struct MapRows {
    const uint32_t* maps;
    double2* spec;
    int nx, ny, sa, sb, lds;
    __device__ __forceinline__ double2 load(int plane, int i, int j) const
    {
        return double2{(double)maps[((int64_t)plane * nx + i) * ny + j], 0.0};
    }
    template <int E, int T>
    __device__ __forceinline__ void store(int plane, int i, int t, const double2 (&x)[E]) const
    {
        double2* row = spec + ((int64_t)plane * nx + i) * lds;
#pragma unroll
        for (int p = 0; p < E; ++p) {
            const int j = t + T * p;
            if (j < sa) row[j] = x[p];
            else if (j >= ny - sb) row[j - ny + sa + sb] = x[p];
        }
    }
};

struct SpeciesCols {
    int inputs;
    double2* spec;
    const double *tmpl, *kx, *ky;
    int nx, ny, sa, sb, lds;
    bool origin; // domain minima at 0: the template's phase is 1
    double xmin, ymin;
    __device__ __forceinline__ double2 load(int plane, int in, int i, int c) const
    {
        return spec[(((int64_t)plane * inputs + in) * nx + i) * lds + c];
    }
    __device__ __forceinline__ double2 mid(int, int in, int i, int c, double2 v) const
    {
        const double f = tmpl[((int64_t)in * nx + i) * lds + c];
        if (origin) return double2{f * v.x, f * v.y};
        const int j = c < sa ? c : c + ny - sa - sb;
        double sn, cs;
        sincos(2 * kPi * (kx[i] * xmin + ky[j] * ymin), &sn, &cs);
        const double2 t{f * cs, f * sn};
        return double2{t.x * v.x - t.y * v.y, t.x * v.y + t.y * v.x};
    }
    __device__ __forceinline__ void store(int plane, int i, int c, double2 v) const
    {
        spec[((int64_t)plane * inputs * nx + i) * lds + c] = v; // over species 0
    }
};

// slice.cpp:1700-1725
struct TransmitRows {
    const double2* spec; // null: no atoms
    double2* band;
    int nsp, nx, ny, sa, sb, lds, ba, bb, ldb;
    bool half;
    double scale;
    __device__ __forceinline__ double2 load(int plane, int i, int j) const
    {
        if (!spec) return double2{0.0, 0.0};
        const double2* row = spec + ((int64_t)plane * nsp * nx + i) * lds;
        if (j < sa) return row[j];
        if (half) {
            if (ny - j >= sa) return double2{0.0, 0.0};
            const double2 v = row[ny - j];
            return double2{v.x, -v.y};
        }
        return j >= ny - sb ? row[j - ny + sa + sb] : double2{0.0, 0.0};
    }
    __device__ __forceinline__ double2 mid(int, int, int, double2 v) const
    {
        const double re = v.x * scale, im = v.y * scale;
        // Im v is rounding of a real sum; exp of so small a value by its
        // series (the next term is below 2e-19)
        const double e = fabs(im) < 1e-6 ? 1.0 - im + 0.5 * im * im : exp(-im);
        double sn, cs;
        sincos(re, &sn, &cs);
        return double2{e * cs, e * sn};
    }
    template <int E, int T>
    __device__ __forceinline__ void store(int plane, int i, int t, const double2 (&x)[E]) const
    {
        double2* row = band + ((int64_t)plane * nx + i) * ldb;
#pragma unroll
        for (int p = 0; p < E; ++p) {
            const int j = t + T * p;
            if (j < ba) row[j] = x[p];
            else if (j >= ny - bb) row[j - ny + ba + bb] = x[p];
        }
    }
};

struct BandCols {
    static constexpr int inputs = 1;
    double2* band;
    const int2* bw;
    int nx, ny, ba, bb, ldb;
    __device__ __forceinline__ double2 load(int plane, int, int i, int c) const
    {
        return band[((int64_t)plane * nx + i) * ldb + c];
    }
    __device__ __forceinline__ double2 mid(int, int, int i, int c, double2 v) const
    {
        const int j = c < ba ? c : c + ny - ba - bb;
        const int2 r = bw[i];
        return (j < r.x || j >= ny - r.y) ? v : double2{0.0, 0.0};
    }
    __device__ __forceinline__ void store(int plane, int i, int c, double2 v) const
    {
        band[((int64_t)plane * nx + i) * ldb + c] = v;
    }
};

// slice.cpp:1741-1748 (/ NxNy).  The FP32 copy used by the slice loop holds
// t - 1: the deviation from vacuum keeps full FP32 relative precision, and the
// 1/sqrtNxNy of adfstem.cpp:1936,1949 is the column pass's.
struct FinishRows {
    const double2* band;
    double2* t64;
    float2* t32;
    int nx, ny, ba, bb, ldb;
    double nxny;
    __device__ __forceinline__ double2 load(int plane, int i, int j) const
    {
        const double2* row = band + ((int64_t)plane * nx + i) * ldb;
        if (j < ba) return row[j];
        return j >= ny - bb ? row[j - ny + ba + bb] : double2{0.0, 0.0};
    }
    template <int E, int T>
    __device__ __forceinline__ void store(int plane, int i, int t, const double2 (&x)[E]) const
    {
        const int64_t r = (int64_t)plane * nx + i;
        double2* row = t64 + r * ny;
        float4* pairs = reinterpret_cast<float4*>(t32 + r * ny); // elements j and j + ny/2 (pair_pos)
#pragma unroll
        for (int p = 0; p < E / 2; ++p) {
            const int j = t + T * p;
            const double2 a{x[p].x / nxny, x[p].y / nxny};
            const double2 b{x[p + E / 2].x / nxny, x[p + E / 2].y / nxny};
            row[j] = a;
            row[j + ny / 2] = b;
            pairs[j] = float4{(float)(a.x - 1.0), (float)a.y, (float)(b.x - 1.0), (float)b.y};
        }
    }
};

hipError_t launch_build(const BuildArgs& a, const double2* twx, const double2* twy, hipStream_t s)
{
    hipError_t e = hipSuccess;
    if (a.nsp > 0) {
        if (a.n_atoms > 0) {
            hipLaunchKernelGGL(scatter_atoms_kernel, dim3((a.n_atoms + 255) / 256), dim3(256), 0, s, a);
            e = hipGetLastError();
        }
        if (e == hipSuccess)
            e = launch_rows64<Fft64::Forward>(
                a.ny, MapRows{a.maps, a.spec, a.nx, a.ny, a.sa, a.sb, a.lds}, a.nx, a.k * a.nsp, twy, s);
        if (e == hipSuccess)
            e = launch_cols64<Fft64::ForwardInverse>(
                a.nx, SpeciesCols{a.nsp, a.spec, a.tmpl, a.kx, a.ky, a.nx, a.ny, a.sa, a.sb, a.lds,
                                  a.xmin == 0.0 && a.ymin == 0.0, a.xmin, a.ymin},
                a.sa + a.sb, a.k, twx, s);
    }
    if (e == hipSuccess)
        e = launch_rows64<Fft64::InverseForward>(
            a.ny, TransmitRows{a.nsp > 0 ? a.spec : nullptr, a.band, a.nsp, a.nx, a.ny, a.sa, a.sb,
                               a.lds, a.ba, a.bb, a.ldb, a.half, 1.0 / a.s},
            a.nx, a.k, twy, s);
    if (e == hipSuccess)
        e = launch_cols64<Fft64::ForwardInverse>(
            a.nx, BandCols{a.band, a.bw, a.nx, a.ny, a.ba, a.bb, a.ldb}, a.ba + a.bb, a.k, twx, s);
    if (e == hipSuccess)
        e = launch_rows64<Fft64::Inverse>(
            a.ny, FinishRows{a.band, a.t64, a.t32, a.nx, a.ny, a.ba, a.bb, a.ldb, a.nxny},
            a.nx, a.k, twy, s);
    return e;
}

__global__ void apply_keep_kernel(double2* a, int nx, int ny, int64_t total, const int2* keep)
{
    const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= total) return;
    const int64_t pix = idx % ((int64_t)nx * ny);
    const int i = (int)(pix / ny), j = (int)(pix % ny);
    const int2 r = keep[i];
    if (!(j < r.x || j >= ny - r.y)) a[idx] = double2{0.0, 0.0};
}

hipError_t launch_apply_keep(double2* a, int nx, int ny, int count, const int2* keep,
                             hipStream_t s)
{
    const int64_t n = (int64_t)nx * ny * count;
    hipLaunchKernelGGL(apply_keep_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, a, nx,
                       ny, n, keep);
    return hipGetLastError();
}

// vacuum slice step (t = 1) in k-space, slice.cpp:1388-1417 with the FFT
// scale folded into `scale`
__global__ void vacuum_step_kernel(double2* a, int nx, int ny, const double2* px,
                                   const double2* py, const int2* keep, double scale)
{
    const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= (int64_t)nx * ny) return;
    const int i = (int)(idx / ny), j = (int)(idx % ny);
    const int2 r = keep[i];
    double2 v{0.0, 0.0};
    if (j < r.x || j >= ny - r.y) {
        const double pr = px[i].x * py[j].x - px[i].y * py[j].y;
        const double pi = px[i].x * py[j].y + px[i].y * py[j].x;
        const double fr = a[idx].x * scale, fi = a[idx].y * scale;
        v = double2{pr * fr - pi * fi, pr * fi + pi * fr};
    }
    a[idx] = v;
}

hipError_t launch_vacuum_step(double2* a, int nx, int ny, const double2* px, const double2* py,
                              const int2* keep, double scale, hipStream_t s)
{
    const int64_t n = (int64_t)nx * ny;
    hipLaunchKernelGGL(vacuum_step_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, a, nx,
                       ny, px, py, keep, scale);
    return hipGetLastError();
}


// -------------------------------------------------------- vacuum waves
int col_stride64(int nc, int ny)
{
    const int pad = (nc + 7) / 8 * 8;
    const int ld = pad % 16 == 8 ? pad : pad + 8;
    return ld <= ny ? ld : nc;
}

// The vacuum wave (t = 1) entering every slice (adfstem.cpp:586-817,
// :1986-2043): u0_0 = s * probe, w_n = M P_n FFT(u0_n) / s^2, u0_{n+1} =
// IFFT(w_n).  FFT(IFFT(w)) = s^2 w, so w_n is H(k) times the product of the
// slices' masks and propagators, and non-zero inside the aperture only: one
// lane per pixel of the aperture's bounding box ([0, ra) U [nx - rb, nx) x
// [0, ca) U [ny - cb, ny)) forms every slice's wave, columns of the box are
// transformed for all slices at once, then the rows, whose last stage writes
// the FP32 shift pairs.  The probe's norm is sqrt(n_ap s^2) by Parseval,
// |H| = 1 on the n_ap aperture pixels, so no sum over the grid is needed.
// A transform pair per slice on one plane at a time took 5 launches a slice
// and a single-workgroup norm: 0.43 ms of set-up at 256^2 with 12 slices and
// 2.7 ms at 1024^2 with 25, bound by launches; now 0.02 and 0.17 ms of kernels.
__global__ void __launch_bounds__(256) vacuum_box_kernel(VacuumArgs a)
{
    const int nc = a.ca + a.cb;
    const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (idx >= (int64_t)(a.ra + a.rb) * nc) return;
    const int ib = (int)(idx / nc), c = (int)(idx - (int64_t)ib * nc);
    const int i = ib < a.ra ? ib : a.nx - a.rb - a.ra + ib;
    const int j = c < a.ca ? c : a.ny - a.cb - a.ca + c;
    const int2 r = a.ap[i];
    double2 v{0.0, 0.0};
    if (j < r.x || j >= a.ny - r.y) v = probe_h(a.kx[i], a.ky[j], a.o);
    v = double2{v.x * a.norm, v.y * a.norm};
    const int2 k = a.keep[i];
    const bool keep = j < k.x || j >= a.ny - k.y;
    double2* __restrict__ out = a.w + (int64_t)i * a.ld + c;
    const int64_t plane = (int64_t)a.nx * a.ld;
#pragma unroll 4
    for (int n = 0; n < a.n1; ++n) {
        if (n >= a.n0) out[(n - a.n0) * plane] = v;
        const double2 px = a.px[(int64_t)n * a.nx + i], py = a.py[(int64_t)n * a.ny + j];
        const double pr = px.x * py.x - px.y * py.y;
        const double pi = px.x * py.y + px.y * py.x;
        v = keep ? double2{pr * v.x - pi * v.y, pr * v.y + pi * v.x} : double2{0.0, 0.0};
    }
    if (a.n1 == a.S) a.psi0[(int64_t)j * a.nx + i] = float2{(float)v.x, (float)v.y};
}

struct VacuumCols {
    static constexpr int inputs = 1;
    double2* w;
    int nx, ld, ra, rb;
    __device__ __forceinline__ double2 load(int plane, int, int i, int c) const
    {
        return (i < ra || i >= nx - rb) ? w[((int64_t)plane * nx + i) * ld + c] : double2{0.0, 0.0};
    }
    __device__ __forceinline__ void store(int plane, int i, int c, double2 v) const
    {
        w[((int64_t)plane * nx + i) * ld + c] = v;
    }
};

// rows from the aperture's columns; out[i][2r + h] = a[i][(r + h ny/2) mod ny]:
// a lane's elements p and p + E/2 are j and j + ny/2, one 16-byte store each
// for the shifts r = j and r = j + ny/2
struct VacuumRows {
    const double2* w;
    float2* u0;
    int nx, ny, ld, ca, cb;
    __device__ __forceinline__ double2 load(int plane, int i, int j) const
    {
        const int c = j < ca ? j : j - ny + ca + cb;
        return (j < ca || j >= ny - cb) ? w[((int64_t)plane * nx + i) * ld + c] : double2{0.0, 0.0};
    }
    template <int E, int T>
    __device__ __forceinline__ void store(int plane, int i, int t, const double2 (&x)[E]) const
    {
        float4* row = reinterpret_cast<float4*>(u0 + ((int64_t)plane * nx + i) * (2 * ny));
#pragma unroll
        for (int p = 0; p < E / 2; ++p) {
            const double2 a = x[p], b = x[p + E / 2];
            const float4 f{(float)a.x, (float)a.y, (float)b.x, (float)b.y};
            row[t + T * p] = f;
            row[t + T * p + ny / 2] = float4{f.z, f.w, f.x, f.y};
        }
    }
};

hipError_t launch_vacuum(const VacuumArgs& a, float2* u0, const double2* twx, const double2* twy,
                         hipStream_t s)
{
    const int64_t box = (int64_t)(a.ra + a.rb) * (a.ca + a.cb);
    const int planes = a.n1 - a.n0;
    if (box <= 0 || planes <= 0) return hipErrorInvalidValue;
    hipLaunchKernelGGL(vacuum_box_kernel, dim3((unsigned)((box + 255) / 256)), dim3(256), 0, s, a);
    hipError_t e = hipGetLastError();
    if (e == hipSuccess)
        e = launch_cols64<Fft64::Inverse>(a.nx, VacuumCols{a.w, a.nx, a.ld, a.ra, a.rb}, a.ca + a.cb,
                                          planes, twx, s);
    if (e == hipSuccess)
        e = launch_rows64<Fft64::Inverse>(a.ny, VacuumRows{a.w, u0, a.nx, a.ny, a.ld, a.ca, a.cb},
                                          a.nx, planes, twy, s);
    return e;
}

// -------------------------------------------------------- detector MTF
// adfstem.cpp:2272-2385: |psi| outside the aperture, BACKWARD FFT, times the
// 2-D MTF / sqrt(NxNy) with the reference's in-place real / imaginary update,
// FORWARD FFT, / sqrt(NxNy), bw_limit.  The input and the band-limited result
// live in the stored columns, so the transforms go columns, rows there and
// back, columns: three passes over 2/3 of a plane, the element-wise steps
// inside them, where separate steps took nine over the whole FP64 plane
// (256 positions of 256^2: 0.62 -> 0.23 ms).
struct MtfMagnitudeCols {
    static constexpr int inputs = 1;
    MtfArgs a;
    __device__ __forceinline__ double2 load(int plane, int, int i, int c) const
    {
        const int j = c < a.ka ? c : c + a.ny - a.ka - a.kb;
        if (!a.outside[i * a.ny + j]) return double2{0.0, 0.0};
        const float2 w = a.psi[((int64_t)plane * a.nx + i) * a.ncp + c];
        const double re = w.x, im = w.y;
        return double2{sqrt((re * re) + (im * im)), 0.0};
    }
    __device__ __forceinline__ void store(int plane, int i, int c, double2 v) const
    {
        a.work[((int64_t)plane * a.nx + i) * a.ld + c] = v;
    }
};

struct MtfRows {
    MtfArgs a;
    __device__ __forceinline__ double2 load(int plane, int i, int j) const
    {
        const double2* row = a.work + ((int64_t)plane * a.nx + i) * a.ld;
        if (j < a.ka) return row[j];
        return j >= a.ny - a.kb ? row[j - a.ny + a.ka + a.kb] : double2{0.0, 0.0};
    }
    __device__ __forceinline__ double2 mid(int, int i, int j, double2 u) const
    {
        const double2 t = a.mtf[i * a.ny + j];
        double2 v;
        v.x = (t.x * u.x - t.y * u.y) / a.s;
        v.y = (t.x * u.y + t.y * v.x) / a.s;
        return v;
    }
    template <int E, int T>
    __device__ __forceinline__ void store(int plane, int i, int t, const double2 (&x)[E]) const
    {
        double2* row = a.work + ((int64_t)plane * a.nx + i) * a.ld;
#pragma unroll
        for (int p = 0; p < E; ++p) {
            const int j = t + T * p;
            if (j < a.ka) row[j] = x[p];
            else if (j >= a.ny - a.kb) row[j - a.ny + a.ka + a.kb] = x[p];
        }
    }
};

struct MtfBandCols {
    static constexpr int inputs = 1;
    MtfArgs a;
    __device__ __forceinline__ double2 load(int plane, int, int i, int c) const
    {
        return a.work[((int64_t)plane * a.nx + i) * a.ld + c];
    }
    __device__ __forceinline__ void store(int plane, int i, int c, double2 w) const
    {
        const int j = c < a.ka ? c : c + a.ny - a.ka - a.kb;
        const int2 k = a.keep[i];
        const bool in = j < k.x || j >= a.ny - k.y;
        a.psi[((int64_t)plane * a.nx + i) * a.ncp + c] =
            in ? float2{(float)(w.x / a.s), (float)(w.y / a.s)} : float2{0.f, 0.f};
    }
};

hipError_t launch_mtf(const MtfArgs& a, const double2* twx, const double2* twy, hipStream_t s)
{
    hipError_t e = launch_cols64<Fft64::Inverse>(a.nx, MtfMagnitudeCols{a}, a.ka + a.kb, a.batch,
                                                 twx, s);
    if (e == hipSuccess)
        e = launch_rows64<Fft64::InverseForward>(a.ny, MtfRows{a}, a.nx, a.batch, twy, s);
    if (e == hipSuccess)
        e = launch_cols64<Fft64::Forward>(a.nx, MtfBandCols{a}, a.ka + a.kb, a.batch, twx, s);
    return e;
}

// FP64 transmission update of one slice on `count` real-space waves
// (adfstem.cpp:1922-1952): mode 0 forms the imaginary part from the already
// updated real part, as the reference's two statements do; mode 1 is the
// complex product.  Both divide by s = sqrt(NxNy).
__global__ void transmit_f64_kernel(double2* a, const double2* t, int64_t m, int count, int mode,
                                    double s)
{
    const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= m * count) return;
    const double2 tt = t[idx % m];
    const double2 u = a[idx];
    double2 v;
    if (mode == 0) {
        v.x = (tt.x * u.x - tt.y * u.y) / s;
        v.y = (tt.x * u.y + tt.y * v.x) / s;
    } else {
        v.x = (tt.x * u.x - tt.y * u.y) / s;
        v.y = (tt.x * u.y + tt.y * u.x) / s;
    }
    a[idx] = v;
}

hipError_t launch_transmit_f64(double2* a, const double2* t, int64_t m, int count, int mode,
                               double s, hipStream_t st)
{
    const int64_t n = m * count;
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(transmit_f64_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, a,
                       t, m, count, mode, s);
    return hipGetLastError();
}

} // namespace msf
