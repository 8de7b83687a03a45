// fft64_passes.hpp -- FP64 row and column passes of the set-up and detector
// MTF transforms, as kernels over an operation (Op) that says where a line's
// elements come from, what happens to them between a forward and an inverse
// transform, and where they go.  A pass so reads and writes only the columns
// that carry data, and the element-wise work before, between and after the
// transforms costs no pass of its own.
//
// Rows run along y (contiguous), columns along x; `plane` counts the planes
// of one launch.  An array of nc < ny columns is kept at a row stride of an
// odd number of 128-byte lines (col_stride64), so that a column's elements
// spread over the memory channels; a power-of-two stride keeps hitting the
// same few (16 planes of 1024^2 at stride 1024: 1.5 TB/s against 4 TB/s for
// the same bytes as rows).
#pragma once
#include <hip/hip_runtime.h>

#include "fft_engine.hpp"
#include "kernels.hpp"

namespace msf {

// which transforms of a line a pass runs
enum class Fft64 { Forward, Inverse, ForwardInverse, InverseForward };

// ------------------------------------------------------------------ rows
// Op: double2 load(int plane, int i, int j);
//     double2 mid(int plane, int i, int j, double2 v)  (two-transform passes);
//     template <int E, int T> void store(int plane, int i, int t, const double2 (&x)[E])
// with x[p] the element at j = t + T p.
// Up to 256 lanes; a line of at most 64 lanes lies in one wavefront and
// exchanges without workgroup barriers.
template <int N, Fft64 MODE, class Op>
__global__ void __launch_bounds__(256) rows64_kernel(Op op, int nx, int rows, const double2* tw)
{
    using P = Plan<N>;
    constexpr int E = P::E, T = P::T, RPW = 256 / T, LEN = lds_len(N);
    constexpr bool WAVE = T <= 64;
    constexpr bool INV0 = MODE == Fft64::Inverse || MODE == Fft64::InverseForward;
    __shared__ double2 s_tw[stage_tw_len<N>()];
    __shared__ double2 s_buf[RPW * LEN];
    for (int e = threadIdx.x; e < stage_tw_len<N>(); e += blockDim.x) s_tw[e] = tw[e];
    __syncthreads();
    const int lr = threadIdx.x / T, t = threadIdx.x % T;
    const int r = (int)blockIdx.x * RPW + lr;
    const bool active = r < rows;
    const int rr = active ? r : rows - 1; // lanes past the last row repeat it and store nothing
    const int plane = rr / nx, i = rr - plane * nx;
    double2* lds = s_buf + lr * LEN;
    double2 x[E];
#pragma unroll
    for (int p = 0; p < E; ++p) x[p] = op.load(plane, i, t + T * p);
    P::template run<INV0, double2, WAVE>(x, lds, s_tw, t);
    if constexpr (MODE == Fft64::ForwardInverse || MODE == Fft64::InverseForward) {
#pragma unroll
        for (int p = 0; p < E; ++p) x[p] = op.mid(plane, i, t + T * p, x[p]);
        P::template run<!INV0, double2, WAVE>(x, lds, s_tw, t);
    }
    if (active) op.template store<E, T>(plane, i, t, x);
}

// --------------------------------------------------------------- columns
// Op: int inputs (ForwardInverse: transformed inputs that mid() turns into
//     terms of one sum);
//     double2 load(int plane, int in, int i, int c);
//     double2 mid(int plane, int in, int i, int c, double2 v);
//     void store(int plane, int i, int c, double2 v)
// with c the stored column.  A workgroup owns W columns: lanes run along the
// columns for loads and stores (128-byte segments for W = 8), the tile passes
// through LDS, and each column is transformed by T neighbouring lanes.  W
// keeps two workgroups' tiles in a CU's 160 KB of LDS (8 x 9.2 KB at 512,
// 4 x 18.4 KB at 1024); twiddles are read from L2, which leaves that room.
// Workgroups are banded over the XCDs: neighbouring tiles share 128-byte
// lines.
template <int N> struct Col64 {
    static constexpr int T = Plan<N>::T;
    static constexpr int W = N >= 768 ? 4 : 8;
    // column stride in the tile: the 8 lanes of a 128-byte LDS access cover W
    // columns x 8/W rows; a stride of 8/W modulo 8 gives each its own slot
    static constexpr int BASE = lds_len(N), WANT = (8 / W) % 8;
    static constexpr int LEN = BASE + ((WANT - BASE % 8) + 8) % 8;
};

template <int N, Fft64 MODE, class Op>
__global__ void __launch_bounds__(Col64<N>::W* Col64<N>::T)
    cols64_kernel(Op op, int ncols, int ntiles, const double2* tw)
{
    using P = Plan<N>;
    constexpr int E = P::E, T = P::T, W = Col64<N>::W, LEN = Col64<N>::LEN;
    constexpr bool WAVE = T <= 64;
    __shared__ double2 s_buf[W * LEN];
    // XCD banding: blocks go round-robin over 8 XCDs; give each a contiguous range
    const int G = (int)gridDim.x, q = G / 8, rem = G % 8;
    const int xc = (int)blockIdx.x % 8, g = xc * q + min(xc, rem) + (int)blockIdx.x / 8;
    const int plane = g / ntiles, j0 = (g - plane * ntiles) * W;
    const int lc = threadIdx.x % W, r0 = threadIdx.x / W; // coalesced phases
    const int c = threadIdx.x / T, t = threadIdx.x % T;   // transform phases
    const bool okc = j0 + lc < ncols;
    const int jl = okc ? j0 + lc : ncols - 1; // columns past the last repeat it and store nothing
    const int jc = min(j0 + c, ncols - 1);
    double2* lds = s_buf + c * LEN;
    double2 x[E];
    auto fetch = [&](int in) {
        double2 v[E];
#pragma unroll
        for (int p = 0; p < E; ++p) v[p] = op.load(plane, in, r0 + T * p, jl);
#pragma unroll
        for (int p = 0; p < E; ++p) s_buf[lc * LEN + lds_pad(r0 + T * p)] = v[p];
        __syncthreads();
#pragma unroll
        for (int p = 0; p < E; ++p) x[p] = lds[lds_pad(t + T * p)];
    };
    if constexpr (MODE == Fft64::ForwardInverse) {
        double2 acc[E];
        for (int in = 0; in < op.inputs; ++in) {
            if (in > 0) __syncthreads(); // the tile's readers are done
            fetch(in);
            P::template run<false, double2, WAVE>(x, lds, tw, t);
#pragma unroll
            for (int p = 0; p < E; ++p) {
                const double2 m = op.mid(plane, in, t + T * p, jc, x[p]);
                acc[p] = in == 0 ? m : double2{acc[p].x + m.x, acc[p].y + m.y};
            }
        }
#pragma unroll
        for (int p = 0; p < E; ++p) x[p] = acc[p];
        P::template run<true, double2, WAVE>(x, lds, tw, t);
    } else {
        fetch(0);
        P::template run<(MODE == Fft64::Inverse), double2, WAVE>(x, lds, tw, t);
    }
    lds_sync<WAVE>();
#pragma unroll
    for (int p = 0; p < E; ++p) lds[lds_pad(t + T * p)] = x[p];
    __syncthreads();
    if (okc) {
#pragma unroll
        for (int p = 0; p < E; ++p)
            op.store(plane, r0 + T * p, j0 + lc, s_buf[lc * LEN + lds_pad(r0 + T * p)]);
    }
}

// ---------------------------------------------------------------- launches
#define MSF_LENGTHS64(CASE)                                                                        \
    CASE(16) CASE(32) CASE(64) CASE(96) CASE(128) CASE(192) CASE(256) CASE(384) CASE(512)          \
    CASE(768) CASE(1024)

template <Fft64 MODE, class Op>
hipError_t launch_rows64(int n, const Op& op, int nx, int planes, const double2* tw, hipStream_t s)
{
    const int64_t rows = (int64_t)nx * planes;
    if (rows <= 0 || rows > (int64_t)1 << 30) return hipErrorInvalidValue;
    switch (n) {
#define MSF_CASE(N)                                                                                \
    case N: {                                                                                      \
        constexpr int RPW = 256 / Plan<N>::T;                                                      \
        hipLaunchKernelGGL((rows64_kernel<N, MODE, Op>), dim3((unsigned)((rows + RPW - 1) / RPW)), \
                           dim3(RPW * Plan<N>::T), 0, s, op, nx, (int)rows, tw);                   \
        return hipGetLastError();                                                                  \
    }
        MSF_LENGTHS64(MSF_CASE)
#undef MSF_CASE
    default:
        return hipErrorInvalidValue;
    }
}

template <Fft64 MODE, class Op>
hipError_t launch_cols64(int n, const Op& op, int ncols, int planes, const double2* tw,
                         hipStream_t s)
{
    if (ncols <= 0 || planes <= 0) return hipErrorInvalidValue;
    switch (n) {
#define MSF_CASE(N)                                                                                \
    case N: {                                                                                      \
        constexpr int W = Col64<N>::W;                                                             \
        const int ntiles = (ncols + W - 1) / W;                                                    \
        hipLaunchKernelGGL((cols64_kernel<N, MODE, Op>), dim3((unsigned)((int64_t)planes * ntiles)), \
                           dim3(W * Plan<N>::T), 0, s, op, ncols, ntiles, tw);                     \
        return hipGetLastError();                                                                  \
    }
        MSF_LENGTHS64(MSF_CASE)
#undef MSF_CASE
    default:
        return hipErrorInvalidValue;
    }
}

} // namespace msf
