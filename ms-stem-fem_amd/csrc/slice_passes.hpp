// slice_passes.hpp -- device code of the FP32 slice-step passes: the row
// pass (inverse transform along y, transmission, forward transform along y)
// and the column pass (forward transform along x, band limit and propagator,
// inverse transform along x, or the exit wave on the last slice), as device
// functions over one workgroup's share and as kernels.  Included by the units
// that launch them one batch at a time (kernels_slice.hip) and grouped over
// several runs (kernels_group.hip).
//
// Reference behaviour restated (paths relative to the reference root):
//   row pass    = adfstem.cpp:1891 (BACKWARD FFT, the y half) + :1922-1952
//                 (transmission multiply, /sqrtNxNy) + :1986 (FORWARD FFT,
//                 y half); the first pass starts from the circularly shifted
//                 real-space probe of adfstem.cpp:1632-1671.
//   column pass = adfstem.cpp:1986-1992 (FORWARD FFT, x half, /sqrtNxNy) +
//                 bw_limit (bw_limit.cpp:30-47) + slice::propagate
//                 (slice.cpp:1366-1421) + the next slice's BACKWARD FFT (x half).
#pragma once

#include <hip/hip_runtime.h>

#include "fft_engine.hpp"
#include "kernels.hpp"

namespace msf {

// Element k of an array whose byte offsets fit 32 bits (a row or one
// position's plane of the wave): the offset is formed in 32 bits, so the
// load or store takes a uniform base and a 32-bit per-lane offset rather
// than a 64-bit address per element.
template <typename T> __device__ __forceinline__ T& elem32(T* base, uint32_t k)
{
    return *reinterpret_cast<T*>(reinterpret_cast<char*>(base) + k * (uint32_t)sizeof(T));
}
template <typename T> __device__ __forceinline__ const T& elem32(const T* base, uint32_t k)
{
    return *reinterpret_cast<const T*>(reinterpret_cast<const char*>(base) + k * (uint32_t)sizeof(T));
}

// Element K past a lane's own (byte offset `lane`) of a uniform base: K goes
// into the instruction, so all elements of a lane share one address register.
template <typename T> __device__ __forceinline__ T& elem_at(T* base, uint32_t lane, int K)
{
    return *reinterpret_cast<T*>(reinterpret_cast<char*>(base) + lane + (int64_t)K * (int)sizeof(T));
}
template <typename T> __device__ __forceinline__ const T& elem_at(const T* base, uint32_t lane, int K)
{
    return *reinterpret_cast<const T*>(reinterpret_cast<const char*>(base) + lane +
                                       (int64_t)K * (int)sizeof(T));
}

// ------------------------------------------------------------------ row pass
// Transmission of one pixel, for the scattered wave u, the vacuum wave u0 and
// U = u + u0, with (tau, ti) = t - 1 and everything times s = sqrt(nx ny)
// (the column pass's P_y carries 1/s^2).  The scattered part of T(U) is
//   A = tau U_re + u_re - ti U_im,
//   B = tau U_im + u_im + ti (A + u0_re) / s     (TMODE 0)
// since the reference's in-place update forms Im from the updated Re, whose
// value is (A + u0_re) / s; TMODE 1 (exact product) has B = tau U_im + u_im +
// ti U_re.  Eight operations a value; with the products of u and u0 taken apart
// they were twelve (32 more instructions of 551 a wave at 512).
template <bool FIRST, int TMODE>
__device__ __forceinline__ float2 transmit_point(float2 u, float2 t, float2 u0, float is)
{
    if constexpr (FIRST) {
        const float a = fmaf(t.x, u0.x, -(t.y * u0.y));
        return float2{a, TMODE == 0 ? fmaf(t.x, u0.y, (t.y * is) * (a + u0.x))
                                    : fmaf(t.x, u0.y, t.y * u0.x)};
    } else {
        const float Ux = u.x + u0.x, Uy = u.y + u0.y;
        const float a = fmaf(t.x, Ux, fmaf(-t.y, Uy, u.x));
        return float2{a, TMODE == 0 ? fmaf(t.x, Uy, fmaf(t.y * is, a + u0.x, u.y))
                                    : fmaf(t.x, Uy, fmaf(t.y, Ux, u.y))};
    }
}

// Lane element p (indices t + T*p) lies entirely inside the middle band
// [3N/8, 5N/8), which the 2/3 band limit leaves empty in k-space (checked on
// the host before a pruned variant is launched).
template <int N, int E> __host__ __device__ constexpr bool in_zero_band(int p)
{
    constexpr int T = N / E;
    return T * p >= (3 * N + 7) / 8 && T * (p + 1) <= (5 * N) / 8;
}

// With PRUNE the host also guarantees ka >= N/4 and kb >= N/4: lane elements
// entirely below N/4 are always in the low kept band, those entirely at or
// above 3N/4 always in the high band; only the elements straddling a band edge
// need a run-time test.
template <int N, int E> __host__ __device__ constexpr bool always_low(int p)
{
    return (N / E) * (p + 1) <= N / 4;
}
template <int N, int E> __host__ __device__ constexpr bool always_high(int p)
{
    return (N / E) * p >= N - N / 4;
}

// Workgroup -> (row i, group of RPW positions).  Consecutive launch indices go
// to different XCDs round-robin; the permutation gives each XCD a contiguous
// band of rows so that the t and u0 rows a band needs are fetched into that
// XCD's L2 once.
__device__ __forceinline__ int xcd_band(int L, int G)
{
    // Workgroups are dispatched round-robin over the 8 XCDs (L % 8).  Give
    // XCD x the contiguous logical range [x*q + min(x, r), ... + q + (x < r))
    // with G = 8q + r, so neighbouring tiles (which share cache lines) meet
    // in one L2.  A bijection on [0, G) for every G.
    constexpr int kXcd = 8;
    const int q = G / kXcd, r = G % kXcd;
    const int x = L % kXcd, k = L / kXcd;
    return x * q + min(x, r) + k;
}

// g / d for uniform 0 <= g < 2^31 by the host's multiplier (2^32 - 1) / d:
// the product's high word is the quotient or one less.  A handful of scalar
// instructions; the compiler's own division of uniform values goes through
// the vector unit and back.
__device__ __forceinline__ int div_by(uint32_t g, uint32_t d, uint32_t mul)
{
    const uint32_t q = __umulhi(g, mul);
    return (int)(g - q * d >= d ? q + 1 : q);
}

// lanes of a row-pass workgroup: RPW = row_threads / T rows share the staged
// twiddle table and transmission row.  At 512 (primary plan) eight rows per
// workgroup halve that staging per row (row pass 41.1 -> 40.4 us per 64
// positions); at 1024 the larger LDS footprint costs more than it saves.
template <int NY, int V> __host__ __device__ constexpr int row_threads()
{
    // the alternate 1024 plan (16 values on 64 lanes, 95 registers): two
    // rows per 128-lane workgroup, 71 us against 76 us on 256 lanes per 17
    // positions
    return (NY == 512 && V == 0) ? 512 : (NY == 1024 && V == 1) ? 128 : 256;
}

// Lean row passes read the twiddle table and the transmission row from
// global memory (L2-resident, shared by the workgroups of a row band) instead
// of staging them in LDS, so that more workgroups fit on a CU.
template <int NY, int V> __host__ __device__ constexpr bool row_lean() { return NY == 1024; }

// Occupancy the row pass asks of the register allocator: 6 waves per SIMD for
// the 8-value plans; the plans with 12 and 16 values per lane need more
// registers, and ask for what their LDS and registers allow (five workgroups
// per CU at 192 and 384, where 98 registers would leave four waves).
template <int NY, int V> __host__ __device__ constexpr int row_waves()
{
    constexpr int E = PlanV<NY, V>::E;
    return E <= 8 ? 6 : (E == 16 ? (NY == 512 ? 3 : 4) : (E == 12 ? (NY == 768 ? 4 : 5) : 2));
}

// RT lanes per workgroup: row_threads() for batches that fill it, or one
// row's T lanes when the batch has fewer positions than a workgroup has rows
// (no lane then computes a row it does not store).
// LDS of a row-pass workgroup in float2 units: the staged twiddle table and
// transmission row (unless lean), and one exchange buffer per row.
template <int NY, int V, int RT> __host__ __device__ constexpr bool row_is_lean()
{
    // one row per workgroup: nothing to share, tables are read from L2
    return row_lean<NY, V>() || RT / PlanV<NY, V>::T == 1;
}
// slots of one row's exchange buffer (padded per exchange, LdsExchange); for
// transforms of 8 lanes the two rows that 16 lanes cover start 8 slots apart
// modulo 16
template <int NY, int V> __host__ __device__ constexpr int row_len()
{
    using P = PlanV<NY, V>;
    return P::T >= 16 ? P::kExchangeLen : (P::kExchangeLen + 7) / 16 * 16 + 8;
}
//
// The row pass waits between load, transforms and store as much as it computes
// (512^2: 551 vector instructions a wave keep the vector unit busy for 63 % of
// the pass, the LDS for 40 %, without bank conflicts), so what is uniform or
// known at compile time stays out of the vector unit: the workgroup's
// division, the row and u0 addresses (a base per wavefront, the element in the
// instruction), the table staging in 16-byte words, the wrap of the shifted
// u0.  Together with transmit_point, and with every t and u0 read of a lane
// issued before the first product, per pass, before and now: 128^2 39.4 ->
// 37.1 us (1024 positions), 192^2 46.8 -> 40.0 (496), 256^2 40.1 -> 35.2
// (272), 384^2 50.8 -> 42.9 (112), 512^2 41.5 -> 37.0 (64), 768^2 36.5 -> 29.9
// (16), 1024^2 50.7 -> 47.9 (16; its tables come from L2, which bounds it).
// Not kept: 16 rows per workgroup at 512 (37.9 -> 39.9), two positions per
// wavefront with the next row prefetched (512 36.3 -> 38.8, 384 42 -> 46,
// 1024 47.9 -> 49.7), for the registers or waves that they cost.
template <int NY, int V, int RT> __host__ __device__ constexpr int row_smem_len()
{
    return (row_is_lean<NY, V, RT>() ? 0 : plan_tw_len<PlanV<NY, V>>() + NY) +
           (RT / PlanV<NY, V>::T) * row_len<NY, V>();
}

// One row-pass workgroup: logical block `blk` of the pass (XCD-banded over
// the pass's own blocks), LDS at smem.
template <int NY, int V, bool FIRST, int TMODE, bool PRUNE, int RT>
__device__ __forceinline__ void row_body(const RowPassArgs& a, int blk, float2* smem)
{
    using P = PlanV<NY, V>;
    constexpr int E = P::E, T = P::T;
    constexpr int RPW = RT / T;
    constexpr int PS = 0, LEN = row_len<NY, V>();
    constexpr bool LEAN = row_is_lean<NY, V, RT>();
    constexpr int TW = plan_tw_len<P>();
    float2* s_tw = smem;
    float2* s_t = smem + (LEAN ? 0 : TW);
    float2* s_buf = smem + (LEAN ? 0 : TW + NY);

    // workgroup-uniform decode (scalar unit)
    const int groups = (a.batch + RPW - 1) / RPW;
    const int g = xcd_band(blk, groups * a.nx);
    const int i = div_by(g, groups, a.div);
    const int b0 = (g - i * groups) * RPW;

    // with T == 64 each row is one wavefront: keep its index in a scalar register
    const int lr = (T % 64 == 0) ? __builtin_amdgcn_readfirstlane(threadIdx.x / T) : threadIdx.x / T;
    const int t = threadIdx.x % T;
    const bool active = b0 + lr < a.batch;
    const int lb = active ? lr : a.batch - 1 - b0; // lanes past the batch repeat its last position
    // rows and u0 pairs by 32-bit offsets from uniform bases: the rows of a
    // workgroup lie within RPW planes, u0 within 16 MB; a row that is a whole
    // wavefront's has its own base
    constexpr bool OWN = T % 64 == 0;
    float2* base = a.psi + ((int64_t)(b0 + (OWN ? lb : 0)) * a.nx + i) * a.ncp;
    const uint32_t lane = ((OWN ? 0u : (uint32_t)lb * (uint32_t)(a.nx * a.ncp)) + (uint32_t)t) * 8u;
    float2* lds = s_buf + lr * LEN;
    const int hi = NY - a.kb;           // first kept column of the negative-ky band
    // compact index = j + (ka + kb - NY) for j >= hi; that band's base
    float2* up = base + (a.ka + a.kb - NY);
    const int2 sh = a.shift[b0 + lb];

    // the wave is asked for before the tables, so that both are on their way
    // when the workgroup meets at the barrier
    float2 x[E];
    if constexpr (!FIRST) {
#pragma unroll
        for (int p = 0; p < E; ++p) {
            const int j = t + T * p;
            if constexpr (PRUNE) {
                // ka and kb lie in [N/4, 3N/8]: elements below N/2 belong to the
                // low band or to none, and a read past its edge stays in the
                // row's ka + kb >= N/2 stored columns, as one below the high
                // band's edge does
                if (in_zero_band<NY, E>(p)) {
                    x[p] = float2{0.f, 0.f};
                } else {
                    const bool low = T * p < NY / 2;
                    x[p] = elem_at(low ? base : up, lane, T * p);
                    if (low ? !always_low<NY, E>(p) && j >= a.ka : !always_high<NY, E>(p) && j < hi)
                        x[p] = float2{0.f, 0.f};
                }
            } else {
                const bool lo = j < a.ka, hi_band = j >= hi;
                // lanes outside the kept band all read element 0 (one shared line)
                const float2 v = elem32(base, lane / 8u - (uint32_t)t + (lo ? (uint32_t)j : hi_band ? (uint32_t)(j + a.ka + a.kb - NY) : 0u));
                x[p] = (lo || hi_band) ? v : float2{0.f, 0.f};
            }
        }
    }

    // twiddles and the transmission row i, shared by the RPW rows of the
    // group: 16 bytes a lane, the two tables one after the other in LDS
    const float2* trow = a.t + (int64_t)i * NY;
    if constexpr (!LEAN) {
        constexpr int NW = TW / 2, N4 = NW + NY / 2;
        static_assert(TW % 2 == 0 && NY % 2 == 0, "tables in 16-byte words");
        float4* dst = reinterpret_cast<float4*>(smem);
#pragma unroll
        for (int k = 0; k < (N4 + RT - 1) / RT; ++k) {
            const int e = (int)threadIdx.x + k * RT;
            if (N4 % RT == 0 || e < N4)
                dst[e] = e < NW ? reinterpret_cast<const float4*>(a.tw)[e]
                                : reinterpret_cast<const float4*>(trow)[e - NW];
        }
        __syncthreads();
    }
    const float2* tw = LEAN ? a.tw : s_tw;
    const float4* tt = reinterpret_cast<const float4*>(LEAN ? trow : s_t);

    if constexpr (!FIRST) P::template run<true, float2, (T <= 64), PS>(x, lds, tw, t);

    // Transmission and u0 rows are stored as pairs (pair_pos): a lane's
    // elements p and p + E/2 are j and j + NY/2, and one 16-byte read fetches
    // both, of t at j and of u0 at the shifted r = (j - sy) mod NY.  All reads
    // are issued before the first product.
    int ii = i - sh.x;
    if (ii < 0) ii += a.nx;
    const uint32_t urow = (uint32_t)ii * (uint32_t)NY, u00 = (uint32_t)(t - sh.y);
    const float4* u0 = reinterpret_cast<const float4*>(a.u0);
    float4 tq[E / 2], uq[E / 2];
#pragma unroll
    for (int p = 0; p < E / 2; ++p) {
        const uint32_t r0 = u00 + (uint32_t)(T * p); // negative (as unsigned: large) below the shift
        const uint32_t r = (NY & (NY - 1)) == 0 ? r0 & (NY - 1) : min(r0, r0 + (uint32_t)NY);
        tq[p] = tt[t + T * p];
        uq[p] = elem32(u0, urow + r);
    }
#pragma unroll
    for (int p = 0; p < E / 2; ++p) {
        x[p] = transmit_point<FIRST, TMODE>(x[p], float2{tq[p].x, tq[p].y},
                                            float2{uq[p].x, uq[p].y}, a.inv_s);
        x[p + E / 2] = transmit_point<FIRST, TMODE>(x[p + E / 2], float2{tq[p].z, tq[p].w},
                                                    float2{uq[p].z, uq[p].w}, a.inv_s);
    }

    P::template run<false, float2, (T <= 64), PS>(x, lds, tw, t);

    if (active) {
#pragma unroll
        for (int p = 0; p < E; ++p) {
            const int j = t + T * p;
            if constexpr (PRUNE) {
                if (in_zero_band<NY, E>(p)) continue;
                const bool low = T * p < NY / 2;
                if (low ? always_low<NY, E>(p) || j < a.ka : always_high<NY, E>(p) || j >= hi)
                    elem_at(low ? base : up, lane, T * p) = x[p];
            } else {
                if (j < a.ka) elem_at(base, lane, T * p) = x[p];
                else if (j >= hi) elem_at(up, lane, T * p) = x[p];
            }
        }
    }
}

template <int NY, int V, bool FIRST, int TMODE, bool PRUNE, int RT>
__global__ void __launch_bounds__(RT)
__attribute__((amdgpu_waves_per_eu((row_waves<NY, V>())))) row_pass_kernel(RowPassArgs a)
{
    __shared__ __align__(16) float2 smem[row_smem_len<NY, V, RT>()];
    row_body<NY, V, FIRST, TMODE, PRUNE, RT>(a, (int)blockIdx.x, smem);
}

// --------------------------------------------------------------- column pass
// A workgroup owns W adjacent kept columns of one position.  The tile is
// loaded with lanes running along the columns (coalesced W*8-byte segments
// per row) into a column-major LDS tile, each column is then transformed by
// T lanes of one wavefront (wave-local exchanges, no workgroup barrier
// between radix stages), and the tile is written back the same coalesced way.
template <int NX, int V = 0> struct ColTile {
    static constexpr int T = PlanV<NX, V>::T;
    static constexpr int WMAX = 16;  // ncp is a multiple of this
    // default tile: keep LDS (W * lds_len * 8 B) near 40 KiB so that several
    // workgroups share a CU
    // The alternate 1024 plan (16 values on 64 lanes, 72 registers) fits two
    // 8-column tiles per CU, and four 4-column tiles with lean tables, which
    // are faster where no second chain runs beside them.
    static constexpr int W = (NX == 1024 && V == 1) ? 4 : (16 * lds_len(NX) * 8 > 48 * 1024) ? 8 : 16;
};

// Slot of row r + T p in a tile's column: the rows as they are where the
// exchanges are swizzled (16 lanes read 16 rows without conflict), else one
// slot more every 16 rows, as after the first stage of radix 8 or 16, whose
// addresses it then shares.
template <typename P> __host__ __device__ constexpr bool col_plain()
{
    return P::T >= 16 && P::kExchangeLen == P::N;
}
template <typename P> __device__ __forceinline__ int col_slot(int r, int p)
{
    if constexpr (col_plain<P>()) return r + P::T * p;
    else return lds_pad_at<P::T, 4>(r, p);
}

// column stride of the LDS tile: a 16-lane group of the coalesced load/store
// phases covers W' = min(W, 16) columns x g = 16/W' rows; a stride that is an
// odd multiple of g puts those 16 lanes on distinct bank pairs
template <int NX, int V, int W> __host__ __device__ constexpr int col_len()
{
    constexpr int tile = col_plain<PlanV<NX, V>>() ? NX : lds_len<4>(NX);
    constexpr int base = PlanV<NX, V>::kExchangeLen > tile ? PlanV<NX, V>::kExchangeLen : tile;
    constexpr int g = 16 / (W < 16 ? W : 16);
    return (base + g - 1) / (2 * g) * (2 * g) + g;
}

// Lean tiles: when the twiddle and propagator tables would keep two
// workgroups from sharing a CU's 160 KB of LDS (1024 rows: a 74 KB tile),
// the tables are read from global memory (L2-resident, shared by every
// workgroup) and only the tile stays in LDS.
template <int NX, int V, int W> __host__ __device__ constexpr bool col_lean()
{
    if (W == 1) return true;      // one column: nothing to share, tables are read from L2
    if (W == 4) return NX >= 512; // small tiles: tables would outweigh the tile
    return 2 * ((size_t)W * col_len<NX, V, W>() * 8 + (size_t)plan_tw_len<PlanV<NX, V>>() * 8 +
                (size_t)NX * 8) > 160 * 1024;
}

// Plans with 12 or more values per lane (the alternate plans, and the
// primary plans of 96, 192, 384 and 768) take the tile's real size as their
// launch bound, so that a 128- to 512-lane tile may use more than the 128
// registers a 1024-lane bound leaves per lane (384: 116 B of spills per lane
// under that bound).
template <int NX, int V, int W> __host__ __device__ constexpr int col_bound()
{
    return (V || PlanV<NX, V>::E >= 12) ? W * PlanV<NX, V>::T : 1024;
}

// Workgroups of a column pass that a CU holds: by its 160 KB of LDS (given
// out in steps of 1,280 bytes) and by waves (8 per SIMD, or 5 with the 75 to
// 96 registers of the plans with 12 and 16 values per lane).
template <int NX, int V, int W> __host__ __device__ constexpr int col_per_cu(bool px)
{
    constexpr int tile = (W * col_len<NX, V, W>() + plan_tw_len<PlanV<NX, V>>()) * 8;
    constexpr int waves = PlanV<NX, V>::E <= 8 ? 32 : 20, lanes = W * PlanV<NX, V>::T;
    const int by_lds = 160 * 1024 / ((tile + (px ? NX * 8 : 0) + 1279) / 1280 * 1280);
    return by_lds < waves * 64 / lanes ? by_lds : waves * 64 / lanes;
}
// The propagator row, read once per element, stays in L2 where the CU then
// holds a workgroup more: tiles of 8 columns of 512 rows take 40,512 bytes
// and run four to a CU instead of three, 37.3 -> 35.0 us per 64 positions.
template <int NX, int V, int W> __host__ __device__ constexpr bool col_px_lean()
{
    return col_lean<NX, V, W>() || col_per_cu<NX, V, W>(false) > col_per_cu<NX, V, W>(true);
}

// LDS of a column-pass workgroup in float2 units: the staged twiddle and
// propagator tables (unless lean), the exit roots (last slice) and the tile.
template <int NX, int V, bool LAST, int W> __host__ __device__ constexpr int col_smem_len()
{
    return (col_lean<NX, V, W>() ? 0 : plan_tw_len<PlanV<NX, V>>()) +
           (col_px_lean<NX, V, W>() ? 0 : NX) + (LAST ? NX : 0) + W * col_len<NX, V, W>();
}

// tile sizes whose LDS and workgroup fit a CU
template <int NX, int V, int W> __host__ __device__ constexpr bool col_fits()
{
    using P = PlanV<NX, V>;
    const size_t tables = col_lean<NX, V, W>() ? (size_t)NX * 8  // s_nat of the last slice
                                                : (size_t)NX * 16 + (size_t)plan_tw_len<P>() * 8;
    return (size_t)W * col_len<NX, V, W>() * 8 + tables <= 160 * 1024 && W * P::T <= 1024;
}

// band limit and propagator P_x[i] * P_y[j] (which carries 1/(nx ny)) of one pixel
__device__ __forceinline__ float2 propagate_point(float2 f, float2 pxi, float2 pyj, bool keep)
{
    const float2 pr = float2{pxi.x * pyj.x - pxi.y * pyj.y, pxi.x * pyj.y + pxi.y * pyj.x};
    return keep ? float2{pr.x * f.x - pr.y * f.y, pr.x * f.y + pr.y * f.x} : float2{0.f, 0.f};
}
// the vacuum exit wave, shifted: psi0(k) e^{-2 pi i (i sx / nx + j sy / ny)}
__device__ __forceinline__ float2 add_vacuum(float2 x, float2 v0, float2 wx, float2 wy)
{
    const float2 w = float2{wx.x * wy.x - wx.y * wy.y, wx.x * wy.y + wx.y * wy.x};
    x.x += v0.x * w.x - v0.y * w.y;
    x.y += v0.x * w.y + v0.y * w.x;
    return x;
}

// One column-pass workgroup: logical block `blk` of `nblk` (XCD-banded over
// the pass's own blocks), LDS at smem.
template <int NX, int V, bool LAST, int W, bool PRUNE>
__device__ __forceinline__ void col_body(const ColPassArgs& a, int blk, int nblk, float2* smem)
{
    using P = PlanV<NX, V>;
    constexpr int E = P::E, T = P::T;
    constexpr int LEN = col_len<NX, V, W>();
    constexpr int PS = 0; // exchanges padded each its own way
    constexpr bool LEAN = col_lean<NX, V, W>(), LEANX = col_px_lean<NX, V, W>();
    // a column transform lies in one wavefront (wave-local exchanges) or
    // spans whole wavefronts (workgroup barriers)
    static_assert(64 % T == 0 || T % 64 == 0, "a column transform must align with wavefronts");
    constexpr bool WAVE = T <= 64;
    float2* s_tw = smem;
    float2* s_px = smem + (LEAN ? 0 : plan_tw_len<P>());
    float2* s_nat = s_px + (LEANX ? 0 : NX); // roots W_nx^e (last slice)
    float2* s_buf = s_nat + (LAST ? NX : 0);

    for (int e = threadIdx.x; e < NX; e += blockDim.x) {
        if constexpr (!LEAN) {
            if (e < plan_tw_len<P>()) s_tw[e] = a.tw[e];
        }
        if constexpr (!LEANX) s_px[e] = a.px[e];
        if constexpr (LAST) s_nat[e] = a.twx_nat[e];
    }
    const float2* tw = LEAN ? a.tw : s_tw;
    const float2* tpx = LEANX ? a.px : s_px;

    // neighbouring tiles share 128-byte lines (W = 8 reads 64 B per row): keep
    // them on one XCD, next to each other in dispatch order
    // tiles cover the stored columns [0, nc); tiles of padding columns only
    // (ncp is rounded up to 16) are not launched
    const int nc = a.ka + a.kb;
    const int ntiles = (nc + W - 1) / W;
    const int g = xcd_band(blk, nblk);
    const int b = div_by(g, ntiles, a.div);
    const int j0 = (g - b * ntiles) * W;
    float2* tile = a.psi + (int64_t)b * NX * a.ncp + j0;

    {   // coalesced load of the tile: one 32-bit lane offset, and a uniform
        // base per element.  Every load is in bounds (b < batch by the grid,
        // padding columns jc >= nc exist in the buffer), so all E loads are
        // issued before the first LDS write and overlap; what the padding
        // columns hold stays in their own tile columns, which nothing stores.
        const int c = threadIdx.x % W, r0 = threadIdx.x / W;
        const uint32_t o0 = (uint32_t)(r0 * a.ncp + c);
        const int64_t step = (int64_t)T * a.ncp;
        float2 v[E];
#pragma unroll
        for (int p = 0; p < E; ++p) v[p] = elem32(tile + p * step, o0);
#pragma unroll
        for (int p = 0; p < E; ++p) s_buf[c * LEN + col_slot<P>(r0, p)] = v[p];
    }
    __syncthreads();

    // with T a multiple of 64 a wavefront's column is uniform
    const int c = T % 64 == 0 ? __builtin_amdgcn_readfirstlane(threadIdx.x / T) : threadIdx.x / T;
    const int t = threadIdx.x % T;
    const int jc = j0 + c;
    const bool active = (b < a.batch) && (jc < nc);
    const int j = (jc < a.ka) ? jc : jc - nc + a.ny;
    float2* lds = s_buf + c * LEN;
    float2 x[E];
#pragma unroll
    for (int p = 0; p < E; ++p) x[p] = lds[col_slot<P>(t, p)];

    P::template run<false, float2, WAVE, PS>(x, lds, tw, t);

    // band limit (bw_limit + propagate's k^2 test, decided on the host) and
    // propagator P_x[i] * P_y[j]; P_y carries the 1/(nx ny) of the transforms and
    // of the transmission, over the FP32 transforms' gain (fp32_gain)
    const float2 pyj = active ? a.py[j] : float2{0.f, 0.f};
    // kept rows of this column, decided on the host (one pair per column
    // instead of a range table per row)
    const int2 ck = active ? a.colkeep[jc] : int2{0, 0};
#pragma unroll
    for (int p = 0; p < E; ++p) {
        if (PRUNE && in_zero_band<NX, E>(p)) {
            x[p] = float2{0.f, 0.f};
            continue;
        }
        // a pruned column keeps nothing of [3N/8, 5N/8), so its elements below
        // N/2 can only be of the low band
        const int i = t + T * p;
        const bool keep = PRUNE ? (T * p < NX / 2 ? i < ck.x : i >= NX - ck.y)
                                : (i < ck.x) || (i >= NX - ck.y);
        x[p] = propagate_point(x[p], elem_at(tpx, (uint32_t)t * 8u, T * p), pyj, keep);
    }

    if constexpr (!LAST) {
        P::template run<true, float2, WAVE, PS>(x, lds, tw, t);
    } else if (active) {
        const int2 sh = a.shift[b];
        const float2 wy = a.twy[((uint32_t)j * (uint32_t)sh.y) % (uint32_t)a.ny];
#pragma unroll
        for (int p = 0; p < E; ++p) {
            if (PRUNE && in_zero_band<NX, E>(p)) continue;
            const uint32_t i = (uint32_t)(t + T * p);
            const float2 wx = s_nat[(i * (uint32_t)sh.x) % (uint32_t)NX];
            x[p] = add_vacuum(x[p], a.psi0[(int64_t)j * NX + i], wx, wy);
        }
    }

    lds_sync<WAVE>();
#pragma unroll
    for (int p = 0; p < E; ++p) lds[col_slot<P>(t, p)] = x[p];
    __syncthreads();

    {   // coalesced store of the tile
        const int c2 = threadIdx.x % W, r0 = threadIdx.x / W;
        const bool ok = (b < a.batch) && (j0 + c2 < nc);
        const uint32_t o0 = (uint32_t)(r0 * a.ncp + c2);
        const int64_t step = (int64_t)T * a.ncp;
        // formed anew: twelve or sixteen bases kept from the loads would not
        // fit the scalar registers
        auto out = (__attribute__((address_space(1))) float2*)tile;
        asm("" : "+s"(out));
        if (ok) {
#pragma unroll
            for (int p = 0; p < E; ++p)
                elem32((float2*)(out + p * step), o0) = s_buf[c2 * LEN + col_slot<P>(r0, p)];
        }
    }
}

template <int NX, int V, bool LAST, int W, bool PRUNE>
__global__ void __launch_bounds__((col_bound<NX, V, W>())) col_pass_kernel(ColPassArgs a)
{
    __shared__ float2 smem[col_smem_len<NX, V, LAST, W>()];
    col_body<NX, V, LAST, W, PRUNE>(a, (int)blockIdx.x, (int)gridDim.x, smem);
}

} // namespace msf
