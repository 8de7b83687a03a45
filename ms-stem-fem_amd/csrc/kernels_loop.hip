// kernels_loop.hip -- the whole slice loop of one position in one workgroup,
// for grids whose wave fits a CU's LDS.
//
// The slice passes read and write every position's wave in memory twice per
// slice and cost two launches a slice (adfstem.cpp:1866-2132 per slice); on
// small grids the launches (4 us each) and the round trips are most of the
// time.  Here a workgroup keeps its position's wave in LDS from the first
// slice to the exit wave: a full row of ny values is the exchange buffer of
// its own row transform, and a column's values that of its column transform,
// so the plane needs no second buffer; transmission, vacuum rows and
// propagators, shared by all positions, come from L2.  The arithmetic per
// value is the passes' own (the same radix plans, transmit_point,
// propagate_point), so results equal theirs bit for bit.
//
// Bound by the latency of one CU working through a position: 64^2 3.3 us a
// slice (4 positions per CU fit the LDS, 2 the registers), 128^2 14.6 us for
// up to 256 positions at once, against 13 and 23 us for a slice's two passes
// over 256 positions.  Tried without gain: 512 instead of 1024 lanes at 128^2
// (17 us), a 16 x 8 plan at 128 (spills, 18 us), the transmission and vacuum
// pairs read ahead of the inverse transform (spills at 128^2, 17 us), 64^2
// held to 80 registers for a third position per CU (4.2 us a slice).
#include "slice_passes.hpp"

namespace msf {

// Rows are LEN slots apart (one padding slot every 8 values) and shifted by
// one slot every 8 rows, which spreads the column accesses over the banks.
template <int NX, int NY, int VX, int VY> struct LoopShape {
    using PX = PlanV<NX, VX>;
    using PY = PlanV<NY, VY>;
    static constexpr int LEN = lds_len(NY);
    static constexpr int PLANE = NX * LEN + NX / 8;
    static constexpr int TWX = plan_tw_len<PX>(), TWY = plan_tw_len<PY>();
    static constexpr int SMEM = PLANE + TWX + TWY;
    // lanes: every row's at once, at most 1024, or 512 for plans of 12 and
    // 24 values per lane, which spill under the 128 registers of 1024 lanes
    static constexpr int CAP = PX::E % 12 == 0 || PY::E % 12 == 0 ? 512 : 1024;
    static constexpr int NT = NX * PY::T < CAP ? NX * PY::T : CAP;
    static constexpr bool fits = (size_t)SMEM * 8 <= 160 * 1024 && NT % 64 == 0 && PX::T <= 64 &&
                                 PY::T <= 64;
};

template <int NX, int NY, int VX, int VY, bool FIRST, int TMODE>
__device__ __forceinline__ void loop_rows(const LoopArgs& a, const float2* t, const float2* u0,
                                          int2 sh, float2* plane, const float2* tw)
{
    using S = LoopShape<NX, NY, VX, VY>;
    using P = typename S::PY;
    constexpr int E = P::E, T = P::T, LEN = S::LEN;
    const RowPassArgs& r = a.row;
    const int hi = NY - r.kb;
    const int l = threadIdx.x % T;
#pragma unroll 1
    for (int i = threadIdx.x / T; i < NX; i += S::NT / T) {
        float2* lds = plane + i * LEN + (i >> 3);
        int ii = i - sh.x;
        if (ii < 0) ii += NX;
        const float2* trow = t + i * NY;
        const float2* urow = u0 + ii * (2 * NY);
        float2 x[E];
        if constexpr (!FIRST) {
#pragma unroll
            for (int p = 0; p < E; ++p) {
                const int j = l + T * p;
                if (in_zero_band<NY, E>(p)) {
                    x[p] = float2{0.f, 0.f};
                } else if (always_low<NY, E>(p) || always_high<NY, E>(p)) {
                    x[p] = lds[lds_pad(j)];
                } else {
                    const float2 v = lds[lds_pad(j)];
                    x[p] = (j < r.ka || j >= hi) ? v : float2{0.f, 0.f};
                }
            }
            P::template run<true, float2, true>(x, lds, tw, l);
        }
#pragma unroll
        for (int p = 0; p < E / 2; ++p) {
            const int j = l + T * p;
            int q = j - sh.y;
            if (q < 0) q += NY;
            const float4 tv = *reinterpret_cast<const float4*>(trow + 2 * j);
            const float4 uv = *reinterpret_cast<const float4*>(urow + 2 * q);
            x[p] = transmit_point<FIRST, TMODE>(x[p], float2{tv.x, tv.y}, float2{uv.x, uv.y}, r.inv_s);
            x[p + E / 2] = transmit_point<FIRST, TMODE>(x[p + E / 2], float2{tv.z, tv.w},
                                                        float2{uv.z, uv.w}, r.inv_s);
        }
        P::template run<false, float2, true>(x, lds, tw, l);
        lds_sync<true>();
#pragma unroll
        for (int p = 0; p < E; ++p) {
            const int j = l + T * p;
            if (in_zero_band<NY, E>(p)) continue;
            if (always_low<NY, E>(p) || always_high<NY, E>(p) || j < r.ka || j >= hi)
                lds[lds_pad(j)] = x[p];
        }
    }
}

template <int NX, int NY, int VX, int VY, bool LAST>
__device__ __forceinline__ void loop_cols(const LoopArgs& a, const float2* px, const float2* py,
                                          int2 sh, float2* plane, const float2* tw)
{
    using S = LoopShape<NX, NY, VX, VY>;
    using P = typename S::PX;
    constexpr int E = P::E, T = P::T, PS = -S::LEN;
    const ColPassArgs& c = a.col;
    const int nc = c.ka + c.kb;
    const int l = threadIdx.x % T;
#pragma unroll 1
    for (int jc = threadIdx.x / T; jc < nc; jc += S::NT / T) {
        const int j = jc < c.ka ? jc : jc - nc + NY;
        float2* lds = plane + lds_pad(j);
        float2 x[E];
#pragma unroll
        for (int p = 0; p < E; ++p) x[p] = lds[lds_pad_at<T, PS>(l, p)];
        P::template run<false, float2, true, PS>(x, lds, tw, l);
        const float2 pyj = py[j];
        const int2 ck = c.colkeep[jc];
#pragma unroll
        for (int p = 0; p < E; ++p) {
            if (in_zero_band<NX, E>(p)) {
                x[p] = float2{0.f, 0.f};
                continue;
            }
            const int i = l + T * p;
            x[p] = propagate_point(x[p], px[i], pyj, i < ck.x || i >= NX - ck.y);
        }
        if constexpr (!LAST) {
            P::template run<true, float2, true, PS>(x, lds, tw, l);
        } else {
            const float2 wy = c.twy[((uint32_t)j * (uint32_t)sh.y) % (uint32_t)NY];
#pragma unroll
            for (int p = 0; p < E; ++p) {
                if (in_zero_band<NX, E>(p)) continue;
                const uint32_t i = (uint32_t)(l + T * p);
                const float2 wx = c.twx_nat[(i * (uint32_t)sh.x) % (uint32_t)NX];
                x[p] = add_vacuum(x[p], c.psi0[j * NX + (int)i], wx, wy);
            }
        }
        lds_sync<true>();
#pragma unroll
        for (int p = 0; p < E; ++p) lds[lds_pad_at<T, PS>(l, p)] = x[p];
    }
}

template <int NX, int NY, int VX, int VY, int TMODE>
__global__ void __launch_bounds__((LoopShape<NX, NY, VX, VY>::NT)) slice_loop_kernel(LoopArgs a)
{
    using S = LoopShape<NX, NY, VX, VY>;
    __shared__ __align__(16) float2 smem[S::SMEM];
    float2 *plane = smem, *twx = smem + S::PLANE, *twy = twx + S::TWX;
    for (int e = threadIdx.x; e < S::TWX; e += S::NT) twx[e] = a.col.tw[e];
    for (int e = threadIdx.x; e < S::TWY; e += S::NT) twy[e] = a.row.tw[e];
    __syncthreads();
    const int b = blockIdx.x;
    const int2 sh = a.row.shift[b];
    const float2 *t = a.row.t, *u0 = a.row.u0, *px = a.col.px, *py = a.col.py;
    loop_rows<NX, NY, VX, VY, true, TMODE>(a, t, u0, sh, plane, twy);
    __syncthreads();
#pragma unroll 1
    for (int n = 1; n < a.slices; ++n) {
        loop_cols<NX, NY, VX, VY, false>(a, px, py, sh, plane, twx);
        t += NX * NY;
        u0 += 2 * NX * NY;
        px += NX;
        py += NY;
        __syncthreads();
        loop_rows<NX, NY, VX, VY, false, TMODE>(a, t, u0, sh, plane, twy);
        __syncthreads();
    }
    loop_cols<NX, NY, VX, VY, true>(a, px, py, sh, plane, twx);
    __syncthreads();
    // the exit wave in the passes' compact layout
    const int ka = a.col.ka, nc = ka + a.col.kb, ncp = a.col.ncp;
    float2* out = a.col.psi + (int64_t)b * NX * ncp;
    for (int e = threadIdx.x; e < NX * nc; e += S::NT) {
        const int i = e / nc, jc = e - i * nc;
        const int j = jc < ka ? jc : jc - nc + NY;
        out[i * ncp + jc] = plane[i * S::LEN + (i >> 3) + lds_pad(j)];
    }
}

// Grids compiled in: sides of 64 to 256 whose plane fits, with the lines
// between the loop and the passes (loop_faster): MIN, MINS, MIN2, A, B, A2, B2.
#define MSF_LOOP_GRIDS(G)                                                                          \
    G(64, 64, 1, 1, 257, 3.98f, 1.19f, 3.98f, 1.19f)                                               \
    G(64, 96, 4, 4, 257, 2.80f, 0.87f, 0.0f, 1.10f)                                                \
    G(96, 64, 4, 4, 257, 2.75f, 0.66f, 0.0f, 0.0f)                                                 \
    G(64, 128, 4, 4, 257, 1.70f, 1.07f, -0.09f, 1.20f)                                             \
    G(128, 64, 4, 4, 257, 1.32f, 1.06f, 0.02f, 1.11f)                                              \
    G(96, 96, 16, 16, 257, 1.22f, 0.79f, 0.05f, 0.91f)                                             \
    G(64, 192, 64, 100, 257, 0.90f, 0.82f, -0.17f, 0.92f)                                          \
    G(192, 64, 64, 64, 257, 1.15f, 0.94f, -0.25f, 1.12f)                                           \
    G(96, 128, 64, 100, 257, 0.77f, 0.93f, -0.34f, 0.99f)                                          \
    G(128, 96, 80, 100, 257, 0.83f, 0.77f, -0.76f, 0.83f)                                          \
    G(64, 256, 128, 128, 257, 1.09f, 0.95f, 0.14f, 1.10f)                                          \
    G(256, 64, 128, 128, 257, 1.10f, 1.02f, 0.14f, 1.21f)                                          \
    G(128, 128, 128, 128, 352, 0.70f, 0.95f, 0.10f, 1.08f)

// the automatic radix plan of a side (256: the alternate)
template <int N> static constexpr int loop_plan() { return N == 256 ? 1 : 0; }

template <int NX, int NY>
static bool loop_ok(const RowPassArgs& r, const ColPassArgs& c)
{
    static_assert(LoopShape<NX, NY, loop_plan<NX>(), loop_plan<NY>()>::fits, "plane over 160 KB");
    return r.plan == loop_plan<NY>() && c.plan == loop_plan<NX>() && r.prune && c.prune;
}

// The loop runs a position on one CU, the passes spread it over all: up to
// 64^2 the loop is always the faster, then from as many positions as fill the
// chip well enough (MIN; MINS of fewer than 4 slices, which leave the loop's
// start and end a larger part).  256 positions are a round of the CUs, and a round
// takes the same time however few of them it has, while the passes grow with
// the positions: a second round pays from MIN2 positions on, and of more than
// two rounds the loop is the faster while rounds <= A + B positions / 256 (the
// passes' fixed and per-position time over a round's, fitted to 30 batches of
// 513 to 2600 positions per grid; wrong by 4 % of the time at most).  On two
// chains one batch's last round and the next one's first run together, and
// the passes fill each other's gaps: there rounds and positions are those of
// all batches together, with A2 and B2 (512 to 7000 positions).  Passes / loop
// in us, sums included, 24 slices: 128^2 257 positions 650 / 772, 384 799 / 767,
// 513 988 / 1117, 640 1162 / 1111, 769 1342 / 1466; 128 x 96 640 994 / 1074, 768
// 1114 / 1077; 64 x 192 513 828 / 954, 704 1004 / 946; 96 x 128 513 882 / 978, 640
// 1019 / 990; 96^2 257 709 / 581, 769 995 / 1087; 256 x 64 513 1048 / 991.  Two
// chains, 12 slices: 128^2 1300 positions 1082 / 1149, 2300 1873 / 1689; 128 x 96
// 2300 1325 / 1611; 96 x 64 4200 1352 / 1538; 64 x 128 1657 / 1421.  40 slices,
// 64 and 80 positions: 64 x 192 568 / 555 and 639 / 553, 96 x 128 594 / 578 and
// 653 / 579, 128 x 96 577 / 627 and 655 / 624; one slice of 64: 39 / 45 each.
struct LoopLine {
    int min, min_short, min2;
    float a, b, a2, b2;
};
static bool loop_faster(const LoopLine& l, int batch, int slices, int64_t together)
{
    if (batch < (slices < 4 ? l.min_short : l.min)) return false;
    const int64_t n = together ? together : batch, rounds = (n + 255) / 256;
    if (together) return (float)rounds <= l.a2 + l.b2 * (float)n / 256.f;
    if (rounds <= 2) return rounds < 2 || batch >= l.min2;
    return (float)rounds <= l.a + l.b * (float)n / 256.f;
}

bool loop_supported(int nx, int ny, const RowPassArgs& r, const ColPassArgs& c, int slices,
                    int64_t together)
{
#define MSF_GRID(NX, NY, ...)                                                                      \
    if (nx == NX && ny == NY)                                                                      \
        return loop_ok<NX, NY>(r, c) && loop_faster(LoopLine{__VA_ARGS__}, r.batch, slices, together);
    MSF_LOOP_GRIDS(MSF_GRID)
#undef MSF_GRID
    return false;
}

hipError_t launch_slice_loop(int nx, int ny, int tmode, const LoopArgs& a, hipStream_t s)
{
    if (a.row.batch <= 0 || a.slices <= 0) return hipErrorInvalidValue;
    const dim3 grid((unsigned)a.row.batch);
#define MSF_GRID(NX, NY, ...)                                                                      \
    if (nx == NX && ny == NY) {                                                                    \
        if (!loop_ok<NX, NY>(a.row, a.col)) return hipErrorNotSupported;                           \
        constexpr int VX = loop_plan<NX>(), VY = loop_plan<NY>();                                  \
        const dim3 block(LoopShape<NX, NY, VX, VY>::NT);                                           \
        if (tmode == 0)                                                                            \
            hipLaunchKernelGGL((slice_loop_kernel<NX, NY, VX, VY, 0>), grid, block, 0, s, a);      \
        else                                                                                       \
            hipLaunchKernelGGL((slice_loop_kernel<NX, NY, VX, VY, 1>), grid, block, 0, s, a);      \
        return hipGetLastError();                                                                  \
    }
    MSF_LOOP_GRIDS(MSF_GRID)
#undef MSF_GRID
    return hipErrorNotSupported;
}

} // namespace msf
