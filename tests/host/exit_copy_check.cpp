// The copy of exit waves to the caller (msf_exit.cpp) on a stand-in for the
// runtime, on the CPU: copies are done when their event or stream is waited
// for and not before, as late as a device may do them, and pinned memory can
// be refused.  Blocks of both sizes, more parts than slots, two callers at
// once; rows hold the kept columns and zeros between them, or the call fails
// without leaving a copy in flight.
#include "../../ms-stem-fem_amd/csrc/msf_internal.hpp"

#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <deque>

namespace {

struct Op {
    void* dst;
    const void* src;
    size_t n;
    hipEvent_t event;
};
struct FakeStream {
    std::mutex m;
    std::deque<Op> queue;
    void run_to(hipEvent_t e) // null: everything
    {
        std::lock_guard<std::mutex> lk(m);
        bool found = !e;
        for (const Op& o : queue) found = found || o.event == e;
        if (!found) return; // already past
        while (!queue.empty()) {
            const Op o = queue.front();
            queue.pop_front();
            if (o.dst) std::memcpy(o.dst, o.src, o.n);
            if (o.event && o.event == e) return;
        }
    }
};
std::mutex g_m;
std::map<hipEvent_t, FakeStream*> g_recorded;
std::atomic<long> g_pinned{0}, g_refuse{0}, g_fail_copy{-1};
FakeStream* fake(hipStream_t s) { return reinterpret_cast<FakeStream*>(s); }

} // namespace

hipError_t hipHostMalloc(void** p, size_t n, unsigned)
{
    if (g_refuse) return hipErrorOutOfMemory;
    ++g_pinned;
    *p = std::malloc(n);
    std::memset(*p, 0xee, n);
    return hipSuccess;
}
hipError_t hipHostFree(void* p)
{
    --g_pinned;
    std::free(p);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t st)
{
    if (g_fail_copy >= 0 && g_fail_copy-- == 0) return hipErrorInvalidValue;
    std::lock_guard<std::mutex> lk(fake(st)->m);
    fake(st)->queue.push_back({d, s, n, nullptr});
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t s)
{
    fake(s)->run_to(nullptr);
    return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned)
{
    *e = reinterpret_cast<hipEvent_t>(new int);
    return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t e)
{
    std::lock_guard<std::mutex> lk(g_m);
    g_recorded.erase(e);
    delete reinterpret_cast<int*>(e);
    return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s)
{
    {
        std::lock_guard<std::mutex> lk(g_m);
        g_recorded[e] = fake(s);
    }
    std::lock_guard<std::mutex> lk(fake(s)->m);
    fake(s)->queue.push_back({nullptr, nullptr, 0, e});
    return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t e)
{
    FakeStream* s;
    {
        std::lock_guard<std::mutex> lk(g_m);
        s = g_recorded.at(e);
    }
    s->run_to(e);
    return hipSuccess;
}
hipError_t hipGetLastError() { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "error"; }

namespace msf_impl {
int fail(msf_ctx*, int code, const std::string&) { return code; }
} // namespace msf_impl

// 1 for a wrong value or a copy left in flight
static long one(int nx, int ny, int ka, int kb, int batch, bool* failed = nullptr)
{
    const int ncp = (ka + kb + 15) / 16 * 16;
    std::vector<float2> psi((size_t)batch * nx * ncp);
    for (size_t k = 0; k < psi.size(); ++k) psi[k] = float2{(float)(k % 100003), -(float)(k % 77)};
    std::vector<float> out((size_t)batch * nx * ny * 2, 1e30f);
    FakeStream s;
    const int rc = msf_impl::copy_exit_waves(nullptr, psi.data(), nx, ny, ncp, ka, kb, batch,
                                             reinterpret_cast<hipStream_t>(&s), out.data());
    long bad = !s.queue.empty();
    if (failed) {
        *failed = rc != MSF_OK;
        return bad;
    }
    if (rc != MSF_OK) return 1;
    for (int64_t r = 0; r < (int64_t)batch * nx; ++r)
        for (int j = 0; j < ny; ++j) {
            const int c = j < ka ? j : j >= ny - kb ? j - ny + ka + kb : -1;
            const float2 want = c >= 0 ? psi[(size_t)r * ncp + c] : float2{0.f, 0.f};
            const float* got = &out[(size_t)(r * ny + j) * 2];
            if (got[0] != want.x || got[1] != want.y) return 1;
        }
    return bad;
}

static long sizes()
{
    // under a small block (256 KB), just over it, one part, and more parts
    // (4 MB) than a block has slots
    return one(64, 64, 22, 21, 2) + one(64, 64, 22, 21, 11) + one(64, 64, 64, 0, 9) +
           one(96, 384, 64, 63, 6) + one(512, 512, 171, 170, 15) + one(16, 16, 0, 0, 3);
}

int main()
{
    msf_impl::exit_context(1);
    const long plain = sizes();
    long both[2] = {0, 0};
    {
        std::thread a([&] { both[0] = sizes(); }), b([&] { both[1] = sizes(); });
        a.join();
        b.join();
    }
    bool failed = false;
    long flight = 0, silent = 0;
    for (long k : {0, 1, 5}) { // a copy of a large block fails
        g_fail_copy = k;
        flight += one(512, 512, 171, 170, 15, &failed);
        silent += !failed;
    }
    g_fail_copy = -1;
    const long kept = g_pinned;
    msf_impl::exit_context(-1);
    const long left = g_pinned;
    msf_impl::exit_context(1);
    g_refuse = 1;
    const long refused = sizes();
    msf_impl::exit_context(-1);
    std::printf("plain %ld both %ld flight %ld silent %ld kept %d left %ld refused %ld\n", plain,
                both[0] + both[1], flight, silent, kept >= 1 && kept <= 4, left, refused);
    return 0;
}
