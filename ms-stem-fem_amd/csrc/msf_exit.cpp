// msf_exit.cpp -- exit waves of a batch to the caller's memory.
//
// The waves are copied as stored (compact columns, 2/3 of a plane) into
// pinned host blocks and spread over the caller's full rows, with the zeros
// between the kept columns, by several threads while the next block is on its
// way.  One pageable copy of the expanded planes ran at 10 GB/s: the runtime
// stages it and a single thread takes the page faults of a fresh caller array
// (30 positions of 512^2, 63 MB: 6.1 ms); the pinned copy runs at 56 GB/s
// (0.8 ms; the call with its 1.0 ms of slices 7.0 -> 2.3 ms into fresh memory).
#include "msf_internal.hpp"

#include <algorithm>
#include <cstdlib>
#include <cstring>
#include <system_error>

namespace msf_impl {

namespace {

// Pinned blocks of two sizes, kept for the next run of any context while a
// context lives, at most two of each; the last context's end frees them.
constexpr size_t kPinnedBytes[2] = {256u << 10, 16u << 20};
constexpr size_t kPinnedKept = 2;
struct PinnedPool {
    std::mutex m;
    std::vector<void*> idle[2];
    int contexts = 0;
};
PinnedPool& pool()
{
    static PinnedPool* p = new PinnedPool; // contexts may end during static destruction
    return *p;
}

struct PinnedBlock {
    int kind;
    char* p = nullptr;
    bool pinned = true;
    explicit PinnedBlock(int k) : kind(k) {}
    PinnedBlock(const PinnedBlock&) = delete;
    PinnedBlock& operator=(const PinnedBlock&) = delete;
    hipError_t get()
    {
        {
            std::lock_guard<std::mutex> lk(pool().m);
            std::vector<void*>& v = pool().idle[kind];
            if (!v.empty()) {
                p = static_cast<char*>(v.back());
                v.pop_back();
                return hipSuccess;
            }
        }
        void* q = nullptr;
        pinned = hipHostMalloc(&q, kPinnedBytes[kind], hipHostMallocPortable) == hipSuccess;
        if (!pinned) { // the copy still works from ordinary memory
            (void)hipGetLastError();
            q = std::malloc(kPinnedBytes[kind]);
        }
        p = static_cast<char*>(q);
        return p ? hipSuccess : hipErrorOutOfMemory;
    }
    ~PinnedBlock()
    {
        if (!p) return;
        if (!pinned) {
            std::free(p);
            return;
        }
        {
            std::lock_guard<std::mutex> lk(pool().m);
            std::vector<void*>& v = pool().idle[kind];
            if (v.size() < kPinnedKept && v.capacity() >= kPinnedKept) {
                v.push_back(p);
                return;
            }
        }
        (void)hipHostFree(p);
    }
};

// Rows of up to kShort values are many and small: a call of memset and two of
// memcpy each cost more than the bytes (837 waves of 16^2, 13,392 rows: the call
// 207 us with them, 153 without).
constexpr int kShort = 64;

void copy_values(float2* d, const float2* s, int n)
{
    if (n > kShort / 2) {
        std::memcpy(d, s, (size_t)n * sizeof(float2));
        return;
    }
    int k = 0;
    for (; k + 4 <= n; k += 4) {
        std::memcpy(d + k, s + k, 4 * sizeof(float2));
        asm volatile("" ::: "memory"); // stays a loop, not a call
    }
    for (; k < n; ++k) d[k] = s[k];
}

// rows [r0, r1): the zeros between the kept columns of full rows (short rows:
// everything, in one go)
void zero_rows(int64_t r0, int64_t r1, int ka, int kb, int ny, float* dst)
{
    if (ny <= kShort) {
        std::memset(dst + r0 * (2 * (int64_t)ny), 0, (size_t)(r1 - r0) * ny * sizeof(float2));
        return;
    }
    for (int64_t r = r0; r < r1; ++r)
        std::memset(dst + r * (2 * (int64_t)ny) + 2 * ka, 0, (size_t)(ny - ka - kb) * sizeof(float2));
}
// rows [r0, r1): the kept columns of a block of compact rows into full rows
void spread_rows(const float2* src, int64_t r0, int64_t r1, int ncp, int ka, int kb, int ny,
                 float* dst)
{
    for (int64_t r = r0; r < r1; ++r) {
        const float2* s = src + r * ncp;
        float2* d = reinterpret_cast<float2*>(dst + r * (2 * (int64_t)ny));
        copy_values(d, s, ka);
        copy_values(d + ny - kb, s + ka, kb);
    }
}

constexpr int kSlots = 4; // parts of a large block in flight

// The copies of one call: the calling thread issues part k into slot k %
// kSlots once part k - kSlots is spread, waits for it and announces it; every
// thread (the caller's too) spreads its share of the rows of each part.
struct Drain {
    std::mutex m;
    std::condition_variable cv;
    int64_t ready = 0;           // parts announced
    std::vector<int64_t> done;   // parts spread, per thread
    bool stop = false;
    int64_t spread()
    {
        return *std::min_element(done.begin(), done.end());
    }
};

} // namespace

void exit_context(int delta)
{
    std::vector<void*> drop;
    {
        std::lock_guard<std::mutex> lk(pool().m);
        for (std::vector<void*>& v : pool().idle) v.reserve(kPinnedKept);
        pool().contexts += delta;
        if (pool().contexts == 0)
            for (std::vector<void*>& v : pool().idle) {
                drop.insert(drop.end(), v.begin(), v.end());
                v.clear();
            }
    }
    for (void* p : drop) (void)hipHostFree(p);
}

int copy_exit_waves(msf_ctx* c, const float2* psi, int nx, int ny, int ncp, int ka, int kb,
                    int64_t batch, hipStream_t s, float* dst)
{
    const int64_t rows = batch * nx;
    const size_t row = (size_t)ncp * sizeof(float2);
    const size_t slot = kPinnedBytes[1] / kSlots;
    PinnedBlock blk((size_t)rows * row <= kPinnedBytes[0] ? 0 : 1);
    HIPCHK(c, blk.get());
    // one part: nothing to overlap, so no events and no threads (34 waves of
    // 32^2 86 -> 76 us)
    if ((size_t)rows * row <= slot) {
        HIPCHK(c, hipMemcpyAsync(blk.p, psi, (size_t)rows * row, hipMemcpyDeviceToHost, s));
        zero_rows(0, rows, ka, kb, ny, dst); // while the GPU works
        HIPCHK(c, hipStreamSynchronize(s));
        spread_rows(reinterpret_cast<const float2*>(blk.p), 0, rows, ncp, ka, kb, ny, dst);
        return MSF_OK;
    }
    const int64_t per = (int64_t)(slot / row); // rows per part
    const int64_t parts = (rows + per - 1) / per;
    struct Events {
        hipEvent_t e[kSlots] = {};
        ~Events()
        {
            for (hipEvent_t x : e)
                if (x) (void)hipEventDestroy(x);
        }
    } ev;
    for (hipEvent_t& e : ev.e) HIPCHK(c, hipEventCreateWithFlags(&e, hipEventDisableTiming));
    // whatever happens, no copy into the block is left in flight when it goes back
    struct Quiet {
        hipStream_t s;
        ~Quiet() { (void)hipStreamSynchronize(s); }
    } quiet{s};

    // a thread per 4 MB, at most 8: more gain nothing over the link's rate
    const unsigned hw = std::max(1u, std::thread::hardware_concurrency());
    const int want = (int)std::min<int64_t>({8, (int64_t)hw, parts});
    Drain d;
    d.done.assign((size_t)want, 0);
    auto work = [&](int64_t k, int w) {
        const int64_t n = std::min(per, rows - k * per);
        const float2* src = reinterpret_cast<const float2*>(blk.p + (size_t)(k % kSlots) * slot);
        spread_rows(src, n * w / want, n * (w + 1) / want, ncp, ka, kb, ny,
                    dst + k * per * (2 * (int64_t)ny));
    };
    // the zeros first: they need no wave, and take most of the page faults of
    // fresh memory while the slices still run
    auto zero = [&](int w) {
        for (int64_t k = 0; k < parts; ++k) {
            const int64_t n = std::min(per, rows - k * per);
            zero_rows(k * per + n * w / want, k * per + n * (w + 1) / want, ka, kb, ny, dst);
        }
    };
    auto run = [&](int w) {
        zero(w);
        for (int64_t k = 0; k < parts; ++k) {
            {
                std::unique_lock<std::mutex> lk(d.m);
                d.cv.wait(lk, [&] { return d.ready > k || d.stop; });
                if (d.ready <= k) return;
            }
            work(k, w);
            {
                std::lock_guard<std::mutex> lk(d.m);
                d.done[(size_t)w] = k + 1;
            }
            d.cv.notify_all();
        }
    };
    struct Threads { // ended before anything they use
        Drain& d;
        std::vector<std::thread> v;
        ~Threads()
        {
            {
                std::lock_guard<std::mutex> lk(d.m);
                d.stop = true;
            }
            d.cv.notify_all();
            for (std::thread& t : v) t.join();
        }
    } threads{d, {}};
    int started = 1; // shares 1 .. started - 1 have threads, the rest are the caller's
    threads.v.reserve((size_t)want);
    try {
        for (; started < want; ++started) threads.v.emplace_back(run, started);
    } catch (const std::system_error&) { // the caller spreads the shares left
    }
    int64_t issued = 0;
    for (int64_t k = 0; k < parts; ++k) {
        for (; issued < parts && issued < k + kSlots; ++issued) {
            {
                std::unique_lock<std::mutex> lk(d.m); // the slot's last part is spread
                if (issued >= kSlots) d.cv.wait(lk, [&] { return d.spread() > issued - kSlots; });
            }
            const int sl = (int)(issued % kSlots);
            const int64_t n = std::min(per, rows - issued * per);
            HIPCHK(c, hipMemcpyAsync(blk.p + (size_t)sl * slot, psi + issued * per * ncp,
                                     (size_t)n * row, hipMemcpyDeviceToHost, s));
            HIPCHK(c, hipEventRecord(ev.e[sl], s));
        }
        if (k == 0) {
            zero(0);
            for (int w = started; w < want; ++w) zero(w);
        }
        HIPCHK(c, hipEventSynchronize(ev.e[k % kSlots]));
        {
            std::lock_guard<std::mutex> lk(d.m);
            d.ready = k + 1;
        }
        d.cv.notify_all();
        work(k, 0);
        for (int w = started; w < want; ++w) work(k, w);
        std::lock_guard<std::mutex> lk(d.m);
        d.done[0] = k + 1;
        for (int w = started; w < want; ++w) d.done[(size_t)w] = k + 1;
    }
    std::unique_lock<std::mutex> lk(d.m);
    d.cv.wait(lk, [&] { return d.spread() >= parts; });
    return MSF_OK;
}

} // namespace msf_impl
