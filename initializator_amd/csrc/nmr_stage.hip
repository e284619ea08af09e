// nmr_stage.hip -- copies between device arrays and a caller's host arrays
// through a ring of pinned slots: the copy engine moves one slot while worker
// threads convert the others.
//
// What bounds a large download is the host: FP32 rows become FP64 arrays whose
// pages the caller has just allocated, so the kernel clears each on its first
// touch, and one thread does 7 GB/s of that behind pageable copies: 256^3, two
// components, 268 MB: 37.3 ms; eight threads on 1 MiB slots: 5.6 (48 GB/s).
// 512x512x130 76 -> 10.5 ms, 203x97x151 3.6-6.6 -> 1.1, 64^3 0.24 -> 0.11.  Up:
// the net's 11.8 MB of features at 96x80x64 (with its pass and the result)
// 0.93 -> 0.73 ms.
#include "nmr_internal.h"

#include <condition_variable>
#include <mutex>
#include <thread>

using nmri::fail;

namespace nmri {

namespace {

constexpr int kWorkers = 8; // threads of a large copy, the caller among them

// The threads of one copy: joined before it returns.
struct Team {
    std::vector<std::thread> t;
    template <typename F>
    void start(int n, const F& f)
    {
        try {
            t.reserve((size_t)n);
            for (int i = 0; i < n; i++) t.emplace_back(f);
        } catch (...) {
            // fewer threads than asked for, or none: the caller works too
        }
    }
    ~Team()
    {
        for (auto& x : t) x.join();
    }
};

} // namespace

HostStage::~HostStage()
{
    if (buf) (void)hipHostFree(buf);
    for (hipEvent_t e : ev)
        if (e) (void)hipEventDestroy(e);
}

int HostStage::open(int slots)
{
    slots = std::min(slots, kSlots);
    for (int i = 0; i < slots; i++)
        if (!ev[i]) HIP_TRY(hipEventCreateWithFlags(&ev[i], hipEventDisableTiming));
    if (slots <= have) return NMR_OK;
    if (buf) (void)hipHostFree(buf);
    buf = nullptr;
    have = 0;
    HIP_TRY(hipHostMalloc((void**)&buf, (size_t)slots * kSlotBytes, hipHostMallocDefault));
    have = slots;
    return NMR_OK;
}

int HostStage::down(hipStream_t s, const float* const* src, int arrays, size_t n,
                    const std::function<void(int, size_t, size_t, const float*)>& use)
{
    if (arrays < 1 || n == 0) {
        HIP_TRY(hipStreamSynchronize(s));
        return NMR_OK;
    }
    // a thread for each 768 KiB (starting one costs 20 us), and pieces of up to
    // a slot that give every thread one
    const size_t total = n * (size_t)arrays;
    const int threads = (int)std::min<size_t>(kWorkers, std::max<size_t>(1, total / ((size_t)3 << 16)));
    const size_t per = std::min(kSlotBytes / sizeof(float), (total + threads - 1) / threads);
    const size_t each = (n + per - 1) / per, chunks = each * (size_t)arrays; // pieces of an array, of all
    if (open((int)std::min<size_t>(chunks, kSlots)) != NMR_OK) { // no pinned memory: through pageable memory
        (void)hipGetLastError();
        std::vector<float> h(n);
        for (int q = 0; q < arrays; q++) {
            HIP_TRY(hipMemcpyAsync(h.data(), src[q], n * sizeof(float), hipMemcpyDeviceToHost, s));
            HIP_TRY(hipStreamSynchronize(s));
            use(q, 0, n, h.data());
        }
        return NMR_OK;
    }
    auto slot = [&](size_t c) { return reinterpret_cast<float*>(buf + (c % have) * kSlotBytes); };
    if (chunks == 1) {
        HIP_TRY(hipMemcpyAsync(slot(0), src[0], n * sizeof(float), hipMemcpyDeviceToHost, s));
        HIP_TRY(hipStreamSynchronize(s));
        use(0, 0, n, slot(0));
        return NMR_OK;
    }
    auto first = [&](size_t c) { return c % each * per; };
    auto count = [&](size_t c) { return std::min(per, n - first(c)); };
    auto issue = [&](size_t c) -> hipError_t {
        hipError_t e = hipMemcpyAsync(slot(c), src[c / each] + first(c), count(c) * sizeof(float), hipMemcpyDeviceToHost, s);
        return e != hipSuccess ? e : hipEventRecord(ev[c % have], s);
    };
    std::mutex mu;
    std::condition_variable cv;
    size_t here = 0, next = 0; // chunks that have arrived; the next one to convert
    std::vector<uint8_t> done(chunks, 0);
    size_t clear = 0;          // chunks before it are converted: their slots are free
    bool stop = false;
    // Converts one arrived chunk; false: nothing to do (wait: until there is).
    auto work = [&](bool wait) {
        size_t c;
        {
            std::unique_lock<std::mutex> l(mu);
            if (wait) cv.wait(l, [&] { return stop || next < here || next == chunks; });
            if (stop || next >= here) return false;
            c = next++;
        }
        use((int)(c / each), first(c), count(c), slot(c));
        {
            std::lock_guard<std::mutex> l(mu);
            done[c] = 1;
            while (clear < chunks && done[clear]) clear++;
        }
        cv.notify_all();
        return true;
    };
    hipError_t e = hipSuccess;
    {
        Team team;
        size_t sent = 0;
        while (e == hipSuccess && sent < std::min<size_t>(chunks, have)) e = issue(sent++);
        if (e == hipSuccess)
            team.start(threads - 1, [&] {
                while (work(true)) {}
            });
        for (size_t c = 0; c < chunks && e == hipSuccess; c++) {
            for (;;) { // copies on their way into every free slot
                size_t free_to;
                {
                    std::lock_guard<std::mutex> l(mu);
                    free_to = std::min(chunks, clear + have);
                }
                while (e == hipSuccess && sent < free_to) e = issue(sent++);
                if (sent > c || e != hipSuccess) break;
                if (!work(false)) { // every slot holds a chunk that another thread converts
                    std::unique_lock<std::mutex> l(mu);
                    cv.wait(l, [&] { return clear + have > c; });
                }
            }
            if (e == hipSuccess) e = hipEventSynchronize(ev[c % have]);
            {
                std::lock_guard<std::mutex> l(mu);
                if (e == hipSuccess) here = c + 1;
                else stop = true;
            }
            cv.notify_all();
        }
        while (e == hipSuccess && work(false)) {}
    }
    if (e != hipSuccess) (void)hipStreamSynchronize(s);
    HIP_TRY(e);
    return NMR_OK;
}

int HostStage::up(hipStream_t s, float* dst, const float* src, size_t n)
{
    constexpr size_t per = kSlotBytes / sizeof(float);
    const size_t chunks = (n + per - 1) / per;
    if (chunks == 0) return NMR_OK;
    if (open((int)std::min<size_t>(chunks, kSlots)) != NMR_OK) {
        (void)hipGetLastError();
        HIP_TRY(hipMemcpyAsync(dst, src, n * sizeof(float), hipMemcpyHostToDevice, s));
        HIP_TRY(hipStreamSynchronize(s));
        return NMR_OK;
    }
    auto slot = [&](size_t c) { return buf + (c % have) * kSlotBytes; };
    auto count = [&](size_t c) { return std::min(per, n - c * per) * sizeof(float); };
    std::mutex mu;
    std::condition_variable cv;
    size_t next = 0, may = std::min<size_t>(chunks, have); // the next chunk to fill; chunks before `may` have a free slot
    std::vector<uint8_t> full(chunks, 0);
    auto work = [&](bool wait) {
        size_t c;
        {
            std::unique_lock<std::mutex> l(mu);
            if (wait) cv.wait(l, [&] { return next < may || next == chunks; });
            if (next >= may) return false;
            c = next++;
        }
        std::memcpy(slot(c), src + c * per, count(c));
        {
            std::lock_guard<std::mutex> l(mu);
            full[c] = 1;
        }
        cv.notify_all();
        return true;
    };
    hipError_t e = hipSuccess;
    {
        Team team;
        if (chunks > 1)
            team.start((int)std::min<size_t>(kWorkers, chunks) - 1, [&] {
                while (work(true)) {}
            });
        for (size_t c = 0; c < chunks; c++) {
            for (;;) {
                {
                    std::lock_guard<std::mutex> l(mu);
                    if (full[c]) break;
                }
                if (!work(false)) {
                    std::unique_lock<std::mutex> l(mu);
                    cv.wait(l, [&] { return full[c] != 0; });
                }
            }
            // (after an error the chunks are still filled, so that every thread ends)
            if (e == hipSuccess) e = hipMemcpyAsync(dst + c * per, slot(c), count(c), hipMemcpyHostToDevice, s);
            if (e == hipSuccess) e = hipEventRecord(ev[c % have], s);
            // two copies stay on their way; the one before them frees its slot
            if (c >= 2 && may < chunks) {
                const size_t old = c - 2;
                if (e == hipSuccess) e = hipEventSynchronize(ev[old % have]);
                {
                    std::lock_guard<std::mutex> l(mu);
                    may = std::max(may, std::min(chunks, old + 1 + have));
                }
                cv.notify_all();
            }
        }
    }
    // the slots are free for the next copy, and the source for its owner
    const hipError_t w = hipStreamSynchronize(s);
    HIP_TRY(e);
    HIP_TRY(w);
    return NMR_OK;
}

int HostStage::down_rows(hipStream_t s, const float* const* src, int arrays, int nx, size_t rows, int pitch,
                         double* const* dst)
{
    return down(s, src, arrays, rows * (size_t)pitch, [=](int q, size_t i, size_t n, const float* p) {
        for (size_t e = i + n; i < e;) { // one row, or what of it the piece holds
            const size_t r = i / (size_t)pitch, x = i % (size_t)pitch, end = std::min(e, (r + 1) * (size_t)pitch);
            const size_t stop = std::min(end, r * (size_t)pitch + (size_t)nx);
            double* d = dst[q] + r * (size_t)nx + x;
            for (size_t k = 0; i + k < stop; k++) d[k] = (double)p[k];
            p += end - i;
            i = end;
        }
    });
}

} // namespace nmri
