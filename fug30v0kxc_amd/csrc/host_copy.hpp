// host_copy.hpp -- host side of the state transfers: copies between a caller's
// pageable array and the pinned staging buffer on several threads, overlapped
// with the DMA of the neighbouring chunks.
//
// One thread copies a fresh (never touched) destination at 1.5-2 GB/s, bound by
// its page faults; the DMA into pinned memory runs at about 50 GB/s.  Fetching
// the 671 MB state of 256^2 x 160 took 74 ms with one thread copying each field
// after its DMA; a stretch of 100 steps and that fetch went from 319 to 272 ms
// with this (512^2 x 64 mixed, 60 steps: 326 -> 240 ms).
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cstring>
#include <thread>
#include <vector>

namespace mhd {

constexpr int XFER_CHUNKS = 16;            // DMA chunks of one field, at most
constexpr int XFER_THREADS = 16;
constexpr long XFER_SERIAL = 1L << 17;     // doubles per thread below which threads do not pay
// Fields from 32 MB on are copied by threads: that is where the C allocator's
// largest threshold for a mapping of its own lies, so their destinations are
// fresh pages.  Smaller ones are mostly memory in use before, which one thread
// copies faster than a team starts: 48 fields of 1.5 to 12 MB took 15 ms longer.
constexpr long XFER_MIN = 1L << 22;

inline int host_threads(long n, long grain)
{
    const long hw = (long)std::thread::hardware_concurrency();
    return (int)std::max(1L, std::min({(long)XFER_THREADS, hw > 0 ? hw : 1L, n / grain}));
}

// runs f(t) for t = 0 .. parts-1 on a thread each (f outlives the team); the
// parts from `started` on, whose threads could not be started, are the caller's
struct HostTeam {
    std::vector<std::thread> th;
    int started = 0;
    template <typename Fn>
    HostTeam(int parts, const Fn& f)
    {
        try {
            th.reserve(parts);
            for (int t = 0; t < parts; ++t) {
                th.emplace_back([&f, t] { f(t); });
                ++started;
            }
        } catch (...) {
        }
    }
    void join()
    {
        for (auto& x : th)
            if (x.joinable()) x.join();
    }
    ~HostTeam() { join(); }
};

// f(begin, end) over [0, n) in contiguous parts
template <typename Fn>
void host_parallel(long n, long grain, Fn&& f)
{
    const int T = host_threads(n, grain);
    auto part = [&](int t) { f(n * t / T, n * (t + 1) / T); };
    if (T == 1) {
        part(0);
        return;
    }
    HostTeam team(T - 1, part);
    for (int t = team.started; t < T; ++t) part(t);
    team.join();
}

// n doubles from the device array `from` to `dst`, through the pinned buffer
// hbuf (n doubles); ev: XFER_CHUNKS events.  Returns with the copy complete.
inline hipError_t fetch_doubles(double* dst, const double* from, long n, double* hbuf, hipEvent_t* ev, hipStream_t s)
{
    const int T = n < XFER_MIN ? 1 : host_threads(n, XFER_SERIAL);
    if (T == 1) {
        // an event to wait for would cost 5 us a call
        hipError_t e = hipMemcpyAsync(hbuf, from, n * sizeof(double), hipMemcpyDeviceToHost, s);
        if (e == hipSuccess) e = hipStreamSynchronize(s);
        if (e == hipSuccess) memcpy(dst, hbuf, n * sizeof(double));
        return e;
    }
    const int C = XFER_CHUNKS;
    auto lo = [&](int c) { return n * c / C; };
    for (int c = 0; c < C; ++c) {
        const long b = lo(c), m = lo(c + 1) - b;
        hipError_t e = hipMemcpyAsync(hbuf + b, from + b, m * sizeof(double), hipMemcpyDeviceToHost, s);
        if (e == hipSuccess) e = hipEventRecord(ev[c], s);
        if (e != hipSuccess) {
            (void)hipStreamSynchronize(s);
            return e;
        }
    }
    std::atomic<int> ready{0};
    auto slice = [&](int t, int c) {
        const long b = lo(c), m = lo(c + 1) - b, p = b + m * t / T, q = b + m * (t + 1) / T;
        memcpy(dst + p, hbuf + p, (q - p) * sizeof(double));
    };
    auto work = [&](int t) {
        for (int c = 0; c < C; ++c) {
            int r;
            while ((r = ready.load(std::memory_order_acquire)) <= c)
                if (r < 0) return;
                else std::this_thread::yield();
            slice(t, c);
        }
    };
    HostTeam team(T, work);
    hipError_t err = hipSuccess;
    for (int c = 0; c < C && err == hipSuccess; ++c) {
        err = hipEventSynchronize(ev[c]);
        ready.store(err == hipSuccess ? c + 1 : -1, std::memory_order_release);
    }
    if (err == hipSuccess)
        for (int t = team.started; t < T; ++t)
            for (int c = 0; c < C; ++c) slice(t, c);
    team.join();
    return err;
}

// n doubles from `src` to the device array `to`; complete on s when it returns
// success and s has been synchronised (hbuf is in use until then)
inline hipError_t send_doubles(double* to, const double* src, long n, double* hbuf, hipStream_t s)
{
    const int T = n < XFER_MIN ? 1 : host_threads(n, XFER_SERIAL);
    const int C = T == 1 ? 1 : XFER_CHUNKS;
    auto lo = [&](int c) { return n * c / C; };
    std::atomic<int> done[XFER_CHUNKS] = {};
    auto slice = [&](int t, int c) {
        const long b = lo(c), m = lo(c + 1) - b, p = b + m * t / T, q = b + m * (t + 1) / T;
        memcpy(hbuf + p, src + p, (q - p) * sizeof(double));
    };
    auto work = [&](int t) {
        for (int c = 0; c < C; ++c) {
            slice(t, c);
            done[c].fetch_add(1, std::memory_order_release);
        }
    };
    HostTeam team(T > 1 ? T : 0, work);
    hipError_t err = hipSuccess;
    for (int c = 0; c < C; ++c) {
        for (int t = team.started; t < T; ++t) slice(t, c);
        while (done[c].load(std::memory_order_acquire) < team.started) std::this_thread::yield();
        const long b = lo(c), m = lo(c + 1) - b;
        if (err == hipSuccess) err = hipMemcpyAsync(to + b, hbuf + b, m * sizeof(double), hipMemcpyHostToDevice, s);
    }
    team.join();
    return err;
}

}  // namespace mhd
