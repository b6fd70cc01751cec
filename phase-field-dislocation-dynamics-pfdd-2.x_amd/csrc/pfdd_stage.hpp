// pfdd_stage.hpp -- fields from device memory to a caller's pageable memory.
//
// A copy to pageable memory is bound by the host: the runtime moves it through
// its own staging with one thread, and a fresh array faults its pages in while
// it is written.  Here the device copies into a ring of pinned slots and several
// threads move (widen, spread) the slots' contents.  33.5 MB to a fresh array:
// 1.9-3.2 -> 1.2 ms; strain and stress fields, 38 MB spread over 75 MB of fresh
// arrays: 5.8 -> 2.8 ms.  Below MIN_BYTES the runtime's own copy is taken: 12.6 MB
// is 0.8 ms that way, 0.5 ms through the ring, and 1.4-2 ms where the threads
// have to win CPUs from a caller's own spinning pool.
// The other direction stays with the runtime: it reads a caller's pages at 30
// GB/s.
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cstddef>
#include <thread>
#include <vector>

namespace pfdd {

struct Stage {
    static constexpr int K = 8, THREADS = 6;
    static constexpr size_t CHUNK = (size_t)2 << 20, MIN_BYTES = (size_t)16 << 20;
    char *mem = nullptr; // as many slots, up to K, as the largest move used; kept until release()
    size_t size = 0;
    hipEvent_t ev[K] = {};

    hipError_t ready(size_t bytes)
    {
        bytes = std::min(bytes, K * CHUNK);
        if (size >= bytes) return hipSuccess;
        release();
        for (hipEvent_t &e : ev) {
            const hipError_t r = hipEventCreateWithFlags(&e, hipEventDisableTiming);
            if (r != hipSuccess) return r;
        }
        const hipError_t r = hipHostMalloc((void **)&mem, bytes, hipHostMallocDefault);
        if (r == hipSuccess) size = bytes;
        return r;
    }
    void release()
    {
        for (hipEvent_t &e : ev)
            if (e) {
                (void)hipEventDestroy(e);
                e = nullptr;
            }
        if (mem) (void)hipHostFree(mem);
        mem = nullptr;
        size = 0;
    }

    // bytes of device memory through the ring; each chunk that has arrived is
    // handed to work(slot, offset, length), on several threads at once.  Returns
    // after the last one.
    template <typename Work>
    hipError_t out(const char *dev, size_t bytes, hipStream_t st, Work work)
    {
        const hipError_t e = ready(bytes);
        if (e != hipSuccess) return e;
        const size_t n = (bytes + CHUNK - 1) / CHUNK;
        std::atomic<size_t> next{0}, issued{0};
        std::atomic<size_t> round[K] = {}; // chunks a worker is done with, per slot
        std::atomic<int> err{hipSuccess};
        int device = 0;
        (void)hipGetDevice(&device);
        auto len = [&](size_t i) { return std::min(CHUNK, bytes - i * CHUNK); };
        auto wait = [&](auto ok) {
            while (!ok() && err.load() == hipSuccess) std::this_thread::yield();
            return err.load() == hipSuccess;
        };
        auto check = [&](hipError_t r) {
            if (r != hipSuccess) err.store(r);
            return r == hipSuccess;
        };
        auto worker = [&] {
            if (!check(hipSetDevice(device))) return;
            for (size_t i; (i = next.fetch_add(1)) < n;) {
                const int k = (int)(i % K);
                if (!wait([&] { return issued.load() > i; }) || !check(hipEventSynchronize(ev[k]))) return;
                work(mem + k * CHUNK, i * CHUNK, len(i));
                round[k].store(i / K + 1);
            }
        };
        std::vector<std::thread> pool;
        try {
            const size_t cpus = std::max(1u, std::thread::hardware_concurrency());
            const size_t want = std::min({n, (size_t)THREADS, cpus});
            pool.reserve(want);
            while (n > 1 && pool.size() < want) pool.emplace_back(worker);
        } catch (...) { // fewer threads than asked for
        }
        for (size_t i = 0; i < n; ++i) {
            const int k = (int)(i % K);
            if (!pool.empty() && !wait([&] { return round[k].load() >= i / K; })) break;
            if (!check(hipMemcpyAsync(mem + k * CHUNK, dev + i * CHUNK, len(i), hipMemcpyDeviceToHost, st)) ||
                !check(hipEventRecord(ev[k], st)))
                break;
            issued.store(i + 1);
            if (!pool.empty()) continue;
            if (!check(hipEventSynchronize(ev[k]))) break;
            work(mem + k * CHUNK, i * CHUNK, len(i));
        }
        for (std::thread &t : pool) t.join();
        return (hipError_t)err.load();
    }
};

} // namespace pfdd
