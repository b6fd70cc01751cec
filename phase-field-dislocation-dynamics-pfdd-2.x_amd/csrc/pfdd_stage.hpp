// pfdd_stage.hpp -- fields from device memory to a caller's pageable memory.
//
// A copy to pageable memory is bound by the host: the runtime moves it through
// its own staging with one thread, and a fresh array faults its pages in while
// it is written.  Here the device copies into a ring of pinned slots and several
// threads move (widen, spread) the slots' contents.  33.5 MB to a fresh array:
// 1.9-3.2 -> 1.2 ms; strain and stress fields, 38 MB spread over 75 MB of fresh
// arrays: 5.8 -> 2.8 ms.  Below STAGE_MIN_BYTES the runtime's own copy is taken: 12.6 MB
// is 0.8 ms that way, 0.5 ms through the ring, and 1.4-2 ms where the threads
// have to win CPUs from a caller's own spinning pool.
// The other direction stays with the runtime: it reads a caller's pages at 30
// GB/s.
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cstddef>
#include <memory>
#include <mutex>
#include <new>
#include <thread>
#include <vector>

namespace pfdd {

// Coherent, and usable by every device of the process.
constexpr unsigned PINNED = hipHostMallocPortable | hipHostMallocMapped;

// A ring of pinned slots with their events, used by one move at a time.
struct Ring {
    static constexpr int K = 8;
    static constexpr size_t CHUNK = (size_t)2 << 20;
    char *mem = nullptr; // as many slots, up to K, as the largest move used
    size_t size = 0;
    int device = 0;
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
        const hipError_t r = hipHostMalloc((void **)&mem, bytes, PINNED);
        if (r == hipSuccess) size = bytes;
        else mem = nullptr;
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
};

// Pinned memory of the process's handles: rings, lent to one move at a time, and
// the small blocks that kernels leave a run's scalars in.  Pinning costs the
// host more than the moves it speeds up (a new 16 MiB ring 1.6 ms and its free 1.0
// ms, a block of its own 50 us, against 2 ms that a ring saves on 33.5 MB), so
// neither is paid per handle.  At most KEEP idle rings are kept; rings and
// blocks are freed with the last handle.
class Pinned {
  public:
    static constexpr size_t BLOCK = 128;
    static Pinned &get()
    {
        static Pinned *p = new Pinned; // never destroyed: handles may outlive static objects
        return *p;
    }
    void enter()
    {
        std::lock_guard<std::mutex> lk(mu);
        ++users;
    }
    void leave()
    {
        std::lock_guard<std::mutex> lk(mu);
        if (--users) return;
        for (Ring *r : idle) drop(r);
        idle.clear();
        for (char *s : slabs) (void)hipHostFree(s);
        slabs.clear();
        blocks.clear();
    }
    // A ring of the device with room for a move of `bytes`; nullptr where none
    // can be had.
    Ring *borrow(int device, size_t bytes)
    {
        Ring *r = nullptr;
        {
            std::lock_guard<std::mutex> lk(mu);
            for (size_t i = 0; i < idle.size() && !r; ++i)
                if (idle[i]->device == device) {
                    r = idle[i];
                    idle.erase(idle.begin() + i);
                }
        }
        if (!r) {
            r = new (std::nothrow) Ring;
            if (!r) return nullptr;
            r->device = device;
        }
        if (r->ready(bytes) == hipSuccess) return r;
        (void)hipGetLastError();
        drop(r);
        return nullptr;
    }
    void give_back(Ring *r)
    {
        {
            std::lock_guard<std::mutex> lk(mu);
            if (idle.size() < KEEP) {
                idle.push_back(r); // room is reserved
                return;
            }
        }
        drop(r);
    }
    // BLOCK bytes for a handle's scalars, between its enter and its leave.
    void *block()
    {
        std::lock_guard<std::mutex> lk(mu);
        if (blocks.empty()) {
            char *s = nullptr;
            if (hipHostMalloc((void **)&s, SLAB * BLOCK, PINNED) != hipSuccess) return nullptr;
            slabs.push_back(s);
            for (size_t i = SLAB; i-- > 0;) blocks.push_back(s + i * BLOCK);
        }
        void *b = blocks.back();
        blocks.pop_back();
        return b;
    }
    void unblock(void *b)
    {
        if (!b) return;
        std::lock_guard<std::mutex> lk(mu);
        blocks.push_back((char *)b);
    }

  private:
    static constexpr size_t KEEP = 2, SLAB = 64;
    std::mutex mu;
    int users = 0;
    std::vector<Ring *> idle;
    std::vector<char *> slabs, blocks;
    Pinned() { idle.reserve(KEEP); }
    static void drop(Ring *r)
    {
        r->release();
        delete r;
    }
};

// Member of a handle: it is one of the pool's users.
struct PinnedUser {
    PinnedUser() { Pinned::get().enter(); }
    ~PinnedUser() { Pinned::get().leave(); }
    PinnedUser(const PinnedUser &) = delete;
    PinnedUser &operator=(const PinnedUser &) = delete;
};

constexpr size_t STAGE_MIN_BYTES = (size_t)16 << 20;
constexpr int STAGE_THREADS = 6;

// bytes of device memory to the host: chunk after chunk is handed to
// work(chunk, offset, length), on several threads at once.  Returns after the
// last one.
template <typename Work> hipError_t stage_out(const char *dev, size_t bytes, hipStream_t st, Work work)
{
    constexpr int K = Ring::K;
    constexpr size_t CHUNK = Ring::CHUNK;
    int device = 0;
    (void)hipGetDevice(&device);
    const size_t n = (bytes + CHUNK - 1) / CHUNK;
    auto len = [&](size_t i) { return std::min(CHUNK, bytes - i * CHUNK); };
    Ring *const ring = Pinned::get().borrow(device, bytes);
    if (!ring) {
        // no pinned memory to be had: chunks through the runtime's own staging
        const std::unique_ptr<char[]> buf(new (std::nothrow) char[std::min(bytes, CHUNK)]);
        if (!buf) return hipErrorOutOfMemory;
        for (size_t i = 0; i < n; ++i) {
            hipError_t e = hipMemcpyAsync(buf.get(), dev + i * CHUNK, len(i), hipMemcpyDeviceToHost, st);
            if (e == hipSuccess) e = hipStreamSynchronize(st);
            if (e != hipSuccess) return e;
            work(buf.get(), i * CHUNK, len(i));
        }
        return hipSuccess;
    }
    std::atomic<size_t> next{0}, issued{0};
    std::atomic<size_t> round[K] = {}; // chunks a worker is done with, per slot
    std::atomic<int> err{hipSuccess};
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
            if (!wait([&] { return issued.load() > i; }) || !check(hipEventSynchronize(ring->ev[k]))) return;
            work(ring->mem + k * CHUNK, i * CHUNK, len(i));
            round[k].store(i / K + 1);
        }
    };
    std::vector<std::thread> pool;
    try {
        const size_t cpus = std::max(1u, std::thread::hardware_concurrency());
        const size_t want = std::min({n, (size_t)STAGE_THREADS, cpus});
        pool.reserve(want);
        while (n > 1 && pool.size() < want) pool.emplace_back(worker);
    } catch (...) { // fewer threads than asked for
    }
    for (size_t i = 0; i < n; ++i) {
        const int k = (int)(i % K);
        if (!pool.empty() && !wait([&] { return round[k].load() >= i / K; })) break;
        if (!check(hipMemcpyAsync(ring->mem + k * CHUNK, dev + i * CHUNK, len(i), hipMemcpyDeviceToHost, st)) ||
            !check(hipEventRecord(ring->ev[k], st)))
            break;
        issued.store(i + 1);
        if (!pool.empty()) continue;
        if (!check(hipEventSynchronize(ring->ev[k]))) break;
        work(ring->mem + k * CHUNK, i * CHUNK, len(i));
    }
    for (std::thread &t : pool) t.join();
    // after an error, copies into the ring may still be under way
    if (err.load() != hipSuccess) (void)hipStreamSynchronize(st);
    Pinned::get().give_back(ring);
    return (hipError_t)err.load();
}

} // namespace pfdd
