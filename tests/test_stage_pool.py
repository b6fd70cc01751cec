"""The pool of pinned memory behind downloads, on the CPU.

pfdd_stage.hpp is compiled against a stand-in for the HIP runtime that copies
at once, counts pinned allocations and events, and fails on demand.  Moves of
many threads at once arrive whole, at most two idle rings stay, everything is
freed with the last handle, a move without pinned memory and one after a
failed move still arrive, and blocks are distinct.
"""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "phase-field-dislocation-dynamics-pfdd-2.x_amd", "csrc")

RUNTIME = r"""
#pragma once
#include <atomic>
#include <cstdlib>
#include <cstring>
typedef int hipError_t;
typedef void *hipStream_t;
typedef void *hipEvent_t;
enum { hipSuccess = 0, hipErrorOutOfMemory = 2, hipErrorUnknown = 999 };
enum { hipEventDisableTiming = 2, hipHostMallocPortable = 1, hipHostMallocMapped = 2, hipMemcpyDeviceToHost = 2 };
inline std::atomic<int> pinned{0}, events{0}, no_pinned{0}, fail_copy{-1};
inline hipError_t hipHostMalloc(void **p, size_t n, unsigned)
{
    if (no_pinned) return hipErrorOutOfMemory;
    ++pinned;
    *p = malloc(n);
    return hipSuccess;
}
inline hipError_t hipHostFree(void *p) { --pinned; free(p); return hipSuccess; }
inline hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { ++events; *e = malloc(1); return hipSuccess; }
inline hipError_t hipEventDestroy(hipEvent_t e) { --events; free(e); return hipSuccess; }
inline hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
inline hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
inline hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
inline hipError_t hipGetLastError() { return hipSuccess; }
inline thread_local int current = 0;
inline hipError_t hipGetDevice(int *d) { *d = current; return hipSuccess; }
inline hipError_t hipSetDevice(int d) { current = d; return hipSuccess; }
inline hipError_t hipMemcpyAsync(void *to, const void *from, size_t n, int, hipStream_t)
{
    if (fail_copy >= 0 && fail_copy-- == 0) return hipErrorUnknown;
    memcpy(to, from, n);
    return hipSuccess;
}
"""

PROGRAM = r"""
#include "pfdd_stage.hpp"
#include <cstdio>
#include <set>
using namespace pfdd;
static int bad = 0;
#define CHECK(x) do { if (!(x)) { std::printf("failed at line %d: %s\n", __LINE__, #x); ++bad; } } while (0)

static bool move(const std::vector<char> &from, size_t n, hipError_t *e = nullptr)
{
    std::vector<char> to(n + 1, 1);
    const hipError_t r = stage_out(from.data(), n, nullptr,
                                   [&](char *c, size_t o, size_t len) { std::memcpy(to.data() + o, c, len); });
    if (e) *e = r;
    return r == hipSuccess && std::memcmp(to.data(), from.data(), n) == 0 && to[n] == 1;
}

int main()
{
    const size_t C = Ring::CHUNK;
    std::vector<char> from(11 * C + 77);
    for (size_t i = 0; i < from.size(); ++i) from[i] = (char)(i * 2654435761u >> 13);
    {
        PinnedUser a;
        for (size_t n : {(size_t)1, C - 1, C, C + 1, 8 * C, 8 * C + 1, from.size()}) CHECK(move(from, n));
        CHECK(pinned == 1 && events == Ring::K); // one ring did it all
        PinnedUser b;
        std::atomic<int> wrong{0};
        std::vector<std::thread> t;
        for (int q = 0; q < 6; ++q)
            t.emplace_back([&, q] {
                current = q % 2;
                PinnedUser u;
                for (int i = 0; i < 6; ++i)
                    if (!move(from, (size_t)(1 + (q * 6 + i) % 11) * C + i)) ++wrong;
            });
        for (auto &x : t) x.join();
        CHECK(wrong == 0);
        CHECK(pinned <= 2 && events <= 2 * Ring::K);
        std::set<void *> blocks;
        for (int i = 0; i < 200; ++i) blocks.insert(Pinned::get().block());
        CHECK(blocks.size() == 200 && !blocks.count(nullptr));
        char *last = nullptr;
        for (void *p : blocks) {
            CHECK(!last || (char *)p - last >= (long)Pinned::BLOCK);
            last = (char *)p;
        }
        for (void *p : blocks) Pinned::get().unblock(p);
        CHECK(blocks.count(Pinned::get().block()));
        hipError_t e;
        for (int at : {0, 3, 9}) { // a copy that fails, then moves as before
            fail_copy = at;
            CHECK(!move(from, from.size(), &e) && e == hipErrorUnknown);
            fail_copy = -1;
            CHECK(move(from, from.size()));
        }
    }
    CHECK(pinned == 0 && events == 0); // with the last handle
    {
        PinnedUser a;
        no_pinned = 1;
        for (size_t n : {(size_t)5, C, 3 * C + 5}) CHECK(move(from, n));
        CHECK(Pinned::get().block() == nullptr);
        no_pinned = 0;
        CHECK(move(from, 3 * C + 5) && pinned == 1);
    }
    CHECK(pinned == 0 && events == 0);
    return bad != 0;
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_pool_of_pinned_memory(tmp_path):
    (tmp_path / "hip").mkdir()
    (tmp_path / "hip" / "hip_runtime.h").write_text(RUNTIME)
    (tmp_path / "main.cpp").write_text(PROGRAM)
    exe = tmp_path / "stage"
    subprocess.run(["g++", "-std=c++17", "-O1", "-pthread", f"-I{tmp_path}", f"-I{CSRC}", "-o", str(exe),
                    str(tmp_path / "main.cpp")], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stdout + r.stderr
