"""The pool that copies large GPU arrays to the caller (csrc/transfer.hpp), built
for the CPU against a stand-in for the HIP calls it makes: who waits for whom,
which device is current, what is copied and what is given back."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

# Streams are numbers; the busy one's synchronize waits until let go. The device
# is a thread's own, as in HIP, and starts as 0.
HIP = r"""
#pragma once
#include <atomic>
#include <condition_variable>
#include <cstdlib>
#include <cstring>
#include <mutex>
typedef int hipError_t;
enum { hipSuccess = 0, hipErrorInvalidValue = 1 };
enum { hipMemcpyDeviceToHost, hipEventDisableTiming, hipHostMallocDefault };
struct FakeStream { int device; bool busy; };
struct FakeEvent { int device; };
typedef FakeStream *hipStream_t;
typedef FakeEvent *hipEvent_t;
inline thread_local int device_now = 0;
inline std::mutex mu;
inline std::condition_variable cv;
inline bool let_go = false, waiting = false;
inline std::atomic<int> live{0}, wrong_device{0};
inline hipError_t hipGetDevice(int *d) { *d = device_now; return hipSuccess; }
inline hipError_t hipSetDevice(int d) { device_now = d; return hipSuccess; }
inline hipError_t hipGetLastError() { return hipSuccess; }
inline hipError_t hipStreamCreate(hipStream_t *s) { *s = new FakeStream{device_now, false}; ++live; return hipSuccess; }
inline hipError_t hipStreamDestroy(hipStream_t s) { delete s; --live; return hipSuccess; }
inline hipError_t hipStreamSynchronize(hipStream_t s)
{
    std::unique_lock<std::mutex> l(mu);
    if (s && s->busy) {
        waiting = true;
        cv.notify_all();
        cv.wait(l, [] { return let_go; });
    }
    return hipSuccess;
}
inline hipError_t hipEventCreateWithFlags(hipEvent_t *e, int) { *e = new FakeEvent{device_now}; ++live; return hipSuccess; }
inline hipError_t hipEventDestroy(hipEvent_t e) { delete e; --live; return hipSuccess; }
inline hipError_t hipEventRecord(hipEvent_t e, hipStream_t s)
{
    if (e->device != s->device || device_now != s->device) ++wrong_device;
    return hipSuccess;
}
inline hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
inline hipError_t hipHostMalloc(void **p, size_t n, int) { *p = std::malloc(n); ++live; return hipSuccess; }
inline hipError_t hipHostFree(void *p) { std::free(p); --live; return hipSuccess; }
inline hipError_t hipMemcpy(void *d, const void *s, size_t n, int) { std::memcpy(d, s, n); return hipSuccess; }
inline hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, int, hipStream_t st)
{
    if (st && st->device != device_now) ++wrong_device;
    std::memcpy(d, s, n);
    return hipSuccess;
}
"""

MAIN = r"""
#include "transfer.hpp"
#include <cstdio>
#include <future>
#include <vector>
using namespace gl;
#define CHECK(c) do { if (!(c)) { std::printf("line %d: %s\n", __LINE__, #c); std::fflush(stdout); std::_Exit(1); } } while (0)
template <class F> bool ends(F f)
{
    auto r = std::make_shared<std::promise<void>>();
    auto got = r->get_future();
    std::thread([=] { f(); r->set_value(); }).detach();
    return got.wait_for(std::chrono::seconds(20)) == std::future_status::ready;
}
int main()
{
    TransferPool &p = TransferPool::get();
    const size_t k = TransferPool::kChunk;
    p.acquire();
    for (size_t n : {(size_t)1, TransferPool::kLeast - 1, TransferPool::kLeast, 5 * k + 3, 9 * k, 16 * k - 1}) {
        std::vector<unsigned char> a(n), b(n, 0);
        for (size_t i = 0; i < n; ++i) a[i] = (unsigned char)(i * 2654435761u >> 13);
        FakeStream s{0, false};
        CHECK(p.to_host(b.data(), a.data(), n, &s, 0) == hipSuccess);
        CHECK(a == b);
    }
    // of another device than the calling thread's: its streams, and the thread's device stays
    {
        std::vector<unsigned char> a(3 * k, 7), b(3 * k);
        FakeStream s{1, false};
        CHECK(p.to_host(b.data(), a.data(), a.size(), &s, 1) == hipSuccess);
        CHECK(a == b && device_now == 0 && wrong_device == 0);
    }
    // while one thread waits for a stream that is not done: others make and give
    // up users, and copy
    std::vector<unsigned char> a(4 * k, 5), b(4 * k), c(4 * k);
    FakeStream busy{0, true}, idle{0, false};
    std::thread t([&] { p.to_host(b.data(), a.data(), a.size(), &busy, 0); });
    {
        std::unique_lock<std::mutex> l(mu);
        cv.wait(l, [] { return waiting; });
    }
    CHECK(ends([&] { p.acquire(); }));
    CHECK(ends([&] { p.to_host(c.data(), a.data(), a.size(), &idle, 0); }));
    CHECK(ends([&] { p.release(); }));
    CHECK(c == a && b != a);
    {
        std::lock_guard<std::mutex> l(mu);
        let_go = true;
    }
    cv.notify_all();
    t.join();
    CHECK(b == a && live > 0);
    p.release();
    CHECK(live == 0);
    std::printf("ok\n");
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="no host compiler")
def test_transfer_pool_waits_and_devices(tmp_path):
    (tmp_path / "hip").mkdir()
    (tmp_path / "hip" / "hip_runtime.h").write_text(HIP)
    (tmp_path / "main.cpp").write_text(MAIN)
    exe = tmp_path / "pool"
    subprocess.run(["g++", "-std=c++17", "-O1", "-pthread", f"-I{tmp_path}",
                    "-I" + os.path.join(ROOT, "gempic.jl_amd", "csrc"), "-o", str(exe), str(tmp_path / "main.cpp")],
                   check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stdout + r.stderr
