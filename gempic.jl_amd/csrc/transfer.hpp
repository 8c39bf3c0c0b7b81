// transfer.hpp -- large copies from GPU memory to a caller's (pageable) array.
//
// The runtime's own copy to pageable memory is one thread that copies out of
// its staging buffers: 17.7 GB/s measured on 1 GiB, against 57 GB/s to pinned
// memory. Here a few threads each copy chunks to their own two pinned buffers
// on their own stream and from there to the caller's array, the next chunk
// under way while the last one is moved on. A splitting's particles (and
// fields) back to the caller, before and after: 1,048,576 particles (32 MiB)
// 2.10 ms, 0.99 ms; 4,194,304 8.1 ms, 3.0 ms (44 GB/s); 12,582,912 23.8 ms,
// 8.6 ms (47 GB/s). Six threads, or chunks of 1 or 4 MiB, measured the same
// within 10 %, eight and twelve less at times.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cstddef>
#include <cstring>
#include <mutex>
#include <new>
#include <system_error>
#include <thread>
#include <vector>

namespace gl {

// One pool for the process: kThreads x 2 buffers of kChunk bytes, made by the
// first large copy and given back with the last handle (acquire/release
// count them). A copy whose stream is done holds the pool's lock, so copies of
// several threads follow one another, as they would on the link; work that is
// still to come, and making or giving up a handle beside others, wait for no copy.
class TransferPool {
public:
    static constexpr size_t kChunk = (size_t)2 << 20;
    static constexpr int kThreads = 4;
    // below this the threads' start outweighs what they save (4 MiB: 0.39 ms and
    // 0.35 ms)
    static constexpr size_t kLeast = (size_t)4 << 20;

    static TransferPool &get()
    {
        static TransferPool *p = new TransferPool();   // never destroyed: handles may outlive static order
        return *p;
    }

    void acquire() { ++users_; }
    void release()
    {
        if (--users_ > 0) return;
        std::lock_guard<std::mutex> g(m_);
        if (users_ == 0) free_all();           // (no other came meanwhile)
    }

    // dst <- src (device memory of `device`, ready once `after` is done);
    // returns when dst is written; the calling thread's device stays as it is
    hipError_t to_host(void *dst, const void *src, size_t bytes, hipStream_t after, int device)
    {
        if (bytes < kLeast) {
            const hipError_t e = hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, after);
            return e != hipSuccess ? e : hipStreamSynchronize(after);
        }
        hipError_t e = hipStreamSynchronize(after);
        if (e != hipSuccess) return e;
        std::lock_guard<std::mutex> g(m_);
        OnDevice here(device);
        if (!make(device)) return hipMemcpy(dst, src, bytes, hipMemcpyDeviceToHost);
        const size_t chunks = (bytes + kChunk - 1) / kChunk;
        std::atomic<size_t> next{0};
        std::atomic<int> err{(int)hipSuccess};
        auto work = [&](int t) {
            Lane &L = lanes_[t];
            hipError_t r = hipSetDevice(device);
            size_t have[2] = {0, 0};               // chunk + 1 under way in each buffer
            auto start = [&](int b) {
                const size_t c = next.fetch_add(1);
                have[b] = 0;
                if (c >= chunks || r != hipSuccess) return;
                const size_t off = c * kChunk, len = std::min(kChunk, bytes - off);
                r = hipMemcpyAsync(L.buf[b], (const char *)src + off, len, hipMemcpyDeviceToHost, L.stream);
                if (r == hipSuccess) r = hipEventRecord(L.done[b], L.stream);
                if (r == hipSuccess) have[b] = c + 1;
            };
            start(0);
            for (int b = 0; have[b]; b ^= 1) {
                start(b ^ 1);
                const hipError_t w = hipEventSynchronize(L.done[b]);
                if (w != hipSuccess) {
                    r = w;
                    break;
                }
                const size_t off = (have[b] - 1) * kChunk;
                std::memcpy((char *)dst + off, L.buf[b], std::min(kChunk, bytes - off));
            }
            if (r != hipSuccess) err.store((int)r);
            (void)hipStreamSynchronize(L.stream);
        };
        std::vector<std::thread> th;
        try {
            th.reserve(kThreads - 1);
            for (int t = 1; t < kThreads; ++t) th.emplace_back(work, t);
        } catch (const std::system_error &) {      // fewer threads: the others take their chunks
        } catch (const std::bad_alloc &) {
        }
        work(0);
        for (auto &t : th) t.join();
        return (hipError_t)err.load();
    }

private:
    struct OnDevice {
        int was = -1, now;
        explicit OnDevice(int d) : now(d)
        {
            if (hipGetDevice(&was) != hipSuccess) was = d;
            if (was != d) (void)hipSetDevice(d);
        }
        ~OnDevice()
        {
            if (was != now) (void)hipSetDevice(was);
        }
    };

    struct Lane {
        hipStream_t stream = nullptr;
        hipEvent_t done[2] = {nullptr, nullptr};
        void *buf[2] = {nullptr, nullptr};
    };

    bool make(int device)
    {
        if (made_ && device_ == device) return true;
        free_all();
        device_ = device;
        made_ = true;
        bool ok = true;
        for (Lane &L : lanes_) {
            ok = ok && hipStreamCreate(&L.stream) == hipSuccess;
            for (int b = 0; b < 2; ++b) {
                ok = ok && hipEventCreateWithFlags(&L.done[b], hipEventDisableTiming) == hipSuccess;
                ok = ok && hipHostMalloc(&L.buf[b], kChunk, hipHostMallocDefault) == hipSuccess;
            }
        }
        if (!ok) {
            (void)hipGetLastError();
            free_all();
        }
        return ok;
    }

    void free_all()
    {
        for (Lane &L : lanes_) {
            if (L.stream) (void)hipStreamDestroy(L.stream);
            for (int b = 0; b < 2; ++b) {
                if (L.done[b]) (void)hipEventDestroy(L.done[b]);
                if (L.buf[b]) (void)hipHostFree(L.buf[b]);
            }
            L = Lane{};
        }
        made_ = false;
    }

    std::mutex m_;
    std::atomic<int> users_{0};
    int device_ = -1;
    bool made_ = false;
    Lane lanes_[kThreads];
};

}  // namespace gl
