// Copies of large device arrays to ordinary host memory.
//
// hipMemcpy to pageable memory moves the data through the runtime's own staging buffer with one
// thread, which also takes the first-touch faults of a fresh destination: 18.5 ms for 200 MB
// (11 GB/s; 11.4 ms into touched memory), where the link carries 56 GB/s into pinned memory.
// Here WORKERS threads each hold a pinned slot and take the next chunk in turn: while one copies
// its slot to the destination, the link fills another's: 6.1 ms for the 201 MB of 48 domains of
// 64^3 (before: 18.6), 4.0 for 147 MB (15.3), 0.33 for 9 MB (0.56).  Slots of 2 and 1 MB took 6.6
// and 7.7 ms; 8 threads with 2 MB 5.9.
#pragma once
#include <hip/hip_runtime.h>
#include <atomic>
#include <cstring>
#include <mutex>
#include <system_error>
#include <thread>

#include "device_lock.h"

namespace mflbm {

// Pinned slots of one handle: made by its first large copy, given back with it.  One copy at a
// time, of all handles: it holds the library's lock, which callers may hold already and which the
// slots' allocation needs (a mutex of the slots' own, taken by a copy before that lock and by a
// caller that held it after, could deadlock two threads).
class HostStaging {
public:
    static constexpr int WORKERS = 4;
    static constexpr size_t SLOT = 4 << 20;
    // below this hipMemcpy is as fast
    static constexpr size_t MIN_BYTES = 6 << 20;

    // dst[0, bytes) = src[0, bytes), after the work queued on `stream`; returns when it is there
    hipError_t copy(void* dst, const void* src, size_t bytes, hipStream_t stream) {
        if (bytes >= MIN_BYTES) {
            std::lock_guard<std::recursive_mutex> lock(device_lock());
            int dev = 0;
            if (make() && hipGetDevice(&dev) == hipSuccess) return staged(static_cast<char*>(dst), static_cast<const char*>(src), bytes, stream, dev);
        }
        const hipError_t r = hipStreamSynchronize(stream);
        return r == hipSuccess ? hipMemcpy(dst, src, bytes, hipMemcpyDeviceToHost) : r;
    }

    void release() {  // under device_lock, with no copy running
        for (int w = 0; w < WORKERS; ++w) {
            if (done_[w]) (void)hipEventDestroy(done_[w]);
            done_[w] = nullptr;
        }
        if (ring_) (void)hipHostFree(ring_);
        ring_ = nullptr;
    }

private:
    bool make() {  // under device_lock
        if (ring_) return true;
        void* p = nullptr;
        bool ok = hipHostMalloc(&p, WORKERS * SLOT, hipHostMallocDefault) == hipSuccess;
        ring_ = ok ? static_cast<char*>(p) : nullptr;
        for (int w = 0; ok && w < WORKERS; ++w) ok = hipEventCreateWithFlags(&done_[w], hipEventDisableTiming) == hipSuccess;
        if (!ok) {
            release();
            (void)hipGetLastError();
        }
        return ok;
    }

    hipError_t staged(char* dst, const char* src, size_t bytes, hipStream_t stream, int dev) {
        // a slot at a time, or a share of the whole to each thread
        const size_t share = (bytes / WORKERS + 4096) & ~(size_t)4095, chunk = share < SLOT ? share : SLOT;
        const size_t chunks = (bytes + chunk - 1) / chunk;
        std::atomic<size_t> next{0};
        std::atomic<int> error{hipSuccess};
        auto work = [&](int w) {
            char* slot = ring_ + w * SLOT;
            hipError_t r = hipSuccess;
            while (r == hipSuccess && error.load() == hipSuccess) {
                const size_t c = next++;
                if (c >= chunks) return;
                const size_t at = c * chunk, len = bytes - at < chunk ? bytes - at : chunk;
                r = hipMemcpyAsync(slot, src + at, len, hipMemcpyDeviceToHost, stream);
                if (r == hipSuccess) r = hipEventRecord(done_[w], stream);
                if (r == hipSuccess) r = hipEventSynchronize(done_[w]);
                if (r == hipSuccess) std::memcpy(dst + at, slot, len);
            }
            if (r != hipSuccess) error = r;
        };
        std::thread other[WORKERS];
        for (int w = 1; w < WORKERS && (size_t)w < chunks; ++w) {
            try {
                other[w] = std::thread([&work, w, dev, &error] {
                    const hipError_t r = hipSetDevice(dev);
                    if (r == hipSuccess) work(w);
                    else error = r;
                });
            } catch (const std::system_error&) {
                break;  // the threads there are take all chunks
            }
        }
        work(0);
        for (std::thread& t : other)
            if (t.joinable()) t.join();
        return static_cast<hipError_t>(error.load());
    }

    char* ring_ = nullptr;
    hipEvent_t done_[WORKERS] = {};
};

}  // namespace mflbm
