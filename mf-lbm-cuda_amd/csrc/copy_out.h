// Copies of large device arrays to ordinary host memory.
//
// hipMemcpy to pageable memory moves the data through the runtime's own staging buffer with one
// thread, which also takes the first-touch faults of a fresh destination: 18.5 ms for 200 MB
// (11 GB/s; 11.4 ms into touched memory), where the link carries 56 GB/s into pinned memory.
// Here the calling thread queues chunks into a ring of pinned slots and waits for them in turn, and
// WORKERS threads copy the slots that have arrived to the destination while the link fills the next
// ones.  Every HIP call is the calling thread's: concurrent HIP calls from many host threads have
// stalled this library's work on the GPU before, and the copies need the threads for memory alone.
// A phi read into a fresh array, hipMemcpy and this: 147 MB 14.0 and 3.9 ms, 20 MB 1.2 and 0.58, 9 MB
// 0.53 and 0.30 (with the HIP calls in each thread 4.5, 0.58 and 0.33).  Into touched memory 201 MB
// take 4.4 ms with 6 or 8 slots of 4 MB, 5.0 with 8 of 2 MB and 6.3 with 12 of 1 MB; 4 slots of 4 MB
// make fresh memory 5 % slower.
#pragma once
#include <hip/hip_runtime.h>
#include <condition_variable>
#include <cstring>
#include <mutex>
#include <thread>

#include "device_lock.h"

namespace mflbm {

// Pinned slots of one handle: made once its large copies are worth them, given back with it.  One
// large copy at a time, of all handles (large_copies).  A copy never waits for the library's lock,
// which its caller may hold and another thread's handle may be created under: where the slots are to
// be made and another thread holds it, the copy is hipMemcpy's.
class HostStaging {
public:
    static constexpr size_t WORKERS = 4, SLOTS = 6;
    static constexpr size_t SLOT = 4 << 20;
    // below this hipMemcpy is as fast
    static constexpr size_t MIN_BYTES = 6 << 20;
    // The slots take 1.6 ms to make, which the copies of fewer bytes than this do not win back (a
    // handle's first read, hipMemcpy and staged with the slots' making: 9 MB 0.9 and 2.2 ms, 20 MB
    // 2.1 and 2.9, 147 MB 15 and 7.4; later reads 0.53 and 0.30, 1.2 and 0.58, 14 and 3.9): until a
    // handle's large copies come to it they are hipMemcpy's.
    static constexpr size_t WORTH_BYTES = 48 << 20;

    // dst[0, bytes) = src[0, bytes), after the work queued on `stream`; returns when it is there
    hipError_t copy(void* dst, const void* src, size_t bytes, hipStream_t stream) {
        std::unique_lock<std::mutex> lock;
        if (bytes >= MIN_BYTES && pageable(dst)) {
            lock = std::unique_lock<std::mutex>(large_copies());
            copied_ = copied_ < WORTH_BYTES ? copied_ + bytes : copied_;
            if (copied_ >= WORTH_BYTES && make()) return staged(static_cast<char*>(dst), static_cast<const char*>(src), bytes, stream);
        }
        const hipError_t r = hipStreamSynchronize(stream);
        return r == hipSuccess ? hipMemcpy(dst, src, bytes, hipMemcpyDeviceToHost) : r;
    }

    void release() {  // under device_lock, with no copy running
        for (size_t w = 0; w < SLOTS; ++w) {
            if (done_[w]) (void)hipEventDestroy(done_[w]);
            done_[w] = nullptr;
        }
        if (ring_) (void)hipHostFree(ring_);
        ring_ = nullptr;
    }

private:
    // Memory that the runtime knows (pinned, managed, a device's) it copies to directly, at the link's
    // rate: 201 MB into pinned memory 3.5 ms, through the slots 25.
    static bool pageable(const void* dst) {
        hipPointerAttribute_t a;
        if (hipPointerGetAttributes(&a, dst) == hipSuccess) return a.type == hipMemoryTypeUnregistered;
        (void)hipGetLastError();  // what runtimes that do not know ordinary memory return for it
        return true;
    }

    static std::mutex& large_copies() {
        static std::mutex m;
        return m;
    }

    bool make() {  // under large_copies
        if (ring_) return true;
        std::unique_lock<std::recursive_mutex> lock(device_lock(), std::try_to_lock);
        if (!lock) return false;
        void* p = nullptr;
        bool ok = hipHostMalloc(&p, SLOTS * SLOT, hipHostMallocDefault) == hipSuccess;
        ring_ = ok ? static_cast<char*>(p) : nullptr;
        for (size_t w = 0; ok && w < SLOTS; ++w) ok = hipEventCreateWithFlags(&done_[w], hipEventDisableTiming) == hipSuccess;
        if (!ok) {
            release();
            (void)hipGetLastError();
        }
        return ok;
    }

    hipError_t staged(char* dst, const char* src, size_t bytes, hipStream_t stream) {
        // a slot at a time, or a share of the whole to each thread
        const size_t share = (bytes / WORKERS + 4096) & ~(size_t)4095, chunk = share < SLOT ? share : SLOT;
        const size_t chunks = (bytes + chunk - 1) / chunk;
        auto slot = [&](size_t c) { return ring_ + c % SLOTS * SLOT; };
        auto length = [&](size_t c) { return bytes - c * chunk < chunk ? bytes - c * chunk : chunk; };
        std::mutex m;
        std::condition_variable ready, freed;
        size_t issued = 0, arrived = 0, taken = 0;  // chunks queued; in their slots; given to a thread
        bool full[SLOTS] = {}, stop = false;        // slots in use
        // copies chunks out of their slots as they arrive, until all are given out
        auto drain = [&] {
            std::unique_lock<std::mutex> lock(m);
            for (;;) {
                ready.wait(lock, [&] { return taken < arrived || taken == chunks || stop; });
                if (taken == arrived) return;
                const size_t c = taken++;
                if (taken == chunks) ready.notify_all();
                lock.unlock();
                std::memcpy(dst + c * chunk, slot(c), length(c));
                lock.lock();
                full[c % SLOTS] = false;
                freed.notify_one();
            }
        };
        auto issue = [&] {
            hipError_t r = hipMemcpyAsync(slot(issued), src + issued * chunk, length(issued), hipMemcpyDeviceToHost, stream);
            if (r == hipSuccess) r = hipEventRecord(done_[issued % SLOTS], stream);
            full[issued++ % SLOTS] = true;
            return r;
        };
        hipError_t r = hipSuccess;
        while (issued < chunks && issued < SLOTS && r == hipSuccess) r = issue();
        // this thread makes the HIP calls and, once all chunks are there, copies with the others
        std::thread other[WORKERS];
        size_t threads = 0;
        try {
            while (threads < WORKERS && threads + 1 < chunks) {
                other[threads] = std::thread(drain);
                ++threads;
            }
        } catch (...) {  // the threads there are take all chunks
        }
        for (size_t c = 0; c < chunks && r == hipSuccess; ++c) {
            r = hipEventSynchronize(done_[c % SLOTS]);
            if (r != hipSuccess) break;
            std::unique_lock<std::mutex> lock(m);
            arrived = c + 1;
            if (threads == 0) {
                std::memcpy(dst + c * chunk, slot(c), length(c));
                full[taken++ % SLOTS] = false;
            }
            ready.notify_one();
            // refill the slots that are free; wait for one only where nothing else is on its way
            while (issued < chunks && r == hipSuccess) {
                if (full[issued % SLOTS]) {
                    if (issued > c + 1) break;
                    freed.wait(lock, [&] { return !full[issued % SLOTS]; });
                }
                r = issue();
            }
        }
        if (r != hipSuccess) {
            std::lock_guard<std::mutex> lock(m);
            stop = true;
            ready.notify_all();
        }
        drain();
        for (size_t t = 0; t < threads; ++t) other[t].join();
        if (r != hipSuccess) (void)hipStreamSynchronize(stream);  // no copy into the slots goes on
        return r;
    }

    size_t copied_ = 0;  // by large copies, up to WORTH_BYTES
    char* ring_ = nullptr;
    hipEvent_t done_[SLOTS] = {};  // a slot's chunk is there
};

}  // namespace mflbm
