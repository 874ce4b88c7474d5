// Host harness of HostStaging (mf-lbm-cuda_amd/csrc/copy_out.h) for tests/test_copy_out_host.py:
// the HIP calls that it makes are defined here, on host memory, so that a CPU runs it.  Built with
// g++; argv[1] names the check, the exit status says whether it held.
#include <atomic>
#include <chrono>
#include <csignal>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <set>
#include <string>
#include <unistd.h>
#include <vector>

#include "copy_out.h"

namespace {
std::mutex book;
std::set<std::thread::id> callers;  // threads that made a HIP call
int made = 0;                       // hipHostMalloc calls
int queued = 0, direct = 0;         // hipMemcpyAsync and hipMemcpy calls
hipMemoryType kind = hipMemoryTypeUnregistered;  // of every destination
hipError_t known = hipSuccess;
int fail_at = 0;  // this queued copy fails
void called() {
    std::lock_guard<std::mutex> lock(book);
    callers.insert(std::this_thread::get_id());
}
}  // namespace

extern "C" {
hipError_t hipHostMalloc(void** p, size_t bytes, unsigned) { called(); ++made; *p = std::malloc(bytes); return hipSuccess; }
hipError_t hipHostFree(void* p) { called(); std::free(p); return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { called(); *e = reinterpret_cast<hipEvent_t>(std::malloc(1)); return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t e) { called(); std::free(reinterpret_cast<void*>(e)); return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { called(); return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { called(); return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { called(); return hipSuccess; }
hipError_t hipGetLastError() { called(); return hipSuccess; }
hipError_t hipGetDevice(int* d) { called(); *d = 0; return hipSuccess; }
hipError_t hipSetDevice(int) { called(); return hipSuccess; }
hipError_t hipPointerGetAttributes(hipPointerAttribute_t* a, const void*) { called(); a->type = kind; return known; }
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) { called(); ++direct; std::memcpy(d, s, n); return hipSuccess; }
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) {
    called();
    if (++queued == fail_at) return hipErrorUnknown;
    std::memcpy(d, s, n);
    return hipSuccess;
}
}

namespace {
using mflbm::HostStaging;

std::vector<unsigned char> pattern(size_t n) {
    std::vector<uint32_t> words(n / 4 + 1);
    for (size_t i = 0; i < words.size(); ++i) words[i] = (uint32_t)(i + n) * 2654435761u;
    std::vector<unsigned char> v(n);
    std::memcpy(v.data(), words.data(), n);
    return v;
}

bool copies(HostStaging& h, size_t n) {
    const auto src = pattern(n);
    std::vector<unsigned char> dst(n + 64, 7);
    if (h.copy(dst.data(), src.data(), n, nullptr) != hipSuccess) return false;
    if (std::memcmp(dst.data(), src.data(), n) != 0) return false;
    for (size_t i = n; i < dst.size(); ++i)
        if (dst[i] != 7) return false;
    return true;
}

// sizes around the least staged one, in whole and broken chunks, on one set of slots
int contents() {
    HostStaging h;
    if (!copies(h, 25 * HostStaging::SLOT)) return 1;  // makes the slots
    for (size_t n : {(size_t)1, HostStaging::MIN_BYTES - 1, HostStaging::MIN_BYTES, HostStaging::MIN_BYTES + 1,
                     4 * HostStaging::SLOT, 4 * HostStaging::SLOT + 1, 9 * HostStaging::SLOT + 4097, 25 * HostStaging::SLOT - 1})
        if (!copies(h, n)) {
            std::printf("%zu bytes differ\n", n);
            return 1;
        }
    h.release();
    return 0;
}

// an entry point that holds the library's lock copies while another thread makes its first copy
int order() {
    HostStaging h;
    bool ok = false;
    std::thread other;
    {
        std::lock_guard<std::recursive_mutex> lock(mflbm::device_lock());
        other = std::thread([&] { ok = copies(h, 25 * HostStaging::SLOT); });
        std::this_thread::sleep_for(std::chrono::milliseconds(300));  // the other is where it waits
        if (!copies(h, 25 * HostStaging::SLOT + 5)) return 1;
    }
    other.join();
    h.release();
    return ok ? 0 : 1;
}

// the threads that copy out of the slots leave the HIP calls to the calling thread
int calls() {
    HostStaging h;
    callers.clear();
    if (!copies(h, 25 * HostStaging::SLOT - 1) || !copies(h, 3 * HostStaging::MIN_BYTES)) return 1;
    h.release();
    std::printf("%zu threads made HIP calls\n", callers.size());
    return callers.size() == 1 && callers.count(std::this_thread::get_id()) ? 0 : 1;
}

// destinations that the runtime copies to directly are left to it
int destinations() {
    HostStaging h;
    for (hipMemoryType k : {hipMemoryTypeHost, hipMemoryTypeManaged, hipMemoryTypeDevice}) {
        kind = k;
        direct = queued = 0;
        if (!copies(h, 25 * HostStaging::SLOT) || direct != 1 || queued) return 1;
    }
    kind = hipMemoryTypeUnregistered;
    for (hipError_t e : {hipSuccess, hipErrorInvalidValue}) {
        known = e;
        direct = queued = 0;
        if (!copies(h, 25 * HostStaging::SLOT) || direct || !queued) return 1;
    }
    h.release();
    return 0;
}

// the slots are made by the copy that is worth them: a first large one, or a later small one
int worth() {
    const size_t small = HostStaging::MIN_BYTES + 3000000, large = 36 * HostStaging::SLOT;
    HostStaging one, many;
    made = 0;
    if (!copies(one, large) || made != 1 || !copies(one, small) || !copies(one, large) || made != 1) return 1;
    made = 0;
    if (!copies(many, small) || made != 0) return 1;
    int n = 1;
    while (made == 0 && n < 100) {
        if (!copies(many, small)) return 1;
        ++n;
    }
    if (made != 1 || (size_t)n * small < (40 << 20) || (size_t)n * small > (60 << 20)) return 1;
    one.release();
    many.release();
    return 0;
}

// a copy that fails at any chunk ends, says so, and leaves the slots fit for the next
int errors() {
    HostStaging h;
    const size_t n = 20 * HostStaging::SLOT + 77;
    if (!copies(h, n)) return 1;
    const auto src = pattern(n);
    std::vector<unsigned char> dst(n);
    for (int k = 1; k <= 21; ++k) {
        queued = 0;
        fail_at = k;
        if (h.copy(dst.data(), src.data(), n, nullptr) != hipErrorUnknown) return 1;
        fail_at = 0;
        if (!copies(h, n)) return 1;
    }
    h.release();
    return 0;
}

// a copy does not wait for a thread that holds the library's lock (a handle that is being created)
int waits() {
    HostStaging h;
    std::atomic<bool> done{false}, ok{false};
    std::thread other;
    bool early = false;
    {
        std::lock_guard<std::recursive_mutex> lock(mflbm::device_lock());
        other = std::thread([&] {
            ok = copies(h, 25 * HostStaging::SLOT);
            done = true;
        });
        for (int t = 0; t < 100 && !early; ++t) {
            std::this_thread::sleep_for(std::chrono::milliseconds(100));
            early = done;
        }
    }
    other.join();
    h.release();
    return early && ok ? 0 : 1;
}

// several threads, each on its own handle's slots or sharing one's
int threads() {
    HostStaging one, two;
    std::atomic<int> good{0};
    std::vector<std::thread> t;
    for (int k = 0; k < 4; ++k)
        t.emplace_back([&, k] {
            for (int r = 0; r < 3; ++r) good += copies(k < 3 ? one : two, (13 + k) * HostStaging::SLOT + r);
        });
    for (auto& x : t) x.join();
    one.release();
    two.release();
    return good == 12 ? 0 : 1;
}
}  // namespace

int main(int argc, char** argv) {
    if (argc != 2) return 2;
    std::signal(SIGALRM, [](int) { _exit(3); });  // a deadlock
    alarm(20);
    const std::string what = argv[1];
    if (what == "contents") return contents();
    if (what == "order") return order();
    if (what == "calls") return calls();
    if (what == "errors") return errors();
    if (what == "waits") return waits();
    if (what == "threads") return threads();
    if (what == "worth") return worth();
    if (what == "destinations") return destinations();
    return 2;
}
