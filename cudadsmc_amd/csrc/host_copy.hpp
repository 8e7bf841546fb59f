// host_copy.hpp -- large copies from device memory to ordinary (pageable) host
// memory.
//
// The runtime copies to pageable memory through its own staging with one
// thread, 17 GB/s where the link does 57: bound by the host's copy.  Here a few
// threads take the range piece by piece, each through a pinned piece of its
// own, so that their host copies and the link overlap: 24 MB 1.40 -> 0.71 ms,
// 96 MB 5.6 -> 2.5 ms (38 GB/s; pieces of 1 MB 31 GB/s, of 4 MB 42 GB/s with
// twice the pinned memory; more than six threads are no faster).  Threads live
// for one copy and the calling thread is one of them.
#pragma once

#include <sched.h>

#include <algorithm>
#include <atomic>
#include <cstring>

#include "dsmc_device.hpp"
#include "dsmc_internal.hpp"
#include "host_threads.hpp"

namespace dsmc {

class HostCopy {
public:
    static constexpr int kThreads = 6;
    static constexpr size_t kPiece = 2u << 20;
    // Smallest copy that goes this way.  Smaller ones gain less (7 MB 0.44 ->
    // 0.29 ms) than a context's first one pays for the pinned pieces (0.8 ms).
    static constexpr size_t kMin = 16u << 20;

    HostCopy() = default;
    HostCopy(const HostCopy &) = delete;
    HostCopy &operator=(const HostCopy &) = delete;
    ~HostCopy()
    {
        for (Slot &s : slot_) {
            if (s.done) (void)hipEventDestroy(s.done);
            if (s.mem) (void)hipHostFree(s.mem);
        }
    }

    // Copies after the work on `st` (a stream of `device`) and returns when
    // the copy is done.
    void to_host(void *host, const void *dev, size_t bytes, int device, hipStream_t st)
    {
        int T = bytes >= kMin ? std::min(cpus(), kThreads) : 0;
        if (T > 1) T = pageable(host) ? ready(T) : 0;
        if (T < 2) {
            // (an asynchronous copy and a wait are 9 us slower up to some 16 KB)
            DSMC_HIP(hipMemcpyWithStream(host, dev, bytes, hipMemcpyDeviceToHost, st));
            return;
        }
        std::atomic<int> error{ (int)hipSuccess };
        std::atomic<size_t> next{ 0 };
        auto work = [&](int k) {
            const Slot &s = slot_[k];
            hipError_t e = k > 0 ? hipSetDevice(device) : hipSuccess;   // (a new thread's)
            while (e == hipSuccess && error.load(std::memory_order_relaxed) == (int)hipSuccess) {
                const size_t at = next.fetch_add(kPiece, std::memory_order_relaxed);
                if (at >= bytes) break;
                const size_t n = std::min(kPiece, bytes - at);
                e = hipMemcpyAsync(s.mem, (const char *)dev + at, n, hipMemcpyDeviceToHost, st);
                if (e == hipSuccess) e = hipEventRecord(s.done, st);
                if (e == hipSuccess) e = hipEventSynchronize(s.done);
                if (e == hipSuccess) std::memcpy((char *)host + at, s.mem, n);
            }
            int none = (int)hipSuccess;
            if (e != hipSuccess) error.compare_exchange_strong(none, (int)e);
        };
        run_threads(T, work);
        DSMC_HIP((hipError_t)error.load());
    }

private:
    struct Slot {
        char *mem = nullptr;   // a pinned piece
        hipEvent_t done = nullptr;
    } slot_[kThreads];

    // Ordinary host memory (pinned memory is copied to directly).
    static bool pageable(const void *p)
    {
        hipPointerAttribute_t a;
        if (hipPointerGetAttributes(&a, p) != hipSuccess) {
            (void)hipGetLastError();
            return true;
        }
        return a.type == hipMemoryTypeUnregistered;
    }

    // Makes the first k slots, as far as there is memory for them; how many.
    int ready(int k)
    {
        for (int i = 0; i < k; ++i) {
            Slot &s = slot_[i];
            if (!s.done && hipEventCreateWithFlags(&s.done, hipEventDisableTiming) != hipSuccess) {
                (void)hipGetLastError();
                s.done = nullptr;
                return i;
            }
            if (!s.mem && hipHostMalloc((void **)&s.mem, kPiece, hipHostMallocDefault) != hipSuccess) {
                (void)hipGetLastError();
                s.mem = nullptr;
                return i;
            }
        }
        return k;
    }

    static int cpus()
    {
        cpu_set_t set;
        return sched_getaffinity(0, sizeof set, &set) == 0 ? CPU_COUNT(&set) : 1;
    }
};

}  // namespace dsmc
