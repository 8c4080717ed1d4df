// qbx_hostcopy.h -- copies of large pageable host arrays.
#pragma once
#include "qbx_common.h"
#include <hip/hip_runtime.h>

#include <sched.h>

#include <algorithm>
#include <atomic>
#include <cstring>
#include <mutex>
#include <system_error>
#include <thread>
#include <vector>

namespace qbx {

// Copies between pageable host arrays and the device through pinned staging
// chunks that several threads fill or empty while the copies run.  The runtime's
// own copy of a pageable array uses one thread, which also takes the page faults
// of a fresh one.  192 MB: to the device 7.2 -> 4.8 ms, to a touched array 10.9 ->
// 5.0 ms, to a fresh one 55.7 -> 9.0 ms (17 ms with 4 threads, 10.7 with 8; chunks
// of 1 MB 6.2 and 6.3 ms, of 4 MB 4.3 and 4.4, at twice the pinned memory).
// One per context, one copy at a time: two chunks of pinned memory for each of up to
// kThreads threads (48 MB), allocated at the first large copy and freed with the context.

// Threads of a staged copy: the CPUs that the calling thread may use, up to `most`.
inline int copy_threads(int most)
{
    cpu_set_t set;
    if (sched_getaffinity(0, sizeof(set), &set) != 0) return most;   // more CPUs than the set holds
    return std::max(1, std::min(most, CPU_COUNT(&set)));
}

class HostCopier {
public:
    HostCopier() = default;
    HostCopier(const HostCopier&) = delete;
    HostCopier& operator=(const HostCopier&) = delete;
    ~HostCopier() { release(); }

    // dst[0, bytes) = device src after the work queued on st; complete on return
    void to_host(int device, void* dst, const void* src, size_t bytes, hipStream_t st)
    {
        std::lock_guard<std::mutex> lk(mu_);
        if (!staged(dst, bytes, kMinToHost)) {
            QBX_HIP(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, st));
            QBX_HIP(hipStreamSynchronize(st));
            return;
        }
        run(device, bytes, [&](Worker& w, size_t n) {
            // two chunks in flight: one is emptied while the other arrives
            size_t c[2] = {n, n};
            for (int s = 0;; s ^= 1) {
                if (c[s] < n) {
                    if (w.check(hipEventSynchronize(w.ev[s]))) return;
                    const size_t o = c[s] * kChunk;
                    std::memcpy((char*)dst + o, w.p[s], std::min(kChunk, bytes - o));
                }
                c[s] = next_.fetch_add(1);
                if (c[s] < n) {
                    const size_t o = c[s] * kChunk;
                    if (w.check(hipMemcpyAsync(w.p[s], (const char*)src + o, std::min(kChunk, bytes - o),
                                               hipMemcpyDeviceToHost, st)) ||
                        w.check(hipEventRecord(w.ev[s], st)))
                        return;
                } else if (c[s ^ 1] >= n) {
                    return;
                }
            }
        });
    }

    // device dst = src[0, bytes) in the order of st; a pageable src may be reused on
    // return, pinned memory once st has come this far
    void to_device(int device, void* dst, const void* src, size_t bytes, hipStream_t st)
    {
        std::lock_guard<std::mutex> lk(mu_);
        if (!staged(src, bytes, kMinToDevice)) {
            QBX_HIP(hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, st));
            return;
        }
        run(device, bytes, [&](Worker& w, size_t n) {
            int s = 0;
            for (size_t c = next_.fetch_add(1); c < n; c = next_.fetch_add(1), s ^= 1) {
                const size_t o = c * kChunk, len = std::min(kChunk, bytes - o);
                if (w.check(hipEventSynchronize(w.ev[s]))) return;   // the chunk's last copy has left it
                std::memcpy(w.p[s], (const char*)src + o, len);
                if (w.check(hipMemcpyAsync((char*)dst + o, w.p[s], len, hipMemcpyHostToDevice, st)) ||
                    w.check(hipEventRecord(w.ev[s], st)))
                    return;
            }
        });
    }

    void release()
    {
        for (Worker& w : workers_)
            for (int s = 0; s < 2; ++s)
                if (w.ev[s]) {
                    (void)hipEventSynchronize(w.ev[s]);
                    (void)hipEventDestroy(w.ev[s]);
                }
        workers_.clear();
        if (mem_) (void)hipHostFree(mem_);
        mem_ = nullptr;
    }

    static constexpr size_t kChunk = 2u << 20;
    static constexpr int kThreads = 12;
    // Smallest staged copies.  Staged against plain, to the host: 17 MiB 1.3 against 1.05
    // ms (with few chunks most calls wait for a thread to wake), 18.1 MiB 0.82/1.10, 24
    // 0.95/1.43, 37 2.0/4.0, 49 2.0/3.5; to the device: 17 MiB 0.72/0.60, 30 1.11/1.08, 42
    // 2.06/2.03, 48 1.85/2.10.  The pinned memory costs a context about 0.7 ms once.
    static constexpr size_t kMinToHost = 19u << 20;
    static constexpr size_t kMinToDevice = 46u << 20;

private:
    struct Worker {
        char* p[2] = {};
        hipEvent_t ev[2] = {};
        hipError_t err = hipSuccess;
        bool check(hipError_t e)
        {
            if (e != hipSuccess && err == hipSuccess) err = e;
            return e != hipSuccess;
        }
    };

    // staging pays, and its memory is there (no pinned memory left: the plain copy runs)
    bool staged(const void* host, size_t bytes, size_t least)
    {
        if (bytes < least) return false;
        threads_ = copy_threads(kThreads);
        if (threads_ < 2) return false;   // one CPU: the threads would take turns
        hipPointerAttribute_t at;
        if (hipPointerGetAttributes(&at, host) == hipSuccess) {
            if (at.type != hipMemoryTypeUnregistered) return false;   // pinned or managed already
        } else {
            (void)hipGetLastError();
        }
        if (threads_ <= (int)workers_.size()) return true;
        release();
        if (hipHostMalloc((void**)&mem_, kChunk * 2 * threads_, hipHostMallocDefault) != hipSuccess) {
            (void)hipGetLastError();
            mem_ = nullptr;
            return false;
        }
        workers_.assign(threads_, Worker());
        for (int t = 0; t < threads_; ++t)
            for (int s = 0; s < 2; ++s) {
                workers_[t].p[s] = mem_ + kChunk * (size_t)(2 * t + s);
                if (hipEventCreateWithFlags(&workers_[t].ev[s], hipEventDisableTiming) != hipSuccess) {
                    (void)hipGetLastError();
                    workers_[t].ev[s] = nullptr;
                    release();
                    return false;
                }
            }
        return true;
    }

    // body on up to threads_ threads, which take the copy's chunks from next_
    template <class Body> void run(int device, size_t bytes, Body body)
    {
        const size_t n = (bytes + kChunk - 1) / kChunk;
        next_ = 0;
        for (Worker& w : workers_) w.err = hipSuccess;
        std::vector<std::thread> pool;
        pool.reserve(threads_);
        for (int t = 1; t < threads_ && (size_t)t < n; ++t) {
            try {
                pool.emplace_back([&, t] {
                    if (!workers_[t].check(hipSetDevice(device))) body(workers_[t], n);
                });
            } catch (const std::system_error&) {
                break;   // fewer threads take all chunks
            }
        }
        body(workers_[0], n);
        for (std::thread& t : pool) t.join();
        for (Worker& w : workers_) QBX_HIP(w.err);
    }

    std::mutex mu_;
    char* mem_ = nullptr;
    std::vector<Worker> workers_;
    int threads_ = 0;   // of the current copy
    std::atomic<size_t> next_{0};
};

}  // namespace qbx
