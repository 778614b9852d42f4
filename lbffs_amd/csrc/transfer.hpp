// transfer.hpp -- copies between pageable host memory and the device.
//
// The host hands over ordinary arrays (std::vector, numpy), which the copy engines cannot reach
// directly: hipMemcpy passes them through a bounce buffer with one thread, and the first touch of a
// fresh destination's pages costs that thread more than the copy (8.6 GB/s into fresh pages,
// 16.6 GB/s into touched ones, against 56.8 GB/s from device to pinned memory).  Here the
// array goes through a ring of pinned chunks: the copy engine fills (or drains) half of them while
// several threads copy the other half from (or to) the array, each faulting its own pages.
//
// The ring is one per process, 16 MiB, made at the first large copy and given back when the
// last context is destroyed.  One copy uses it at a time; a copy that finds it taken by another
// thread, any copy below kStageMin, and memory the runtime knows (pinned, device, managed)
// take hipMemcpy.  Threads live for one copy.  What bounds it is the bus (56.8 GB/s) and,
// into fresh pages, the system's zeroing of them.  With eight threads, chunks of 2 MiB: 75 MB
// up at 36 GB/s, down into a fresh array at 26 GB/s, 21 MB at 25 and 23; an output step of
// 160x128x128 cells (six fields and the FP32 populations, 252 MB) 23 -> 10 ms.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <condition_variable>
#include <cstring>
#include <deque>
#include <mutex>
#include <system_error>
#include <thread>
#include <vector>

namespace lbffs {

constexpr size_t kStageChunk = size_t(2) << 20;  // bytes of one pinned chunk
constexpr int kStageSlots = 8;                   // chunks of the ring
constexpr int kStageThreads = 8;                 // copying threads at most
constexpr size_t kStageMin = size_t(4) << 20;    // below this hipMemcpy (threads would cost more)
constexpr size_t kStageLone = size_t(64) << 20;  // the same while no context keeps the ring

class HostStage
{
public:
    // contexts alive: the ring is kept while there is one
    void retain()
    {
        std::lock_guard<std::mutex> l(mu_);
        users_++;
    }
    void release()
    {
        std::lock_guard<std::mutex> l(mu_);
        if (--users_ <= 0) free_ring();
    }

    // copy `bytes` between host and device memory on `st`, after the work queued there; returns
    // when the data is in place
    hipError_t copy(void *dst, const void *src, size_t bytes, hipMemcpyKind kind, hipStream_t st)
    {
        if (bytes >= kStageMin && pageable(kind == hipMemcpyDeviceToHost ? dst : src)) {
            std::unique_lock<std::mutex> l(mu_, std::try_to_lock);
            if (l.owns_lock() && (users_ > 0 || bytes >= kStageLone) && make_ring()) {
                const hipError_t e = staged((char *)dst, (const char *)src, bytes, kind, st);
                if (users_ <= 0) free_ring();
                return e;
            }
        }
        const hipError_t e = hipStreamSynchronize(st);
        return e != hipSuccess ? e : hipMemcpy(dst, src, bytes, kind);
    }

private:
    std::mutex mu_;
    int users_ = 0;
    int device_ = -1;
    char *buf_ = nullptr;
    hipEvent_t ev_[kStageSlots] = {};

    // ordinary memory, which the runtime has no record of
    static bool pageable(const void *p)
    {
        hipPointerAttribute_t a;
        if (hipPointerGetAttributes(&a, p) != hipSuccess) {
            (void)hipGetLastError();  // "invalid value" stands for unknown memory
            return true;
        }
        return a.type == hipMemoryTypeUnregistered;
    }

    void free_ring()
    {
        for (hipEvent_t &e : ev_) {
            if (e) (void)hipEventDestroy(e);
            e = nullptr;
        }
        if (buf_) (void)hipHostFree(buf_);
        buf_ = nullptr;
        device_ = -1;
    }
    // the ring for the current device (its events belong to one); false if there is no memory
    bool make_ring()
    {
        int dev = 0;
        if (hipGetDevice(&dev) != hipSuccess) return false;
        if (buf_ && dev == device_) return true;
        free_ring();
        bool ok = hipHostMalloc((void **)&buf_, kStageSlots * kStageChunk, hipHostMallocPortable) == hipSuccess;
        if (!ok) buf_ = nullptr;
        for (int s = 0; s < kStageSlots && ok; s++) {
            ok = hipEventCreateWithFlags(&ev_[s], hipEventDisableTiming) == hipSuccess;
            if (!ok) ev_[s] = nullptr;
        }
        if (!ok) {
            free_ring();
            (void)hipGetLastError();
            return false;
        }
        device_ = dev;
        return true;
    }

    struct Job {
        char *dst;
        const char *src;
        size_t bytes;
        int slot;
    };
    // host-side copies of one transfer: jobs in order, their slots' states under one mutex
    struct Crew {
        std::mutex mu;
        std::condition_variable todo, done;
        std::deque<Job> jobs;
        bool busy[kStageSlots] = {};
        bool over = false;
        std::vector<std::thread> threads;

        void work()
        {
            std::unique_lock<std::mutex> l(mu);
            for (;;) {
                todo.wait(l, [&] { return over || !jobs.empty(); });
                if (jobs.empty()) return;
                const Job j = jobs.front();
                jobs.pop_front();
                l.unlock();
                std::memcpy(j.dst, j.src, j.bytes);
                l.lock();
                busy[j.slot] = false;
                done.notify_all();
            }
        }
        void give(const Job &j)
        {
            {
                std::lock_guard<std::mutex> l(mu);
                busy[j.slot] = true;
                jobs.push_back(j);
            }
            todo.notify_one();
        }
        void wait_slot(int s)
        {
            std::unique_lock<std::mutex> l(mu);
            done.wait(l, [&] { return !busy[s]; });
        }
        void finish()
        {
            {
                std::lock_guard<std::mutex> l(mu);
                over = true;
            }
            todo.notify_all();
            for (std::thread &t : threads) t.join();
        }
    };

    hipError_t staged(char *dst, const char *src, size_t bytes, hipMemcpyKind kind, hipStream_t st)
    {
        const long n = (long)((bytes + kStageChunk - 1) / kStageChunk);
        const bool down = kind == hipMemcpyDeviceToHost;
        Crew crew;
        const unsigned cpus = std::max(1u, std::thread::hardware_concurrency());
        const int want = (int)std::min<long>(std::min<long>(kStageThreads, cpus), n);
        try {
            for (int t = 0; t < want; t++) crew.threads.emplace_back([&crew] { crew.work(); });
        } catch (const std::system_error &) {
            // fewer threads than asked for
        }
        if (crew.threads.empty()) {
            const hipError_t e = hipStreamSynchronize(st);
            return e != hipSuccess ? e : hipMemcpy(dst, src, bytes, kind);
        }
        auto size_of = [&](long c) { return std::min(kStageChunk, bytes - (size_t)c * kStageChunk); };
        auto slot_buf = [&](long c) { return buf_ + (size_t)(c % kStageSlots) * kStageChunk; };
        constexpr int lag = kStageSlots / 2;  // chunks between the first and the second leg
        hipError_t e = hipSuccess;
        for (long c = 0; c < n + lag && e == hipSuccess; c++) {
            const int s = (int)(c % kStageSlots);
            if (c < n) {  // first leg: device to chunk, or array to chunk
                if (down) {
                    crew.wait_slot(s);
                    e = hipMemcpyAsync(slot_buf(c), src + (size_t)c * kStageChunk, size_of(c), kind, st);
                    if (e == hipSuccess) e = hipEventRecord(ev_[s], st);
                } else {
                    if (c >= kStageSlots) e = hipEventSynchronize(ev_[s]);
                    if (e == hipSuccess) crew.give({slot_buf(c), src + (size_t)c * kStageChunk, size_of(c), s});
                }
            }
            const long b = c - lag;
            if (b >= 0 && e == hipSuccess) {  // second leg: chunk to array, or chunk to device
                const int sb = (int)(b % kStageSlots);
                if (down) {
                    e = hipEventSynchronize(ev_[sb]);
                    if (e == hipSuccess) crew.give({dst + (size_t)b * kStageChunk, slot_buf(b), size_of(b), sb});
                } else {
                    crew.wait_slot(sb);
                    e = hipMemcpyAsync(dst + (size_t)b * kStageChunk, slot_buf(b), size_of(b), kind, st);
                    if (e == hipSuccess) e = hipEventRecord(ev_[sb], st);
                }
            }
        }
        crew.finish();  // the copies in hand end in any case
        const hipError_t es = hipStreamSynchronize(st);
        return e != hipSuccess ? e : es;
    }
};

}  // namespace lbffs
