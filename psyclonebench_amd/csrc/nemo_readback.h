// Read-back of an FP32 device field into a caller's FP64 array.
//
// The caller's array is ordinary memory, often fresh from the allocator, and
// one host thread widens values into it at 6 GB/s (less while its pages are
// new), a tenth of the link. The FP32 values come into pinned memory chunk by
// chunk, half the bytes of the FP64 ones, and several threads widen a chunk
// while the next ones arrive. The threads live for one call and touch memory
// only; they poll for a chunk while it may come within the next microseconds
// and sleep while steps before it still run. The stage belongs to the handle.
//
// us a field, pageable copy and one loop / staged, one thread / staged, team:
//   ssh         25 k values 32 / 30 / -;  81 k 62 / 52 / -;  0.18 M 118 / - / 84;
//               1.2 M 790 / - / 370
//   velocities  25 k 17 / 18 / -;  81 k 32 / 34 / -;  0.18 M 60 / - / 58;  1.2 M
//               430 / - / 240
// so a thread for every 128 k values, and below that the pageable copy for a
// field of one word. A single chunk waits for the stream: an event costs 8 us
// more (25 k values of ssh 40, of u 28).
#pragma once

#include <algorithm>
#include <atomic>
#include <chrono>
#include <condition_variable>
#include <exception>
#include <mutex>
#include <thread>
#include <vector>

#include "nemo_hip_common.h"

namespace nemo {

class ReadBack {
public:
    ReadBack() = default;
    ReadBack(const ReadBack &) = delete;
    ReadBack &operator=(const ReadBack &) = delete;
    ~ReadBack()
    {
        for (hipEvent_t e : ready_)
            if (e) (void)hipEventDestroy(e);
        if (stage_) (void)hipHostFree(stage_);
    }

    // out[k] = hi[k] (+ lo[k], where lo is not null), k < n, device arrays as
    // work on stream s leaves them.
    void read(hipStream_t s, const float *hi, const float *lo, size_t n, double *out)
    {
        if (n == 0) return;
        if (!lo && n <= kOneThread) {
            std::vector<float> a(n);
            NEMO_HIP_CHECK(hipStreamSynchronize(s));
            NEMO_HIP_CHECK(hipMemcpy(a.data(), hi, n * sizeof(float), hipMemcpyDeviceToHost));
            for (size_t k = 0; k < n; k++) out[k] = (double)a[k];
            return;
        }
        // threads may read one handle at the same time; they share the stage
        const std::lock_guard<std::mutex> one(mutex_);
        if (!stage_) {
            NEMO_HIP_CHECK(hipHostMalloc((void **)&stage_, kSlots * 2 * kChunk * sizeof(float),
                                         hipHostMallocDefault));
            for (hipEvent_t &e : ready_)
                NEMO_HIP_CHECK(hipEventCreateWithFlags(&e, hipEventDisableTiming));
        }
        const size_t chunks = (n + kChunk - 1) / kChunk;
        auto count = [&](size_t c) { return std::min(kChunk, n - c * kChunk); };
        auto copy = [&](size_t c) {
            float *const d = stage_ + c % kSlots * 2 * kChunk;
            const size_t bytes = count(c) * sizeof(float);
            NEMO_HIP_CHECK(hipMemcpyAsync(d, hi + c * kChunk, bytes, hipMemcpyDeviceToHost, s));
            if (lo)
                NEMO_HIP_CHECK(hipMemcpyAsync(d + kChunk, lo + c * kChunk, bytes,
                                              hipMemcpyDeviceToHost, s));
        };
        auto queue = [&](size_t c) {
            copy(c);
            NEMO_HIP_CHECK(hipEventRecord(ready_[c % kSlots], s));
        };
        // thread t of `threads` widens its part of every chunk
        Arrivals arrived;
        int nt = 1;  // known before the first arrival
        Done done[kMaxThreads];
        auto part = [&](size_t c, int t) {
            const size_t m = count(c), a = m * t / nt, b = m * (t + 1) / nt;
            const float *const d = stage_ + c % kSlots * 2 * kChunk;
            double *const o = out + c * kChunk;
            if (lo)
                for (size_t k = a; k < b; k++) o[k] = (double)d[k] + (double)d[kChunk + k];
            else
                for (size_t k = a; k < b; k++) o[k] = (double)d[k];
            done[t].chunks.store(c + 1, std::memory_order_release);
        };
        auto helper = [&](int t) {
            for (size_t c = 0; c < chunks; c++) {
                arrived.wait(c);
                part(c, t);
            }
        };
        if (n <= kOneThread) {  // no event, no team
            copy(0);
            NEMO_HIP_CHECK(hipStreamSynchronize(s));
            part(0, 0);
            return;
        }
        for (size_t c = 0; c < std::min(chunks, kSlots); c++) queue(c);
        // a thread for every kPerThread values, as far as there are processors
        const size_t want = std::min({(size_t)kMaxThreads, n / kPerThread + 1,
                                      (size_t)std::max(1u, std::thread::hardware_concurrency())});
        std::vector<std::thread> team;
        try {
            team.reserve(want);
            while (team.size() + 1 < want) team.emplace_back(helper, (int)team.size() + 1);
        } catch (const std::exception &) {  // no more threads: fewer will do
        }
        nt = (int)team.size() + 1;
        for (size_t c = 0; c < chunks; c++) {
            NEMO_HIP_CHECK(hipEventSynchronize(ready_[c % kSlots]));
            arrived.add();
            part(c, 0);
            if (c + kSlots >= chunks) continue;
            for (int t = 1; t < nt; t++)  // the slot is free when every part is out
                while (done[t].chunks.load(std::memory_order_acquire) <= c)
                    std::this_thread::yield();
            queue(c + kSlots);
        }
        for (std::thread &t : team) t.join();
    }

private:
    static constexpr size_t kChunk = 1 << 18, kSlots = 3;  // 2 MB, with lo
    static constexpr size_t kPerThread = 1 << 17, kOneThread = kPerThread - 1;
    static_assert(kOneThread <= kChunk, "one chunk");
    static constexpr int kMaxThreads = 8;
    static constexpr std::chrono::microseconds kPoll{200};  // ten chunks' time on the link
    struct alignas(64) Done {
        std::atomic<size_t> chunks{0};
    };
    // Chunks that have arrived.
    class Arrivals {
    public:
        void add()
        {
            {
                const std::lock_guard<std::mutex> hold(mutex_);
                count_.store(count_.load(std::memory_order_relaxed) + 1,
                             std::memory_order_release);
            }
            more_.notify_all();
        }
        void wait(size_t c)  // until chunk c is there
        {
            auto there = [&] { return count_.load(std::memory_order_acquire) > c; };
            const auto until = std::chrono::steady_clock::now() + kPoll;
            while (!there() && std::chrono::steady_clock::now() < until)
                std::this_thread::yield();
            if (there()) return;
            std::unique_lock<std::mutex> hold(mutex_);
            more_.wait(hold, there);
        }

    private:
        std::mutex mutex_;
        std::condition_variable more_;
        std::atomic<size_t> count_{0};
    };
    std::mutex mutex_;
    float *stage_ = nullptr;
    hipEvent_t ready_[kSlots] = {};
};

}  // namespace nemo
