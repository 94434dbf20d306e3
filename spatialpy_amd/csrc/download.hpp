// Copies of results to the caller's (pageable) arrays.
//
// A plain device-to-host copy into fresh pageable memory runs on one thread: the
// runtime copies through its own pinned buffer, and every page is first touched
// there; particle-major [n][3] arrays take a second pass over a temporary.  From
// DOWNLOAD_MIN bytes on, the data comes through a ring of pinned slots instead,
// and some threads move the slots' contents to their places (interleaving the
// three components on the way) while the next ones arrive.
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>
#include <condition_variable>
#include <cstring>
#include <exception>
#include <mutex>
#include <thread>
#include <vector>

#include "engine.hpp"

namespace ssa {

// 16 MiB, allocated by the first large copy of its owner, given back with it
class PinnedRing {
  public:
    static constexpr int SLOTS = 8;
    static constexpr size_t SLOT = 2u << 20;
    PinnedRing() = default;
    PinnedRing(const PinnedRing &) = delete;
    PinnedRing &operator=(const PinnedRing &) = delete;
    ~PinnedRing() { release(); }
    bool ready() {
        if (base_) return true;
        if (hipHostMalloc((void **)&base_, SLOTS * SLOT, hipHostMallocDefault) != hipSuccess) {
            (void)hipGetLastError();
            base_ = nullptr;
            return false;
        }
        for (int k = 0; k < SLOTS; k++)
            if (hipEventCreateWithFlags(&ev_[k], hipEventDisableTiming) != hipSuccess) {
                (void)hipGetLastError();
                release();
                return false;
            }
        return true;
    }
    void release() {
        for (auto &e : ev_) {
            if (e) (void)hipEventDestroy(e);
            e = nullptr;
        }
        if (base_) (void)hipHostFree(base_);
        base_ = nullptr;
    }
    char *slot(int k) { return base_ + k * SLOT; }
    hipEvent_t event(int k) { return ev_[k]; }

  private:
    char *base_ = nullptr;
    hipEvent_t ev_[SLOTS] = {};
};

// A plain copy into fresh memory moves 9 GB/s: 1 ms for 8 MiB, about what the
// ring's allocation (0.4 ms) and the threads cost.  Above it: two snapshots of a
// million particles (184 MB with the interleaving) 45 -> 18 ms, 262 MB of counts
// 60 -> 25 ms.
constexpr size_t DOWNLOAD_MIN = 8u << 20;
constexpr int DOWNLOAD_THREADS = 8;

// The copies of one call, in stream order; a source may be overwritten by work
// enqueued after its put().  finish() returns when all have arrived.
class Download {
  public:
    // total: bytes that will be put, about
    Download(hipStream_t s, PinnedRing &ring, size_t total) : s_(s), ring_(ring) {
        if (total < DOWNLOAD_MIN || !ring.ready()) return;
        const int hw = (int)std::thread::hardware_concurrency();
        const int want = std::max(1, std::min(DOWNLOAD_THREADS, hw / 2));
        try {
            team_.reserve(want);
            for (int k = 0; k < want; k++) team_.emplace_back([this] { work(); });
        } catch (const std::exception &) {
            // (std::system_error or std::bad_alloc: an exception that left here
            // would destroy running threads.)  As many as there are; with none
            // the copies are plain ones
        }
    }
    Download(const Download &) = delete;
    Download &operator=(const Download &) = delete;
    ~Download() { close(); }

    template <class T> void put(T *dst, const T *src, size_t count) {
        const size_t bytes = sizeof(T) * count;
        if (team_.empty()) {
            if (bytes) check(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, s_));
            return;
        }
        for (size_t at = 0; at < bytes; at += PinnedRing::SLOT) {
            const size_t len = std::min(PinnedRing::SLOT, bytes - at);
            const int k = claim();
            check(hipMemcpyAsync(ring_.slot(k), (const char *)src + at, len, hipMemcpyDeviceToHost, s_));
            publish(k, (char *)dst + at, len, false);
        }
    }
    // component-major [3][n] to particle-major [n][3]
    void put3(double *dst, const double *src, size_t n) {
        if (team_.empty()) {
            tmp_.resize(3 * n);
            check(hipMemcpyAsync(tmp_.data(), src, sizeof(double) * 3 * n, hipMemcpyDeviceToHost, s_));
            check(hipStreamSynchronize(s_));
            interleave(dst, tmp_.data(), n);
            return;
        }
        const size_t most = PinnedRing::SLOT / (3 * sizeof(double));
        for (size_t at = 0; at < n; at += most) {
            const size_t m = std::min(most, n - at);
            const int k = claim();
            for (int c = 0; c < 3; c++)
                check(hipMemcpyAsync(ring_.slot(k) + c * m * sizeof(double), src + c * n + at, m * sizeof(double),
                                     hipMemcpyDeviceToHost, s_));
            publish(k, (char *)(dst + 3 * at), m, true);
        }
    }
    void finish() {
        check(hipStreamSynchronize(s_));
        close();
        check(err_);
    }

  private:
    struct Job {
        char *dst;
        size_t len;      // bytes, or particles
        bool three;
        int slot;
    };
    static void check(hipError_t e) { HIP_OK(e); }
    static void interleave(double *dst, const double *src, size_t m) {
        for (size_t i = 0; i < m; i++)
            for (int c = 0; c < 3; c++) dst[3 * i + c] = src[c * m + i];
    }
    // the next slot in turn, once its last contents have been moved
    int claim() {
        const int k = (int)(sent_++ % PinnedRing::SLOTS);
        std::unique_lock<std::mutex> l(mx_);
        room_.wait(l, [&] { return !busy_[k]; });
        return k;
    }
    void publish(int k, char *dst, size_t len, bool three) {
        check(hipEventRecord(ring_.event(k), s_));
        {
            std::lock_guard<std::mutex> l(mx_);
            busy_[k] = true;
            jobs_.push_back(Job{dst, len, three, k});
        }
        ready_.notify_one();
    }
    void work() {
        std::unique_lock<std::mutex> l(mx_);
        for (;;) {
            ready_.wait(l, [&] { return taken_ < jobs_.size() || closed_; });
            if (taken_ == jobs_.size()) return;
            const Job j = jobs_[taken_++];
            l.unlock();
            const hipError_t e = hipEventSynchronize(ring_.event(j.slot));
            if (e == hipSuccess) {
                const char *from = ring_.slot(j.slot);
                if (j.three) interleave((double *)j.dst, (const double *)from, j.len);
                else memcpy(j.dst, from, j.len);
            }
            l.lock();
            if (e != hipSuccess && err_ == hipSuccess) err_ = e;
            busy_[j.slot] = false;
            room_.notify_one();
        }
    }
    void close() {
        {
            std::lock_guard<std::mutex> l(mx_);
            closed_ = true;
        }
        ready_.notify_all();
        for (auto &t : team_) t.join();
        team_.clear();
    }

    hipStream_t s_;
    PinnedRing &ring_;
    std::vector<double> tmp_;
    std::vector<std::thread> team_;
    std::mutex mx_;
    std::condition_variable ready_, room_;
    std::vector<Job> jobs_;
    size_t taken_ = 0, sent_ = 0;
    bool busy_[PinnedRing::SLOTS] = {};
    bool closed_ = false;
    hipError_t err_ = hipSuccess;
};

}  // namespace ssa
