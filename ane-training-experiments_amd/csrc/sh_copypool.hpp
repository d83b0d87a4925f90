// sh_copypool.hpp — host copies spread over a few threads (host code only).
//
// One thread moves about 16 GB/s between host buffers and faults fresh pages in at 25 GB/s at
// best, a third of what PCIe brings. The pool's owner starts a job, may do something else, and
// finishes it: helpers and, in finish(), the owner itself take the job's parts one by one, so a
// helper that gets no CPU (a container's quota, other programs, other pools of the process) takes
// no part and holds nobody up beyond the part it is in. Nobody waits by spinning for longer than
// kSpin: with helpers and the owner spinning without a limit, three models called in turn (18
// helpers on 16 CPUs) took 848 us for a call whose 0.9 MB take the runtime's copy 210 us.
#pragma once

#include <stddef.h>
#include <stdint.h>
#include <string.h>
#include <sys/mman.h>
#include <unistd.h>

#include <algorithm>
#include <atomic>
#include <chrono>
#include <condition_variable>
#include <exception>
#include <mutex>
#include <thread>
#include <vector>

#ifndef MADV_POPULATE_WRITE
#define MADV_POPULATE_WRITE 23   // Linux 5.14; older kernels answer EINVAL
#endif

namespace sh {

// Used by one thread at a time, its owner.
class CopyPool {
  public:
    // Up to `helpers` threads; fewer where the system refuses one (the owner then does more).
    explicit CopyPool(int helpers) {
        try {
            threads_.reserve(helpers);
            for (int i = 0; i < helpers; i++) threads_.emplace_back([this] { work(); });
        } catch (const std::exception &) {
        }
    }
    CopyPool(const CopyPool &) = delete;
    CopyPool &operator=(const CopyPool &) = delete;
    ~CopyPool() {
        finish();
        {
            std::lock_guard<std::mutex> lk(mu_);
            stop_ = true;
        }
        wake_.notify_all();
        for (auto &t : threads_) t.join();
    }

    // dst[0, n) copied from src or, without a src, its pages faulted in (the contents stay), beside
    // what the caller does until finish(). The job before it is finished first.
    void start(void *dst, const void *src, size_t n) {
        finish();
        if (n == 0) return;
        dst_ = (uint8_t *)dst;
        src_ = (const uint8_t *)src;
        n_ = n;
        size_ = (std::max(kPart, n / kMaxParts) + 4095) & ~(size_t)4095;
        parts_ = (int)((n + size_ - 1) / size_);
        done_ = 0;
        left_ = parts_;   // publishes the job
        if (sleeping_.load() > 0) {
            std::lock_guard<std::mutex> lk(mu_);
            wake_.notify_all();
        }
    }
    // Returns once every part of the job is done, taking those that nobody has begun.
    void finish() {
        while (take()) {
        }
        spin([&] { return done_.load() == parts_; });
        if (done_.load() == parts_) return;
        std::unique_lock<std::mutex> lk(mu_);
        waiting_ = true;
        all_done_.wait(lk, [&] { return done_.load() == parts_; });
        waiting_ = false;
    }

  private:
    static constexpr size_t kPart = 32u << 10;   // about 2 us of copying, eight in the ring's least chunk
    static constexpr size_t kMaxParts = 64;
    static constexpr std::chrono::microseconds kSpin{50};   // about the time PCIe takes for a 2 MiB chunk

    template <class Ready>
    static void spin(Ready ready) {
        const auto until = std::chrono::steady_clock::now() + kSpin;
        while (!ready()) {
            for (int i = 0; i < 32; i++) __builtin_ia32_pause();
            if (std::chrono::steady_clock::now() >= until) return;
        }
    }
    // Does one part, if one is left. The job's fields stay as they are while a part is not done.
    bool take() {
        int left = left_.load();
        do {
            if (left == 0) return false;
        } while (!left_.compare_exchange_weak(left, left - 1));
        const int parts = parts_;
        const size_t a = (size_t)(parts - left) * size_, m = std::min(size_, n_ - a);
        if (src_) memcpy(dst_ + a, src_ + a, m);
        else fault_in(dst_ + a, m);
        // from here on the owner may return from finish() and write the next job
        if (done_.fetch_add(1) + 1 == parts && waiting_.load()) {
            std::lock_guard<std::mutex> lk(mu_);
            all_done_.notify_all();
        }
        return true;
    }
    static void fault_in(uint8_t *p, size_t m) {
        const uintptr_t page = (uintptr_t)sysconf(_SC_PAGESIZE);
        const uintptr_t lo = (uintptr_t)p & ~(page - 1), hi = ((uintptr_t)p + m + page - 1) & ~(page - 1);
        (void)madvise((void *)lo, hi - lo, MADV_POPULATE_WRITE);   // a failure leaves the faults to the copy
    }
    void work() {
        for (;;) {
            spin([&] { return left_.load() > 0 || stop_.load(); });
            if (left_.load() == 0 && !stop_.load()) {
                std::unique_lock<std::mutex> lk(mu_);
                sleeping_++;
                wake_.wait(lk, [&] { return left_.load() > 0 || stop_.load(); });
                sleeping_--;
            }
            if (stop_.load()) return;
            while (take()) {
            }
        }
    }

    std::vector<std::thread> threads_;
    std::mutex mu_;
    std::condition_variable wake_, all_done_;
    uint8_t *dst_ = nullptr;       // the job: written while none is left undone, read after a part is taken
    const uint8_t *src_ = nullptr;
    size_t n_ = 0, size_ = 0;
    int parts_ = 0;
    std::atomic<int> left_{0};     // parts nobody has taken
    std::atomic<int> done_{0};
    std::atomic<int> sleeping_{0};
    std::atomic<bool> waiting_{false}, stop_{false};
};

}  // namespace sh
