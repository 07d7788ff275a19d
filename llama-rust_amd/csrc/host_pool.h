// Worker threads for the host side of a call: comparing weight bytes, attention heads, element-wise rows.
//
// The pieces of work here are short (5-500 us) and follow each other closely, so what counts is how soon a worker
// begins and how little the caller waits at the end:
//   - a worker that has run out of items watches for the next call for SPIN_US before it sleeps in the kernel: a woken
//     thread starts 5-50 us late, one that watches in well under 1 us;
//   - items are handed out one by one from a single word that also holds the call's number and item count, and run()
//     returns when every item is done, not when every worker has woken up: a late worker finds the word spent and
//     goes back to sleep.
// A pool belongs to one object and is driven by one thread at a time; it ends with its owner.  All pools of a process
// together have a bounded number of workers: a pool that finds fewer left, or whose threads the system refuses, has as
// many as it got, down to none (the calling thread then does all the work).
#ifndef NATIVE_HIP_HOST_POOL_H
#define NATIVE_HIP_HOST_POOL_H

#include <linux/futex.h>
#include <sys/syscall.h>
#include <unistd.h>

#include <atomic>
#include <chrono>
#include <climits>
#include <cstddef>
#include <cstdint>
#include <exception>
#include <thread>
#include <vector>

namespace nh {

class HostPool {
  public:
    // Threads of a pool, the caller included: the reference spreads host work over few threads too, and a process may
    // hold several pools.
    static size_t default_threads() {
        const unsigned hw = std::thread::hardware_concurrency();
        return hw < 2 ? 1 : (hw > 16 ? 16 : hw);
    }
    // Workers of all pools together: four whole pools.  A program that calls from more threads than that keeps its
    // processors busy without them.
    static size_t most_workers() { return 4 * (default_threads() - 1); }
    // Never throws: this is reached from C entry points, and a thread that cannot be made is no failure of the call.
    explicit HostPool(size_t workers = default_threads() - 1) noexcept {
        size_t used = live().load(std::memory_order_relaxed), want;
        do {
            const size_t left = most_workers() > used ? most_workers() - used : 0;
            want = workers < left ? workers : left;
        } while (!live().compare_exchange_weak(used, used + want, std::memory_order_relaxed));
        try {
            threads_.reserve(want);
            while (threads_.size() < want) threads_.emplace_back([this] { loop(); });
        } catch (const std::exception &) {  // the system's limit on threads or memory: those made so far do
        }
        live().fetch_sub(want - threads_.size(), std::memory_order_relaxed);
    }
    HostPool(const HostPool &) = delete;
    HostPool &operator=(const HostPool &) = delete;
    ~HostPool() {
        stop_.store(true, std::memory_order_relaxed);
        ring(INT_MAX);
        for (auto &t : threads_) t.join();
        live().fetch_sub(threads_.size(), std::memory_order_relaxed);
    }
    size_t threads() const { return threads_.size() + 1; }

    // Calls fn(i) once for every i < n, on the workers and on the calling thread; returns when all are done.
    template <typename F> void run(size_t n, const F &fn) {
        while (n > MAX_ITEMS) {  // the item count has 20 bits of the word
            run_some(MAX_ITEMS, [&](size_t i) { fn(n - MAX_ITEMS + i); });
            n -= MAX_ITEMS;
        }
        run_some(n, fn);
    }
    // Calls fn(begin, end) over pieces of [0, n) of at least `grain`.
    template <typename F> void run_ranges(size_t n, size_t grain, const F &fn) {
        if (n == 0) return;
        size_t pieces = (n + grain - 1) / (grain ? grain : 1);
        const size_t most = 4 * threads();  // a few per thread: they do not all run at one speed
        if (pieces > most) pieces = most;
        run(pieces, [&](size_t i) { fn(n * i / pieces, n * (i + 1) / pieces); });
    }

  private:
    static std::atomic<size_t> &live() {
        static std::atomic<size_t> count{0};
        return count;
    }

    static constexpr size_t MAX_ITEMS = (1u << 20) - 1;
    static constexpr int SPIN_US = 60;  // about the time a product call of a host session keeps its caller away

    using Call = void (*)(const void *, size_t);
    template <typename F> void run_some(size_t n, const F &fn) {
        if (threads_.empty() || n < 2) {
            for (size_t i = 0; i < n; i++) fn(i);
            return;
        }
        call_ = [](const void *f, size_t i) { (*static_cast<const F *>(f))(i); };
        arg_ = &fn;
        done_.store(0, std::memory_order_relaxed);
        epoch_ = (epoch_ + 1) & 0xffffffu;
        word_.store(((uint64_t)epoch_ << 40) | ((uint64_t)n << 20), std::memory_order_release);
        ring((int)(n - 1));
        work(epoch_);
        for (uint32_t spins = 0; done_.load(std::memory_order_acquire) != n;) pause(spins);
    }
    // Takes items of call `epoch` until there are none left.  An item taken belongs to a call whose run() has not
    // returned (it waits for that item), so call_ and arg_ are that call's.
    void work(uint32_t epoch) {
        uint64_t w = word_.load(std::memory_order_acquire);
        for (;;) {
            const uint64_t n = (w >> 20) & MAX_ITEMS, next = w & MAX_ITEMS;
            if ((uint32_t)(w >> 40) != epoch || next >= n) return;
            if (!word_.compare_exchange_weak(w, w + 1, std::memory_order_acq_rel, std::memory_order_acquire)) continue;
            call_(arg_, (size_t)next);
            done_.fetch_add(1, std::memory_order_release);
            w = word_.load(std::memory_order_acquire);
        }
    }
    void loop() {
        uint32_t seen = 0;
        for (;;) {
            const uint32_t bell = bell_.load(std::memory_order_acquire);
            if (stop_.load(std::memory_order_relaxed)) return;
            if (bell == seen) {
                const auto until = std::chrono::steady_clock::now() + std::chrono::microseconds(SPIN_US);
                uint32_t spins = 0;
                do {
                    for (int k = 0; k < 32 && bell_.load(std::memory_order_relaxed) == seen; k++) pause(spins);
                } while (bell_.load(std::memory_order_relaxed) == seen && std::chrono::steady_clock::now() < until);
                if (bell_.load(std::memory_order_acquire) == seen) {
                    sleepers_.fetch_add(1, std::memory_order_seq_cst);
                    syscall(SYS_futex, reinterpret_cast<uint32_t *>(&bell_), FUTEX_WAIT_PRIVATE, seen, nullptr, nullptr, 0);
                    sleepers_.fetch_sub(1, std::memory_order_relaxed);
                }
                continue;
            }
            seen = bell;
            work((uint32_t)(word_.load(std::memory_order_acquire) >> 40));
        }
    }
    void ring(int sleepers) {
        bell_.fetch_add(1, std::memory_order_seq_cst);
        if (sleepers_.load(std::memory_order_seq_cst) != 0)  // a worker about to sleep re-reads the bell in the futex call
            syscall(SYS_futex, reinterpret_cast<uint32_t *>(&bell_), FUTEX_WAKE_PRIVATE, sleepers, nullptr, nullptr, 0);
    }
    static void pause(uint32_t &spins) {
        if (++spins % 4096 == 0) std::this_thread::yield();  // more threads than processors: let the owner of an item run
        __builtin_ia32_pause();
    }

    std::vector<std::thread> threads_;
    std::atomic<uint64_t> word_{0};  // call number (24 bits) | items (20) | next item (20)
    alignas(64) std::atomic<size_t> done_{0};
    alignas(64) std::atomic<uint32_t> bell_{0};
    std::atomic<uint32_t> sleepers_{0};
    std::atomic<bool> stop_{false};
    Call call_ = nullptr;
    const void *arg_ = nullptr;
    uint32_t epoch_ = 0;
};

}  // namespace nh
#endif
