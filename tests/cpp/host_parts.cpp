// Checks of the library's host-only parts (llama-rust_amd/csrc/*.h that need no device), for the host compiler alone.
// Prints "OK" and returns 0, or says what failed and returns 1.
#include <sys/resource.h>
#include <sys/wait.h>
#include <unistd.h>

#include <atomic>
#include <cstdio>
#include <memory>
#include <thread>
#include <vector>

#include "../../llama-rust_amd/csrc/device_once.h"
#include "../../llama-rust_amd/csrc/host_pool.h"
#include "../../llama-rust_amd/csrc/host_range.h"
#include "../../llama-rust_amd/csrc/host_route.h"
#include "../../llama-rust_amd/csrc/step_replays.h"

static int failures = 0;
#define CHECK(cond)                                                         \
    do {                                                                    \
        if (!(cond)) {                                                      \
            std::printf("%s:%d: %s\n", __FILE__, __LINE__, #cond);          \
            failures++;                                                     \
        }                                                                   \
    } while (0)

// A buffer is used in place only where one mapping holds all of it.
static void host_range() {
    char *const host = reinterpret_cast<char *>(0x10000), *const device = reinterpret_cast<char *>(0x7000000);
    // [host + 4096, host + 12288) is pinned, and so is, on its own, what follows directly
    auto find = [&](const void *p, nh::HostMapping *m) {
        const size_t at = (size_t)(static_cast<const char *>(p) - host);
        if (at < 4096 || at >= 16384) return false;
        m->device = device + at;
        m->base = device + (at < 12288 ? 4096 : 12288);
        m->size = at < 12288 ? 8192 : 4096;
        return true;
    };
    CHECK(nh::device_view(host + 4096, 8192, find) == device + 4096);
    CHECK(nh::device_view(host + 5000, 7288, find) == device + 5000);
    CHECK(nh::device_view(host + 12287, 1, find) == device + 12287);
    CHECK(nh::device_view(host + 4096, 8193, find) == nullptr);   // the first part is pinned only
    CHECK(nh::device_view(host + 5000, 7289, find) == nullptr);
    CHECK(nh::device_view(host + 4096, 12288, find) == nullptr);  // two mappings
    CHECK(nh::device_view(host, 8192, find) == nullptr);          // the last part is pinned only
    CHECK(nh::device_view(host + 4096, SIZE_MAX, find) == nullptr);
    CHECK(nh::device_view(host + 4096, 16, [](const void *, nh::HostMapping *) { return true; }) == nullptr);
}

// Which host calls' kernels use pinned memory; the caller's own y only where one launch writes the whole of it, so that a call
// of several launches that fails has left it alone.
static void host_route() {
    constexpr uint32_t F16 = 1, Q4_0 = 2, Q4_K = 12, Q6_K = 14;
    auto route = [](const std::vector<nh::HostProduct> &p, bool shared_x, bool y_in_place) {
        size_t x = 0;
        for (const nh::HostProduct &q : p) x = shared_x ? q.tokens * q.cols : x + q.tokens * q.cols;
        const nh::HostRoute r = nh::host_route(p.size(), shared_x, x, y_in_place, [&](size_t g) { return p[g]; });
        return (r.x ? 1 : 0) + (r.y ? 2 : 0);
    };
    for (bool own : {false, true}) {
        CHECK(route({{1, 20000, 4096, Q4_K}}, false, own) == 3);
        CHECK(route({{1, 20000, 8192, Q4_K}}, false, own) == 3);
        CHECK(route({{1, 20000, 8448, Q4_K}}, false, own) == 2);
        CHECK(route({{1, 20000, 16384, Q4_K}}, false, own) == 2);
        CHECK(route({{1, 20000, 16640, Q4_K}}, false, own) == 0);
        CHECK(route({{3, 20000, 256, Q4_K}}, false, own) == 0);
        CHECK(route({{1, 14336, 4096, Q4_K}, {1, 14336, 4096, Q4_K}}, true, own) == 3);                     // one launch
        CHECK(route(std::vector<nh::HostProduct>(8, {1, 4096, 4096, Q4_K}), true, own) == 3);
        CHECK(route({{1, 4096, 4096, Q4_K}, {1, 16384, 4096, Q6_K}}, true, own) == (own ? 0 : 3));          // two dtypes
        CHECK(route({{1, 8192, 4096, Q4_K}, {1, 8192, 4096, Q4_K}}, false, own) == (own ? 0 : 3));          // two inputs
        CHECK(route({{1, 8192, 4096, Q4_K}, {1, 0, 4096, Q4_K}}, true, own) == (own ? 0 : 3));
        CHECK(route(std::vector<nh::HostProduct>(9, {1, 4096, 4096, Q4_K}), true, own) == (own ? 0 : 3));
        CHECK(route({{2, 8192, 1024, Q4_0}}, false, own) == (own ? 0 : 3));                                 // a launch per token
        CHECK(route({{2, 8192, 1024, F16}}, false, own) == (own ? 0 : 3));
        CHECK(route({{1, 8192, 1024, Q4_0}, {2, 8192, 1024, Q4_0}}, false, own) == (own ? 0 : 3));
    }
}

// Every step once, in whole replays where there is the longer graph, which is made when single replays have lost what it costs
// and never asked for again where it cannot be made.
static void step_replays() {
    constexpr size_t STEPS = nh::StepReplays::STEPS;
    for (bool can : {true, false}) {
        nh::StepReplays r;
        r.set_nodes(20);
        const size_t worth = r.worth();
        CHECK(worth > STEPS && worth < 400);
        size_t steps = 0, singles = 0, wholes = 0, makes = 0;
        auto run = [&](size_t n) {
            steps = singles = wholes = 0;
            const int rc = r.run(n, [&] { return steps++, singles++, 0; }, [&] { return steps += STEPS, wholes++, 0; });
            CHECK(rc == 0 && steps == n && singles + STEPS * wholes == n);
        };
        auto offer = [&] { r.offer([&] { return makes++, can ? 0 : 1; }); };
        for (size_t i = 0; i < 1000; i++) run(STEPS - 1), offer();  // runs that it could not serve
        CHECK(makes == 0);
        run(worth - 1 + STEPS - 1), offer();  // one step short
        CHECK(makes == 0 && wholes == 0);
        run(STEPS);
        CHECK(wholes == 0);
        offer();
        CHECK(makes == 1);
        for (size_t n : {size_t(0), size_t(1), STEPS - 1, STEPS, STEPS + 1, 5 * STEPS, 5 * STEPS + 3, 4 * worth}) {
            run(n), offer();
            CHECK(wholes == (can ? n / STEPS : 0));
        }
        CHECK(makes == 1);
    }
    nh::StepReplays none;  // a graph without nodes is no reason either
    none.set_nodes(0);
    none.offer([] { failures++; return 0; });
    // what fails ends the run
    nh::StepReplays r;
    size_t calls = 0;
    CHECK(r.run(5, [&] { return ++calls == 3 ? 7 : 0; }, [] { return 0; }) == 7 && calls == 3);
}

// Every item exactly once, seen by the caller afterwards, over calls of changing size that follow each other closely or
// after the workers have gone to sleep.
static void pool_items(nh::HostPool &pool) {
    std::vector<int> seen;
    const size_t sizes[] = {0, 1, 2, 3, 15, 16, 17, 64, 1000, 5, 2, 40000};
    for (int round = 0; round < 300; round++) {
        const size_t n = sizes[(size_t)round % 12];
        seen.assign(n, 0);
        pool.run(n, [&](size_t i) { seen[i]++; });
        size_t wrong = 0;
        for (size_t i = 0; i < n; i++) wrong += seen[i] != 1;
        CHECK(wrong == 0);
        if (round % 50 == 49) usleep(2000);
    }
    for (size_t n : {1, 7, 96, 97, 1000, 100003})
        for (size_t grain : {1, 10, 96, 200000}) {
            seen.assign(n, 0);
            std::atomic<size_t> pieces{0};
            pool.run_ranges(n, grain, [&](size_t begin, size_t end) {
                for (size_t i = begin; i < end; i++) seen[i]++;
                pieces++;
            });
            size_t wrong = 0;
            for (size_t i = 0; i < n; i++) wrong += seen[i] != 1;
            CHECK(wrong == 0);
            CHECK(pieces >= 1 && pieces <= 4 * pool.threads() && pieces <= (n + grain - 1) / grain);
        }
    size_t calls = 0;
    pool.run_ranges(0, 16, [&](size_t, size_t) { calls++; });
    CHECK(calls == 0);
    std::atomic<uint64_t> sum{0};  // more items than one word of the pool counts
    const size_t many = (1u << 20) + 5;
    pool.run(many, [&](size_t i) { sum.fetch_add(i, std::memory_order_relaxed); });
    CHECK(sum == (uint64_t)many * (many - 1) / 2);
}

static void pools() {
    {
        nh::HostPool pool(3), none(0);
        CHECK(none.threads() == 1);
        pool_items(pool);
        pool_items(none);
    }
    // pools of several threads at once, more of them than there are workers for
    std::vector<std::unique_ptr<nh::HostPool>> held;
    size_t workers = 0;
    for (int i = 0; i < 9; i++) {
        held.push_back(std::make_unique<nh::HostPool>(nh::HostPool::most_workers() / 4 + 1));
        workers += held.back()->threads() - 1;
    }
    CHECK(workers == nh::HostPool::most_workers());
    std::vector<std::thread> callers;
    for (auto &p : held) callers.emplace_back([&p] { pool_items(*p); });
    for (auto &t : callers) t.join();
    held.clear();
    nh::HostPool again(nh::HostPool::most_workers());  // given back
    CHECK(again.threads() == nh::HostPool::most_workers() + 1);
}

// A pool in a process that may have few or no further threads: no exception, no end of the process.
static void pool_without_threads() {
    const pid_t child = fork();
    if (child == 0) {
        long pages = 0;
        if (std::FILE *f = std::fopen("/proc/self/statm", "r")) {
            if (std::fscanf(f, "%ld", &pages) != 1) pages = 0;
            std::fclose(f);
        }
        const rlim_t limit = (rlim_t)pages * (rlim_t)sysconf(_SC_PAGESIZE) + (20u << 20);  // a few stacks, not sixteen
        const rlimit r = {limit, limit};
        if (pages == 0 || setrlimit(RLIMIT_AS, &r) != 0) _exit(2);
        {
            nh::HostPool pool(16);
            if (pool.threads() > 16) _exit(3);
            size_t seen[64] = {};
            pool.run(64, [&](size_t i) { seen[i]++; });
            for (size_t s : seen)
                if (s != 1) _exit(4);
        }
        _exit(0);
    }
    int status = -1;
    CHECK(child > 0 && waitpid(child, &status, 0) == child);
    CHECK(WIFEXITED(status) && WEXITSTATUS(status) == 0);
}

// Once for every device, again after a failure, and never skipped by a thread for which it has not been done.
static void device_once() {
    nh::DeviceOnce once;
    int calls = 0;
    auto works = [&] { return ++calls, 0; };
    auto fails = [&] { return ++calls, 7; };
    CHECK(once.run(0, fails) == 7 && once.run(0, works) == 0 && calls == 2);
    CHECK(once.run(0, fails) == 0 && calls == 2);
    CHECK(once.run(3, fails) == 7 && once.run(3, works) == 0 && once.run(63, works) == 0 && calls == 5);
    CHECK(once.run(3, works) == 0 && once.run(0, works) == 0 && once.run(63, works) == 0 && calls == 5);
    CHECK(once.run(64, works) == 0 && once.run(64, works) == 0 && once.run(-1, works) == 0 && calls == 8);  // not remembered
    for (int round = 0; round < 200; round++) {
        nh::DeviceOnce shared;
        int set[4] = {0, 0, 0, 0};  // not atomic: the flag is what orders it for the threads that skip
        std::atomic<int> missing{0}, first{0};
        std::vector<std::thread> threads;
        for (int t = 0; t < 4; t++)
            threads.emplace_back([&, t] {
                const int d = t % 2;
                shared.run(d, [&] { return first.fetch_add(1), set[2 * d + t / 2] = 1, 0; });
                if (shared.run(d, [] { return 1; }) != 0) missing++;
            });
        for (auto &t : threads) t.join();
        CHECK(missing == 0 && first >= 2 && first <= 4 && set[0] + set[1] >= 1 && set[2] + set[3] >= 1);
    }
}

int main() {
    pool_without_threads();  // first: a forked child has only the thread that forked
    host_range();
    host_route();
    step_replays();
    device_once();
    pools();
    if (failures == 0) std::printf("OK\n");
    return failures != 0;
}
