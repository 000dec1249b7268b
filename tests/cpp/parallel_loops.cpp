// so_parallel (csrc/parallel.h): `parallel_loops ranges | throws | no_threads`, exit status 0 when it behaves.
#include "parallel.h"

#include <atomic>
#include <cstdio>
#include <cstring>
#include <stdexcept>
#include <sys/resource.h>

static bool covers(uint32_t count, uint64_t work, uint64_t scratch, int *most_threads = nullptr)
{
    std::vector<std::atomic<int>> seen(count);
    std::atomic<int> calls{0};
    so_parallel(count, work, [&](uint32_t a, uint32_t b) {
        ++calls;
        for (uint32_t i = a; i < b; ++i) ++seen[i];
    }, scratch);
    if (most_threads) *most_threads = calls;
    for (auto &s : seen)
        if (s != 1) return false;
    return true;
}

// An exception from the range that holds `where` comes out, after every other range has ended.
static bool throws(uint32_t where)
{
    std::atomic<int> running{0};
    try {
        so_parallel(1000, 100000000ull, [&](uint32_t a, uint32_t b) {
            ++running;
            struct Leave { std::atomic<int> &n; ~Leave() { --n; } } leave{running};
            std::this_thread::sleep_for(std::chrono::milliseconds(10));
            if (a <= where && where < b) throw std::bad_alloc();
        });
    } catch (const std::bad_alloc &) {
        return running == 0;
    }
    return false;
}

int main(int, char **argv)
{
    if (!std::strcmp(argv[1], "ranges")) {
        int ranges = 0;
        for (uint32_t count : {0u, 1u, 2u, 15u, 16u, 17u, 1000u})
            for (uint64_t work : {0ull, 99999ull, 250000ull, 100000000ull})
                if (!covers(count, work, 1)) return 1;
        if (!covers(1000, 100000000ull, 100ull << 20, &ranges) || ranges > 2) return 2;
        return covers(1000, 100000000ull, ~0ull, &ranges) && ranges == 1 ? 0 : 3;
    }
    if (!std::strcmp(argv[1], "throws")) return throws(0) && throws(500) && throws(999) ? 0 : 1;
    // no address space left for another thread's stack
    rlimit lim{64u << 20, 64u << 20};
    if (setrlimit(RLIMIT_AS, &lim) != 0) return 9;
    void *const hog = std::malloc(54u << 20);
    const bool ok = covers(1000, 100000000ull, 1);
    std::printf("%p\n", hog);
    return ok ? 0 : 1;
}
