// Loops of the layout builders on several host threads.
#pragma once
#include <algorithm>
#include <cstdint>
#include <exception>
#include <mutex>
#include <thread>
#include <vector>

// f(first, last) over ranges of 0 .. count on up to 16 threads.  `work` = elements that the whole loop touches: a thread
// costs some 30 us to start, which 100 000 elements repay.  `scratch` = bytes of memory that every range needs for
// itself: there are no more ranges at a time than share 256 MB.  An exception in any range is thrown to the caller (the
// first, if there are several) once no thread is running any more; a thread that cannot be started has its range done by
// the caller.
template <class F>
void so_parallel(uint32_t count, uint64_t work, F &&f, uint64_t scratch = 1)
{
    const uint64_t most = std::min<uint64_t>({std::max(1u, std::thread::hardware_concurrency()), 16u, count, work / 100000u + 1u,
                                              (256ull << 20) / std::max<uint64_t>(scratch, 1u)});
    const uint32_t nt = (uint32_t)std::max<uint64_t>(1u, most);
    std::exception_ptr failure;
    std::mutex failure_mutex;
    const auto range = [&](uint32_t t) {
        try {
            f((uint32_t)((uint64_t)count * t / nt), (uint32_t)((uint64_t)count * (t + 1) / nt));
        } catch (...) {
            const std::lock_guard<std::mutex> lock(failure_mutex);
            if (!failure) failure = std::current_exception();
        }
    };
    std::vector<std::thread> threads;
    uint32_t started = 1;
    try {
        for (threads.reserve(nt - 1); started < nt; ++started) threads.emplace_back(range, started);
    } catch (...) {
    }
    range(0);
    for (; started < nt; ++started) range(started);
    for (auto &t : threads) t.join();
    if (failure) std::rethrow_exception(failure);
}
