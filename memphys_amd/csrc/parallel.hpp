// Host threads over an index range.
#pragma once
#include <algorithm>
#include <exception>
#include <mutex>
#include <thread>
#include <vector>

namespace mp {

// body(i0, i1, q) for the contiguous ranges q = 0 .. t-1 of [0, n), a thread each
// (range 0 on the caller's).  An exception of any range is thrown again here,
// once every thread has ended; ranges whose thread cannot be started run on the
// caller's.
template <typename F>
void parallel_ranges(int n, int t, F&& body) {
    std::exception_ptr error;
    std::mutex lock;
    auto run = [&](int q) {
        try {
            body((int)((long)n * q / t), (int)((long)n * (q + 1) / t), q);
        } catch (...) {
            const std::lock_guard<std::mutex> hold(lock);
            if (!error) error = std::current_exception();
        }
    };
    std::vector<std::thread> pool;
    pool.reserve(t);
    int q = 1;
    try {
        for (; q < t; ++q) pool.emplace_back(run, q);
    } catch (...) {  // (no thread for range q)
    }
    run(0);
    for (; q < t; ++q) run(q);
    for (std::thread& w : pool) w.join();
    if (error) std::rethrow_exception(error);
}

// f(i) for i in [0, n) on up to 16 threads.
template <typename F>
void parallel_for(int n, F&& f) {
    const int t = (int)std::max(1u, std::min({16u, std::thread::hardware_concurrency(),
                                              (unsigned)(n / 64 + 1)}));
    parallel_ranges(n, t, [&](int i0, int i1, int) {
        for (int i = i0; i < i1; ++i) f(i);
    });
}

}  // namespace mp
