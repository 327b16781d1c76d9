/*
 * mdz_host_parallel.h -- loops over host data on a few threads.
 */
#pragma once

#include <algorithm>
#include <exception>
#include <mutex>
#include <thread>
#include <vector>

/* fn(begin, end) over chunks of [0, n) on up to eight host threads (the
 * caller's alone below two grains, or where no thread can be started); an
 * exception of a chunk is thrown again here after every chunk has ended */
template <class Fn>
void mdz_host_parallel(long long n, long long grain, Fn &&fn) {
    const long long most = std::min<long long>(8, std::max(1u, std::thread::hardware_concurrency()));
    const int nt = (int)std::max<long long>(1, std::min(most, n / std::max<long long>(grain, 1)));
    std::mutex mu;
    std::exception_ptr failed;
    auto chunk = [&](int t) {
        try {
            fn(n * t / nt, n * (t + 1) / nt);
        } catch (...) {
            std::lock_guard<std::mutex> g(mu);
            failed = std::current_exception();
        }
    };
    std::vector<std::thread> th;
    th.reserve((size_t)nt);
    int started = 1;
    try {
        for (; started < nt; started++) th.emplace_back(chunk, started);
    } catch (...) { /* no thread, or no memory for one */
    }
    chunk(0);
    for (int t = started; t < nt; t++) chunk(t);
    for (auto &x : th) x.join();
    if (failed) std::rethrow_exception(failed);
}
