// Host threads for parts of one call.
#pragma once
#include <exception>
#include <mutex>
#include <thread>
#include <vector>

// Calls work(0) .. work(parts - 1), each on a thread of its own and the first
// on this one; the parts whose threads cannot be started run here after it.
// Returns when all have ended; what a part threw is thrown here then (the
// first of them).
template <typename F>
void tsg_parallel(int parts, F work) {
    std::exception_ptr thrown;
    std::mutex m;
    auto part = [&](int p) {
        try {
            work(p);
        } catch (...) {
            std::lock_guard<std::mutex> lock(m);
            if (!thrown) thrown = std::current_exception();
        }
    };
    std::vector<std::thread> pool;
    int started = 1;
    try {
        pool.reserve(parts > 1 ? parts - 1 : 0);
        for (; started < parts; started++) pool.emplace_back(part, started);
    } catch (...) {  // (no more threads, or no memory for one)
    }
    if (parts > 0) part(0);
    for (int p = started; p < parts; p++) part(p);
    for (std::thread &t : pool) t.join();
    if (thrown) std::rethrow_exception(thrown);
}
