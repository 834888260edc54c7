// Host work on several threads.
#pragma once
#include <cstddef>
#include <exception>
#include <thread>
#include <vector>

namespace xpbd {

// Runs work() on n threads, this one among them, and returns when all have ended.
// work takes its share from a common counter and throws nothing.  With no thread to
// be had, or no memory for one, those there are do it all.
template <typename Work>
void on_threads(size_t n, const Work& work)
{
    std::vector<std::thread> pool;
    try {
        pool.reserve(n);
        for (size_t i = 1; i < n; i++) pool.emplace_back([&work] { work(); });
    } catch (const std::exception&) {
    }
    work();
    for (auto& t : pool) t.join();
}

}  // namespace xpbd
