// dtb_parts.hpp -- host passes over neurons on several threads.
#pragma once

#include <algorithm>
#include <cstdint>
#include <exception>
#include <thread>
#include <vector>

namespace dtb {

// Threads for a pass over n neurons' property rows (88 bytes each, so one
// thread waits for memory): 200k neurons' parameters re-derived took 1.1 ms
// on one thread.
inline uint32_t host_parts(uint32_t n)
{
    const uint32_t hw = std::thread::hardware_concurrency();
    return std::max(1u, std::min({hw ? hw : 4u, 8u, n / 16384u}));
}

// f(0) .. f(parts - 1), each on a thread of its own; rethrows the first error.
template <typename F>
void for_parts(uint32_t parts, F &&f)
{
    std::vector<std::exception_ptr> err(parts);
    std::vector<std::thread> th;
    th.reserve(parts);
    auto run = [&](uint32_t k) {
        try {
            f(k);
        } catch (...) {
            err[k] = std::current_exception();
        }
    };
    uint32_t k = 1;
    try {
        for (; k < parts; ++k)
            th.emplace_back(run, k);
    } catch (...) {
        // no more threads, or no memory for one (thrown past the running
        // ones it would end the process): this one does the rest
    }
    for (; k < parts; ++k)
        run(k);
    run(0);
    for (auto &t : th)
        t.join();
    for (auto &e : err)
        if (e)
            std::rethrow_exception(e);
}

}  // namespace dtb
