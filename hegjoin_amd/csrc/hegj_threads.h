// hegj_threads.h -- host work shared by several threads.
#pragma once

#include <cstddef>
#include <thread>
#include <vector>

namespace hegj {

// work(0) on the calling thread and work(1) .. work(extra) on threads of their
// own, all of it done on return.  Where the system refuses a thread the ones
// that run are all there are, so the work must be taken from a common queue.
template <typename F>
void run_on_threads(size_t extra, F &&work) {
    std::vector<std::thread> pool;
    try {
        pool.reserve(extra);
        for (size_t t = 1; t <= extra; t++) pool.emplace_back([&work, t] { work(t); });
    } catch (...) {  // no thread or no memory for one
    }
    work(0);
    for (auto &t : pool) t.join();
}

}  // namespace hegj
