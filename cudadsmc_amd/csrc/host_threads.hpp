// host_threads.hpp -- a piece of work done by several host threads for the
// length of one call.
#pragma once

#include <exception>
#include <functional>
#include <thread>
#include <vector>

namespace dsmc {

// work(0) on the calling thread and work(1) .. work(threads - 1) on new ones;
// returns when all are done.  Fewer run when a thread cannot be made (out of
// threads or of memory), so the work is shared out as it goes; it must not
// throw.
template <class Work>
void run_threads(int threads, const Work &work)
{
    std::vector<std::thread> pool;
    try {
        pool.reserve((size_t)(threads > 1 ? threads - 1 : 0));
        for (int k = 1; k < threads; ++k) pool.emplace_back(std::cref(work), k);
    } catch (const std::exception &) {   // those that run are joined below
    }
    work(0);
    for (std::thread &t : pool) t.join();
}

}  // namespace dsmc
