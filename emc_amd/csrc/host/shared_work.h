// Work shared by a few threads of one call.
#pragma once
#include <thread>

namespace emc {

// work(0), ..., work(N - 1), or up to `threads` of them, each in a thread of its own but the first, which runs here.  What
// no thread can be had for (any exception of its making: no thread, no memory) runs here as well, and every thread has
// ended on return: the callers are C entries, which no exception may leave.  work itself must not throw.
template <int N, typename F>
void run_shared(int threads, const F &work)
{
    std::thread helper[N - 1];
    for (int t = 1; t < threads; ++t) {
        try {
            helper[t - 1] = std::thread([&work, t] { work(t); });
        } catch (...) {
        }
    }
    work(0);
    for (int t = 1; t < threads; ++t) {
        if (helper[t - 1].joinable()) helper[t - 1].join();
        else work(t);
    }
}

}  // namespace emc
