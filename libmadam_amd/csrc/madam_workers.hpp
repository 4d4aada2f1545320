// Several workers on one queue of pieces.
#pragma once
#include <exception>
#include <thread>
#include <vector>

namespace madam {

// work(0) on the calling thread and work(1) .. work(n - 1) on threads of their
// own, all ended on return.  The workers share one queue, so that work(0) alone
// empties it: a thread that cannot be made (the process or its container has
// too many) is a worker less, not an error.
template <typename F>
void run_workers(int n, F &&work)
{
    struct Joined {
        std::vector<std::thread> th;
        ~Joined()
        {
            for (std::thread &t : th) t.join();
        }
    } j;
    try {
        j.th.reserve(n > 1 ? n - 1 : 0);
        for (int i = 1; i < n; ++i) j.th.emplace_back([&work, i] { work(i); });
    } catch (const std::exception &) {
    }
    work(0);
}

}  // namespace madam
