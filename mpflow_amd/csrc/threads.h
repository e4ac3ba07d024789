// Work shared by a few host threads.
#pragma once

#include <thread>
#include <vector>

namespace mpf {

// work(0) on this thread and work(1) .. work(n - 1) on others, all ended on return.  The work is shared,
// not split by number: where a thread cannot be started (none left, no memory for its state), those
// that run do its part.
template <class F>
void on_threads(int n, F&& work) {
    struct Joined {
        std::vector<std::thread> t;
        ~Joined() {
            for (auto& x : t) x.join();
        }
    } others;
    try {
        others.t.reserve(n);
        for (int i = 1; i < n; ++i) others.t.emplace_back([&work, i] { work(i); });
    } catch (...) {
    }
    work(0);
}

}  // namespace mpf
