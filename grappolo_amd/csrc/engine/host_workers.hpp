// host_workers.hpp -- a piece of host work shared by short-lived threads.
#pragma once

#include <system_error>
#include <thread>
#include <vector>

namespace glv {

// worker() on the calling thread and on up to n - 1 others, joined on return:
// each call takes what is left of the work.  Where the system gives no more
// threads, those there are do it (an exception past a running std::thread would
// end the program).  worker throws nothing.
template <class F>
void run_workers(int n, const F &worker) {
    std::vector<std::thread> pool;
    pool.reserve(n > 1 ? n - 1 : 0);
    try {
        for (int t = 1; t < n; t++) pool.emplace_back([&] { worker(); });
    } catch (const std::system_error &) {
    }
    worker();
    for (auto &t : pool) t.join();
}

}  // namespace glv
