// Host work shared by threads.
#pragma once
#include <algorithm>
#include <exception>
#include <mutex>
#include <thread>
#include <vector>

namespace hfh {

// work(t) on up to `nt` threads, this one among them: on fewer when no more
// can start (the work is shared out as it goes).  The first exception of any
// of them is rethrown here when all have ended.
template <typename F>
void run_parallel(int nt, F &&work) {
    std::exception_ptr err;
    std::mutex mu;
    auto body = [&](int t) {
        try {
            work(t);
        } catch (...) {
            std::lock_guard<std::mutex> lk(mu);
            if (!err) err = std::current_exception();
        }
    };
    std::vector<std::thread> th;
    try {
        th.reserve(std::max(nt - 1, 0));
        for (int t = 1; t < nt; t++) th.emplace_back(body, t);
    } catch (...) {
    }
    body(0);
    for (auto &t : th) t.join();
    if (err) std::rethrow_exception(err);
}

}  // namespace hfh
