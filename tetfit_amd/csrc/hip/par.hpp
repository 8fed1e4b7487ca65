// par.hpp - host loops over several threads (no HIP in here).
#pragma once

#include <algorithm>
#include <atomic>
#include <cstdint>
#include <exception>
#include <mutex>
#include <thread>
#include <vector>

namespace tfd {

// Runs f(lo, hi) over [0, n) in chunks of `chunk` entries on up to 16 host
// threads, the caller among them (chunk boundaries do not depend on the thread
// count). The first exception f throws ends the loop and is thrown here once
// every thread has stopped; threads that cannot be started are done without.
template <class Fn>
void par_chunks(int64_t n, int64_t chunk, const Fn& f) {
    const int64_t nc = (n + chunk - 1) / chunk;
    const int64_t hw = std::max(1u, std::thread::hardware_concurrency());
    const int nt = (int)std::min<int64_t>(nc, std::min<int64_t>(hw, 16));
    if (nt <= 1) {
        for (int64_t k = 0; k < nc; ++k) f(k * chunk, std::min(n, (k + 1) * chunk));
        return;
    }
    std::atomic<int64_t> next{0};
    std::exception_ptr err;
    std::mutex err_lock;
    auto work = [&] {
        try {
            for (int64_t k; (k = next++) < nc;) f(k * chunk, std::min(n, (k + 1) * chunk));
        } catch (...) {
            std::lock_guard<std::mutex> g(err_lock);
            if (!err) err = std::current_exception();
            next = nc;
        }
    };
    std::vector<std::thread> th;
    try {
        th.reserve(nt - 1);
        for (int t = 1; t < nt; ++t) th.emplace_back(work);
    } catch (const std::exception&) {
    }
    work();
    for (auto& t : th) t.join();
    if (err) std::rethrow_exception(err);
}

}  // namespace tfd
