// ftdma_threads.h -- parts of a host job on threads (internal, host only).
#pragma once

#include <thread>

namespace ftd {

// part(0) .. part(N - 1), each on a thread of its own but the caller's part 0;
// returns after the last. A part whose thread cannot be had (no thread, no
// memory for one) runs on the caller's: nothing leaves this as an exception,
// since its callers are C entries and threads may be running by then.
template <int N, typename F>
void run_parts(const F& part) noexcept {
    std::thread th[N];
    for (int t = 1; t < N; ++t) {
        try {
            th[t] = std::thread([&part, t] { part(t); });
        } catch (...) {
            part(t);
        }
    }
    part(0);
    for (int t = 1; t < N; ++t)
        if (th[t].joinable()) th[t].join();
}

}  // namespace ftd
