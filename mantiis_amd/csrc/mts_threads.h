// Host threads for short parallel sections.
#pragma once
#include <algorithm>
#include <thread>

namespace mts {

constexpr int MAX_HOST_THREADS = 8;
inline int host_threads() { return std::max(1, std::min(MAX_HOST_THREADS, (int)std::thread::hardware_concurrency())); }

// Runs work(0) .. work(n - 1), n <= MAX_HOST_THREADS, on up to n threads, the
// caller's among them.  A thread that cannot be started (no memory, no thread)
// leaves its share to the others: work items are taken from a common counter by
// whoever runs.  Throws nothing if work does not.
template <class Work>
inline void on_threads(int n, const Work& work) noexcept {
    std::thread pool[MAX_HOST_THREADS];
    int k = 0;
    for (int t = 1; t < n && t < MAX_HOST_THREADS; t++) {
        try {
            pool[k] = std::thread([&work, t] { work(t); });
        } catch (...) {
            break;
        }
        k++;
    }
    work(0);
    for (int i = 0; i < k; i++) pool[i].join();
}

}  // namespace mts
