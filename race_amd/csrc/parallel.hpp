// parallel.hpp -- contiguous parts of a range on host threads.
#pragma once
#include <algorithm>
#include <exception>
#include <system_error>
#include <thread>
#include <vector>

namespace race {

// f(lo, hi) over [0, n) in contiguous parts of at least `grain`, on up to 8
// host threads; an exception of a part reaches the caller once all have ended
template <class F>
void parallelRanges(int n, int grain, F&& f) {
    const int want = std::max(
        1, std::min({8, (int)std::max(1u, std::thread::hardware_concurrency()), n / std::max(1, grain)}));
    std::vector<std::exception_ptr> bad(want);
    auto part = [&](int t) {
        try {
            f((int)((long)n * t / want), (int)((long)n * (t + 1) / want));
        } catch (...) {
            bad[t] = std::current_exception();
        }
    };
    std::vector<std::thread> ts;
    ts.reserve(want);
    int started = 1;  // part 0 runs here, and so do those no thread was left for
    try {
        for (; started < want; ++started) ts.emplace_back(part, started);
    } catch (const std::system_error&) {
    }
    part(0);
    for (int t = started; t < want; ++t) part(t);
    for (std::thread& t : ts) t.join();
    for (const std::exception_ptr& e : bad)
        if (e) std::rethrow_exception(e);
}

}  // namespace race
