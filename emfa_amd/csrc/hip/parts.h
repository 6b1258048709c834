// Host work in parts on threads.
#pragma once
#include <exception>
#include <functional>
#include <thread>
#include <vector>

namespace emfa {

// work(0) .. work(parts - 1), one host thread each where the system grants it.
// All parts have ended when it returns or throws; the first part's exception, if
// any threw, is the caller's.
inline void run_parts(int parts, const std::function<void(int)> &work) {
    std::vector<std::exception_ptr> thrown(parts);
    auto part = [&](int t) {
        try {
            work(t);
        } catch (...) {
            thrown[t] = std::current_exception();
        }
    };
    std::vector<std::thread> pool;
    pool.reserve(parts);
    int t = 1;
    try {
        for (; t < parts; ++t) pool.emplace_back(part, t);
    } catch (...) {  // no more threads: the rest here
    }
    for (; t < parts; ++t) part(t);
    part(0);
    for (auto &th : pool) th.join();
    for (auto &e : thrown)
        if (e) std::rethrow_exception(e);
}

}  // namespace emfa
