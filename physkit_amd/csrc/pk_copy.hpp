// Host memory parts copied together, split over a few threads when large (a fresh array's
// pages are faulted in by whoever writes them first).
#pragma once
#include <algorithm>
#include <cstddef>
#include <cstring>
#include <thread>
#include <vector>

namespace pk
{

struct host_part
{
    char *dst;
    const char *src;
    size_t bytes;
};

inline void copy_parts(const std::vector<host_part> &parts)
{
    size_t total = 0;
    for (const host_part &p : parts) total += p.bytes;
    auto range = [&](size_t lo, size_t hi)
    {
        size_t at = 0;
        for (const host_part &p : parts)
        {
            const size_t a = std::max(lo, at), e = std::min(hi, at + p.bytes);
            if (a < e) std::memcpy(p.dst + (a - at), p.src + (a - at), e - a);
            at += p.bytes;
        }
    };
    const size_t n = std::min<size_t>(std::min<size_t>(8, std::thread::hardware_concurrency()), total >> 20);
    if (n < 2) return range(0, total);
    std::vector<std::thread> team;
    size_t done = 0; // parts given to threads
    // A thread that cannot start, for want of threads or of memory, is no error: what is left is
    // copied here, and the threads that did start are joined.
    try
    {
        team.reserve(n - 1);
        for (; done + 1 < n; ++done) team.emplace_back(range, total / n * done, total / n * (done + 1));
    }
    catch (...)
    {
    }
    range(total / n * done, total);
    for (std::thread &t : team) t.join();
}

} // namespace pk
