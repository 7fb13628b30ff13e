// copy_parts (physkit_amd/csrc/pk_copy.hpp) where a thread cannot start: operator new throws
// from its `fail`-th call on, so the thread's state (or the list of threads) cannot be
// allocated. The copy is whole all the same, with every started thread joined.
#include "pk_copy.hpp"

#include <cstdio>
#include <cstdlib>
#include <new>

static long calls_left = -1; // -1: never fail

void *operator new(std::size_t n)
{
    if (calls_left == 0) throw std::bad_alloc();
    if (calls_left > 0) --calls_left;
    if (void *p = std::malloc(n ? n : 1)) return p;
    throw std::bad_alloc();
}
void operator delete(void *p) noexcept { std::free(p); }
void operator delete(void *p, std::size_t) noexcept { std::free(p); }

int main()
{
    const size_t sizes[3] = {5 << 20, 1, (3 << 20) + 17};
    for (long fail = -1; fail < 12; ++fail)
    {
        std::vector<std::vector<char>> src, dst;
        std::vector<pk::host_part> parts;
        for (size_t n : sizes)
        {
            src.emplace_back(n);
            dst.emplace_back(n);
            for (size_t i = 0; i < n; ++i) src.back()[i] = static_cast<char>(i * 2654435761u >> 13);
        }
        for (size_t k = 0; k < src.size(); ++k) parts.push_back({dst[k].data(), src[k].data(), src[k].size()});
        calls_left = fail;
        pk::copy_parts(parts);
        calls_left = -1;
        if (src != dst) return std::printf("parts differ at fail %ld\n", fail), 1;
    }
    std::printf("copy_parts ok\n");
    return 0;
}
