// for_parts where the host runs out of memory at its n-th allocation: every
// part is done, or the error is thrown with none running; the process goes on.
#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <new>

#include "dtb_parts.hpp"

namespace {
std::atomic<int> g_left{-1};   // allocations until one fails (-1: none does)
}

void *operator new(std::size_t n)
{
    if (g_left >= 0 && g_left-- == 0)
        throw std::bad_alloc();
    if (void *p = std::malloc(n ? n : 1))
        return p;
    throw std::bad_alloc();
}
void operator delete(void *p) noexcept { std::free(p); }
void operator delete(void *p, std::size_t) noexcept { std::free(p); }

int main()
{
    int whole = 0, thrown = 0;
    for (int n = 0; n < 24; ++n) {
        std::atomic<int> done[8] = {};
        g_left = n;
        bool all = true;
        try {
            dtb::for_parts(8, [&](uint32_t k) { ++done[k]; });
        } catch (const std::bad_alloc &) {
            all = false;
        }
        g_left = -1;
        for (auto &d : done)
            if (d != (all ? 1 : 0)) {
                std::printf("allocation %d: a part ran %d times\n", n, (int)d);
                return 1;
            }
        ++(all ? whole : thrown);
    }
    // an error in a part reaches the caller after all parts ended
    std::atomic<int> ran{0};
    try {
        dtb::for_parts(8, [&](uint32_t k) {
            ++ran;
            if (k == 5)
                throw 7;
        });
        return 1;
    } catch (int) {
    }
    std::puts(whole > 8 && thrown > 0 && ran == 8 ? "ok" : "counts");
    return 0;
}
