// run_parts (csrc/ftdma_threads.h): every part runs once and the call returns,
// also where the memory for a thread cannot be had (test_host_checks.py).
#include "../../filtered_tdma_amd/csrc/ftdma_threads.h"

#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <new>

static std::atomic<int> g_left{-1};  // allocations until one fails; -1: none does

void* operator new(std::size_t n) {
    if (g_left.load() >= 0 && g_left.fetch_sub(1) == 0) throw std::bad_alloc();
    if (void* p = std::malloc(n ? n : 1)) return p;
    throw std::bad_alloc();
}
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, std::size_t) noexcept { std::free(p); }

int main() {
    for (int fail = -1; fail < 6; ++fail) {
        std::atomic<int> ran[6] = {};
        g_left = fail;
        ftd::run_parts<6>([&](int t) { ++ran[t]; });
        g_left = -1;
        for (int t = 0; t < 6; ++t)
            if (ran[t] != 1) {
                std::printf("fail=%d part=%d ran %d times\n", fail, t, ran[t].load());
                return 1;
            }
    }
    std::puts("ok");
    return 0;
}
