// fft_make (csrc/ftdma_fft.h) over a hipFFT of this file's own in which each
// call fails in turn: the pair is ready only with both plans made and set to the
// stream, a failed attempt leaves no plan, and the next attempt works
// (test_host_checks.py).
#include "../../filtered_tdma_amd/csrc/ftdma_fft.h"

#include <cstdio>
#include <map>

static int g_calls = 0, g_fail = -1;
static std::map<hipfftHandle, hipStream_t> g_plans;  // live plans and their streams

static hipfftResult next() { return g_calls++ == g_fail ? HIPFFT_INTERNAL_ERROR : HIPFFT_SUCCESS; }

extern "C" {
hipfftResult hipfftPlanMany(hipfftHandle* plan, int, int*, int*, int, int, int*, int, int,
                            hipfftType, int) {
    static size_t made = 0;
    if (next() != HIPFFT_SUCCESS) return HIPFFT_ALLOC_FAILED;
    *plan = (hipfftHandle)(++made * 64);
    g_plans[*plan] = nullptr;
    return HIPFFT_SUCCESS;
}
hipfftResult hipfftSetStream(hipfftHandle plan, hipStream_t s) {
    if (next() != HIPFFT_SUCCESS) return HIPFFT_INTERNAL_ERROR;
    g_plans.at(plan) = s;
    return HIPFFT_SUCCESS;
}
hipfftResult hipfftDestroy(hipfftHandle plan) {
    return g_plans.erase(plan) == 1 ? HIPFFT_SUCCESS : HIPFFT_INVALID_PLAN;
}
}

int main() {
    const hipStream_t stream = (hipStream_t)0x40;
    for (int fail = 0; fail < 4; ++fail) {
        ftd::FftPair p;
        g_calls = 0;
        g_fail = fail;
        const bool said = ftd::fft_make(p, 8, 6, 5, 5, stream) != nullptr;
        if (!said || p.ready || !g_plans.empty()) {
            std::printf("call %d failed: said=%d ready=%d plans left=%zu\n", fail, said, p.ready,
                        g_plans.size());
            return 1;
        }
        g_fail = -1;
        if (ftd::fft_make(p, 8, 6, 5, 5, stream) || !p.ready || g_plans.size() != 2 ||
            g_plans.at(p.fwd) != stream || g_plans.at(p.bwd) != stream) {
            std::printf("after call %d failed: no ready pair on the stream\n", fail);
            return 1;
        }
        ftd::fft_free(p);
        if (!g_plans.empty()) return 1;
    }
    std::puts("ok");
    return 0;
}
