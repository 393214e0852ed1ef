// ftdma_fft.h -- a pair of 2-D FFT plans of the channel solver (internal, host
// only).
#pragma once

#include <hipfft/hipfft.h>

namespace ftd {

// Real [ny][nx] to lines of `pitch` complex modes and back, nz planes at once.
struct FftPair {
    hipfftHandle fwd = 0, bwd = 0;
    bool ready = false;  // both made, and set to the stream
};

inline void fft_free(FftPair& p) {
    if (p.fwd) (void)hipfftDestroy(p.fwd);
    if (p.bwd) (void)hipfftDestroy(p.bwd);
    p = FftPair{};
}

// nullptr, or what failed: then no plan is left, and the next call makes them
inline const char* fft_make(FftPair& p, int nx, int ny, int nz, int pitch, hipStream_t stream) {
    if (p.ready) return nullptr;
    int n2[2] = {ny, nx}, real[2] = {ny, nx}, modes[2] = {ny, pitch};
    const int dr = nx * ny, dm = pitch * ny;
    const char* failed = nullptr;
    if (hipfftPlanMany(&p.fwd, 2, n2, real, 1, dr, modes, 1, dm, HIPFFT_D2Z, nz) !=
        HIPFFT_SUCCESS) {
        p.fwd = 0;
        failed = "hipfftPlanMany (D2Z) failed";
    } else if (hipfftPlanMany(&p.bwd, 2, n2, modes, 1, dm, real, 1, dr, HIPFFT_Z2D, nz) !=
               HIPFFT_SUCCESS) {
        p.bwd = 0;
        failed = "hipfftPlanMany (Z2D) failed";
    } else if (hipfftSetStream(p.fwd, stream) != HIPFFT_SUCCESS ||
               hipfftSetStream(p.bwd, stream) != HIPFFT_SUCCESS) {
        failed = "hipfftSetStream failed";
    }
    if (failed)
        fft_free(p);
    else
        p.ready = true;
    return failed;
}

}  // namespace ftd
