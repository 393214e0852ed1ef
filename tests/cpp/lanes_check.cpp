// lane_offsets_fit (csrc/ftdma_lanes.h) against the offsets of every wave
// (test_host_checks.py).
#include "../../filtered_tdma_amd/csrc/ftdma_lanes.h"

#include <algorithm>
#include <cstdio>

// the largest offset from a wave's first lane, waves starting anywhere
static size_t spread(int nx, size_t pitch) {
    size_t most = 0;
    for (int first = 0; first < nx; ++first)
        for (int s = first; s < first + 64; ++s)
            most = std::max(most, (size_t)(s / nx) * pitch + 8 * (size_t)(s % nx) - 8 * (size_t)first);
    return most;
}

int main() {
    const size_t two32 = (size_t)1 << 32;
    for (int nx = 3; nx < 300; ++nx)
        for (size_t pitch = (nx + 17) * 8; pitch < 4 * two32; pitch += pitch / 7 + 8)
            if (ftd::lane_offsets_fit(nx, pitch) && spread(nx, pitch) >= two32) {
                std::printf("nx=%d pitch=%zu accepted\n", nx, pitch);
                return 1;
            }
    // planes of the y sweep: lines of nx + 2 values in whole 128 bytes, ny + 2 of them
    auto plane = [](size_t nx, size_t ny) { return (nx + 2 + 15) / 16 * 128 * (ny + 2); };
    if (ftd::lane_offsets_fit(524288, plane(524288, 1024)) ||       // 4.3 GB
        !ftd::lane_offsets_fit(500000, plane(500000, 1024)) ||      // 4.1 GB
        !ftd::lane_offsets_fit(1 << 28, plane(1 << 28, 0) / 2)) {   // a line of 2 GiB
        std::puts("planes");
        return 1;
    }
    for (int n = 3; n <= 4096; ++n)
        if (!ftd::lane_offsets_fit(n, plane(n, 1024))) {
            std::puts("ordinary");
            return 1;
        }
    std::puts("ok");
    return 0;
}
