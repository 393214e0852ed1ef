// ftdma_lanes.h -- whether a wave's lanes are within 32 bits of its first
// one's cell in the heat sweeps along y and z (internal, host only).
#pragma once

#include <stddef.h>
#include <stdint.h>

namespace ftd {

// The 64 lanes of a wave hold consecutive systems, nx to a run, the next run
// `pitch` bytes on: a line in the z sweep, a plane in the y sweep.
inline bool lane_offsets_fit(int nx, size_t pitch) {
    const size_t runs = (63 + (size_t)nx - 1) / nx;  // crossed by 64 systems at most
    return runs * pitch + sizeof(double) * (size_t)(nx < 64 ? nx : 64) <= UINT32_MAX;
}

}  // namespace ftd
