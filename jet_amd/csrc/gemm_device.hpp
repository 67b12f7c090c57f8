// gemm_device.hpp -- device helpers shared by the GEMM kernel files (gfx950).
#pragma once

#include "common.hpp"

#include <cstdint>

namespace jet_hip {

// Map the linear work-group id to an output tile.  Work-groups are dispatched
// round-robin over the 8 XCDs (each with its own L2), so first give every XCD
// a contiguous range of tile indices, then order tiles in groups of
// kGroupM tile-rows so that the work-groups resident on one XCD share A and B
// panels in its L2.
constexpr int kXcds = 8;
constexpr int kGroupM = 8;

__device__ __forceinline__ void tile_coords(int64_t id, int64_t tiles_m, int64_t tiles_n,
                                            int64_t &tm, int64_t &tn)
{
    const int64_t total = tiles_m * tiles_n;
    const int64_t q = total / kXcds, r = total % kXcds;
    const int64_t x = id % kXcds, k = id / kXcds;
    const int64_t j = x * q + (x < r ? x : r) + k;
    const int64_t per_group = int64_t(kGroupM) * tiles_n;
    const int64_t group = j / per_group;
    const int64_t first_m = group * kGroupM;
    const int64_t gsz = (tiles_m - first_m) < kGroupM ? (tiles_m - first_m) : kGroupM;
    const int64_t w = j % per_group;
    tm = first_m + w % gsz;
    tn = w / gsz;
}

} // namespace jet_hip
