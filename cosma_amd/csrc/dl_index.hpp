// Index arithmetic of the direct-LDS DGEMM kernels (dgemm_dl.hip): the tile that
// a workgroup takes.  Plain constexpr functions of integers (callable on both
// sides), so that a host test can walk every workgroup of a launch.
#pragma once
#include <cstdint>

namespace cosma_amd {
namespace dl {

constexpr int NXCD = 8;

// ---- tile rasterisation: XCD-aware, group_m rows of tiles walked before moving along n
struct TileAt {
    uint32_t m, n;
};
// group_m in [1, tiles_m], so that no product here exceeds the number of tiles.
constexpr TileAt raster(uint32_t block, uint32_t blocks, uint32_t tiles_m, uint32_t tiles_n, uint32_t group_m) {
    const uint32_t q8 = blocks / NXCD, r8 = blocks % NXCD, xcd = block % NXCD, loc = block / NXCD;
    const uint32_t bid = xcd * q8 + (xcd < r8 ? xcd : r8) + loc;
    const uint32_t per_group = group_m * tiles_n, grp = bid / per_group, in_group = bid - grp * per_group;
    const uint32_t rest = tiles_m - grp * group_m, gsize = group_m < rest ? group_m : rest;
    return {grp * group_m + in_group % gsize, in_group / gsize};
}

// The group of a launch: a larger one walks the same way as tiles_m rows.
constexpr int clamp_group(int group_m, int64_t tiles_m) { return group_m < tiles_m ? group_m : (int)tiles_m; }

}  // namespace dl
}  // namespace cosma_amd
