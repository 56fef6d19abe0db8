// The direct-LDS DGEMM kernels (dgemm_dl.hip): tile shapes and launch.
#pragma once
#include "common.hpp"

namespace cosma_amd {

enum DlTile { DL_128x128, DL_64x128, DL_64x64, DL_64x32, DL_32x32 };

// Whether the kernels can address the problem.
bool dl_fits(int64_t m, int64_t n, int64_t k, int64_t lda, int64_t ldb);
// The tile expected to be fastest (all give bit-identical results).
DlTile pick_dl_tile(int64_t m, int64_t n, int64_t k);
int launch_dl(DlTile tile, char ta, char tb, int64_t m, int64_t n, int64_t k, double alpha, const double *a,
              int64_t lda, const double *b, int64_t ldb, double beta, double *c, int64_t ldc, int group_m,
              hipStream_t s);

// Grouped tiles with the same kernels: cfg 1, 2, 3, 5 (grouped_tile_shape); the
// descriptors are followed by their tile starts and the owner of every tile.
// trans: the transposes (flags & 3) that all problems share, else 4.
int launch_grouped_dl(int cfg, const GroupedProblem *probs, int nprob, int64_t total_tiles, int grid, int trans,
                      hipStream_t s);

// Grouped launches walk virtual tile ids v = blockIdx.x + i * gridDim.x; the
// hardware places workgroup b on XCD b % 8.  Consecutive tiles (of one
// problem, which share A and B panels) are kept on one XCD and its L2 by
// handing out chunks of GROUP_CHUNK consecutive tiles: XCD x takes chunks x,
// x + 8, x + 16, ... in dispatch order, so the decreasing-cost order of the
// problems is kept at chunk granularity.  Bijective on [0, T): ids beyond
// the last whole round of 8 chunks map to themselves.
constexpr int64_t GROUP_CHUNK = 32;
__device__ __forceinline__ int64_t grouped_tile_of(int64_t v, int64_t T) {
    constexpr int64_t NXCD = 8, span = NXCD * GROUP_CHUNK;
    if (v >= T / span * span) return v;
    const int64_t xcd = v % NXCD, local = v / NXCD;
    return ((local / GROUP_CHUNK) * NXCD + xcd) * GROUP_CHUNK + local % GROUP_CHUNK;
}

}  // namespace cosma_amd
