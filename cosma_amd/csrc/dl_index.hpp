// Index arithmetic of the direct-LDS DGEMM kernels (dgemm_dl.hip): the tile that
// a workgroup takes and the elements that a lane loads.  Plain constexpr
// functions of integers (callable on both sides), so that a host test can walk
// every workgroup, lane and step of a shape.
#pragma once
#include <cstdint>

namespace cosma_amd {
namespace dl {

constexpr int BK = 16;       // k-step
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

// ---- loads of one operand tile: R rows, k-contiguous or row-contiguous, NW waves
// Last row of the tile at r0 inside the matrix.
template <int R>
constexpr int last_row(int64_t ext, int64_t r0) {
    return (int)(ext - 1 - r0 < R - 1 ? ext - 1 - r0 : R - 1);
}
// Slot (of eight) of k-pair kp in row r of a k-contiguous tile is kp ^ row_swz(r).
constexpr int row_swz(int r) { return ((r >> 2) & 3) | ((r & 2) << 1); }
// The first of the two elements that a lane's 16-byte load q takes (the second
// is the next k of a k-contiguous operand, else the next row).  A row-contiguous
// operand's k counts from wave * K_PER_WAVE + q * K_PER_ROUND.
struct Element {
    int row, k;
};
template <int R>
constexpr int K_PER_WAVE = 128 / R;
template <int R, int NW>
constexpr int K_PER_ROUND = 128 * NW / R;
template <int R, bool KCONTIG, int NW>
constexpr Element lane_load(int q, int wave, int lane, int last) {
    if (KCONTIG) {
        const int row = 8 * (wave + NW * q) + (lane >> 3);
        return {row < last ? row : last, 2 * ((lane & 7) ^ row_swz(row))};
    }
    const int e = 2 * lane;                                  // position in the 128 doubles of an instruction
    const int odd_kp = R == 128 ? (wave >> 1) & 1 : R == 64 ? wave & 1 : lane >> 5;
    const int row = (e % R) ^ (16 * odd_kp);
    return {row < (last & ~1) ? row : last & ~1, e / R};
}

// Full k-steps.  A row-contiguous operand with an odd extent keeps the last k
// out of them: the 16-byte load of its last row reads one element beyond the
// row, which only inside the matrix is the next column's.
constexpr int full_steps(int64_t M, int64_t N, int64_t K, bool a_kcontig, bool b_kcontig) {
    const bool hold_last = (!a_kcontig && (M & 1)) || (!b_kcontig && (N & 1));
    return (int)((hold_last ? K - 1 : K) / BK);
}

}  // namespace dl
}  // namespace cosma_amd
