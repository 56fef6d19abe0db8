// Host test of the direct-LDS DGEMM kernels' index arithmetic
// (cosma_amd/csrc/dl_index.hpp), driven by tests/test_dl_index.py.
//
//   dl_index_test raster   workgroup -> tile is a bijection onto the tile grid,
//                          the 64-bit walk's, for every group_m that the tuning
//                          entry point takes
//   dl_index_test loads    every 16-byte load of the full k-steps ends inside
//                          the operand, at its tightest leading dimension, and
//                          together they take every element of a step
// Prints "ok <what>" / "FAIL <what>" lines; exit status 1 on any failure.
#include <algorithm>
#include <cstdint>
#include <cstdio>
#include <string>
#include <vector>

#include "dl_index.hpp"

namespace dl = cosma_amd::dl;

namespace {

int failures = 0;

void expect(bool ok, const std::string &what) {
    std::printf("%s %s\n", ok ? "ok" : "FAIL", what.c_str());
    if (!ok) ++failures;
}

// The same walk in 64 bits, for any group_m.
void walk64(int64_t block, int64_t tiles_m, int64_t tiles_n, int64_t group_m, int64_t &m, int64_t &n) {
    const int64_t blocks = tiles_m * tiles_n, xcd = block % 8;
    const int64_t bid = xcd * (blocks / 8) + std::min(xcd, blocks % 8) + block / 8;
    const int64_t grp = bid / (group_m * tiles_n), in_group = bid % (group_m * tiles_n);
    const int64_t rows = std::min(group_m, tiles_m - grp * group_m);
    m = grp * group_m + in_group % rows;
    n = in_group / rows;
}

bool every_tile_once(uint32_t tiles_m, uint32_t tiles_n, int group_m) {
    const uint32_t blocks = tiles_m * tiles_n;
    const uint32_t rows = (uint32_t)dl::clamp_group(group_m, tiles_m);
    if (rows * tiles_n == 0) return false;   // the walk would divide by zero
    std::vector<char> seen(blocks, 0);
    for (uint32_t b = 0; b < blocks; ++b) {
        const dl::TileAt t = dl::raster(b, blocks, tiles_m, tiles_n, rows);
        int64_t m, n;
        walk64(b, tiles_m, tiles_n, group_m, m, n);
        if (t.m != m || t.n != n || t.m >= tiles_m || t.n >= tiles_n || seen[t.m + (size_t)t.n * tiles_m]++) return false;
    }
    return true;
}

void run_raster() {
    const uint32_t grids[][2] = {{1, 1}, {8, 4}, {1, 1024}, {1024, 1}, {16, 64}, {4, 4096}, {37, 53}, {2897, 2895}};
    const int groups[] = {1, 2, 7, 8, 9, 36, 37, 1000, 1 << 20, 1 << 22, 1 << 26, (1 << 26) + 1, 1 << 30, 0x7fffffff};
    for (const auto &g : grids)
        for (int group_m : groups)
            expect(every_tile_once(g[0], g[1], group_m), "raster " + std::to_string(g[0]) + " x " + std::to_string(g[1]) +
                                                       " tiles, group_m " + std::to_string(group_m));
}

// Whether a 16-byte load of a full step reaches beyond the operand: rows r0 ..
// of an ext x K operand with the tightest leading dimension, `steps` steps.
// Counts the elements inside that are taken.
template <int R, bool KCONTIG, int NW>
bool beyond(int64_t ext, int64_t r0, int64_t K, int steps, int64_t &taken) {
    const int64_t ld = KCONTIG ? K : ext, end = KCONTIG ? (K - 1) + (ext - 1) * ld : (ext - 1) + (K - 1) * ld;
    const int last = dl::last_row<R>(ext, r0);
    bool out = false;
    for (int s = 0; s < steps; ++s) {
        std::vector<char> seen(R * dl::BK, 0);
        for (int wave = 0; wave < NW; ++wave)
            for (int lane = 0; lane < 64; ++lane)
                for (int q = 0; q < R / 8 / NW; ++q) {
                    // a row-contiguous operand's lane offset does not depend on q
                    const dl::Element e = dl::lane_load<R, KCONTIG, NW>(KCONTIG ? q : 0, wave, lane, last);
                    const int k = KCONTIG ? e.k : e.k + wave * dl::K_PER_WAVE<R> + q * dl::K_PER_ROUND<R, NW>;
                    const int64_t kk = (int64_t)s * dl::BK + k, row = r0 + e.row;
                    const int64_t at = KCONTIG ? kk + row * ld : row + kk * ld;
                    out |= k < 0 || k + (KCONTIG ? 1 : 0) >= dl::BK || e.row < 0 || row >= ext || at + 1 > end;
                    seen[e.row * dl::BK + k] = 1;
                    if (KCONTIG) seen[e.row * dl::BK + k + 1] = 1;
                    else if (e.row + 1 < R) seen[(e.row + 1) * dl::BK + k] = 1;
                }
        for (int r = 0; r <= last; ++r)
            for (int k = 0; k < dl::BK; ++k) taken += seen[r * dl::BK + k];
    }
    return out;
}

template <int R, bool KCONTIG, int NW>
void run_operand() {
    const std::string name = std::to_string(R) + (KCONTIG ? " k-contiguous, " : " row-contiguous, ") + std::to_string(NW) + " waves";
    bool inside = true, whole = true, hold_matters = false;
    for (int64_t ext : {1, 2, 3, 15, 16, 17, 31, 32, 33, 63, 64, 65, 100, 127, 128, 129, 255, 257})
        for (int64_t K = 1; K <= 50; ++K)
            for (int64_t r0 = 0; r0 < ext; r0 += R)
                for (int other = 0; other < 3; ++other) {   // the other operand: k-contiguous, row-contiguous even, odd
                    // this operand as A, then as B
                    const int64_t n = other == 2 ? 7 : 8;
                    const int steps = dl::full_steps(ext, n, K, KCONTIG, other == 0);
                    if (steps != dl::full_steps(n, ext, K, other == 0, KCONTIG)) whole = false;
                    if (K - (int64_t)steps * dl::BK < 0 || K - (int64_t)steps * dl::BK > dl::BK) whole = false;   // the partial step
                    int64_t taken = 0, unheld = 0;
                    inside &= !beyond<R, KCONTIG, NW>(ext, r0, K, steps, taken);
                    whole &= taken == (int64_t)steps * dl::BK * (dl::last_row<R>(ext, r0) + 1);
                    hold_matters |= beyond<R, KCONTIG, NW>(ext, r0, K, (int)(K / dl::BK), unheld);
                }
    expect(inside, "loads inside: " + name);
    expect(whole, "loads complete: " + name);
    // the check sees the over-read that holding back the last k prevents
    expect(hold_matters == !KCONTIG, "over-read seen: " + name);
}

void run_loads() {
    run_operand<128, true, 8>();
    run_operand<128, false, 8>();
    run_operand<128, true, 4>();
    run_operand<128, false, 4>();
    run_operand<64, true, 8>();
    run_operand<64, false, 8>();
    run_operand<64, true, 4>();
    run_operand<64, false, 4>();
    run_operand<32, true, 4>();
    run_operand<32, false, 4>();
}

}  // namespace

int main(int argc, char **argv) {
    const std::string what = argc > 1 ? argv[1] : "";
    if (what == "raster") run_raster();
    else if (what == "loads") run_loads();
    else return 2;
    return failures ? 1 : 0;
}
