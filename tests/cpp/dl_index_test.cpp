// Host test of the direct-LDS DGEMM kernels' index arithmetic
// (cosma_amd/csrc/dl_index.hpp), driven by tests/test_dl_index.py.
//
//   dl_index_test raster   workgroup -> tile is a bijection onto the tile grid,
//                          the 64-bit walk's, for every group_m that the tuning
//                          entry point takes
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

}  // namespace

int main(int argc, char **argv) {
    const std::string what = argc > 1 ? argv[1] : "";
    if (what == "raster") run_raster();
    else return 2;
    return failures ? 1 : 0;
}
