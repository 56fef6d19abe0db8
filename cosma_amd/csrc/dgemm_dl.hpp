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

}  // namespace cosma_amd
