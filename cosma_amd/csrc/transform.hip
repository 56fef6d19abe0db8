// Local block transform: dst <- alpha * op(src) + beta * dst (column-major).
//
// Replaces COSTA's local block copy/transpose (costa::memory::copy_and_transpose,
// call site benchmarks/transpose.cpp:46-47) and the per-block alpha/beta update
// that costa::transformer applies when COSMA reshuffles operands between the
// ScaLAPACK layout and its own (src/cosma/cosma_pxgemm.cpp:338-364,
// src/cosma/multiply.cpp:186-204).  On one rank a ScaLAPACK block-cyclic local
// array is the global matrix in column-major order with leading dimension lld
// (numroc with one process returns the full extent, src/cosma/scalapack.cpp:49-87),
// so the reorder reduces to this strided copy / transpose.
//
// The bound is HBM.  With a leading dimension that is no multiple of 16 the
// columns of dst start anywhere in a 128-byte line, and the lines at the ends
// of a tile's column runs are written in parts by two workgroups.  So the
// copies and the large transposes give every column of dst its own row
// window, which starts where a line does, and use 16-byte accesses at the
// 8-byte alignment of a double (8191 x 12289, ld 12291 / 8193: 'T' 421 us
// element by element, 358 us in 16-byte accesses, 283 us in shifted windows =
// 5.7 TB/s; 'N' 351 -> 250 us = 6.4 TB/s).
//
// op = 'N': a workgroup covers 512 rows of one or two columns, a thread two
//           consecutive doubles of each.
// op = 'T': tiles staged through LDS (odd row pitch, so that the column reads
//           spread over all banks): read along src columns, written along dst
//           columns.  Three forms: operands that the last-level cache holds in
//           64 x 64 tiles (with aligned pointers and even leading dimensions
//           16-byte accesses, and several tiles per workgroup, the next loaded
//           during the stores of the current one); larger ones in shifted
//           windows, which need 16 more src columns than they write rows (the
//           next tile's too, from L2: their loads are cached); and larger ones
//           with all columns in whole lines in 128 x 64 tiles that stream past
//           the caches on both sides.
// alpha == 1 and beta == 0 copies values bit-for-bit (no arithmetic at all);
// beta == 0 never reads dst.
#include "common.hpp"

namespace cosma_amd {
namespace {

constexpr int LINE = 16;     // doubles per 128-byte line
constexpr int NT = 256;      // threads per workgroup

typedef double f64x2u __attribute__((ext_vector_type(2), aligned(8)));

__device__ __forceinline__ double combine(double x, double alpha, double beta, const double *d, int mode) {
    // mode 0: pure copy; 1: alpha*x (dst not read); 2: alpha*x + beta*dst
    if (mode == 0) return x;
    if (mode == 1) return alpha * x;
    return fma(beta, *d, alpha * x);
}
__device__ __forceinline__ f64x2u combine2(f64x2u x, double alpha, double beta, f64x2u old, int mode) {
    if (mode == 0) return x;
    if (mode == 1) return f64x2u{alpha * x.x, alpha * x.y};
    return f64x2u{fma(beta, old.x, alpha * x.x), fma(beta, old.y, alpha * x.y)};
}
// Position of an element in its 128-byte line.
__device__ __forceinline__ int phase(const double *p) { return (int)(reinterpret_cast<uintptr_t>(p) >> 3) & (LINE - 1); }

// 16-byte load, streaming past the caches or not.
template <bool NONTEMPORAL>
__device__ __forceinline__ f64x2u load2(const double *p) {
    const f64x2u *q = reinterpret_cast<const f64x2u *>(p);
    return NONTEMPORAL ? __builtin_nontemporal_load(q) : *q;
}

// dst(rows x cols) <- f(src(rows x cols)).  Grid: x over 512-row windows, y
// over groups of U columns.  SHIFT: row windows by dst's lines.  SRC_NT,
// DST_NT: loads that stream past the caches (streamed()); the stores always do.
// U pieces per thread are loaded before one is stored: two, but one where all
// streams, except from short columns and from so many that a workgroup walks
// several (10000 x 13400, beta = 1/2: 539 and 518 us; 300 x 446666: 564 and 620 us).
template <bool SHIFT, bool SRC_NT, bool DST_NT, int U>
__global__ __launch_bounds__(NT) void copy_kernel(int64_t rows, int64_t cols, double alpha,
                                                  const double *__restrict__ src, int64_t lds, double beta,
                                                  double *__restrict__ dst, int64_t ldd, int mode) {
    const int64_t r0 = 2 * ((int64_t)blockIdx.x * NT + threadIdx.x);
    if (r0 - (SHIFT ? LINE - 1 : 0) >= rows) return;   // no row of any column (3 x 300000: 84 us with these waves in the loop, 59 us)
    for (int64_t c0 = U * (int64_t)blockIdx.y; c0 < cols; c0 += U * (int64_t)gridDim.y) {
        f64x2u v[U], old[U];
        int64_t r[U];
        bool in[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int64_t c = c0 + u;
            r[u] = r0 - (SHIFT ? phase(dst + c * ldd) : 0);
            in[u] = c < cols && r[u] >= 0 && r[u] + 1 < rows;
            if (!in[u]) continue;
            v[u] = load2<SRC_NT>(src + r[u] + c * lds);
            if (mode == 2) old[u] = load2<DST_NT>(dst + r[u] + c * ldd);
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int64_t c = c0 + u;
            double *d = dst + r[u] + c * ldd;
            if (in[u]) {
                __builtin_nontemporal_store(combine2(v[u], alpha, beta, old[u], mode), reinterpret_cast<f64x2u *>(d));
            } else if (c < cols) {
                const double *q = src + r[u] + c * lds;
                if (r[u] >= 0 && r[u] < rows) d[0] = combine(q[0], alpha, beta, d, mode);
                if (r[u] + 1 >= 0 && r[u] + 1 < rows) d[1] = combine(q[1], alpha, beta, d + 1, mode);
            }
        }
    }
}

// The same for many blocks in one launch: a workgroup takes 2048 consecutive
// pairs of one block (row pairs of its columns, columns one after another).
// The block list travels in the kernel arguments: nothing to allocate, upload
// or keep alive.
constexpr int LIST = 72;     // blocks per launch (3.5 KB of the 4 KB of arguments)
constexpr int ITEMS = 8;     // pairs per thread
constexpr int64_t LIST_PAIRS = 1 << 26;   // most pairs of one block
struct BlockList {
    struct {
        const double *src;
        double *dst;
        int64_t lds, ldd;
        int rows, cols;
        uint32_t first;      // first workgroup
        uint32_t pairs;      // row pairs per column, with the window's shift
    } b[LIST];
    int n;
};
template <bool SRC_NT, bool DST_NT>
__global__ __launch_bounds__(NT) void copy_list_kernel(BlockList list, double alpha, double beta, int mode) {
    int lo = 0, hi = list.n - 1;   // last block with first <= this workgroup
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (list.b[mid].first <= blockIdx.x) lo = mid;
        else hi = mid - 1;
    }
    const double *__restrict__ src = list.b[lo].src;
    double *__restrict__ dst = list.b[lo].dst;
    const int64_t lds = list.b[lo].lds, ldd = list.b[lo].ldd;
    const int rows = list.b[lo].rows, cols = list.b[lo].cols;
    const uint32_t pairs = list.b[lo].pairs, base = (blockIdx.x - list.b[lo].first) * (NT * ITEMS) + threadIdx.x;
    f64x2u v[ITEMS], old[ITEMS];
    int r[ITEMS], c[ITEMS];
    bool in[ITEMS];
#pragma unroll
    for (int q = 0; q < ITEMS; ++q) {
        const uint32_t idx = base + NT * q;
        c[q] = (int)min(idx / pairs, (uint32_t)cols);
        r[q] = (int)(2 * (idx - (uint32_t)c[q] * pairs)) - phase(dst + c[q] * ldd);
        in[q] = c[q] < cols && r[q] >= 0 && r[q] + 1 < rows;
        if (!in[q]) continue;
        v[q] = load2<SRC_NT>(src + r[q] + c[q] * lds);
        if (mode == 2) old[q] = load2<DST_NT>(dst + r[q] + c[q] * ldd);
    }
#pragma unroll
    for (int q = 0; q < ITEMS; ++q) {
        double *d = dst + r[q] + c[q] * ldd;
        if (in[q]) {
            __builtin_nontemporal_store(combine2(v[q], alpha, beta, old[q], mode), reinterpret_cast<f64x2u *>(d));
        } else if (c[q] < cols) {
            const double *s = src + r[q] + c[q] * lds;
            if (r[q] >= 0 && r[q] < rows) d[0] = combine(s[0], alpha, beta, d, mode);
            if (r[q] + 1 >= 0 && r[q] + 1 < rows) d[1] = combine(s[1], alpha, beta, d + 1, mode);
        }
    }
}

constexpr int TT = 64;       // edge of the cached kernels' tiles

// dst(rows x cols)[i, j] <- f(src[j, i]); src is cols x rows with leading dim lds.
// blockIdx.x -> 64-row block of dst (= 64-column block of src),
// blockIdx.y -> 64-column block of dst (= 64-row block of src).
__global__ __launch_bounds__(NT) void transpose_cached_kernel(int64_t rows, int64_t cols, double alpha,
                                                        const double *__restrict__ src, int64_t lds,
                                                        double beta, double *__restrict__ dst,
                                                        int64_t ldd, int mode) {
    __shared__ double tile[TT][TT + 1];
    const int tx = threadIdx.x & 63, ty = threadIdx.x >> 6;
    const int64_t i0 = (int64_t)blockIdx.x * TT;   // dst rows / src cols
    for (int64_t j0 = (int64_t)blockIdx.y * TT; j0 < cols; j0 += (int64_t)gridDim.y * TT) {
        // read: src rows j0+tx (contiguous), src cols i0+ty+4r
#pragma unroll
        for (int r = 0; r < TT / 4; ++r) {
            const int il = ty + 4 * r;
            const int64_t i = i0 + il, j = j0 + tx;
            if (i < rows && j < cols) tile[il][tx] = src[j + i * lds];
        }
        __syncthreads();
        // write: dst rows i0+tx (contiguous), dst cols j0+ty+4r
#pragma unroll
        for (int r = 0; r < TT / 4; ++r) {
            const int jl = ty + 4 * r;
            const int64_t i = i0 + tx, j = j0 + jl;
            if (i < rows && j < cols) {
                double *d = dst + i + j * ldd;
                *d = combine(tile[tx][jl], alpha, beta, d, mode);
            }
        }
        __syncthreads();
    }
}

// Same transpose with 16-byte global accesses: every load takes two
// consecutive src elements of one src column, every store writes two
// consecutive dst elements of one dst column.  Needs 16-byte aligned
// pointers and even leading dimensions; tiles that cross the matrix edge take
// the element-wise path.
__global__ __launch_bounds__(NT) void transpose_cached_vec_kernel(int64_t rows, int64_t cols, double alpha,
                                                            const double *__restrict__ src, int64_t lds,
                                                            double beta, double *__restrict__ dst,
                                                            int64_t ldd, int mode) {
    __shared__ double tile[TT][TT + 1];
    const int t = threadIdx.x;
    const int64_t i0 = (int64_t)blockIdx.x * TT;   // dst rows / src cols
    const int64_t jstep = (int64_t)gridDim.y * TT;
    auto full = [&](int64_t j0) { return (i0 + TT <= rows) && (j0 + TT <= cols); };
    // src column i0 + il, rows j0 + c2, c2 + 1
    auto load = [&](int64_t j0, f64x2 (&v)[8]) {
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            const int idx = t + NT * q, il = idx >> 5, c2 = (idx & 31) * 2;
            v[q] = __builtin_nontemporal_load(reinterpret_cast<const f64x2 *>(src + (j0 + c2) + (i0 + il) * lds));
        }
    };
    // A workgroup walks the tiles j0, j0 + jstep, ... of its column of
    // tiles; the loads of the next full tile are issued right after the
    // current one is in LDS, so they are in flight during its stores.
    f64x2 v[8];
    int64_t j0 = (int64_t)blockIdx.y * TT;
    if (j0 < cols && full(j0)) load(j0, v);
    for (; j0 < cols; j0 += jstep) {
        if (full(j0)) {
#pragma unroll
            for (int q = 0; q < 8; ++q) {
                const int idx = t + NT * q, il = idx >> 5, c2 = (idx & 31) * 2;
                tile[il][c2] = v[q].x;
                tile[il][c2 + 1] = v[q].y;
            }
            __syncthreads();
            if (j0 + jstep < cols && full(j0 + jstep)) load(j0 + jstep, v);
#pragma unroll
            for (int q = 0; q < 8; ++q) {     // dst column j0 + jl, rows i0 + r2, r2 + 1
                const int idx = t + NT * q, jl = idx >> 5, r2 = (idx & 31) * 2;
                f64x2 *d = reinterpret_cast<f64x2 *>(dst + (i0 + r2) + (j0 + jl) * ldd);
                f64x2 o;
                if (mode == 0) {
                    o.x = tile[r2][jl];
                    o.y = tile[r2 + 1][jl];
                } else if (mode == 1) {
                    o.x = alpha * tile[r2][jl];
                    o.y = alpha * tile[r2 + 1][jl];
                } else {
                    const f64x2 old = *d;
                    o.x = fma(beta, old.x, alpha * tile[r2][jl]);
                    o.y = fma(beta, old.y, alpha * tile[r2 + 1][jl]);
                }
                __builtin_nontemporal_store(o, d);
            }
        } else {
            const int tx = t & 63, ty = t >> 6;
#pragma unroll
            for (int r = 0; r < TT / 4; ++r) {
                const int il = ty + 4 * r;
                const int64_t i = i0 + il, j = j0 + tx;
                if (i < rows && j < cols) tile[il][tx] = src[j + i * lds];
            }
            __syncthreads();
            if (j0 + jstep < cols && full(j0 + jstep)) load(j0 + jstep, v);
#pragma unroll
            for (int r = 0; r < TT / 4; ++r) {
                const int jl = ty + 4 * r;
                const int64_t i = i0 + tx, j = j0 + jl;
                if (i < rows && j < cols) {
                    double *d = dst + i + j * ldd;
                    *d = combine(tile[tx][jl], alpha, beta, d, mode);
                }
            }
        }
        __syncthreads();
    }
}

// dst(rows x cols)[i, j] <- f(src[j, i]); src is cols x rows with leading dim
// lds.  Tiles of TR dst rows x TC dst columns, SHIFT: each column's rows start
// at its own line boundary at or up to 15 rows after the tile's first.  BETA:
// dst is read (mode 2), by loads in flight together with those of src.
template <int TR, int TC, bool SHIFT, bool BETA>
__global__ __launch_bounds__(NT) void transpose_kernel(int64_t rows, int64_t cols, double alpha,
                                                       const double *__restrict__ src, int64_t lds,
                                                       double beta, double *__restrict__ dst,
                                                       int64_t ldd, int mode, uint32_t nx, uint32_t tiles) {
    constexpr int S = SHIFT ? LINE : 0, LR = TR + S, H = TC / 2;
    static_assert(TR % LINE == 0 && LR * H % NT == 0 && TR * TC % (2 * NT) == 0 && LR * TC % NT == 0, "whole rounds of the workgroup");
    __shared__ double tile[LR][TC + 1];
    const int t = threadIdx.x;
    for (uint32_t b = blockIdx.x; b < tiles; b += gridDim.x) {
        const int64_t i0 = (int64_t)(b % nx) * TR - S, j0 = (int64_t)(b / nx) * TC;
        auto shift = [&](const double *col) { return SHIFT ? (LINE - phase(col)) & (LINE - 1) : 0; };
        if (i0 >= 0 && i0 + LR <= rows && j0 + TC <= cols) {
            constexpr int OUT = TR * TC / 2 / NT;
            f64x2u v[LR * H / NT], old[OUT];
            auto dst_pair = [&](int q, int &jl, int &r) {
                const int e = t + NT * q;
                jl = e / (TR / 2);
                double *col = dst + (j0 + jl) * ldd + i0;
                r = (e % (TR / 2)) * 2 + shift(col);
                return reinterpret_cast<f64x2u *>(col + r);
            };
#pragma unroll
            for (int q = 0; q < LR * H / NT; ++q) {
                const int e = t + NT * q, il = e / H, c2 = (e % H) * 2;
                const f64x2u *p = reinterpret_cast<const f64x2u *>(src + (j0 + c2) + (i0 + il) * lds);
                v[q] = SHIFT ? *p : __builtin_nontemporal_load(p);
            }
            if (BETA) {
#pragma unroll
                for (int q = 0; q < OUT; ++q) {
                    int jl, r;
                    old[q] = *dst_pair(q, jl, r);
                }
            }
#pragma unroll
            for (int q = 0; q < LR * H / NT; ++q) {
                const int e = t + NT * q, il = e / H, c2 = (e % H) * 2;
                tile[il][c2] = v[q].x;
                tile[il][c2 + 1] = v[q].y;
            }
            __syncthreads();
#pragma unroll
            for (int q = 0; q < OUT; ++q) {
                int jl, r;
                f64x2u *d = dst_pair(q, jl, r);
                __builtin_nontemporal_store(combine2(f64x2u{tile[r][jl], tile[r + 1][jl]}, alpha, beta, old[q], BETA ? 2 : mode), d);
            }
        } else {
            // Edge tile: by element, from addresses clamped into the matrix so
            // that a batch of loads is in flight together (one element at a time, two edge
            // tiles in 24 made 2601 x 12501 take 308 us with beta = 1/2, 177 us in
            // batches of 8, 152 us in one; without beta, whose tiles need fewer
            // registers, batches keep 8191 x 12289 at 283 us, one batch 322 us).
            constexpr int IN = LR * TC / NT, OUT = TR * TC / NT;
            constexpr int UI = BETA ? IN : 8, UO = BETA ? OUT : OUT % 7 == 0 ? 7 : 8;   // loads per batch
            static_assert(IN % UI == 0 && OUT % UO == 0, "whole batches");
#pragma unroll 1
            for (int e0 = t; e0 < LR * TC; e0 += NT * UI) {
                double v[UI];
#pragma unroll
                for (int q = 0; q < UI; ++q) {
                    const int e = e0 + NT * q;
                    const int64_t i = min(max(i0 + e / TC, (int64_t)0), rows - 1), j = min(j0 + e % TC, cols - 1);
                    v[q] = src[j + i * lds];
                }
#pragma unroll
                for (int q = 0; q < UI; ++q) tile[(e0 + NT * q) / TC][(e0 + NT * q) % TC] = v[q];
            }
            __syncthreads();
#pragma unroll 1
            for (int e0 = t; e0 < TR * TC; e0 += NT * UO) {
                double old[UO];
#pragma unroll
                for (int q = 0; q < UO; ++q) {
                    const int e = e0 + NT * q;
                    double *col = dst + min(j0 + e / TR, cols - 1) * ldd;
                    old[q] = BETA ? col[min(max(i0 + e % TR + shift(col + i0), (int64_t)0), rows - 1)] : 0.0;
                }
#pragma unroll
                for (int q = 0; q < UO; ++q) {
                    const int e = e0 + NT * q, jl = e / TR;
                    double *col = dst + (j0 + jl) * ldd + i0;
                    const int r = e % TR + shift(col);
                    if (j0 + jl < cols && i0 + r >= 0 && i0 + r < rows)
                        col[r] = combine(tile[r][jl], alpha, beta, &old[q], BETA ? 2 : mode);
                }
            }
        }
        __syncthreads();
    }
}

template <int TR, int TC, bool SHIFT>
void launch_transpose(int64_t rows, int64_t cols, double alpha, const double *src, int64_t lds, double beta,
                      double *dst, int64_t ldd, int mode, hipStream_t s) {
    const int64_t nx = (rows + (SHIFT ? LINE : 0) + TR - 1) / TR, tiles = nx * ((cols + TC - 1) / TC);
    const dim3 grid((unsigned)std::min<int64_t>(tiles, 1 << 23));
#define CA_TRANSPOSE(BETA)                                                                                          \
    hipLaunchKernelGGL((transpose_kernel<TR, TC, SHIFT, BETA>), grid, dim3(NT), 0, s, rows, cols, alpha, src, lds, beta, \
                       dst, ldd, mode, (uint32_t)nx, (uint32_t)tiles)
    if (mode == 2) CA_TRANSPOSE(true);
    else CA_TRANSPOSE(false);
#undef CA_TRANSPOSE
}

inline bool aligned16(const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }
inline int phase_of(const void *p) { return (int)(reinterpret_cast<uintptr_t>(p) & (8 * LINE - 1)); }   // bytes into its line

// Which loads of a copy of so many elements stream past the 256 MB last-level
// cache: none while it holds what is read, src's while it still holds dst, else
// both (1000 x 20000: 51.6 us streamed, 46.4 us cached, 1000 x 50000: 127 and
// 135 us; with beta = 1/2, 4096 x 4882: 73 us streamed, 67.5 us cached, 1000 x
// 30000: 116 and 128 us, 104 us with src streamed, 3000 x 15000: 186 us so, 163
// us all streamed).
struct Streamed {
    bool src, dst;
};
Streamed streamed(int64_t elements, int mode) {
    if (mode != 2) return {elements >= 38000000, elements >= 38000000};
    return {elements >= 21000000, elements >= 34000000};
}

int mode_of(double alpha, double beta) { return (alpha == 1.0 && beta == 0.0) ? 0 : (beta == 0.0 ? 1 : 2); }

}  // namespace

int launch_block_transform(char op, int64_t rows, int64_t cols, double alpha,
                           const double *src, int64_t lds, double beta,
                           double *dst, int64_t ldd, hipStream_t s) {
    if (rows == 0 || cols == 0) return COSMA_AMD_OK;
    const int mode = mode_of(alpha, beta);
    const bool in_phase = ldd % LINE == 0 && phase_of(dst) == 0;   // every column of dst starts at a line
    const bool src_in_phase = lds % LINE == 0 && phase_of(src) == 0;
    // src and dst together exceed the 256 MB last-level cache, which hides
    // shared lines (8191 x 12289 'T': 421 us, in shifted windows 283 us, 5000 x
    // 5001: 111 and 79 us, with beta = 1/2 157 and 116 us, but 3000 x 5000: 46 and 53 us)
    const bool large = rows * cols >= 20000000;
    const bool vec = aligned16(src) && aligned16(dst) && (lds % 2 == 0) && (ldd % 2 == 0);
    if (op == 'N') {
        // Many columns of few rows: a workgroup per two columns leaves most of
        // its threads idle, but what counts up to some 2^14 columns is that
        // there are many (33 x 7943: 4.2 us, 6.9 us as a list, x 31775: 9.6 and
        // 8.2 us; 1 x 10^8: 9.2 and 2.4 ms).  Fuller windows are as fast (128 x
        // 65536: 22.1 and 21.4 us, with beta = 1/2 33.3 and 37.1 us).
        if (rows <= (mode == 2 ? 48 : 64) && cols >= (1 << 14) + rows * (1 << 7)) {
            const CopyBlock one{src, dst, lds, ldd, rows, cols};
            return launch_block_copies(&one, 1, alpha, beta, s);
        }
        const bool shift = !in_phase && rows >= 1024;
        const Streamed st = streamed(rows * cols, mode);
        const int64_t bx = (rows + (shift ? LINE - 1 : 0) + 2 * NT - 1) / (2 * NT);
        const int u = st.dst && rows >= 3 * NT / 2 && cols <= 100000 ? 1 : 2;
        const int64_t by = std::min<int64_t>((cols + u - 1) / u, 65535);
        if (bx > 0x7fffffffLL) {
            set_error("block_transform: %lld rows exceed the grid limit", (long long)rows);
            return COSMA_AMD_ERR_UNSUPPORTED;
        }
        const dim3 grid((unsigned)bx, (unsigned)by);
#define CA_COPY(SHIFT, SRC_NT, DST_NT, U)                                                                            \
    hipLaunchKernelGGL((copy_kernel<SHIFT, SRC_NT, DST_NT, U>), grid, dim3(NT), 0, s, rows, cols, alpha, src, lds,  \
                       beta, dst, ldd, mode)
        if (u == 1 && shift) CA_COPY(true, true, true, 1);
        else if (u == 1) CA_COPY(false, true, true, 1);
        else if (st.dst && shift) CA_COPY(true, true, true, 2);
        else if (st.dst) CA_COPY(false, true, true, 2);
        else if (st.src && shift) CA_COPY(true, true, false, 2);
        else if (st.src) CA_COPY(false, true, false, 2);
        else if (shift) CA_COPY(true, false, false, 2);
        else CA_COPY(false, false, false, 2);
#undef CA_COPY
    } else if (in_phase && src_in_phase && rows >= 4096 && rows * cols >= ((int64_t)1 << 26)) {
        // both sides in whole lines (16384^2: 769 us in 64 x 64 tiles, 700 us;
        // slower below 4096 rows, 2000 x 16000: 90 and 112 us)
        launch_transpose<128, 64, false>(rows, cols, alpha, src, lds, beta, dst, ldd, mode, s);
    } else if (!(in_phase && (src_in_phase || (vec && (mode != 2 || rows * cols < 32000000)))) && large && rows >= 1024 &&
               cols >= 1024) {
        // with dst in whole lines the windows' extra columns buy nothing until
        // dst is also read from beyond the cache (2000 x 30002: 177 us in 64 x
        // 64 tiles, 195 us; with beta = 1/2 410 and 272 us, 4096 x 6002: 103 and 110 us)
        launch_transpose<112, 64, true>(rows, cols, alpha, src, lds, beta, dst, ldd, mode, s);
    } else {
        const int64_t bx = (rows + TT - 1) / TT;
        int64_t by = (cols + TT - 1) / TT;
        if (by > 65535) by = 65535;
        if (bx > 0x7fffffffLL) {
            set_error("block_transform: %lld rows exceed the grid limit", (long long)rows);
            return COSMA_AMD_ERR_UNSUPPORTED;
        }
        // with plenty of workgroups, four tiles each (the vectorised kernel
        // prefetches the next tile of a workgroup during the current one)
        if (vec && bx * by > 4096) by = (by + 3) / 4;
        if (vec)
            hipLaunchKernelGGL(transpose_cached_vec_kernel, dim3((unsigned)bx, (unsigned)by), dim3(NT), 0, s,
                               rows, cols, alpha, src, lds, beta, dst, ldd, mode);
        else
            hipLaunchKernelGGL(transpose_cached_kernel, dim3((unsigned)bx, (unsigned)by), dim3(NT), 0, s,
                               rows, cols, alpha, src, lds, beta, dst, ldd, mode);
    }
    CA_HIP(hipGetLastError());
    return COSMA_AMD_OK;
}

int launch_block_copies(const CopyBlock *blocks, int64_t n, double alpha, double beta, hipStream_t s) {
    const int mode = mode_of(alpha, beta);
    BlockList list;
    list.n = 0;
    uint32_t groups = 0;
    int64_t elements = 0;   // of the blocks that read whole lines; others share them (33 x 2033601: 228 us cached, 364 us)
    for (int64_t i = 0; i < n; ++i)
        if (blocks[i].rows >= NT / 2) elements += blocks[i].rows * blocks[i].cols;
    const Streamed st = streamed(elements, mode);
    auto flush = [&]() -> int {
        if (list.n == 0) return COSMA_AMD_OK;
#define CA_LIST(SRC_NT, DST_NT) \
    hipLaunchKernelGGL((copy_list_kernel<SRC_NT, DST_NT>), dim3(groups), dim3(NT), 0, s, list, alpha, beta, mode)
        if (st.dst) CA_LIST(true, true);
        else if (st.src) CA_LIST(true, false);
        else CA_LIST(false, false);
#undef CA_LIST
        CA_HIP(hipGetLastError());
        list.n = 0;
        groups = 0;
        return COSMA_AMD_OK;
    };
    int rc;
    for (int64_t i = 0; i < n; ++i) {
        const CopyBlock &b = blocks[i];
        if (b.rows == 0 || b.cols == 0) continue;
        const int64_t pairs = (b.rows + LINE) / 2;
        if (b.rows > NT && pairs * b.cols > LIST_PAIRS) {   // 1 GiB fills the chip by itself
            rc = launch_block_transform('N', b.rows, b.cols, alpha, b.src, b.lds, beta, b.dst, b.ldd, s);
            if (rc) return rc;
            continue;
        }
        // Narrow blocks stay here whatever their length (launch_block_transform
        // sends them to this list), cut to the kernel's 32-bit indexes.
        const int64_t piece = b.rows > NT ? b.cols : LIST_PAIRS / pairs;
        for (int64_t c0 = 0; c0 < b.cols; c0 += piece) {
            const int64_t nc = std::min(piece, b.cols - c0);
            list.b[list.n++] = {b.src + c0 * b.lds, b.dst + c0 * b.ldd, b.lds, b.ldd, (int)b.rows, (int)nc, groups,
                                (uint32_t)pairs};
            groups += (uint32_t)((pairs * nc + NT * ITEMS - 1) / (NT * ITEMS));
            if (list.n == LIST && (rc = flush())) return rc;
        }
    }
    return flush();
}

}  // namespace cosma_amd
