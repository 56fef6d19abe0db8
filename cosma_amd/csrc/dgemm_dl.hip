// FP64 DGEMM on the gfx950 matrix cores with operand tiles loaded straight
// from global memory into LDS (global_load_lds_dwordx4: lane l of a wave
// instruction writes the 16 bytes at the instruction's LDS base + 16 l), for
// any extents, leading dimensions and transposes.  The default kernel of
// cosma_amd_dgemm.
//
//   * A workgroup of 2 x 4 waves (2 x 2 below 64 x 64) owns a BM x BN tile of C,
//     a wave its part in 16 x 16 MFMA blocks.  Five tile shapes, 128 x 128 to 32 x 32, all
//     summing k in the order of dgemm.hip's gemm_tile: the choice of a tile
//     (pick_dl_tile) never changes a bit of the result.
//   * What bounds it: the FP64 MFMA pipe (a v_mfma_f64_16x16x4 takes 64
//     cycles of a SIMD).  Two to four workgroups per CU share the pipe, so one's
//     barrier and fragment reads overlap the others' MFMAs, and eight waves of
//     half the accumulators in place of four put twice the waves on a SIMD
//     (128 x 128 tiles, two workgroups per CU: 8192^3 TN 72.3 -> 73.4 TF, NT 70.1 ->
//     72.3; one workgroup per CU, 2048 x 2048 x 65536 TN: 69.4 -> 71.6; 64 x 64,
//     1537 x 1021 x 2999 NT: 193 -> 177 us).  NS LDS stages keep the loads of the
//     next NS - 1 steps in flight; small tiles need more than one (1024 x 1024 x
//     32768 TN, one 64 x 64 tile per CU: 1332 us with two stages, 1000 us with
//     three).
//   * Fragment registers are double-buffered by half-step, and each batch of
//     reads is waited for before the next one is issued (by then as many MFMAs
//     old as a half-step holds: 16 per wave at 128 x 128, 2 at 32 x 32).  Left to the compiler, the wait stood behind the next batch
//     and covered it too, idling the wave for an LDS round trip per half-step
//     (8192^3 TN 70.6 -> 73.0 TF, NN 70.7 -> 72.1 with the scalar addresses).
//   * LDS layout per operand and stage, every eight lanes of a fragment read on
//     distinct 16-byte bank groups (SQ_LDS_BANK_CONFLICT still counts 1.3
//     cycles per LDS instruction at 16384^3 TN, in total what the former slot
//     function kp ^ (r & 7), two-way by that measure, counted):
//     k-contiguous (A 'T', B 'N'): row r holds its eight k-pairs in 128 bytes,
//     pair kp in slot kp ^ row_swz(r); a fragment is one 16-byte read.
//     Row-contiguous (A 'N', B 'T'): k-row k holds the tile's rows, row r at
//     r ^ (16 if its k-pair is odd); a fragment is two 8-byte reads.
//     The loads' global addresses apply the permutations.
//   * Edges: rows beyond the matrix are read from its last row (or row pair)
//     and their results never stored, so full steps need no masks; the
//     partial last step is loaded by element, zero beyond K.  16-byte accesses
//     need no more than the 8-byte alignment of a double.
#include <algorithm>

#include "common.hpp"
#include "dgemm_dl.hpp"
#include "dl_index.hpp"

namespace cosma_amd {
namespace {

using dl::BK;
using dl::row_swz;

typedef double f64x2u __attribute__((ext_vector_type(2), aligned(8)));   // 16-byte access at 8-byte alignment

// s_waitcnt immediates (gfx9 fields: vmcnt bits 3:0 and 15:14, expcnt 6:4, lgkmcnt 11:8)
constexpr int wait_vm(int n) { return (n & 15) | ((n >> 4) << 14) | 0x0F70; }
constexpr int WAIT_LGKM0 = 0xC07F;
constexpr int WAIT_VM0_LGKM0 = 0x0070;

template <int R, bool KCONTIG, int NW>
struct Operand {
    static constexpr int NT = 64 * NW;
    static constexpr int SIZE = R * BK;          // doubles per stage
    static constexpr int LOADS = R / 8 / NW;     // 1 KB wave instructions per wave and step
    static_assert(R % (8 * NW) == 0 && NW % 4 == 0, "whole wave instructions, one k-pair parity per wave");
    static constexpr int NOFF = KCONTIG ? LOADS : 1;
    static constexpr int TAIL = R * BK / NT;     // elements per thread of the partial step
    const char *base;                            // wave-uniform
    int64_t ldb;                                 // leading dimension in bytes
    uint32_t off[NOFF];                          // per-lane byte offsets

    __device__ __forceinline__ Operand(const double *x, int64_t ld, int64_t r0, int64_t ext, int wave, int lane) {
        ldb = ld * 8;
        const int last = dl::last_row<R>(ext, r0);
        base = KCONTIG ? reinterpret_cast<const char *>(x + r0 * ld)
                       : reinterpret_cast<const char *>(x + r0) + (int64_t)(wave * dl::K_PER_WAVE<R>) * ldb;
#pragma unroll
        for (int q = 0; q < NOFF; ++q) {
            const dl::Element e = dl::lane_load<R, KCONTIG, NW>(q, wave, lane, last);
            off[q] = KCONTIG ? (uint32_t)e.row * (uint32_t)ldb + (uint32_t)e.k * 8
                             : (uint32_t)e.k * (uint32_t)ldb + (uint32_t)e.row * 8;
        }
    }
    __device__ __forceinline__ void issue(int k0, double *tile, int wave) const {
#pragma unroll
        for (int q = 0; q < LOADS; ++q) {
            // scalar base + 32-bit lane offset (the asm keeps the compiler from
            // folding the lane offset into 64-bit vector adds per load)
            const char *u = KCONTIG ? base + (int64_t)k0 * 8 : base + (int64_t)(k0 + q * dl::K_PER_ROUND<R, NW>) * ldb;
            asm("" : "+s"(u));
            __builtin_amdgcn_global_load_lds(static_cast<const void *>(u + off[KCONTIG ? q : 0]),
                                             (__attribute__((address_space(3))) void *)(tile + 128 * (wave + NW * q)),
                                             16, 0, 0);
        }
    }
    // The partial step: elements (row, k) with k < kt, zero beyond.
    __device__ __forceinline__ static void tail_rk(int e, int &row, int &k) {
        const int idx = threadIdx.x + NT * e;
        if (KCONTIG) { row = idx >> 4; k = idx & 15; }
        else { row = idx % R; k = idx / R; }
    }
    __device__ __forceinline__ static void tail_load(const double *x, int64_t ld, int64_t r0, int64_t ext, int64_t k0,
                                                     int kt, double (&v)[TAIL]) {
        const int last = dl::last_row<R>(ext, r0);
#pragma unroll
        for (int e = 0; e < TAIL; ++e) {
            int row, k;
            tail_rk(e, row, k);
            const int64_t r = r0 + min(row, last);
            v[e] = k < kt ? (KCONTIG ? x[k0 + k + r * ld] : x[r + (k0 + k) * ld]) : 0.0;
        }
    }
    __device__ __forceinline__ static void tail_store(double *tile, const double (&v)[TAIL]) {
#pragma unroll
        for (int e = 0; e < TAIL; ++e) {
            int row, k;
            tail_rk(e, row, k);
            tile[KCONTIG ? 2 * (row * 8 + ((k >> 1) ^ row_swz(row))) + (k & 1) : k * R + (row ^ (16 * ((k >> 1) & 1)))] =
                v[e];
        }
    }
};

// Fragment reads of one operand: row rbase + 16 i, lane group g, sub-step ks
// (k-pair kp = 4 ks + g).  Several blocks per wave (COUNT > 1) start at a
// multiple of 32 rows.
template <int R, bool KCONTIG, int COUNT>
struct Frag {
    int o0, o1;
    __device__ __forceinline__ Frag(int rbase, int g) {
        if (KCONTIG) {
            o0 = 2 * (rbase * 8 + (g ^ row_swz(rbase)));
            o1 = 2 * (rbase * 8 + ((g + 4) ^ row_swz(rbase)));
        } else {
            const int gb = 16 * (g & 1);
            o0 = 2 * g * R + (COUNT == 1 ? rbase ^ gb : rbase + gb);   // even i
            o1 = 2 * g * R + rbase - gb;                            // odd i
        }
    }
    __device__ __forceinline__ f64x2 read(const double *tile, int i, int ks) const {
        if (KCONTIG) return *reinterpret_cast<const f64x2 *>(tile + (ks ? o1 : o0) + 256 * i);
        const double *p = tile + ((i & 1) ? o1 : o0) + 16 * i + 8 * ks * R;
        return f64x2{p[0], p[R]};
    }
};

// One BM x BN tile of C at (m0, n0) with NS LDS stages in sm.  EDGE: the MFMAs
// of 16 x 16 blocks that lie wholly outside C are skipped.
template <int BM, int BN, int NS, int WM, int WN, bool AK, bool BKC, bool EDGE>
__device__ __forceinline__ void dl_tile(int64_t M, int64_t N, int64_t K, double alpha, const double *__restrict__ A,
                                        int64_t lda, const double *__restrict__ B, int64_t ldb, double beta,
                                        double *__restrict__ C, int64_t ldc, int64_t m0, int64_t n0, double *sm) {
    using OA = Operand<BM, AK, WM * WN>;
    using OB = Operand<BN, BKC, WM * WN>;
    constexpr int STAGE = OA::SIZE + OB::SIZE;
    constexpr int LOADS = OA::LOADS + OB::LOADS;
    constexpr int FM = BM / 16 / WM, FN = BN / 16 / WN;
    constexpr bool EARLY_TAIL = BM * BN <= 64 * 64;

    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wm = wave % WM, wn = wave / WM;
    const int g = lane >> 4, li = lane & 15;
    const OA oa(A, lda, m0, M, wave, lane);
    const OB ob(B, ldb, n0, N, wave, lane);
    const Frag<BM, AK, FM> fra(wm * (BM / WM) + 4 * (li & 3) + (li >> 2), g);
    const Frag<BN, BKC, FN> frb(wn * (BN / WN) + li, g);

    const int nk = dl::full_steps(M, N, K, AK, BKC);
    const int kt = (int)(K - (int64_t)nk * BK);   // 0..16
    double ta[OA::TAIL], tb[OB::TAIL];
    auto tail_load = [&]() {
        OA::tail_load(A, lda, m0, M, (int64_t)nk * BK, kt, ta);
        OB::tail_load(B, ldb, n0, N, (int64_t)nk * BK, kt, tb);
    };

    f64x4 acc[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) acc[i][j] = f64x4{0.0, 0.0, 0.0, 0.0};
    f64x2 af[2][FM], bf[2][FN];
    auto read_frags = [&](const double *tile, int ks) {
#pragma unroll
        for (int i = 0; i < FM; ++i) af[ks][i] = fra.read(tile, i, ks);
#pragma unroll
        for (int j = 0; j < FN; ++j) bf[ks][j] = frb.read(tile + OA::SIZE, j, ks);
    };
    const int rows_in = EDGE ? (int)min((int64_t)FM, (M - m0 - wm * (BM / WM) + 15) >> 4) : FM;   // may be <= 0
    const int cols_in = EDGE ? (int)min((int64_t)FN, (N - n0 - wn * (BN / WN) + 15) >> 4) : FN;
    auto mfmas = [&](int h) {
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
            for (int j = 0; j < FN; ++j)
                if (!EDGE || (i < rows_in && j < cols_in))
                    acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(af[h][i].x, bf[h][j].x, acc[i][j], 0, 0, 0);
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
            for (int j = 0; j < FN; ++j)
                if (!EDGE || (i < rows_in && j < cols_in))
                    acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(af[h][i].y, bf[h][j].y, acc[i][j], 0, 0, 0);
    };
    auto issue = [&](int kt_, double *tile) {
        oa.issue(kt_ * BK, tile, wave);
        ob.issue(kt_ * BK, tile + OA::SIZE, wave);
    };
    auto barrier = [&]() {
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
    if (EARLY_TAIL && kt > 0) tail_load();

    if (nk > 0) {
#pragma unroll
        for (int s = 0; s < NS; ++s) issue(min(s, nk - 1), sm + s * STAGE);
        __builtin_amdgcn_s_waitcnt(wait_vm((NS - 1) * LOADS));
        barrier();
        read_frags(sm, 0);
        auto iteration = [&](int k, double *cur, double *next) {
            __builtin_amdgcn_s_waitcnt(WAIT_LGKM0);
            __builtin_amdgcn_sched_barrier(0);
            read_frags(cur, 1);
            __builtin_amdgcn_sched_barrier(0);
            mfmas(0);
            __builtin_amdgcn_sched_barrier(0);
            __builtin_amdgcn_s_waitcnt(wait_vm((NS - 2) * LOADS) & WAIT_LGKM0);
            barrier();
            issue(min(k + NS, nk - 1), cur);
            __builtin_amdgcn_sched_barrier(0);
            read_frags(next, 0);
            __builtin_amdgcn_sched_barrier(0);
            mfmas(1);
            __builtin_amdgcn_sched_barrier(0);
        };
        int k = 0;
        for (; k + NS <= nk; k += NS) {
#pragma unroll
            for (int s = 0; s < NS; ++s) iteration(k + s, sm + s * STAGE, sm + ((s + 1) % NS) * STAGE);
        }
#pragma unroll
        for (int s = 0; s < NS - 1; ++s)
            if (k + s < nk) iteration(k + s, sm + s * STAGE, sm + ((s + 1) % NS) * STAGE);
    }
    if (kt > 0) {
        if (!EARLY_TAIL) tail_load();
        __builtin_amdgcn_s_waitcnt(WAIT_VM0_LGKM0);   // no load into LDS outstanding
        barrier();
        OA::tail_store(sm, ta);
        OB::tail_store(sm + OA::SIZE, tb);
        __syncthreads();
        read_frags(sm, 0);
        if (kt > BK / 2) read_frags(sm, 1);
        mfmas(0);
        if (kt > BK / 2) mfmas(1);
    }
    __builtin_amdgcn_s_waitcnt(wait_vm(0));   // no LDS writes outstanding at exit

    // ---- epilogue: lane holds rows 4g..4g+3 (contiguous) of column li
    const bool beta0 = (beta == 0.0);
#pragma unroll
    for (int i = 0; i < FM; ++i) {
        const int64_t row = m0 + wm * (BM / WM) + 16 * i + 4 * g;
#pragma unroll
        for (int j = 0; j < FN; ++j) {
            const int64_t col = n0 + wn * (BN / WN) + 16 * j + li;
            if (col >= N) continue;
            double *cp = C + row + col * ldc;
            const f64x4 r = acc[i][j];
            if (row + 3 < M) {
                f64x2u *cv = reinterpret_cast<f64x2u *>(cp);
                f64x2u lo = {alpha * r[0], alpha * r[1]};
                f64x2u hi = {alpha * r[2], alpha * r[3]};
                if (!beta0) {
                    const f64x2u clo = cv[0], chi = cv[1];
                    lo.x = fma(beta, clo.x, lo.x); lo.y = fma(beta, clo.y, lo.y);
                    hi.x = fma(beta, chi.x, hi.x); hi.y = fma(beta, chi.y, hi.y);
                }
                cv[0] = lo;
                cv[1] = hi;
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    if (row + e < M) {
                        double val = alpha * r[e];
                        if (!beta0) val = fma(beta, cp[e], val);
                        cp[e] = val;
                    }
                }
            }
        }
    }
}

// NS: LDS stages; WPE: waves per SIMD it is built for; WM x WN waves.
template <int BM, int BN, int NS, int WPE, int WM, int WN, bool AK, bool BKC>
__global__ __launch_bounds__(64 * WM * WN) __attribute__((amdgpu_waves_per_eu(WPE, WPE))) void dgemm_dl_kernel(
    int64_t M, int64_t N, int64_t K, double alpha,
    const double *__restrict__ A, int64_t lda,
    const double *__restrict__ B, int64_t ldb,
    double beta, double *__restrict__ C, int64_t ldc, int group_m) {
    __shared__ __attribute__((aligned(16))) double sm[NS * (BM + BN) * BK];
    const dl::TileAt t = dl::raster(blockIdx.x, gridDim.x, (uint32_t)((M + BM - 1) / BM),
                                    (uint32_t)((N + BN - 1) / BN), (uint32_t)group_m);
    const int64_t m0 = (int64_t)t.m * BM, n0 = (int64_t)t.n * BN;
    dl_tile<BM, BN, NS, WM, WN, AK, BKC, false>(M, N, K, alpha, A, lda, B, ldb, beta, C, ldc, m0, n0, sm);
}

// Grouped tiles: workgroup w takes the virtual ids w, w + G, ... of all
// problems' tiles, mapped to tiles by grouped_tile_of.  TRANS: the problems'
// common transposes (GroupedProblem::flags), or MIXED, whose four loops in one
// kernel need registers for three workgroups per CU in place of four.
// What bounds it: a tile takes about 1.9 us of its CU before and after its
// k-steps (owner, descriptor and first loads in a chain, C's stores), as much
// as four 64 x 64 steps, and the batch's 2 GB from HBM take 0.4 ms; one
// workgroup per tile overlaps these best.  4096 NN products, m, n, k log-uniform
// in [16, 512], tuned: 889 us register-staged with a search for the owner,
// 728 us here, 690 us with the blocks outside C skipped and the kernel of one
// transpose.  Cutting a tile into four rows or columns of blocks, whichever
// balances its waves better at an edge, spilled and lost (774 us).
constexpr int MIXED = 4;
template <int BM, int BN, int NS, int WPE, int TRANS>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(WPE, WPE))) void dgemm_dl_grouped_kernel(
    const GroupedProblem *__restrict__ probs, const int *__restrict__ owner, int64_t total_tiles) {
    __shared__ __attribute__((aligned(16))) double sm[NS * (BM + BN) * BK];
    for (int64_t v = blockIdx.x; v < total_tiles; v += gridDim.x) {
        const int64_t t = grouped_tile_of(v, total_tiles);
        const GroupedProblem &q = probs[owner[t]];
        const uint32_t local = (uint32_t)(t - q.tile_start), tiles_m = (uint32_t)((q.m + BM - 1) / BM);
        const int64_t m0 = (int64_t)(local % tiles_m) * BM, n0 = (int64_t)(local / tiles_m) * BN;
        const bool scale_only = (q.k == 0 || q.alpha == 0.0);
        const int64_t K = scale_only ? 0 : q.k;
        const double alpha = scale_only ? 0.0 : q.alpha;
        if (v >= gridDim.x) __syncthreads();   // the previous tile's last LDS reads are done
#define CA_TILE(X, Y)                                                                                           \
    dl_tile<BM, BN, NS, 2, 2, X, Y, true>(q.m, q.n, K, alpha, q.a, q.lda, q.b, q.ldb, q.beta, q.c, q.ldc, m0, n0, sm)
        switch (TRANS == MIXED ? q.flags & 3 : TRANS) {   // bit 0: A transposed, bit 1: B transposed
        case 0: CA_TILE(false, true); break;
        case 1: CA_TILE(true, true); break;
        case 2: CA_TILE(false, false); break;
        default: CA_TILE(true, false); break;
        }
#undef CA_TILE
    }
}

template <int BM, int BN, int NS, int WPE, int WM, int WN>
void launch(char ta, char tb, int64_t m, int64_t n, int64_t k, double alpha, const double *a, int64_t lda,
            const double *b, int64_t ldb, double beta, double *c, int64_t ldc, int group_m, hipStream_t s) {
    const int64_t tiles_m = (m + BM - 1) / BM;
    const dim3 grid((unsigned)(tiles_m * ((n + BN - 1) / BN))), block(64 * WM * WN);
    const int rows = dl::clamp_group(group_m, tiles_m);
#define CA_LAUNCH_DL(X, Y)                                                                                        \
    hipLaunchKernelGGL((dgemm_dl_kernel<BM, BN, NS, WPE, WM, WN, X, Y>), grid, block, 0, s, m, n, k, alpha, a, lda, b,   \
                       ldb, beta, c, ldc, rows)
    // template flags: operand k-contiguous (A 'T', B 'N')
    if (ta == 'T' && tb == 'N') CA_LAUNCH_DL(true, true);
    else if (ta == 'N' && tb == 'N') CA_LAUNCH_DL(false, true);
    else if (ta == 'N' && tb == 'T') CA_LAUNCH_DL(false, false);
    else CA_LAUNCH_DL(true, false);
#undef CA_LAUNCH_DL
}

}  // namespace

namespace {
constexpr int N_CU = 256;
struct TileModel {
    int bm, bn;
    double extra;     // prologue and epilogue of a tile, in k
    double busy[3];   // MFMA utilisation with one, two, and more tiles per CU
    double beyond;    // its factor when the operands exceed the last-level cache
};
// Fitted to 420 shapes (m, n 32 to 8192, k 8 to 65536, all transposes and
// alignments, every tile timed): the choice is 0.4% slower than the fastest
// tile on average, 12% at most.
constexpr TileModel MODEL[] = {
    {128, 128, 97, {0.866, 0.924, 0.925}, 1.0}, {64, 128, 66, {0.689, 0.886, 0.912}, 0.977},
    {64, 64, 66, {0.715, 0.804, 0.862}, 0.999}, {64, 32, 55, {0.623, 0.707, 0.774}, 0.784},
    {32, 32, 52, {0.539, 0.622, 0.678}, 0.786},
};
constexpr double LLC_DOUBLES = 256.0 * (1 << 20) / 8;
int64_t tiles_of(DlTile t, int64_t m, int64_t n) {
    return ((m + MODEL[t].bm - 1) / MODEL[t].bm) * ((n + MODEL[t].bn - 1) / MODEL[t].bn);
}
}  // namespace

// The busiest CU computes ceil(tiles / CUs) tiles, each bm * bn * (k + extra)
// products at the tile's MFMA utilisation: large tiles move less data per
// product, small ones leave less of the chip idle and pad less.  1000^3 NN:
// 125 us in 128 x 128 tiles (64 of 256 CUs busy), 35 us in 64 x 64; 700 x 700 x
// 16384 TN: 1914 us, 269 us in 64 x 32; 8192^3 TN: 14.8 ms, 18.6 ms in 32 x 32.
DlTile pick_dl_tile(int64_t m, int64_t n, int64_t k) {
    DlTile best = DL_128x128;
    double least = 0.0;
    const bool beyond = (double)(m + n) * (double)k > LLC_DOUBLES;
    for (int t = DL_128x128; t <= DL_32x32; ++t) {
        const TileModel &x = MODEL[t];
        const int64_t per_cu = (tiles_of(static_cast<DlTile>(t), m, n) + N_CU - 1) / N_CU;
        const double busy = x.busy[std::min<int64_t>(per_cu, 3) - 1] * (beyond ? x.beyond : 1.0);
        const double cost = (double)(per_cu * x.bm * x.bn) * ((double)k + x.extra) / busy;
        if (t == DL_128x128 || cost < least) {
            least = cost;
            best = static_cast<DlTile>(t);
        }
    }
    return best;
}

bool dl_fits(int64_t m, int64_t n, int64_t k, int64_t lda, int64_t ldb) {
    // 32-bit byte offsets over 128 rows, 32-bit step counts, and the 2^32
    // work-items of a launch
    return (m + 31) / 32 * ((n + 31) / 32) < ((int64_t)1 << 23) && k < ((int64_t)1 << 31) &&
           lda < ((int64_t)1 << 22) && ldb < ((int64_t)1 << 22);
}

int launch_dl(DlTile tile, char ta, char tb, int64_t m, int64_t n, int64_t k, double alpha, const double *a, int64_t lda,
              const double *b, int64_t ldb, double beta, double *c, int64_t ldc, int group_m, hipStream_t s) {
#define CA_DL(BM, BN, NS, WPE, WM, WN) \
    launch<BM, BN, NS, WPE, WM, WN>(ta, tb, m, n, k, alpha, a, lda, b, ldb, beta, c, ldc, group_m, s)
    switch (tile) {
    case DL_128x128: CA_DL(128, 128, 2, 4, 2, 4); break;
    case DL_64x128: CA_DL(64, 128, 2, 6, 2, 4); break;
    case DL_64x64: CA_DL(64, 64, 3, 6, 2, 4); break;
    case DL_64x32: CA_DL(64, 32, 3, 4, 2, 2); break;
    default: CA_DL(32, 32, 4, 4, 2, 2); break;
    }
#undef CA_DL
    CA_HIP(hipGetLastError());
    return COSMA_AMD_OK;
}

int launch_grouped_dl(int cfg, const GroupedProblem *probs, int nprob, int64_t total_tiles, int grid, int trans,
                      hipStream_t s) {
    const int *owner = reinterpret_cast<const int *>(reinterpret_cast<const int64_t *>(probs + nprob) + nprob);
    const dim3 g((unsigned)grid), b(256);
#define CA_GROUPED(BM, BN, NS, WPE, TRANS) \
    hipLaunchKernelGGL((dgemm_dl_grouped_kernel<BM, BN, NS, WPE, TRANS>), g, b, 0, s, probs, owner, total_tiles)
    switch (cfg) {
    case 1:
        switch (trans) {
        case 0: CA_GROUPED(64, 64, 2, 4, 0); break;
        case 1: CA_GROUPED(64, 64, 2, 4, 1); break;
        case 2: CA_GROUPED(64, 64, 2, 4, 2); break;
        case 3: CA_GROUPED(64, 64, 2, 4, 3); break;
        default: CA_GROUPED(64, 64, 2, 3, MIXED); break;
        }
        break;
    case 2: CA_GROUPED(128, 64, 2, 2, MIXED); break;
    case 3: CA_GROUPED(128, 128, 2, 2, MIXED); break;
    default: CA_GROUPED(32, 32, 2, 6, MIXED); break;
    }
#undef CA_GROUPED
    CA_HIP(hipGetLastError());
    return COSMA_AMD_OK;
}

}  // namespace cosma_amd
