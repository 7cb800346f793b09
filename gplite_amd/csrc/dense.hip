// Dense FP64 linear algebra for gfx950: MFMA GEMM, 64x64 diagonal-block Cholesky
// with in-LDS inverse, blocked triangular solves and matrix-vector products.
//
// Every matrix is column-major with a leading dimension that is a multiple of 64
// and logical sizes padded to multiples of 64 (padding is identity / zero), so the
// kernels only ever see whole 64x64 tiles.
#include "gpl_internal.h"

#include <cmath>
#include <type_traits>

namespace gpl {

typedef double d4 __attribute__((ext_vector_type(4)));

// Map the hardware block id so that each XCD (blocks are dealt round-robin over
// 8 XCDs) receives a contiguous range of logical tiles: neighbouring tiles share
// operand panels, which then stay in that XCD's L2.
__device__ __forceinline__ int64_t xcd_remap(int64_t b, int64_t nb) {
    const int64_t per = nb / 8, rem = nb % 8;
    const int64_t x = b % 8, q = b / 8;
    return (x < rem) ? x * (per + 1) + q : rem * (per + 1) + (x - rem) * per + q;
}

__device__ __forceinline__ void lower_tile(int64_t t, int64_t& ti, int64_t& tj) {
    int64_t r = (int64_t)((sqrt(8.0 * (double)t + 1.0) - 1.0) * 0.5);
    while ((r + 1) * (r + 2) / 2 <= t) ++r;
    while (r * (r + 1) / 2 > t) --r;
    ti = r;
    tj = t - r * (r + 1) / 2;
}

// ---------------------------------------------------------------------------
// FP64-compute GEMM, operands straight from global memory to registers.
//
// A workgroup of 2 x 2 waves; each wave owns a WT x WT block of C as 16x16 tiles
// of v_mfma_f64_16x16x4 and loads its own operand fragments, PF - 1 chunks of 16
// k ahead, into registers: no LDS, no barrier, so a wave never waits for another
// and the loads of several chunks are in flight while one is multiplied.  The
// waves of a workgroup share their operands through L1, the workgroups of an XCD
// through its L2.  (The staged form this replaces, 64x64 or 128x128 tiles double
// buffered in LDS, took about 1 us per 16-k chunk whatever the size, the load
// latency and two barriers; measured alone, us staged -> here:
// 512 x 256 x 256: 20.1 -> 7.1, 1024 x 512 x 512: 35.7 -> 18.5, 4096 x 512 x 512:
// 60 -> 52, lower 7168, k = 512: 587 -> 507, X^T X at 8192: 3186 -> 2890.)
//
// Within a chunk lane (li, g) holds k = 4g + s of step s (s < 4), so an operand
// that is contiguous in k is read as 32 bytes per lane and whole 128-byte lines
// per 16 rows; one that is contiguous in m is read as pairs of rows (lane li: rows
// 2li and 2li + 1, which belong to two tiles).  Sums run over k in one fixed order,
// whatever the tile.
// M, N and K are multiples of 64, operand addresses of 16 bytes.
//
// SUB: C -= op(A) op(B) (alpha = -1, beta = 1), where every 64 k's products are summed on
// their own and subtracted.
//
// INP: C is B (a solve against a 64x64 inverse, M = 64).  A workgroup of 64x64 then
// covers the whole contraction of its columns, and stores only after all of its waves
// have read.
// ---------------------------------------------------------------------------
template <typename T> struct vec2_of;
template <> struct vec2_of<double> { typedef double2 type; };
template <> struct vec2_of<float> { typedef float2 type; };

// row (column) of a WT-wide block that lane li of tile i holds
template <bool KC, int NB>
__device__ __forceinline__ int frag_row(int i, int li) {
    return (KC || NB == 1) ? 16 * i + li : 32 * (i >> 1) + 2 * li + (i & 1);
}

// One chunk of an operand: p at the lane's element (its row of tile 0, k = 4g).
template <bool KC, int NB, typename T>
__device__ __forceinline__ void frag_load(T (&f)[NB][4], const T* p, int64_t ld) {
    typedef typename vec2_of<T>::type V2;
    if (KC) {
#pragma unroll
        for (int i = 0; i < NB; ++i) {
            const V2* q = reinterpret_cast<const V2*>(p + 16 * i * ld);
            const V2 a = q[0], b = q[1];
            f[i][0] = a.x;
            f[i][1] = a.y;
            f[i][2] = b.x;
            f[i][3] = b.y;
        }
    } else if (NB == 1) {
#pragma unroll
        for (int s = 0; s < 4; ++s) f[0][s] = p[s * ld];
    } else {
#pragma unroll
        for (int i = 0; i < NB; i += 2)
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                const V2 a = *reinterpret_cast<const V2*>(p + 16 * i + s * ld);
                f[i][s] = a.x;
                f[i + 1 < NB ? i + 1 : i][s] = a.y;
            }
    }
}

// C = beta*C + alpha*op(A) op(B); A, B and C may be stored as float or double.
// KS: op(A) diag(ks) op(B), where the problems of the batch are consecutive ranges
// of K of one contraction of length kall (the last may be shorter).
template <int TA, int TB, int WT, int PF, bool INP, bool KS, bool SUB, typename TAs, typename TBs, typename TCs>
__global__ __launch_bounds__(256) void k_gemm_reg(int64_t M, int64_t N, int64_t K, int64_t tilesM, double alpha,
                                                  const TAs* A, int64_t lda, const TBs* B, int64_t ldb, double beta,
                                                  TCs* C, int64_t ldc, int tiles, int64_t sA, int64_t sB, int64_t sC,
                                                  const double* ks, int64_t kall) {
    constexpr int NB = WT / 16, BM = 2 * WT;
    constexpr bool KA = TA != 0, KB = TB == 0;  // contiguous in k
    A += blockIdx.y * sA;  // batch: one problem per grid row
    B += blockIdx.y * sB;
    C += blockIdx.y * sC;
    if (KS) {
        ks += blockIdx.y * K;
        const int64_t left = kall - (int64_t)blockIdx.y * K;
        K = left < K ? left : K;
    }
    // Contiguous tile ranges per XCD share operand panels in L2; with a k range
    // that depends on the tile row (tiles == 2, 5) or column (tiles == 4, whose
    // columns are contiguous in the tile order) work per tile varies widely, so
    // the hardware's round-robin placement is kept there to balance the XCDs.
    const int64_t bid = (tiles == 2 || tiles >= 4) ? (int64_t)blockIdx.x : xcd_remap(blockIdx.x, gridDim.x);
    int64_t ti, tj;
    if (tiles != 1 && tiles != 2) {
        ti = bid % tilesM;
        tj = bid / tilesM;
        if (tiles == 3) ti = tilesM - 1 - ti;  // the longest k ranges first
    } else if (BM >= 64) {
        lower_tile(bid, ti, tj);
    } else {  // the lower 64x64 tiles, 2 x 2 workgroups each
        lower_tile(bid >> 2, ti, tj);
        ti = 2 * ti + (bid & 1);
        tj = 2 * tj + ((bid >> 1) & 1);
    }
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int li = lane & 15, g = lane >> 4;
    const int64_t row0 = ti * BM + (w & 1) * WT, col0 = tj * BM + (w >> 1) * WT;
    if (row0 >= M || col0 >= N) return;
    if ((tiles == 1 || tiles == 2) && row0 / 64 < col0 / 64) return;  // above the diagonal tiles
    const int64_t kbeg = (tiles == 2 || tiles == 5) ? row0 / 64 * 64 : (tiles == 4) ? col0 / 64 * 64 : 0;
    const int64_t kend = (tiles == 3) ? (row0 / 64 + 1) * 64 < K ? (row0 / 64 + 1) * 64 : K : K;
    const int nch = kend > kbeg ? (int)((kend - kbeg) / 16) : 0;
    const int64_t ra = row0 + frag_row<KA, NB>(0, li), rb = col0 + frag_row<KB, NB>(0, li);
    const TAs* pa = KA ? A + (kbeg + 4 * g) + ra * lda : A + ra + (kbeg + 4 * g) * lda;
    const TBs* pb = KB ? B + (kbeg + 4 * g) + rb * ldb : B + rb + (kbeg + 4 * g) * ldb;
    const int64_t stepa = KA ? 16 : 16 * lda, stepb = KB ? 16 : 16 * ldb;
    d4 acc[NB][NB];
#pragma unroll
    for (int i = 0; i < NB; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j) acc[i][j] = d4{0.0, 0.0, 0.0, 0.0};
    TAs fa[PF][NB][4];
    TBs fb[PF][NB][4];
    double2 fs[KS ? PF : 1][2];
    const double* pk = KS ? ks + kbeg + 4 * g : nullptr;
    auto load = [&](int st) {
        frag_load<KA, NB>(fa[st], pa, lda);
        frag_load<KB, NB>(fb[st], pb, ldb);
        if (KS) {
            fs[st][0] = reinterpret_cast<const double2*>(pk)[0];
            fs[st][1] = reinterpret_cast<const double2*>(pk)[1];
            pk += 16;
        }
        pa += stepa;
        pb += stepb;
    };
    typedef typename vec2_of<TCs>::type C2;
    constexpr bool PAIR = !KA && NB > 1;  // rows 2li, 2li + 1 of tiles i, i + 1
    constexpr int RI = PAIR ? 2 : 1;
    TCs cv[NB][NB][4];
    auto addr = [&](int i, int j, int v) {
        return C + (row0 + frag_row<KA, NB>(i, li)) + (col0 + frag_row<KB, NB>(j, g + 4 * v)) * ldc;
    };
    auto load_c = [&]() {
#pragma unroll
        for (int i = 0; i < NB; i += RI)
#pragma unroll
            for (int j = 0; j < NB; ++j)
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    if (PAIR) {
                        const C2 x = *reinterpret_cast<const C2*>(addr(i, j, v));
                        cv[i][j][v] = x.x;
                        cv[i + RI - 1][j][v] = x.y;
                    } else {
                        cv[i][j][v] = *addr(i, j, v);
                    }
                }
    };
    auto take = [&]() {
#pragma unroll
        for (int i = 0; i < NB; ++i)
#pragma unroll
            for (int j = 0; j < NB; ++j) {
#pragma unroll
                for (int v = 0; v < 4; ++v) cv[i][j][v] -= (TCs)acc[i][j][v];
                acc[i][j] = d4{0.0, 0.0, 0.0, 0.0};
            }
    };
    // the tiles are formed transposed: D lane (li, g) holds columns g + 4v of row li
    auto mult = [&](int st) {
        if (KS) {
#pragma unroll
            for (int j = 0; j < NB; ++j) {
                fb[st][j][0] *= fs[st][0].x;
                fb[st][j][1] *= fs[st][0].y;
                fb[st][j][2] *= fs[st][1].x;
                fb[st][j][3] *= fs[st][1].y;
            }
        }
#pragma unroll
        for (int s = 0; s < 4; ++s)
#pragma unroll
            for (int i = 0; i < NB; ++i)
#pragma unroll
                for (int j = 0; j < NB; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64((double)fb[st][j][s], (double)fa[st][i][s],
                                                                     acc[i][j], 0, 0, 0);
    };
#pragma unroll
    for (int q = 0; q < PF - 1; ++q)
        if (q < nch) load(q);
    int c = 0;
    if (SUB) load_c();
    static_assert(!SUB || PF == 4, "a pass is the 64 k whose sum is subtracted");
    for (; c + 2 * PF - 1 <= nch; c += PF) {  // every load of this pass exists
#pragma unroll
        for (int q = 0; q < PF; ++q) {
            load((q + PF - 1) % PF);
            mult(q);
        }
        if (SUB) take();
    }
    for (; c < nch; c += PF) {
#pragma unroll
        for (int q = 0; q < PF; ++q) {
            if (c + q + PF - 1 < nch) load((q + PF - 1) % PF);
            if (c + q < nch) mult(q);
        }
        if (SUB) take();
    }
    // With beta != 0 every C value is loaded before the first store (a load placed
    // after a store that may alias it waits for that store's round trip).
    if (!SUB && beta != 0.0) load_c();
    if (INP) __syncthreads();
    auto out = [&](int i, int j, int v) {
        if (SUB) return cv[i][j][v];
        const double o = alpha * acc[i][j][v];
        return (TCs)((beta == 0.0) ? o : beta * (double)cv[i][j][v] + o);
    };
#pragma unroll
    for (int i = 0; i < NB; i += RI)
#pragma unroll
        for (int j = 0; j < NB; ++j)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                if (PAIR) {
                    C2 x;
                    x.x = out(i, j, v);
                    x.y = out(i + RI - 1, j, v);
                    *reinterpret_cast<C2*>(addr(i, j, v)) = x;
                } else {
                    *addr(i, j, v) = out(i, j, v);
                }
            }
}

template <int WT, int PF, bool INP, typename TAs, typename TBs, typename TCs>
static void gemm_reg_launch(hipStream_t s, int ta, int tb, int64_t M, int64_t N, int64_t K, double alpha,
                            const TAs* A, int64_t lda, const TBs* B, int64_t ldb, double beta, TCs* C, int64_t ldc,
                            int tiles, int batch, int64_t sA, int64_t sB, int64_t sC) {
    constexpr int BM = 2 * WT;
    const int64_t tm = (M + BM - 1) / BM, tn = (N + BM - 1) / BM, t64 = M / 64;
    const int64_t nblk = (tiles != 1 && tiles != 2) ? tm * tn : BM < 64 ? 4 * (t64 * (t64 + 1) / 2) : tm * (tm + 1) / 2;
    dim3 grid((unsigned)nblk, (unsigned)batch), block(256);
#define GPL_GR(TAv, TBv)                                                                                           \
    hipLaunchKernelGGL((k_gemm_reg<TAv, TBv, WT, PF, INP, false, false, TAs, TBs, TCs>), grid, block, 0, s, M, N, K, tm,    \
                       alpha, A, lda, B, ldb, beta, C, ldc, tiles, sA, sB, sC, (const double*)nullptr, (int64_t)0)
    if constexpr (INP || sizeof(TAs) == 4) GPL_GR(0, 0);  // the only forms that are called
    else if (!ta && !tb) GPL_GR(0, 0);
    else if (!ta && tb) GPL_GR(0, 1);
    else if (ta && !tb) GPL_GR(1, 0);
    else GPL_GR(1, 1);
#undef GPL_GR
}

// Wave tile by the number of 64x64 output tiles (all problems of the launch), t64,
// and their number of 128x128 ones, t128; times staged LDS / 16 / 32 / 64 measured
// alone, in us.  Fewer than 128: 16-wide waves (32x32 workgroups), so that a small
// product spreads over the chip and its k loop is a quarter as long (512 x 256 x
// 256: 20 / 7.0 / 12 / 37; X B at 512: 32 / 14 / 21 / 67; 128 tiles, 1024 x 512 x
// 512: 36 / 20 / 22 / 68).  Else 32-wide ones (2048 x 512 x 512: 38 / 36 / 25 / 70;
// lower 7168, k = 512: 558 / 769 / 458 / 496).  Long k with enough tiles to
// fill the chip more than twice over: 64-wide ones, half the operand traffic per
// flop (X B at 4096: 1562 / 2857 / 1278 / 1146; X^T X at 8192: 3213 / 9711 / 4902 /
// 2943, at 3072: 423 / 542 / 297 / 377; long is the mean range, half of K with a
// triangular operand: X B with 1024 x 131072, 32 / 64: 2921 / 3155).  With both operands contiguous in k the
// 32-wide waves are bound by their loads (37 TFLOP/s), so a product whose tiles
// all have the same k range takes the 64-wide ones as soon as they fill the chip
// once (1024 x 1024 x 32768 in four parts).
template <typename TAs, typename TBs, typename TCs>
static void gemm_any(hipStream_t s, int ta, int tb, int64_t M, int64_t N, int64_t K, double alpha, const TAs* A,
                     int64_t lda, const TBs* B, int64_t ldb, double beta, TCs* C, int64_t ldc, int tiles, int batch,
                     int64_t sA, int64_t sB, int64_t sC) {
    if (M <= 0 || N <= 0 || batch <= 0) return;
#define GPL_GA(WT, PF, INP) \
    gemm_reg_launch<WT, PF, INP>(s, ta, tb, M, N, K, alpha, A, lda, B, ldb, beta, C, ldc, tiles, batch, sA, sB, sC)
    if constexpr (sizeof(TAs) == 8) {
        if (B == C) {
            GPL_GA(32, 3, true);
            return;
        }
    }
    const bool low = tiles == 1 || tiles == 2;
    const int64_t m = M / 64, n = N / 64, m2 = (m + 1) / 2, n2 = (n + 1) / 2;
    const int64_t t64 = (low ? m * (m + 1) / 2 : m * n) * batch, t128 = (low ? m2 * (m2 + 1) / 2 : m2 * n2) * batch;
    if (t64 < 128) GPL_GA(16, 4, false);
    else if ((tiles >= 3 ? K / 2 : K) >= 1024 && t128 >= (ta && !tb && !tiles ? 256 : 600)) GPL_GA(64, 3, false);
    else GPL_GA(32, 3, false);
#undef GPL_GA
}

void gemm2_f64(hipStream_t s, int ta, int tb, int64_t M, int64_t N, int64_t K, double alpha, const double* A,
               int64_t lda, const double* B, int64_t ldb, double beta, double* C, int64_t ldc, int tiles) {
    gemm_any(s, ta, tb, M, N, K, alpha, A, lda, B, ldb, beta, C, ldc, tiles, 1, 0, 0, 0);
}

// `batch` independent FP64 GEMMs (strides in elements), one grid row per problem
void gemm2_f64_batched(hipStream_t s, int ta, int tb, int64_t M, int64_t N, int64_t K, double alpha, const double* A,
                       int64_t lda, const double* B, int64_t ldb, double beta, double* C, int64_t ldc, int tiles,
                       int batch, int64_t sA, int64_t sB, int64_t sC) {
    gemm_any(s, ta, tb, M, N, K, alpha, A, lda, B, ldb, beta, C, ldc, tiles, batch, sA, sB, sC);
}

// C -= A B^T (A: M x K, B: N x K), the sums of 64 k subtracted one by one: the update of
// a panel's later columns by its earlier ones.  One sum of all 256 rounds each element at
// the size of that sum 256 times; the solutions' error is then 1.15 to 1.45 times as large.
void gemm_sub_f64(hipStream_t s, int64_t M, int64_t N, int64_t K, const double* A, int64_t lda, const double* B,
                  int64_t ldb, double* C, int64_t ldc) {
    if (M <= 0 || N <= 0) return;
#define GPL_GS(WT)                                                                                                  \
    hipLaunchKernelGGL((k_gemm_reg<0, 1, WT, 4, false, false, true, double, double, double>),                       \
                       dim3((unsigned)(((M + 2 * WT - 1) / (2 * WT)) * ((N + 2 * WT - 1) / (2 * WT)))), dim3(256), 0, \
                       s, M, N, K, (M + 2 * WT - 1) / (2 * WT), -1.0, A, lda, B, ldb, 1.0, C, ldc, 0, (int64_t)0,     \
                       (int64_t)0, (int64_t)0, (const double*)nullptr, (int64_t)0)
    if (M / 64 * (N / 64) < 128) GPL_GS(16);  // the line of gemm_any
    else GPL_GS(32);
#undef GPL_GS
}

// Lower 64x64 tiles of A diag(ks) A^T, A (M x K): `parts` partial products over kp
// columns each, C + p * sC (fitc_part_cols chooses their number).  32-wide waves with
// three chunks in flight whatever the size (16 / 32 / 64 wide, products and their sum, us:
// K = 131072 with M = 1024 5454 / 2698 / 3568, M = 512 1563 / 762 / 1034, M = 128 137 / 90 /
// 272; K = 32768 with M = 512 389 / 216 / 229).
void gemm_gram_f64(hipStream_t s, int64_t M, int64_t K, const double* A, int64_t lda, const double* ks, int parts,
                   int64_t kp, double* C, int64_t ldc, int64_t sC) {
    const int64_t t = M / 64;
    hipLaunchKernelGGL((k_gemm_reg<0, 1, 32, 4, false, true, false, double, double, double>),
                       dim3((unsigned)(t * (t + 1) / 2), (unsigned)parts), dim3(256), 0, s, M, M, kp, t, 1.0, A, lda, A,
                       lda, 0.0, C, ldc, 1, kp * lda, kp * lda, sC, ks, K);
}

// FP64-compute GEMM on FP32 storage of A (prediction)
void gemm_mixed_f32f64f64(hipStream_t s, int64_t M, int64_t N, int64_t K, double alpha, const float* A,
                          int64_t lda, const double* B, int64_t ldb, double beta, double* C, int64_t ldc, int tiles) {
    gemm_any(s, 0, 0, M, N, K, alpha, A, lda, B, ldb, beta, C, ldc, tiles, 1, 0, 0, 0);
}

// A failing row + 1 into info, the lowest of all that are reported: the workgroups of
// one launch that factor different diagonal blocks report in no fixed order, and past a
// failing pivot every later block holds NaN and reports too.  A time-out stays.
__device__ __forceinline__ void report_minor(int* info, int minor) {
    int old = atomicCAS(info, 0, minor);
    while (old > minor && old != kPanelWaitTimeout) {  // old only falls, or becomes the time-out
        const int seen = atomicCAS(info, old, minor);
        if (seen == old) return;
        old = seen;
    }
}

// ---------------------------------------------------------------------------
// Cholesky of a 64-column block held in LDS, FP64.  The block is a trapezoid
// S[col][row] (64 columns, row stride kTP): rows 0..63 the diagonal block and,
// optionally, rows 64..127 a 64-row block below it, which leaves as
// A_below L^-T in the same pass.
//
// It runs in four phases of 16 columns.  In a phase one wave per 64 rows keeps
// its rows' 16 columns in registers, and beside them a copy of the phase's
// 16x16 diagonal tile, one copy per 16-lane row.  Every wave factors that tile
// for itself: the pivot and the multipliers of a column are then 16-lane row
// broadcasts (v_mov_b64_dpp row_newbcast) of its own registers, so a column
// costs no LDS round trip, no readlane and no exchange between waves, and the
// rows below are solved by the same instructions.  The four waves then apply
// the rank-16 update to the columns to the right on v_mfma_f64_16x16x4.
//
// Bound by the dependent FP64 chain of a column (rsq, two Newton steps, a
// scale, one update).
// ---------------------------------------------------------------------------
constexpr int kPanelThreads = 512;
constexpr int kTP = 144;  // row stride: 4 k-rows apart is 32 banks, so both halves of an MFMA operand read are conflict-free
static_assert(kTP >= 128 + 16, "trapezoid_factor parks a tile's rows in the padding");

// 1/sqrt(d) for d > 0 from the hardware estimate y (good to 2^-24).  CUBIC: one
// cubic step, y (1 + e/2 + 3e^2/8) with e = 1 - d y^2: four dependent operations,
// of which only the last rounds at the result's size.  Otherwise two Newton
// steps y (3 - d y^2) / 2, six operations (the FP32-storage forms: their factors
// are rounded to FP32, and results stay bit for bit what they were).
// Non-positive or NaN d gives NaN or a value the pivot check reports.
template <bool CUBIC>
__device__ __forceinline__ double rsqrt_f64(double d) {
    double y = __builtin_amdgcn_rsq(d);
    if (CUBIC) {
        const double e = fma(-(d * y), y, 1.0);
        return fma(y * e, fma(e, 0.375, 0.5), y);
    }
    const double h = 0.5 * d;
    y = y * fma(-h * y, y, 1.5);
    y = y * fma(-h * y, y, 1.5);
    return y;
}

template <int KQ>
__device__ __forceinline__ double quad_bcast_f64(double v) {
    constexpr int ctrl = KQ | (KQ << 2) | (KQ << 4) | (KQ << 6);  // quad_perm [KQ,KQ,KQ,KQ]
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_mov_dpp((int)(b & 0xffffffffLL), ctrl, 0xf, 0xf, false);
    const int hi = __builtin_amdgcn_mov_dpp((int)(b >> 32), ctrl, 0xf, 0xf, false);
    return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}

template <int LANE>
__device__ __forceinline__ double row_bcast_f64(double v) {  // lane LANE of every 16-lane row
    return __longlong_as_double(
        __builtin_amdgcn_update_dpp((long long)0, __double_as_longlong(v), 0x150 | LANE, 0xf, 0xf, true));
}

// acc += (lane C of the 16-lane row of src) * m.  src needs two wait states
// after the VALU instruction that wrote it (dpp_ready).
template <int C>
__device__ __forceinline__ void fnmac_bcast_f64(double& acc, double src, double m) {  // acc -= the same
    asm("v_fmac_f64_dpp %0, %1, -%2 row_newbcast:%3 row_mask:0xf bank_mask:0xf" : "+v"(acc) : "v"(src), "v"(m), "n"(C));
}
template <int C>
__device__ __forceinline__ void fmac_bcast_f64(double& acc, double src, double m) {
    asm("v_fmac_f64_dpp %0, %1, %2 row_newbcast:%3 row_mask:0xf bank_mask:0xf" : "+v"(acc) : "v"(src), "v"(m), "n"(C));
}
__device__ __forceinline__ void dpp_ready(double& v) { asm("s_nop 1" : "+v"(v)); }

// Columns J..15 of a phase: d the 16x16 diagonal tile (lane % 16 = row), a this
// lane's own row, whose columns go to out (row stride kTP) as they are done (rows above
// the tile's diagonal leave what is not read).  PIV: piv and rinv receive the pivot of
// column lane % 16 and its 1/sqrt.  The updates
// take their multipliers inside the multiply-add (4 cycles; a separate broadcast
// costs another 6 per multiplier).
template <int C>
__device__ __forceinline__ void factor16_update(double (&a)[16], double (&d)[16], double l, double dl) {
    if constexpr (C < 16) {
        fnmac_bcast_f64<C>(d[C], dl, dl);
        fnmac_bcast_f64<C>(a[C], dl, l);
        factor16_update<C + 1>(a, d, l, dl);
    }
}

template <int J, bool PIV, bool CUBIC>
__device__ __forceinline__ void factor16(double (&a)[16], double (&d)[16], int li, double& piv, double& rinv,
                                         double* out) {
    if constexpr (J < 16) {
        const double pv = row_bcast_f64<J>(d[J]);
        const double inv = rsqrt_f64<CUBIC>(pv);
        if (PIV) {
            piv = (li == J) ? pv : piv;
            rinv = (li == J) ? inv : rinv;
        }
        d[J] *= inv;
        a[J] *= inv;
        out[J * kTP] = a[J];
        dpp_ready(d[J]);
        factor16_update<J + 1>(a, d, a[J], d[J]);
        factor16<J + 1, PIV, CUBIC>(a, d, li, piv, rinv, out);
    }
}

// Tile (rt, ct) of the rank-16 update by phase p's columns (from j0):
// S(r, c) -= sum_k L(r, j0 + k) L(c, j0 + k).  The product is formed transposed:
// D lane (li, g) holds columns c = g + 4v of row r = li.  (The MFMA rounds like
// sequential multiply-adds in k.)  SUM: the products are summed first and the
// sum subtracted.
template <bool SUM>
__device__ __forceinline__ void trapezoid_tile(double (*S)[kTP], int j0, int rt, int ct, int li, int g) {
    double ac[4], br[4], cv[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        ac[k] = S[j0 + 4 * k + g][16 * ct + li];
        br[k] = S[j0 + 4 * k + g][16 * rt + li];
    }
#pragma unroll
    for (int v = 0; v < 4; ++v) cv[v] = S[16 * ct + g + 4 * v][16 * rt + li];
    d4 acc;
#pragma unroll
    for (int v = 0; v < 4; ++v) acc[v] = SUM ? 0.0 : cv[v];
#pragma unroll
    for (int k = 0; k < 4; ++k)
        acc = __builtin_amdgcn_mfma_f64_16x16x4f64(SUM ? ac[k] : -ac[k], br[k], acc, 0, 0, 0);
#pragma unroll
    for (int v = 0; v < 4; ++v) S[16 * ct + g + 4 * v][16 * rt + li] = SUM ? cv[v] - acc[v] : acc[v];
}

// Factor of S by kPanelThreads threads (eight waves).  RT row tiles of 16 (4: the
// diagonal block alone, its pivots and their 1/sqrt into piv[64], rinv[64]; 8:
// with the block below).  After a
// phase all waves update the next phase's columns, one tile each; the tiles
// further right are updated by the waves of the other two SIMDs while the
// factoring waves run the next phase.  Ends with a barrier.
template <int RT, bool CUBIC, bool SUM>
__device__ __forceinline__ void trapezoid_factor(double (*S)[kTP], double* piv, double* rinv) {
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int li = lane & 15, g = lane >> 4;
#pragma unroll 1
    for (int p = 0; p < 4; ++p) {
        const int j0 = 16 * p;
        if (w < RT / 4) {
            const int row = 64 * w + lane;
            double a[16], d[16], pv = 0.0, ri = 0.0;
#pragma unroll
            for (int q = 0; q < 16; ++q) {
                d[q] = S[j0 + q][j0 + li];
                a[q] = S[j0 + q][row];
            }
            // The other factoring wave may still be loading the diagonal tile, and with a
            // block below nobody reads that tile's factor: its rows go to the padding.
            const int orow = (RT == 8 && row >> 4 == p) ? 128 + li : row;
            factor16<0, RT == 4, CUBIC>(a, d, li, pv, ri, &S[j0][orow]);
            if (RT == 4 && lane < 16) {
                piv[j0 + lane] = pv;
                rinv[j0 + lane] = ri;
            }
        } else if (p > 0 && (w & 2)) {
            // waves 2, 3, 6, 7: the last phase's updates of the columns from tile p + 1
            int u = (w & 1) + 2 * (w >> 2);
#pragma unroll 1
            for (int ct = p + 1; ct < 4; ++ct)
#pragma unroll 1
                for (int rt = ct; rt < RT; ++rt, ++u)
                    if ((u & 3) == 0) trapezoid_tile<SUM>(S, j0 - 16, rt, ct, li, g);
        }
        __syncthreads();
        if (p < 3) {
            if (p + 1 + w < RT) trapezoid_tile<SUM>(S, j0, p + 1 + w, p + 1, li, g);
            __syncthreads();
        }
    }
}

// Blocks handed to other workgroups are stored with relaxed agent-scope atomics
// (write-through), so publishing one needs no cache write-back: every wave waits
// until its stores have been performed, then one thread sets the flag (0.9 us;
// 3.5 us with a release fence in every wave).  Their readers take one acquire
// fence after the flag and load plainly, so that the workgroups of an XCD share
// the block in its L2 (loads that bypass it took 1.9 us instead of 0.7 us with 32
// workgroups reading one block).
template <typename T>
__device__ __forceinline__ void put_shared(T* p, T v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// After trapezoid_factor<4>: the factor of diagonal block k to global memory
// (blk, leading dimension ld; the upper triangle as zeros), ldiag[64k + i] =
// log L_ii, info = lowest failing row + 1, and the block's inverse to Dinv (FP64,
// 64x64 column-major) by 16x16 blocks: DPP substitution inside the diagonal
// blocks, f64 MFMA for the block rows.  The inverse is left in rows 64..127 of
// S, S[c][64 + r] = X(r, c).  rinv, piv: 64 doubles of LDS each.  SH: other
// workgroups of the launch read Dinv (put_shared).  Without `put` nothing is stored.
template <typename T, bool SH = false>
__device__ __forceinline__ void diag_finish(T* __restrict__ blk, int64_t ld, int64_t k, double* __restrict__ Dinv,
                                            double* __restrict__ ldiag, int* __restrict__ info, double (*S)[kTP],
                                            const double* rinv, const double* piv, bool put = true) {
    const int t = threadIdx.x, i = t & 63, w = t >> 6;
#pragma unroll
    for (int q = 0; q < 8; ++q) {
        const int c = 8 * w + q;
        if (i < c) S[c][i] = 0.0;  // what the factorization left above the diagonal
        if (put) blk[i + (int64_t)c * ld] = (i < c) ? (T)0 : (T)S[c][i];
    }
    __syncthreads();
    if (t < 64) S[t][t] = 0.0;  // the substitution uses the strictly lower part
    if (put && t < 64) {
        ldiag[k * 64 + t] = 0.5 * log(piv[t]);
        const unsigned long long bad = __ballot(!(piv[t] > 0.0));
        if (t == 0 && bad) report_minor(info, (int)(k * 64 + __ffsll((long long)bad)));
    }
    __syncthreads();
    // Inverse by 16x16 blocks.  (1) Each wave inverts its diagonal block by
    // forward substitution, four lanes per column exchanging values by DPP (16
    // dependent steps).  (2) Block rows bi = 1..3 in turn, wave j < bi forming
    // X_{bi,j} = -X_{bi,bi} T, T = sum_{j <= kb < bi} L_{bi,kb} X_{kb,j}, on
    // v_mfma_f64_16x16x4.  T is left in the D layout (lane (li, g) holds rows
    // g + 4v of column li), which is the A-operand layout of T^T with k = g + 4v,
    // so the product is taken as Y^T = T^T X_{bi,bi}^T without leaving registers.
    const int lane = t & 63, li = lane & 15, g = lane >> 4;
    if (w < 4) {
        const int c = lane >> 2, q = lane & 3, base = 16 * w;
        double b[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) b[r] = (4 * r + q == c) ? 1.0 : 0.0;
#pragma unroll
        for (int kk = 0; kk < 16; ++kk) {
            const int kr = kk >> 2;
            double xk = b[kr] * rinv[base + kk];
            switch (kk & 3) {
                case 0: xk = quad_bcast_f64<0>(xk); break;
                case 1: xk = quad_bcast_f64<1>(xk); break;
                case 2: xk = quad_bcast_f64<2>(xk); break;
                default: xk = quad_bcast_f64<3>(xk); break;
            }
            if (q == (kk & 3)) b[kr] = xk;
#pragma unroll
            for (int r = 0; r < 4; ++r) b[r] -= S[base + kk][base + 4 * r + q] * xk;
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) S[base + c][64 + base + 4 * r + q] = b[r];
        for (int r = q; r < base; r += 4) S[base + c][64 + r] = 0.0;  // above the diagonal block
    }
    __syncthreads();
#pragma unroll
    for (int bi = 1; bi < 4; ++bi) {
        if (w < bi) {
            const int r0 = 16 * bi, c0 = 16 * w;
            d4 acc = d4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
            for (int kb = 0; kb < r0; kb += 4)  // X is zero above its diagonal blocks
                acc = __builtin_amdgcn_mfma_f64_16x16x4f64(S[kb + g][r0 + li], S[c0 + li][64 + kb + g], acc, 0, 0, 0);
            d4 y = d4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
            for (int v = 0; v < 4; ++v)
                y = __builtin_amdgcn_mfma_f64_16x16x4f64(acc[v], S[r0 + g + 4 * v][64 + r0 + li], y, 0, 0, 0);
#pragma unroll
            for (int v = 0; v < 4; ++v) S[c0 + g + 4 * v][64 + r0 + li] = -y[v];
        }
        __syncthreads();
    }
    if (!put) return;
    double* D = Dinv + k * 64 * 64;
    for (int e = t; e < 64 * 64; e += kPanelThreads) {
        if (SH) put_shared(D + e, S[e >> 6][64 + (e & 63)]);
        else D[e] = S[e >> 6][64 + (e & 63)];
    }
}

// One 64x64 diagonal block per problem of a batch: FP32 storage, factored from
// its FP64 tile (Dsrc, the layout of Dinv).  SOLVE: with the rows below it, A = A Dinv^T;
// then every 64-row block below has a workgroup, which factors the block for itself (the
// first stores it), and the solve's launch and load latency leave the chain.
template <bool SOLVE>
__global__ __launch_bounds__(kPanelThreads) void k_potrf_diag(float* __restrict__ A, int64_t ld, int64_t k,
                                                    double* __restrict__ Dinv, double* __restrict__ ldiag,
                                                    int* __restrict__ info, int64_t sA, int64_t sD, int64_t sL,
                                                    const double* __restrict__ Dsrc) {
    __shared__ double S[64][kTP];
    __shared__ double rinv[64];
    __shared__ double piv[64];
    const int64_t pr = blockIdx.y;
    Dsrc += pr * sD + k * 64 * 64;
    A += pr * sA + k * 64 * (ld + 1);
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int li = lane & 15, g = lane >> 4;
    float* const p = A + 64 * ((int64_t)blockIdx.x + 1) + 16 * (w & 3) + li;  // wave w: rows 16 (w % 4) .. of its block
    float a[4][4];
    if (SOLVE)
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
            for (int s = 0; s < 4; ++s) a[q][s] = p[(16 * q + 4 * g + s) * ld];
    for (int e = threadIdx.x; e < 64 * 64; e += kPanelThreads) S[e >> 6][e & 63] = Dsrc[e];
    __syncthreads();
    trapezoid_factor<4, false, true>(S, piv, rinv);
    diag_finish(A, ld, k, Dinv + pr * sD, ldiag + pr * sL, info + pr, S, rinv, piv, !SOLVE || blockIdx.x == 0);
    if (!SOLVE) return;
    // as k_panel_solve; waves 0 - 3 the 16 columns of tiles 0 and 3, the others of 1 and 2
    d4 acc[2] = {d4{0.0, 0.0, 0.0, 0.0}, d4{0.0, 0.0, 0.0, 0.0}};
    const int j0 = w < 4 ? 0 : 1, j1 = 3 - j0;
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            const double* X = &S[16 * q + 4 * g + s][64 + li];
            if (q <= j0) acc[0] = __builtin_amdgcn_mfma_f64_16x16x4f64(X[16 * j0], (double)a[q][s], acc[0], 0, 0, 0);
            if (q <= j1) acc[1] = __builtin_amdgcn_mfma_f64_16x16x4f64(X[16 * j1], (double)a[q][s], acc[1], 0, 0, 0);
        }
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        p[(16 * j0 + g + 4 * v) * ld] = (float)acc[0][v];
        p[(16 * j1 + g + 4 * v) * ld] = (float)acc[1][v];
    }
}

// The rows below a diagonal block of a batch's factorization: A = A Dinv^T in place, A (M x
// 64, FP32), Dinv the block's inverse (FP64, lower triangular), FP64 products with one
// rounding.  A wave per 16 rows, all of its operand loaded at once; Dinv's lower tiles go
// to LDS once per workgroup and its zero tiles are skipped.
// Bound by A's traffic for many rows, by one load latency and 40 matrix instructions for few.
// (As a general product in place, a wave with 32 rows and half of the columns loading two
// chunks ahead: 112 us for 16 problems of up to 8128 rows beside the other streams' products,
// 47 here; 6.1 and 4.5 in a batch of 64 .. 2048 points.)
__global__ __launch_bounds__(256) void k_panel_solve(float* __restrict__ A, int64_t ld,
                                                     const double* __restrict__ Dinv, int64_t sA, int64_t sD) {
    constexpr int LP = 68;  // 4 rows of k are 32 banks apart: both halves of an operand read are conflict-free
    __shared__ double S[64][LP];
    A += blockIdx.y * sA + 64 * (int64_t)blockIdx.x;
    Dinv += blockIdx.y * sD;
    const int t = threadIdx.x, lane = t & 63, w = __builtin_amdgcn_readfirstlane(t >> 6);
    const int li = lane & 15, g = lane >> 4;
    float* p = A + 16 * w + li;
    float a[4][4];
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
        for (int s = 0; s < 4; ++s) a[q][s] = p[(16 * q + 4 * g + s) * ld];
    double d[16];
#pragma unroll
    for (int u = 0; u < 16; ++u) {  // column w + 4u: rows from its 16-block down
        const int k = w + 4 * u;
        d[u] = lane >= (k & ~15) ? Dinv[lane + 64 * k] : 0.0;
    }
#pragma unroll
    for (int u = 0; u < 16; ++u) S[w + 4 * u][lane] = d[u];
    __syncthreads();
    // lane (li, g) of the (transposed) product holds columns g + 4v of row li; the
    // sums run over k in the order of the other products (k = 4g + s of each 16 in step s)
    d4 acc[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[j] = d4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
        for (int s = 0; s < 4; ++s)
#pragma unroll
            for (int j = q; j < 4; ++j)
                acc[j] = __builtin_amdgcn_mfma_f64_16x16x4f64(S[16 * q + 4 * g + s][16 * j + li], (double)a[q][s],
                                                              acc[j], 0, 0, 0);
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int v = 0; v < 4; ++v) p[(16 * j + g + 4 * v) * ld] = (float)acc[j][v];
}

// Up to this many row blocks, a workgroup to a CU, the two are one launch (a batch of 128, 64 ..
// 2048 points: 21.3 ms as two, 20.5 with any line from 64 to 1024; one of 2048 problems: 62.6, and
// 62.3 with a line at 256, 63.0 at 512, 63.7 at 4096, as the factors are then repeated on a full chip).
static const int64_t kStepFused = 256;
void potrf_step_f32_batched(hipStream_t s, float* A, int64_t ld, int64_t k, int64_t M, double* Dinv, double* ldiag,
                            int* info, int batch, int64_t sA, int64_t sD, int64_t sL, const double* Dacc) {
    if (batch <= 0) return;
    if (M > 0 && M / 64 * batch <= kStepFused) {
        hipLaunchKernelGGL(k_potrf_diag<true>, dim3((unsigned)(M / 64), (unsigned)batch), dim3(kPanelThreads), 0, s, A, ld,
                           k, Dinv, ldiag, info, sA, sD, sL, Dacc);
        return;
    }
    hipLaunchKernelGGL(k_potrf_diag<false>, dim3(1, (unsigned)batch), dim3(kPanelThreads), 0, s, A, ld, k, Dinv, ldiag,
                       info, sA, sD, sL, Dacc);
    if (M > 0)
        hipLaunchKernelGGL(k_panel_solve, dim3((unsigned)(M / 64), (unsigned)batch), dim3(256), 0, s,
                           A + (k + 1) * 64 + k * 64 * ld, ld, Dinv + k * 64 * 64, sA, sD);
}

// ---------------------------------------------------------------------------
// One outer panel of the blocked Cholesky in a single launch: columns
// [K0, K0 + 64nc), nc <= kPanelMaxBlocks column blocks, all rows from K0.
// Workgroup rb owns the 64-row block rb (rows K0 + 64rb ..) for the whole
// panel.  For each column block c < rb it
//   (1) waits for the updated (not yet factored) diagonal block c,
//   (2) factors it for itself together with its own block A_{rb,c}
//       (trapezoid_factor), which leaves L_{rb,c},
//   (3) subtracts L_{rb,c} L_{rb,c}^T from its own diagonal block (kept in
//       registers) and L_{rb,c} L_{c2,c}^T from its blocks in the later panel
//       columns, reading L_{c2,c} once workgroup c2 has published it.  The block
//       of column c + 1 stays in LDS for the next step.
// Workgroup c + 1 publishes its diagonal block right after its update by column
// c, before it is factored: no factor, inverse or solve of another workgroup is
// on the chain from one diagonal block to the next, only one 64-column
// trapezoid factor, one 64x64 update, and the hand-over of a 64x64 block.  (With
// one factor and inverse per block, handed to the workgroups below to multiply
// by, the chain was 24-26 us per 64 columns.)  The diagonal block's own
// workgroup stores its factor and inverse beside that chain.
//
// T = float (the mixed-precision form): A is FP32; the diagonal blocks come
// from, and are published in, their FP64 copies Dpub = Dacc (64x64 column-major,
// tile j at 4096j).  Block products are FP64 on the stored FP32 values with one
// rounding to FP32 per stored result.  T = double: Dpub is workspace for the
// panel's blocks 1 .. nc - 1 (tile c at 4096c); block 0 is read from A by every
// workgroup, so its factor goes to tile 0 of Dpub first and the last workgroup
// to report its read (or, for workgroup 0, that tile) copies it into A.
//
// rhs (optional, FP64 storage only): a vector b of N rows that leaves as
// y = L^-1 b, the forward solve carried along one column block behind:
// workgroup c stores y_c = Dinv_c b_c and publishes it, every workgroup below
// subtracts L_{rb,c} y_c from its block of b.
//
// Ordering: each workgroup takes a ticket (atomic counter) as its logical row
// block, so block rb is held by a workgroup that started after those of every
// lower block; all waits are on lower blocks, which have started and do not
// wait on higher ones, so every wait ends.  Flags carry the launch's epoch.
// A wait that outlasts maxpoll polls (2^20 by default: a second or more, far
// beyond any legitimate wait) stores kPanelWaitTimeout in info and leaves the
// kernel; the callers report it as a device error.
//
// sync (kPanelSyncWords words), P = kPanelMaxBlocks: [0, P) diagonal-block flags,
// [P, P + P^2) flags of L_{c2,c} (P + P c2 + c), then P flags of y_c, the counter
// of block 0's readers and the ticket counter; base: tickets handed out before
// this launch (both counters advance by the grid size per launch).
// ---------------------------------------------------------------------------
__device__ __forceinline__ bool panel_wait(unsigned* f, unsigned epoch, int* info, int* s_ok, unsigned maxpoll) {
    if (threadIdx.x == 0) {
        int ok = 0;
        for (unsigned n = 0; n < maxpoll; ++n) {
            ok = __hip_atomic_load(f, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == epoch;
            if (ok) break;
            __builtin_amdgcn_s_sleep(1);
        }
        if (!ok) atomicCAS(info, 0, kPanelWaitTimeout);
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
        *s_ok = ok;
    }
    __syncthreads();
    return *s_ok != 0;
}

// the same for the flags f[stride * i], lo <= i < hi (hi - lo <= 64): one lane each
__device__ __forceinline__ bool panel_wait_all(unsigned* f, int stride, int lo, int hi, unsigned epoch, int* info,
                                               int* s_ok, unsigned maxpoll) {
    if (threadIdx.x < 64) {
        unsigned* fi = f + stride * (lo + ((int)threadIdx.x < hi - lo ? (int)threadIdx.x : 0));
        int ok = 0;
        for (unsigned n = 0; n < maxpoll; ++n) {
            ok = !__ballot(__hip_atomic_load(fi, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != epoch);
            if (ok) break;
            __builtin_amdgcn_s_sleep(1);
        }
        if (!ok && threadIdx.x == 0) atomicCAS(info, 0, kPanelWaitTimeout);
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
        if (threadIdx.x == 0) *s_ok = ok;
    }
    __syncthreads();
    return *s_ok != 0;
}

__device__ __forceinline__ void panel_publish(unsigned* f, unsigned epoch) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (threadIdx.x == 0) __hip_atomic_store(f, epoch, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// sum_k M(e, k) y_k over a 64x64 block M (element (e, k) at M[e + k ld]), e < 64 in
// threads t < 64; red: kPanelThreads doubles of LDS.  Ends with a barrier.
__device__ __forceinline__ double blk_matvec(const double* M, int64_t ld, const double* y, double* red) {
    const int e = threadIdx.x & 63, pq = threadIdx.x >> 6;
    double sum = 0.0;
#pragma unroll
    for (int u = 0; u < 8; ++u) sum += M[e + (int64_t)(8 * pq + u) * ld] * y[8 * pq + u];
    red[threadIdx.x] = sum;
    __syncthreads();
    sum = 0.0;
    if (threadIdx.x < 64)
#pragma unroll
        for (int q = 0; q < 8; ++q) sum += red[e + 64 * q];
    __syncthreads();
    return sum;
}

// The lower 16x16 tiles of a 64x64 block over eight waves: tile u of wave w (two
// tiles for waves 0 and 1) is (row, column) (diag_rt, diag_ct).
__device__ __forceinline__ int diag_rt(int w, int u) { return u ? 3 : w < 1 ? 0 : w < 3 ? 1 : w < 6 ? 2 : 3; }
__device__ __forceinline__ int diag_ct(int w, int u) { return u ? 2 + w : w < 1 ? 0 : w < 3 ? w - 1 : w < 6 ? w - 3 : w - 6; }

template <typename T, int NC>
__global__ __launch_bounds__(kPanelThreads) void k_potrf_panel(
    T* A, int64_t ld, int64_t K0, int nc, double* Dinv, double* __restrict__ ldiag, int* __restrict__ info,
    unsigned* __restrict__ sync, unsigned epoch, unsigned base, double* Dpub,
    unsigned maxpoll, double* rhs) {
    constexpr bool kF64 = sizeof(T) == 8;
    constexpr int P = kPanelMaxBlocks;
    __shared__ double S[64][kTP];
    __shared__ double rinv[64];
    __shared__ double piv[64];
    __shared__ double red[kPanelThreads];
    __shared__ unsigned s_id;
    __shared__ int s_ok;
    if (threadIdx.x == 0) s_id = atomicAdd(&sync[kPanelSyncWords - 1], 1u) - base;
    __syncthreads();
    const int rb = __builtin_amdgcn_readfirstlane((int)s_id);
    unsigned* const yflag = sync + P + P * P;
    unsigned* const readers = yflag + P;
    const int t = threadIdx.x, lane = t & 63, w = __builtin_amdgcn_readfirstlane(t >> 6);
    const int li = lane & 15, g = lane >> 4, r64 = t & 63;
    const int64_t kb0 = K0 / 64;
    T* const A0 = A + K0 + K0 * ld;           // the panel's first block
    T* const Arow = A0 + 64 * (int64_t)rb;    // row block rb, column 0
    if (!kF64) Dpub += kb0 * 4096;
    // what column block c is solved with: FP64 storage, the diagonal block as
    // published (block 0 is read from A); FP32 storage, its inverse
    double dv[8];
    auto diag_fetch = [&](int c) {
        const bool ina = kF64 && c == 0;
        const double* D = ina ? (const double*)A0 : kF64 ? Dpub + 4096 * c : Dinv + 4096 * (kb0 + c);
        const int64_t ldd = ina ? ld : 64;
#pragma unroll
        for (int q = 0; q < 8; ++q) dv[q] = D[r64 + (int64_t)(w + 8 * q) * ldd];
    };
    auto diag_put = [&]() {
#pragma unroll
        for (int q = 0; q < 8; ++q) S[w + 8 * q][r64] = dv[q];
    };
    // the last workgroup to report copies block 0's factor into A
    auto report_read = [&]() {
        if (!kF64) {  // (nothing is held back; the counter advances with the tickets)
            if (t == 0) atomicAdd(readers, 1u);
            return;
        }
        __syncthreads();
        if (t == 0) {
            const unsigned n = __hip_atomic_fetch_add(readers, 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT) - base;
            s_ok = n + 1 == gridDim.x;
        }
        __syncthreads();
        if (s_ok) {
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
#pragma unroll
            for (int q = 0; q < 8; ++q) A0[r64 + (int64_t)(w + 8 * q) * ld] = (T)Dpub[r64 + 64 * (w + 8 * q)];
        }
    };
    const int cend = rb < nc ? rb : nc;  // columns left of the own diagonal block
    // The own blocks of columns c + 1 .. c + NC - 1 stay in registers as transposed
    // 16x16 MFMA tiles until their column is reached: wave w has rows 16(w%4)..,
    // columns 32(w/4).. of each (two tiles).  (Read and written back in global
    // memory on every step, an update took 4 us against 1.7 us of products.)
    const int r0 = 16 * (w & 3) + li, q0 = 32 * (w >> 2);
    T own[NC - 1][2][4];
    d4 dacc[2];
    if (rb > 0) {
#pragma unroll
        for (int q = 0; q < 8; ++q) S[w + 8 * q][64 + r64] = (double)Arow[r64 + (int64_t)(w + 8 * q) * ld];
        if (kF64) {
            diag_fetch(0);
            diag_put();
        }
#pragma unroll
        for (int i = 0; i < NC - 1; ++i)
            if (i + 1 < cend)
#pragma unroll
                for (int j = 0; j < 2; ++j)
#pragma unroll
                    for (int v = 0; v < 4; ++v)
                        own[i][j][v] = Arow[r0 + (int64_t)(64 * (i + 1) + q0 + 16 * j + g + 4 * v) * ld];
        if (rb < nc) {  // the own diagonal block's lower tiles
            const double* D = kF64 ? (const double*)(Arow + 64 * (int64_t)rb * ld) : Dpub + 4096 * rb;
            const int64_t ldd = kF64 ? ld : 64;
#pragma unroll
            for (int u = 0; u < 2; ++u)
                if (u < 1 || w < 2)
#pragma unroll
                    for (int v = 0; v < 4; ++v)
                        dacc[u][v] = D[(16 * diag_rt(w, u) + li) + (int64_t)(16 * diag_ct(w, u) + g + 4 * v) * ldd];
        }
        report_read();
        if (!kF64) {
            if (!panel_wait(&sync[0], epoch, info, &s_ok, maxpoll)) return;
            diag_fetch(0);
            diag_put();
        }
    }
#pragma unroll 1
    for (int c = 0; c < cend; ++c) {
        __syncthreads();
        if constexpr (kF64) {
            trapezoid_factor<8, true, false>(S, piv, rinv);
        } else {
            // L_{rb,c} = A_{rb,c} Dinv_c^T
            d4 acc[2] = {d4{0.0, 0.0, 0.0, 0.0}, d4{0.0, 0.0, 0.0, 0.0}};
#pragma unroll 8
            for (int k0 = 0; k0 < 64; k0 += 4) {
                const double b = S[k0 + g][64 + r0];
#pragma unroll
                for (int j = 0; j < 2; ++j)
                    acc[j] = __builtin_amdgcn_mfma_f64_16x16x4f64(S[k0 + g][q0 + 16 * j + li], b, acc[j], 0, 0, 0);
            }
            __syncthreads();
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int v = 0; v < 4; ++v) S[q0 + 16 * j + g + 4 * v][64 + r0] = acc[j][v];
            __syncthreads();
        }
        // L_{rb,c} to global memory, rounded to T; LDS keeps the stored values
        {
            T* Ab = Arow + 64 * (int64_t)c * ld;
#pragma unroll
            for (int q = 0; q < 8; ++q) {
                const T v = (T)S[w + 8 * q][64 + r64];
                if (rb < nc) put_shared(Ab + r64 + (int64_t)(w + 8 * q) * ld, v);
                else Ab[r64 + (int64_t)(w + 8 * q) * ld] = v;
                if (!kF64) S[w + 8 * q][64 + r64] = (double)v;
            }
            if (!kF64) __syncthreads();
        }
        if (rb < nc) panel_publish(&sync[P + P * rb + c], epoch);
        // the own diagonal block: D -= L_{rb,c} L_{rb,c}^T, lower tiles (here and below the
        // products are summed before they are subtracted: one rounding at the block's size
        // for 64, where accumulating into the block took the log-determinant's error to twice)
        auto diag_update = [&]() {
            d4 sum[2] = {d4{0.0, 0.0, 0.0, 0.0}, d4{0.0, 0.0, 0.0, 0.0}};
#pragma unroll 8
            for (int k0 = 0; k0 < 64; k0 += 4) {
                const double* Sk = &S[k0 + g][64 + li];
#pragma unroll
                for (int u = 0; u < 2; ++u)
                    if (u < 1 || w < 2)
                        sum[u] = __builtin_amdgcn_mfma_f64_16x16x4f64(Sk[16 * diag_ct(w, u)], Sk[16 * diag_rt(w, u)],
                                                                      sum[u], 0, 0, 0);
            }
#pragma unroll
            for (int u = 0; u < 2; ++u) dacc[u] -= sum[u];
        };
        if (rb == c + 1 && rb < nc) {
            // the next diagonal block: published before it is factored
            diag_update();
            double* D = Dpub + 4096 * rb;
#pragma unroll
            for (int u = 0; u < 2; ++u)
                if (u < 1 || w < 2)
#pragma unroll
                    for (int v = 0; v < 4; ++v) {
                        const int row = 16 * diag_rt(w, u) + li, col = 16 * diag_ct(w, u) + g + 4 * v;
                        if (kF64) put_shared(D + row + 64 * col, (double)dacc[u][v]);
                        S[col][row] = dacc[u][v];
                    }
            if (kF64) panel_publish(&sync[rb], epoch);
        }
        // The own blocks of the later panel columns, nearest last: its result
        // goes to LDS as the next step's block.  One wait for all of them; the
        // next L_{c2,c} is loaded while the current one is multiplied.
        if (cend - 1 > c) {
            if (!panel_wait_all(sync + P + c, P, c + 1, cend, epoch, info, &s_ok, maxpoll)) return;
            T lv[8];
            auto fetch = [&](int c2) {
                const T* Lc2 = A0 + 64 * (int64_t)c2 + 64 * (int64_t)c * ld;
#pragma unroll
                for (int q = 0; q < 8; ++q) lv[q] = Lc2[r64 + (int64_t)(w + 8 * q) * ld];
            };
            fetch(cend - 1);
#pragma unroll
            for (int i = NC - 2; i >= 0; --i) {
                const int c2 = c + 1 + i;
                if (c2 >= cend) continue;
#pragma unroll
                for (int q = 0; q < 8; ++q) S[w + 8 * q][r64] = (double)lv[q];
                __syncthreads();
                if (i > 0) fetch(c2 - 1);
                d4 acc[2] = {d4{0.0, 0.0, 0.0, 0.0}, d4{0.0, 0.0, 0.0, 0.0}};
#pragma unroll 8
                for (int k0 = 0; k0 < 64; k0 += 4) {
                    const double b = S[k0 + g][64 + r0];
#pragma unroll
                    for (int j = 0; j < 2; ++j)
                        acc[j] = __builtin_amdgcn_mfma_f64_16x16x4f64(S[k0 + g][q0 + 16 * j + li], b, acc[j], 0, 0, 0);
                }
#pragma unroll
                for (int j = 0; j < 2; ++j)
#pragma unroll
                    for (int v = 0; v < 4; ++v) own[i][j][v] = (T)((double)own[i][j][v] - acc[j][v]);
                if (i > 0) __syncthreads();  // the operand is free
            }
        }
        if (c + 1 < cend) {
            // the next diagonal block (published long before this workgroup gets
            // here, unless it is the next but one): its load is covered by the
            // update of the own diagonal block
            if (!panel_wait(&sync[c + 1], epoch, info, &s_ok, maxpoll)) return;
            diag_fetch(c + 1);
            if (rb < nc) diag_update();
            __syncthreads();  // S is no longer read
            diag_put();
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int v = 0; v < 4; ++v) S[q0 + 16 * j + g + 4 * v][64 + r0] = (double)own[0][j][v];
#pragma unroll
            for (int i = 0; i + 1 < NC - 1; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j)
#pragma unroll
                    for (int v = 0; v < 4; ++v) own[i][j][v] = own[i + 1][j][v];
        }
        if (rhs && c > 0) {
            if (!panel_wait(&yflag[c - 1], epoch, info, &s_ok, maxpoll)) return;
            const double u = blk_matvec((const double*)(Arow + 64 * (int64_t)(c - 1) * ld), ld, rhs + K0 + 64 * (c - 1), red);
            if (t < 64) rhs[K0 + 64 * (int64_t)rb + t] -= u;
        }
    }
    if (rb < nc) {
        // diagonal block rb with all its updates: in S (left there by the last
        // column), or for rb = 0 as stored
        const int64_t kc = kb0 + rb;
        if (rb == 0) {
            if (kF64) {
                diag_fetch(0);
                diag_put();
            } else {
#pragma unroll
                for (int q = 0; q < 8; ++q) S[w + 8 * q][r64] = Dpub[r64 + 64 * (w + 8 * q)];
            }
        }
        __syncthreads();
        trapezoid_factor<4, kF64, false>(S, piv, rinv);
        const bool hold = kF64 && rb == 0;  // A's block 0 may still be read
        diag_finish<T, !kF64>(hold ? (T*)Dpub : Arow + 64 * (int64_t)rb * ld, hold ? 64 : ld, kc, Dinv, ldiag, info, S,
                              rinv, piv);
        if (!kF64) panel_publish(&sync[rb], epoch);
        if (rb == 0) {
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
            report_read();
        }
        if (rhs) {  // y_c = L_cc^-1 b_c from the inverse left in S
            double* bc = rhs + K0 + 64 * (int64_t)rb;
            if (rb > 0) {
                if (!panel_wait(&yflag[rb - 1], epoch, info, &s_ok, maxpoll)) return;
                const double u = blk_matvec((const double*)(Arow + 64 * (int64_t)(rb - 1) * ld), ld, bc - 64, red);
                if (t < 64) bc[t] -= u;
                __syncthreads();
            }
            const double y = blk_matvec(&S[0][64], kTP, bc, red);
            if (t < 64) put_shared(bc + t, y);
            panel_publish(&yflag[rb], epoch);
        }
    } else if (rhs) {
        if (!panel_wait(&yflag[nc - 1], epoch, info, &s_ok, maxpoll)) return;
        const double u = blk_matvec((const double*)(Arow + 64 * (int64_t)(nc - 1) * ld), ld, rhs + K0 + 64 * (nc - 1), red);
        if (t < 64) rhs[K0 + 64 * (int64_t)rb + t] -= u;
    }
}

void potrf_panel_f64(hipStream_t s, double* A, int64_t ld, int64_t K0, int nc, int64_t nrb, double* Dinv,
                     double* ldiag, int* info, unsigned* sync, unsigned epoch, unsigned base, double* Dpub,
                     unsigned maxpoll, double* rhs) {
    hipLaunchKernelGGL((k_potrf_panel<double, kPanelBlocksF64>), dim3((unsigned)nrb), dim3(kPanelThreads), 0, s, A, ld, K0, nc, Dinv, ldiag, info,
                       sync, epoch, base, Dpub, maxpoll, rhs);
}

void potrf_panel_mixed(hipStream_t s, float* A, int64_t ld, int64_t K0, int nc, int64_t nrb, double* Dinv,
                       double* ldiag, int* info, unsigned* sync, unsigned epoch, unsigned base, double* Dacc,
                       unsigned maxpoll) {
    hipLaunchKernelGGL((k_potrf_panel<float, kPanelBlocksF32>), dim3((unsigned)nrb), dim3(kPanelThreads), 0, s, A, ld, K0, nc, Dinv, ldiag, info,
                       sync, epoch, base, Dacc, maxpoll, (double*)nullptr);
}

// ---------------------------------------------------------------------------
// FP64 diagonal tiles of the mixed-precision factorization.  Every FP32 update
// A -= P P^T that reaches diagonal tiles is also applied to their FP64 copies
// D_j -= P_j P_j^T, where P_j is the FP32 panel's rows of block j: the products
// of FP32 values are exact in FP64 and are accumulated in FP64, so the diagonal
// blocks that are factored carry no FP32 accumulation error.
// D: first tile to update (64x64 column-major tiles, consecutive), P: the panel
// rows of that tile (leading dimension ldp), kdepth: panel width (multiple of 64).
//
// A wave per lower 16x16 tile (ten per block; the strictly upper ones are never
// read), straight from global memory with 64 k loaded ahead: bound by its chain of
// kdepth / 4 matrix instructions, 0.11 us per 16 k.  (A workgroup per block that
// staged 16 k at a time in LDS took a load latency and two barriers for each, about
// 1 us: depth 64 / 128 / 256 / 512 on eight blocks 7.7 / 12 / 18.5 / 36 us.)
// The sums run over k in order and are subtracted at the end.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_dacc_update(double* __restrict__ D, const float* __restrict__ P, int64_t ldp,
                                                     int64_t kdepth, int64_t nwaves, int64_t sD, int64_t sP) {
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int64_t id = (int64_t)blockIdx.x * 4 + w;
    if (id >= nwaves) return;
    const int64_t j = id / 10;
    const int u = (int)(id - 10 * j);
    const int rt = u < 1 ? 0 : u < 3 ? 1 : u < 6 ? 2 : 3, ct = u - rt * (rt + 1) / 2;
    D += blockIdx.y * sD + j * 64 * 64;
    P += blockIdx.y * sP + j * 64;
    const int l16 = lane & 15, lk = lane >> 4;
    // lane (l16, lk) of the (transposed) product holds columns lk + 4v of row l16
    double* d = D + (16 * rt + l16) + (16 * ct + lk) * 64;
    double old[4];
#pragma unroll
    for (int v = 0; v < 4; ++v) old[v] = d[4 * v * 64];
    const float* pr = P + 16 * rt + l16 + lk * ldp;
    const float* pc = P + 16 * ct + l16 + lk * ldp;
    float r[2][16], c[2][16];
    auto load = [&](int st) {
#pragma unroll
        for (int q = 0; q < 16; ++q) {
            r[st][q] = pr[4 * q * ldp];
            c[st][q] = pc[4 * q * ldp];
        }
        pr += 64 * ldp;
        pc += 64 * ldp;
    };
    d4 acc = d4{0.0, 0.0, 0.0, 0.0};
    auto mult = [&](int st) {
#pragma unroll
        for (int q = 0; q < 16; ++q)
            acc = __builtin_amdgcn_mfma_f64_16x16x4f64((double)c[st][q], (double)r[st][q], acc, 0, 0, 0);
    };
    const int nch = (int)(kdepth / 64);
    load(0);
    int q = 0;
    for (; q + 2 < nch; q += 2) {
        load(1);
        mult(0);
        load(0);
        mult(1);
    }
    if (q + 1 < nch) {
        load(1);
        mult(0);
        mult(1);
    } else {
        mult(0);
    }
#pragma unroll
    for (int v = 0; v < 4; ++v) d[4 * v * 64] = old[v] - acc[v];
}

void dacc_update(hipStream_t s, double* D, const float* P, int64_t ldp, int64_t ntiles, int64_t kdepth, int batch,
                 int64_t sD, int64_t sP) {
    if (ntiles <= 0 || batch <= 0 || kdepth <= 0) return;
    const int64_t nwaves = 10 * ntiles;
    hipLaunchKernelGGL(k_dacc_update, dim3((unsigned)((nwaves + 3) / 4), (unsigned)batch), dim3(256), 0, s, D, P, ldp,
                       kdepth, nwaves, sD, sP);
}

// ---------------------------------------------------------------------------
// Blocked triangular solves with one vector (L y = b, L^T x = b).  Step i:
// every workgroup forms x_i = Dinv_i b_i (Dinv_i^T b_i for the transpose) and
// workgroup w updates the pending block r of b with the tile L(r,i) (or L(i,r)^T).
// ---------------------------------------------------------------------------
__device__ __forceinline__ double block_sum4(double v, double* red) {
    // 256 threads: thread t holds the partial of element (t & 63), part (t >> 6)
    const int t = threadIdx.x;
    red[t] = v;
    __syncthreads();
    double s = 0.0;
    if (t < 64) s = red[t] + red[t + 64] + red[t + 128] + red[t + 192];
    __syncthreads();
    return s;
}

__global__ __launch_bounds__(256) void k_trsv_step(const double* __restrict__ L, int64_t ld,
                                                   const double* __restrict__ Dinv, int64_t T, int64_t i,
                                                   double* __restrict__ b, double* __restrict__ x, int trans) {
    __shared__ double red[256];
    __shared__ double xi[64];
    const int t = threadIdx.x, e = t & 63, p = t >> 6;
    const double* D = Dinv + i * 64 * 64;
    // x_i = D b_i (trans: D^T b_i); element e, columns/rows p*16..p*16+15
    double s = 0.0;
#pragma unroll
    for (int u = 0; u < 16; ++u) {
        const int c = p * 16 + u;
        s += (trans ? D[c + e * 64] : D[e + c * 64]) * b[i * 64 + c];
    }
    s = block_sum4(s, red);
    if (t < 64) xi[t] = s;
    __syncthreads();
    if (blockIdx.x == 0 && t < 64) x[i * 64 + t] = xi[t];
    // pending block for this workgroup
    const int64_t w = blockIdx.x;
    int64_t r;
    if (!trans) { r = i + 1 + w; if (r >= T) return; }
    else        { r = i - 1 - w; if (r < 0) return; }
    double u2 = 0.0;
    if (!trans) {
        const double* Lt = L + r * 64 + i * 64 * ld;  // tile (r, i)
#pragma unroll
        for (int u = 0; u < 16; ++u) {
            const int c = p * 16 + u;
            u2 += Lt[e + (int64_t)c * ld] * xi[c];
        }
    } else {
        const double* Lt = L + i * 64 + r * 64 * ld;  // tile (i, r): (L^T)(r,i) = tile^T
#pragma unroll
        for (int u = 0; u < 16; ++u) {
            const int c = p * 16 + u;
            u2 += Lt[c + (int64_t)e * ld] * xi[c];
        }
    }
    u2 = block_sum4(u2, red);
    if (t < 64) b[r * 64 + t] -= u2;
}

void trsv_lower_f64(hipStream_t s, const double* L, int64_t ld, const double* Dinv, int64_t N, double* b,
                    double* x, int trans) {
    // b is consumed as workspace; the solution is written to x.
    const int64_t T = N / 64;
    for (int64_t st = 0; st < T; ++st) {
        const int64_t i = trans ? (T - 1 - st) : st;
        const int64_t pend = trans ? i : (T - 1 - i);
        hipLaunchKernelGGL(k_trsv_step, dim3((unsigned)(pend > 0 ? pend : 1)), dim3(256), 0, s, L, ld, Dinv,
                           T, i, b, x, trans);
    }
}

// ---------------------------------------------------------------------------
// The transposed solve L^T x = b in one launch: workgroup k (ticket order) owns
// block i = T - 1 - k and waits only on blocks of lower tickets, whose workgroups
// have started, so every wait ends; the summation order is fixed.
//
// Bound by the chain from block to block.  So (1) a solved block is handed over as
// data alone: the 64 values lie in `pub`, which holds a signalling NaN that no
// arithmetic returns (kUnsolved) until they are stored, and every wave of a consumer
// polls the values it multiplies, one per lane, with no flag, fence or barrier in
// between; (2) a wave keeps 16 rows, lane (li, p) the row li and the columns 16p ..
// 16p + 15 of it, whose multipliers are then 16-lane row broadcasts of the polled
// register (v_fmac_f64_dpp row_newbcast), and only the product with Dinv_i needs an
// exchange between the waves.  1.25 us per block: n = 4096 82 us, 1200 26, 500 12.
// (With a flag per block, a fence and LDS reductions 2.9: 188, 55, 22.  With Dinv_i
// L_{i,i-1} formed beforehand, so that the last block's values meet one product
// instead of two: 85, 34, 21, as its operands' cold loads stand in front of the
// chain.)  pub: N doubles, all kUnsolved; the launch sets the first 64 nreset
// of `reset`, the other of the context's two such arrays, back for the next one.
// With `scaled` the launch also leaves scale .* x there (zero beyond n), unless the
// gate's flags say NaN or V <= 0.  ticket: one word.
// ---------------------------------------------------------------------------
template <int C = 0>
__device__ __forceinline__ void fmac16(double (&acc)[2], double src, const double (&m)[16]) {
    if constexpr (C < 16) {
        fmac_bcast_f64<C>(acc[C & 1], src, m[C]);
        fmac16<C + 1>(acc, src, m);
    }
}

// this lane's value of a published block; a wave that has timed out waits no more
__device__ __forceinline__ double take_solved(const double* p, bool& ok, unsigned maxpoll) {
    unsigned long long v = 0;
    if (ok) {
        ok = false;
        for (unsigned n = 0; n < maxpoll; ++n) {
            v = __hip_atomic_load(reinterpret_cast<const unsigned long long*>(p), __ATOMIC_RELAXED,
                                  __HIP_MEMORY_SCOPE_AGENT);
            ok = !__ballot(v == kUnsolved);
            if (ok) break;
            __builtin_amdgcn_s_sleep(1);
        }
    }
    double d = __longlong_as_double((long long)v);
    dpp_ready(d);
    return d;
}

__global__ __launch_bounds__(256) void k_trsv_persist(const double* __restrict__ L, int64_t ld,
                                                      const double* __restrict__ Dinv, int64_t T,
                                                      const double* __restrict__ b, double* __restrict__ x,
                                                      double* pub, double* __restrict__ reset, int64_t nreset,
                                                      unsigned* __restrict__ ticket, unsigned base,
                                                      int* __restrict__ info, unsigned maxpoll,
                                                      const double* __restrict__ scale, int64_t n,
                                                      double* __restrict__ scaled, const int* __restrict__ gate) {
    __shared__ double sv[64];
    __shared__ unsigned s_id;
    const int t = threadIdx.x, lane = t & 63, w = __builtin_amdgcn_readfirstlane(t >> 6);
    if (t == 0) s_id = atomicAdd(ticket, 1u) - base;
    __syncthreads();
    const int64_t k = __builtin_amdgcn_readfirstlane((int)s_id);
    const int64_t i = T - 1 - k;
    for (int64_t q = k; q < nreset; q += T)
        if (t < 64) reinterpret_cast<unsigned long long*>(reset)[64 * q + t] = kUnsolved;
    const int li = lane & 15, p = lane >> 4, row = 16 * w + li;
    const double* D = Dinv + i * 64 * 64;
    double dv[16];
#pragma unroll
    for (int u = 0; u < 16; ++u) dv[u] = D[(16 * p + u) + row * 64];
    const double bi = b[64 * i + row];
    bool ok = true;
    double acc[2] = {0.0, 0.0};
    for (int64_t m = 0; m < k; ++m) {
        const int64_t j = T - 1 - m;  // the blocks solved before i, in their order
        double lt[16];
#pragma unroll
        for (int u = 0; u < 16; ++u) lt[u] = L[(64 * j + 16 * p + u) + (64 * i + row) * ld];
        const double xv = take_solved(pub + 64 * j + lane, ok, maxpoll);
        fmac16(acc, xv, lt);
    }
    double s = acc[0] + acc[1];
    s += __shfl_xor(s, 16, 64);
    s += __shfl_xor(s, 32, 64);
    if (p == 0) sv[row] = bi - s;
    __syncthreads();
    double rv = sv[lane];
    dpp_ready(rv);
    double out[2] = {0.0, 0.0};
    fmac16(out, rv, dv);
    double xi = out[0] + out[1];
    xi += __shfl_xor(xi, 16, 64);
    xi += __shfl_xor(xi, 32, 64);
    if (!ok) {  // nothing is published, so the blocks that wait for this one time out too
        if (lane == 0) atomicCAS(info, 0, kPanelWaitTimeout);
        return;
    }
    if (p != 0) return;
    put_shared(pub + 64 * i + row, xi);
    x[64 * i + row] = xi;
    if (scaled && !(gate && (*gate & 6))) scaled[64 * i + row] = 64 * i + row < n ? scale[64 * i + row] * xi : 0.0;
}

void trsv_persist_f64(hipStream_t s, const double* L, int64_t ld, const double* Dinv, int64_t N, const double* b,
                      double* x, double* pub, double* reset, int64_t nreset, unsigned* ticket,
                      unsigned base, int* info, unsigned maxpoll, const double* scale, int64_t n, double* scaled,
                      const int* gate) {
    const int64_t T = N / 64;
    if (T <= 0) return;
    hipLaunchKernelGGL(k_trsv_persist, dim3((unsigned)T), dim3(256), 0, s, L, ld, Dinv, T, b, x, pub, reset,
                           nreset, ticket, base, info, maxpoll, scale, n, scaled, gate);
}

// ---------------------------------------------------------------------------
// L Y = S B for many right-hand sides in one launch, in place (B: ldb x M, column
// major, M a multiple of 64; S = diag(sv) on the first n rows, or none).  A
// workgroup per 64-row block i and WN columns j, in ticket order of the row
// blocks: it subtracts L_{ik} Y_{kj} from S_i B_{ij} for k < i as the blocks
// Y_{kj} are published (operands straight from global memory, those of the next
// block loaded ahead), multiplies what is left by Dinv_i and publishes it.  Every
// wait is on a block of a lower ticket; the order of the sums is fixed.
//
// Every 64-k block's product is summed on its own and subtracted as a whole: the
// longest chain of roundings is then 64 + n / 64.  One sum over all k < 64 i made it n
// and the variances' error 2.3 and 3.6 times as large (n = 640, 1500).
//
// Bound by N/64 dependent blocks (a hand-over, one 64 x 64 x WN product and one
// with the inverse each) for few columns, by its products for many.  In launches
// of their own, two per 64 rows, the same steps took 7 us (13 before the products
// lost their LDS staging) each: 1000 points on n = 4096 1.18 ms of the 1.47.
//
// sync: flags [0, T ncol) (i ncol + j), ncol = M / WN, the ticket counter at
// sync[kTrsmFlags].
// ---------------------------------------------------------------------------
template <int WN>
__global__ __launch_bounds__(256) void k_trsm_persist(const double* __restrict__ L, int64_t ld,
                                                      const double* __restrict__ Dinv, double* B, int64_t ldb,
                                                      int ncol, const double* __restrict__ sv, int64_t n,
                                                      unsigned* __restrict__ sync, unsigned epoch, unsigned base,
                                                      int* __restrict__ info, unsigned maxpoll) {
    constexpr int NR = WN == 16 ? 1 : 2, NC = WN == 16 ? 1 : 2;  // 16x16 tiles of a wave
    constexpr int RP = 66;
    __shared__ double R[WN][RP];
    __shared__ unsigned s_id;
    __shared__ int s_ready;
    const int t = threadIdx.x, lane = t & 63, w = __builtin_amdgcn_readfirstlane(t >> 6);
    if (t == 0) s_id = atomicAdd(&sync[kTrsmFlags], 1u) - base;
    __syncthreads();
    const int id = __builtin_amdgcn_readfirstlane((int)s_id), i = id / ncol, j = id % ncol;
    const int li = lane & 15, g = lane >> 4;
    // this wave's rows and columns of the 64 x WN block
    const int r0 = WN == 16 ? 16 * w : 32 * (w & 1), c0 = WN == 16 ? 0 : 32 * (w >> 1);
    const int ra = r0 + frag_row<false, NR>(0, li);
    const double* pa = L + 64 * (int64_t)i + ra + 4 * g * ld;                // row ra of L_{i,0}, k = 4g
    const double* pb = B + 4 * g + (WN * (int64_t)j + c0 + li) * ldb;        // column of Y_{0,j}, k = 4g
    const double* pd = Dinv + 4096 * (int64_t)i + ra + 4 * g * 64;
    double* pc = B + 64 * (int64_t)i + (WN * (int64_t)j) * ldb;
    double bv[NR][NC][4];
#pragma unroll
    for (int a = 0; a < NR; ++a)
#pragma unroll
        for (int b = 0; b < NC; ++b)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int row = r0 + frag_row<false, NR>(a, li), col = c0 + 16 * b + g + 4 * v;
                const int64_t gr = 64 * (int64_t)i + row;
                bv[a][b][v] = pc[row + col * ldb] * (sv && gr < n ? sv[gr] : 1.0);
            }
    d4 acc[2][NR][NC];  // the products of this block and the last one
#pragma unroll
    for (int a = 0; a < NR; ++a)
#pragma unroll
        for (int b = 0; b < NC; ++b) acc[0][a][b] = acc[1][a][b] = d4{0.0, 0.0, 0.0, 0.0};
    double fa[2][4][NR][4], fb[2][4][NC][4];  // two 64-k blocks of each operand, in 16-k chunks
    auto load_a = [&](int st, int k, int c) {  // L_{ik}; for k = i the inverse of the diagonal block
        const double* q = k < i ? pa + 64 * (int64_t)k * ld : pd;
        const int64_t l = k < i ? ld : 64;
        frag_load<false, NR>(fa[st][c], q + 16 * c * l, l);
    };
    auto load_b = [&](int st, int k, int c) { frag_load<true, NC>(fb[st][c], pb + 64 * k + 16 * c, ldb); };
    auto take = [&](int st, int a, int b) {
#pragma unroll
        for (int v = 0; v < 4; ++v) bv[a][b][v] -= acc[st][a][b][v];
    };
    // Block k's product.  Between its matrix instructions the last block's product is
    // subtracted and the next block's operands are requested, a chunk's at a time: all of
    // them in a row hold the wave up until the memory path has taken them (4096 points on
    // n = 8192: 8.3 ms with all ahead of the product, 5.7 behind its first instruction,
    // 5.0 here).
    auto mult = [&](int st, int k, bool have, auto last) {  // last: the product with the inverse
#pragma unroll
        for (int a = 0; a < NR; ++a)
#pragma unroll
            for (int b = 0; b < NC; ++b) acc[st][a][b] = d4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int c = 0; c < 4; ++c)
#pragma unroll
            for (int s = 0; s < 4; ++s) {
#pragma unroll
                for (int a = 0; a < NR; ++a)
#pragma unroll
                    for (int b = 0; b < NC; ++b)
                        acc[st][a][b] = __builtin_amdgcn_mfma_f64_16x16x4f64(fb[st][c][b][s], fa[st][c][a][s],
                                                                             acc[st][a][b], 0, 0, 0);
                if (!last && s == 0) {
                    __builtin_amdgcn_sched_barrier(0);
                    load_a(st ^ 1, k + 1, c);
                    if (have) load_b(st ^ 1, k + 1, c);
                    __builtin_amdgcn_sched_barrier(0);
                }
                if (!last && c == 1 && s < NR * NC) take(st ^ 1, s / NC, s % NC);
            }
    };
#pragma unroll
    for (int c = 0; c < 4; ++c) load_a(0, 0, c);
    int ready = 0;  // blocks below this one are published
    bool have = false;
    for (int k0 = 0; k0 < i; k0 += 2)
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const int k = k0 + u;
            if (k >= i) break;
            if (k >= ready) {
                if (t < 64) {  // how many blocks from k on are published
                    const int kk = k + lane < i ? k + lane : i - 1;
                    unsigned long long miss = ~0ull;
                    for (unsigned p = 0; p < maxpoll; ++p) {
                        miss = __ballot(__hip_atomic_load(&sync[kk * ncol + j], __ATOMIC_RELAXED,
                                                          __HIP_MEMORY_SCOPE_AGENT) != epoch);
                        if (!(miss & 1)) break;
                        __builtin_amdgcn_s_sleep(1);
                    }
                    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
                    const int cnt = miss ? __ffsll((long long)miss) - 1 : 64;
                    if (t == 0) {
                        s_ready = cnt ? (k + cnt < i ? k + cnt : i) : -1;
                        if (!cnt) atomicCAS(info, 0, kPanelWaitTimeout);
                    }
                }
                __syncthreads();
                ready = __builtin_amdgcn_readfirstlane(s_ready);
                __syncthreads();
                if (ready < 0) return;
            }
            if (!have)
#pragma unroll
                for (int c = 0; c < 4; ++c) load_b(u, k, c);
            have = k + 1 < ready;
            mult(u, k, have, std::false_type());
        }
#pragma unroll
    for (int a = 0; a < NR; ++a)
#pragma unroll
        for (int b = 0; b < NC; ++b)
            if (i & 1) take(0, a, b);
            else take(1, a, b);
    // R = S_i B_ij less every block's product, then Y_ij = Dinv_i R (the inverse's operand was loaded last)
#pragma unroll
    for (int a = 0; a < NR; ++a)
#pragma unroll
        for (int b = 0; b < NC; ++b)
#pragma unroll
            for (int v = 0; v < 4; ++v)
                R[c0 + 16 * b + g + 4 * v][r0 + frag_row<false, NR>(a, li)] = bv[a][b][v];
    __syncthreads();
#pragma unroll
    for (int c = 0; c < 4; ++c)
#pragma unroll
        for (int b = 0; b < NC; ++b)
#pragma unroll
            for (int s = 0; s < 4; ++s) fb[0][c][b][s] = R[c0 + 16 * b + li][16 * c + 4 * g + s];
    if (i & 1) {
#pragma unroll
        for (int c = 0; c < 4; ++c)
#pragma unroll
            for (int a = 0; a < NR; ++a)
#pragma unroll
                for (int s = 0; s < 4; ++s) fa[0][c][a][s] = fa[1][c][a][s];
    }
    mult(0, i, false, std::true_type());
#pragma unroll
    for (int a = 0; a < NR; ++a)
#pragma unroll
        for (int b = 0; b < NC; ++b)
#pragma unroll
            for (int v = 0; v < 4; ++v)
                put_shared(pc + r0 + frag_row<false, NR>(a, li) + (c0 + 16 * b + g + 4 * v) * ldb,
                           (double)acc[0][a][b][v]);
    panel_publish(&sync[i * ncol + j], epoch);
}

// ---------------------------------------------------------------------------
// The same solve for a few right-hand sides, a wave per 64-row block i and column
// j.  Bound by the chain of blocks, so they are handed over as data (pub, reset and
// ticket as in k_trsv_persist; block k of column j at 64 (k ncol + j)): every wave
// polls the 64 values it multiplies, replicated over its 16-lane rows, and adds
// them with row-broadcast multiply-adds, one row of L to a lane, the next block's
// loaded ahead.  1.3 us a block against 3.5 with 16 columns on the matrix units (one
// point on n = 640: 34.8 -> 14.4 us).  The sums run in the order of the matrix
// instructions (k = 4g + s of each 16 in step s, g ascending), whose rounding is that
// of sequential multiply-adds: a column's result has the same bits whatever the
// number of columns.
// ---------------------------------------------------------------------------
template <int E = 0>
__device__ __forceinline__ void fmac64(double& acc, const double (&y)[4], const double (&m)[64]) {
    if constexpr (E < 64) {
        constexpr int c = E / 16, k = 4 * (E % 4) + (E % 16) / 4;  // the E-th term: chunk c, step (E % 16) / 4, g = E % 4
        fmac_bcast_f64<k>(acc, y[c], m[16 * c + k]);
        fmac64<E + 1>(acc, y, m);
    }
}

__global__ __launch_bounds__(64) void k_trsm_few(const double* __restrict__ L, int64_t ld,
                                                 const double* __restrict__ Dinv, double* __restrict__ B, int64_t ldb,
                                                 int ncol, const double* __restrict__ sv, int64_t n, double* pub,
                                                 double* __restrict__ reset, int64_t nreset,
                                                 unsigned* __restrict__ ticket, unsigned base, int* __restrict__ info,
                                                 unsigned maxpoll) {
    __shared__ double R[64];
    const int lane = threadIdx.x, li = lane & 15;
    unsigned tk = 0;
    if (lane == 0) tk = atomicAdd(ticket, 1u) - base;
    const int id = __builtin_amdgcn_readfirstlane((int)tk), i = id / ncol, j = id % ncol;
    for (int64_t q = id; q < nreset; q += gridDim.x)
        reinterpret_cast<unsigned long long*>(reset)[64 * q + lane] = kUnsolved;
    const int64_t row = 64 * (int64_t)i + lane;
    const double* Lr = L + row;
    const double* Dr = Dinv + 4096 * (int64_t)i + lane;
    double* b = B + row + j * ldb;
    double bv = *b * (sv && row < n ? sv[row] : 1.0);
    double lt[2][64], y[4];
    auto load = [&](int st, int k) {  // L_{ik}; for k = i the inverse of the diagonal block
        const double* q = k < i ? Lr + 64 * (int64_t)k * ld : Dr;
        const int64_t l = k < i ? ld : 64;
#pragma unroll
        for (int e = 0; e < 64; ++e) lt[st][e] = q[e * l];
    };
    load(0, 0);
    for (int k0 = 0; k0 < i; k0 += 2)
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const int k = k0 + u;
            if (k >= i) break;
            load(u ^ 1, k + 1);
            const unsigned long long* q = reinterpret_cast<const unsigned long long*>(pub) + 64 * ((int64_t)k * ncol + j);
            unsigned long long v[4];
            bool ok = false;
            for (unsigned p = 0; p < maxpoll; ++p) {
                bool miss = false;
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    v[c] = __hip_atomic_load(q + 16 * c + li, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    miss = miss || v[c] == kUnsolved;
                }
                ok = !__ballot(miss);
                if (ok) break;
                __builtin_amdgcn_s_sleep(1);
            }
            if (!ok) {  // nothing is published, so the blocks that wait for this one time out too
                if (lane == 0) atomicCAS(info, 0, kPanelWaitTimeout);
                return;
            }
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                y[c] = __longlong_as_double((long long)v[c]);
                dpp_ready(y[c]);
            }
            double acc = 0.0;
            fmac64(acc, y, lt[u]);
            bv -= acc;
        }
    R[lane] = bv;
    __syncthreads();
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        y[c] = R[16 * c + li];
        dpp_ready(y[c]);
    }
    double acc = 0.0;
    if (i & 1) fmac64(acc, y, lt[1]);
    else fmac64(acc, y, lt[0]);
    put_shared(pub + 64 * ((int64_t)i * ncol + j) + lane, acc);
    *b = acc;
}

void trsm_few_f64(hipStream_t s, const double* L, int64_t ld, const double* Dinv, int64_t N, double* B, int64_t ldb,
                  int ncol, const double* sv, int64_t n, double* pub, double* reset, int64_t nreset, unsigned* ticket,
                  unsigned base, int* info, unsigned maxpoll) {
    hipLaunchKernelGGL(k_trsm_few, dim3((unsigned)(N / 64 * ncol)), dim3(64), 0, s, L, ld, Dinv, B, ldb, ncol, sv, n, pub,
                       reset, nreset, ticket, base, info, maxpoll);
}

// 16 columns a workgroup while the chain of row blocks is what takes the time, 64 once
// the products are (a quarter of the reads of L).  A whole prediction with 16 / 64, us:
// n = 640 m = 2000 161 / 182, m = 4096 220 / 217; n = 1000 m = 1400 189 / 211, m = 3000
// 245 / 217; n = 2048 m = 1000 312 / 310, m = 1400 373 / 332; n = 4096 m = 500 532 / 540,
// m = 700 641 / 563, m = 4096 2936 / 1518; n = 8192 m = 256 984 / 1021, m = 500 1593 /
// 1084, m = 4096 11131 / 5320; n = 16384 m = 128 1924 / 2109, m = 256 3185 / 2157, m =
// 4096 44191 / 20916.
int trsm_cols(int64_t N, int64_t M) { return N * M <= 2400000 ? 16 : 64; }

void trsm_persist_f64(hipStream_t s, const double* L, int64_t ld, const double* Dinv, int64_t N, double* B, int64_t ldb,
                      int64_t M, const double* sv, int64_t n, unsigned* sync, unsigned epoch, unsigned base, int* info,
                      unsigned maxpoll) {
    const int wn = trsm_cols(N, M), ncol = (int)(M / wn);
    const dim3 grid((unsigned)(N / 64 * ncol));
    if (wn == 16)
        hipLaunchKernelGGL(k_trsm_persist<16>, grid, dim3(256), 0, s, L, ld, Dinv, B, ldb, ncol, sv, n, sync, epoch,
                           base, info, maxpoll);
    else
        hipLaunchKernelGGL(k_trsm_persist<64>, grid, dim3(256), 0, s, L, ld, Dinv, B, ldb, ncol, sv, n, sync, epoch,
                           base, info, maxpoll);
}

// ---------------------------------------------------------------------------
// Triangular / symmetric matrix-vector products over lower tiles.  One
// workgroup per 64-row output block, fixed summation order (deterministic).
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_trmv(const double* __restrict__ X, int64_t ld, int64_t T,
                                              const double* __restrict__ b, double* __restrict__ y,
                                              int trans) {
    __shared__ double red[256];
    const int64_t ti = blockIdx.x;
    const int t = threadIdx.x, e = t & 63, p = t >> 6;
    double s = 0.0;
    if (!trans) {
        // y[ti] = sum_{tj <= ti} X(ti,tj) b[tj]
        for (int64_t tj = 0; tj <= ti; ++tj) {
            const double* Xt = X + ti * 64 + tj * 64 * ld;
#pragma unroll 4
            for (int u = 0; u < 16; ++u) {
                const int c = p * 16 + u;
                s += Xt[e + (int64_t)c * ld] * b[tj * 64 + c];
            }
        }
    } else {
        // y[ti] = sum_{tr >= ti} X(tr,ti)^T b[tr]; element e = column of the tile
        for (int64_t tr = ti; tr < T; ++tr) {
            const double* Xt = X + tr * 64 + ti * 64 * ld;
#pragma unroll 4
            for (int u = 0; u < 16; ++u) {
                const int r = p * 16 + u;
                s += Xt[r + (int64_t)e * ld] * b[tr * 64 + r];
            }
        }
    }
    s = block_sum4(s, red);
    if (t < 64) y[ti * 64 + t] = s;
}

void trmv_lower_f64(hipStream_t s, const double* X, int64_t ld, int64_t N, const double* b, double* y, int trans,
                    double* part) {
    (void)part;
    const int64_t T = N / 64;
    hipLaunchKernelGGL(k_trmv, dim3((unsigned)T), dim3(256), 0, s, X, ld, T, b, y, trans);
}

__global__ __launch_bounds__(256) void k_symv(const double* __restrict__ K, int64_t ld, int64_t T,
                                              const double* __restrict__ v, double* __restrict__ y) {
    __shared__ double red[256];
    const int64_t ti = blockIdx.x;
    const int t = threadIdx.x, e = t & 63, p = t >> 6;
    double s = 0.0;
    for (int64_t tj = 0; tj < T; ++tj) {
        if (tj <= ti) {
            const double* Kt = K + ti * 64 + tj * 64 * ld;
#pragma unroll 4
            for (int u = 0; u < 16; ++u) {
                const int c = p * 16 + u;
                const double kv = (tj == ti && c > e) ? Kt[c + (int64_t)e * ld] : Kt[e + (int64_t)c * ld];
                s += kv * v[tj * 64 + c];
            }
        } else {
            const double* Kt = K + tj * 64 + ti * 64 * ld;  // tile (tj, ti), use transposed
#pragma unroll 4
            for (int u = 0; u < 16; ++u) {
                const int c = p * 16 + u;
                s += Kt[c + (int64_t)e * ld] * v[tj * 64 + c];
            }
        }
    }
    s = block_sum4(s, red);
    if (t < 64) y[ti * 64 + t] = s;
}

void symv_lower_f64(hipStream_t s, const double* K, int64_t ld, int64_t N, const double* v, double* y,
                    double* part) {
    (void)part;
    hipLaunchKernelGGL(k_symv, dim3((unsigned)(N / 64)), dim3(256), 0, s, K, ld, N / 64, v, y);
}

// y = A v for a symmetric FP64 matrix held as its lower 64x64 tiles (column-
// major, leading dimension ld; diagonal tiles complete), reading every stored
// tile once.  The lower tiles are grouped into G x G super-tiles; block
// (RI, CJ) of the lower super-tile grid (RI >= CJ) takes tiles (ti, tj) of its
// super-tile with tj <= ti.  An off-diagonal tile serves both triangles: A_ij v_j
// goes to output block i (the "row" role) and A_ij^T v_i to output block j (the
// "column" role); a diagonal tile serves the row role alone.  Thread (r, p)
// reads row r of columns 16p..16p+15 of each tile, so every load is a 512-byte
// column segment per wave.  Row-role sums are kept per row tile and reduced over
// the four waves at the end; column-role sums are kept for one column tile at a
// time (16 per thread) and reduced over the 64 rows by a butterfly that halves
// the values held per lane at each exchange.  Both go to partial slots of their
// own: part[CJ][i] (row role of column group CJ) and part[S + RI][j] (column role
// of row group RI), S = number of super-tile rows.  A second pass adds the slots
// that exist for each output block in a fixed order, so the result does not
// depend on scheduling.
static int symv_group(int batch) { return batch >= 4 ? 4 : 2; }

int symv_slots(int64_t N, int batch) {
    const int64_t T = N / 64, G = symv_group(batch), S = (T + G - 1) / G;
    return (int)(2 * (S > 0 ? S : 1));
}

// Sum of v over the 64 lanes for 16 values per lane: after the exchanges with
// lanes l^32, l^16, l^8, l^4 a lane holds one value, the partial of value
// u(l) = 8 b5 + 4 b4 + 2 b3 + b2 (bk = bit k of l) over the 16 lanes that agree
// with it in bits 2..5; the exchanges with l^2 and l^1 complete the sum.
__device__ __forceinline__ double butterfly16(double (&v)[16], int lane) {
#pragma unroll
    for (int u = 0; u < 8; ++u) {
        const bool hi = (lane & 32) != 0;
        const double keep = hi ? v[u + 8] : v[u], give = hi ? v[u] : v[u + 8];
        v[u] = keep + __shfl_xor(give, 32, 64);
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        const bool hi = (lane & 16) != 0;
        const double keep = hi ? v[u + 4] : v[u], give = hi ? v[u] : v[u + 4];
        v[u] = keep + __shfl_xor(give, 16, 64);
    }
#pragma unroll
    for (int u = 0; u < 2; ++u) {
        const bool hi = (lane & 8) != 0;
        const double keep = hi ? v[u + 2] : v[u], give = hi ? v[u] : v[u + 2];
        v[u] = keep + __shfl_xor(give, 8, 64);
    }
    {
        const bool hi = (lane & 4) != 0;
        const double keep = hi ? v[1] : v[0], give = hi ? v[0] : v[1];
        v[0] = keep + __shfl_xor(give, 4, 64);
    }
    double x = v[0];
    x += __shfl_xor(x, 2, 64);
    x += __shfl_xor(x, 1, 64);
    return x;
}

template <int G>
__global__ __launch_bounds__(256) void k_symv2(const double* __restrict__ A, int64_t ld, int64_t T,
                                               const double* __restrict__ v, double* __restrict__ part, int64_t sA,
                                               int64_t sV) {
    const int64_t b = blockIdx.y, S = (T + G - 1) / G;
    A += b * sA;
    v += b * sV;
    part += b * 2 * S * T * 64;
    int64_t RI, CJ;
    lower_tile(blockIdx.x, RI, CJ);
    const int64_t ti0 = RI * G, tj0 = CJ * G;
    const int ni = (int)((ti0 + G <= T) ? G : T - ti0), nj = (int)((tj0 + G <= T) ? G : T - tj0);
    const int t = threadIdx.x, r = t & 63, p = t >> 6;
    __shared__ double vc[G][64];  // v over the column tiles
    __shared__ double red[4][64];
    if (t < 64) {
#pragma unroll
        for (int q = 0; q < G; ++q) vc[q][t] = (q < nj) ? v[(tj0 + q) * 64 + t] : 0.0;
    }
    double vr[G], rowacc[G];
#pragma unroll
    for (int q = 0; q < G; ++q) {
        vr[q] = (q < ni) ? v[(ti0 + q) * 64 + r] : 0.0;
        rowacc[q] = 0.0;
    }
    __syncthreads();
    // the column role's output: lane l of wave p ends with column 16p + u(l)
    const int uo = ((r >> 5) & 1) * 8 + ((r >> 4) & 1) * 4 + ((r >> 3) & 1) * 2 + ((r >> 2) & 1);
    double* pcol = part + (S + RI) * T * 64;
#pragma unroll
    for (int qj = 0; qj < G; ++qj) {
        if (qj >= nj) break;  // block-uniform
        const int64_t tj = tj0 + qj;
        double colacc[16];
#pragma unroll
        for (int u = 0; u < 16; ++u) colacc[u] = 0.0;
#pragma unroll
        for (int qi = 0; qi < G; ++qi) {
            const int64_t ti = ti0 + qi;
            if (qi >= ni || tj > ti) continue;  // block-uniform
            const double* At = A + ti * 64 + r + (tj * 64 + 16 * p) * ld;
            double a[16];
#pragma unroll
            for (int u = 0; u < 16; ++u) a[u] = At[(int64_t)u * ld];
            double s = 0.0;
#pragma unroll
            for (int u = 0; u < 16; ++u) s += a[u] * vc[qj][16 * p + u];
            rowacc[qi] += s;
            if (tj < ti) {
#pragma unroll
                for (int u = 0; u < 16; ++u) colacc[u] += a[u] * vr[qi];
            }
        }
        const double cs = butterfly16(colacc, r);
        if ((r & 3) == 0) pcol[tj * 64 + 16 * p + uo] = cs;
    }
    // row role: sum over the four waves, per row tile
    double* prow = part + CJ * T * 64;
#pragma unroll
    for (int qi = 0; qi < G; ++qi) {
        red[p][r] = rowacc[qi];
        __syncthreads();
        if (t < 64 && qi < ni) prow[(ti0 + qi) * 64 + t] = red[0][t] + red[1][t] + red[2][t] + red[3][t];
        __syncthreads();
    }
}

// y[i] = sum of the row-role slots CJ <= I and the column-role slots RI >= I of
// output block i (I = its super-tile row), in that order
// Sums of the partial vectors in a fixed order, a thread per row: bound by the chain of
// loads, so sixteen are in flight and a workgroup is one wave (n = 4096: 11.8 -> 4.6 us).
__global__ void k_symv2_sum(const double* __restrict__ part, int64_t T, int G, double* __restrict__ y, int64_t sV,
                            const int* __restrict__ gate) {
    if (gate && (*gate & 6)) return;
    const int64_t b = blockIdx.y, S = (T + G - 1) / G, N = T * 64;
    part += b * 2 * S * N;
    y += b * sV;
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= N) return;
    const int64_t I = (i / 64) / G;
    // S + 1 terms: the row sums' slots up to I, the column sums' from I on
    double s = 0.0;
#pragma unroll 16
    for (int64_t u = 0; u <= S; ++u) s += part[(u <= I ? u : S + u - 1) * N + i];
    y[i] = s;
}

__global__ void k_chunk_sum(const double* __restrict__ part, int64_t N, int nchunk, double* __restrict__ y,
                            int64_t sV) {
    const int64_t b = blockIdx.y;
    part += b * (int64_t)nchunk * N;
    y += b * sV;
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= N) return;
    double s = 0.0;
#pragma unroll 16
    for (int c = 0; c < nchunk; ++c) s += part[(int64_t)c * N + i];
    y[i] = s;
}

// part: batch * symv_slots(N, batch) * N doubles (nchunk is not used)
void chunk_sum_f64(hipStream_t s, const double* part, int64_t N, int nchunk, double* y, int batch, int64_t sV);
void symv_lt_f64(hipStream_t s, const double* A, int64_t N, const double* v, double* y, double* part, int nchunk,
                 int batch, int64_t sA, int64_t sV, const int* gate) {
    (void)nchunk;
    const int64_t T = N / 64;
    const int G = symv_group(batch);
    const int64_t S = (T + G - 1) / G;
    const dim3 grid((unsigned)(S * (S + 1) / 2), (unsigned)batch);
    if (G == 4) hipLaunchKernelGGL(k_symv2<4>, grid, dim3(256), 0, s, A, N, T, v, part, sA, sV);
    else hipLaunchKernelGGL(k_symv2<2>, grid, dim3(256), 0, s, A, N, T, v, part, sA, sV);
    hipLaunchKernelGGL(k_symv2_sum, dim3((unsigned)(N / 64), (unsigned)batch), dim3(64), 0, s, part, T, G, y,
                       sV, gate);
}

// y[b][i] = sum_c part[b][c][i] (fixed order)
void chunk_sum_f64(hipStream_t s, const double* part, int64_t N, int nchunk, double* y, int batch, int64_t sV) {
    hipLaunchKernelGGL(k_chunk_sum, dim3((unsigned)(N / 64), (unsigned)batch), dim3(64), 0, s, part, N,
                       nchunk, y, sV);
}

// The weight matrix of the latent-likelihood gradient, in place over the lower
// tiles of B^-1 (every element of a lower tile, diagonal tiles complete):
// W_ik = s_i B^-1_ik s_k - (t_i u_k + u_i t_k) for i, k < n (t, u may be null:
// no rank-two term), zero where i or k is padding.  With s = V^-1/2,
// s B^-1 s = (K + V)^-1.
__global__ __launch_bounds__(256) void k_form_wgrad(double* __restrict__ B, int64_t ld, int64_t n,
                                                    const double* __restrict__ sv, const double* __restrict__ t,
                                                    const double* __restrict__ u) {
    int64_t ti, tj;
    lower_tile(blockIdx.x, ti, tj);
    const int e = threadIdx.x & 63, p = threadIdx.x >> 6;
    const int64_t i = ti * 64 + e;
    const double si = (i < n) ? sv[i] : 0.0;
    const double tii = (t && i < n) ? t[i] : 0.0, ui = (u && i < n) ? u[i] : 0.0;
#pragma unroll 4
    for (int q = 0; q < 16; ++q) {
        const int64_t k = tj * 64 + 16 * p + q;
        double* b = B + i + k * ld;
        if (i < n && k < n) {
            double w = si * (*b) * sv[k];
            if (t) w -= tii * u[k] + ui * t[k];
            *b = w;
        } else {
            *b = 0.0;
        }
    }
}

void form_wgrad_f64(hipStream_t s, double* B, int64_t N, int64_t n, const double* sv, const double* t,
                    const double* u) {
    const int64_t T = N / 64;
    hipLaunchKernelGGL(k_form_wgrad, dim3((unsigned)(T * (T + 1) / 2)), dim3(256), 0, s, B, N, n, sv, t, u);
}

// one wave per column: out[j] = sum_i A[i + j*ld]^2; lower != 0 starts at the
// column's diagonal tile (the upper tiles of a lower-triangular buffer are never written)
__global__ __launch_bounds__(256) void k_colsumsq(const double* __restrict__ A, int64_t ld, int64_t nrow,
                                                  int64_t ncol, double* __restrict__ out, int lower) {
    const int lane = threadIdx.x & 63;
    const int64_t j = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (j >= ncol) return;
    const double* col = A + j * ld;
    double s = 0.0;
    for (int64_t i = (lower ? (j / 64) * 64 : 0) + lane; i < nrow; i += 64) {
        const double v = col[i];
        s += v * v;
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
    if (lane == 0) out[j] = s;
}

__global__ __launch_bounds__(256) void k_gemv_t(const double* __restrict__ A, int64_t ld, int64_t nrow,
                                                int64_t ncol, const double* __restrict__ v, double* __restrict__ out) {
    const int lane = threadIdx.x & 63;
    const int64_t j = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (j >= ncol) return;
    const double* col = A + j * ld;
    double s = 0.0;
    for (int64_t i = lane; i < nrow; i += 64) s += col[i] * v[i];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
    if (lane == 0) out[j] = s;
}

void gemv_t_f64(hipStream_t s, const double* A, int64_t ld, int64_t nrow, int64_t ncol, const double* v,
                double* out) {
    if (ncol <= 0) return;
    hipLaunchKernelGGL(k_gemv_t, dim3((unsigned)((ncol + 3) / 4)), dim3(256), 0, s, A, ld, nrow, ncol, v, out);
}

void colsumsq_f64(hipStream_t s, const double* A, int64_t ld, int64_t nrow, int64_t ncol, double* out, int lower) {
    if (ncol <= 0) return;
    hipLaunchKernelGGL(k_colsumsq, dim3((unsigned)((ncol + 3) / 4)), dim3(256), 0, s, A, ld, nrow, ncol, out, lower);
}

// ---------------------------------------------------------------------------
// Elementwise helpers over lower tiles / vectors
// ---------------------------------------------------------------------------
// Column j = c0 + blockIdx.x of X (N x N, ld N): the block's column from Dinv
// (64x64 column-major per block, zero above its diagonal) on its 64x64 diagonal
// block and, with `clear`, zero above it; the rows below are left to the caller.
__global__ __launch_bounds__(256) void k_trtri_leaves(double* __restrict__ X, int64_t N,
                                                      const double* __restrict__ Dinv, int64_t c0, int clear) {
    const int64_t j = c0 + blockIdx.x, kb = j / 64, r0 = kb * 64;
    const double* D = Dinv + kb * 4096 + (j - r0) * 64;
    for (int64_t i = (clear ? 0 : r0) + threadIdx.x; i < r0 + 64; i += 256) X[i + j * N] = (i < r0) ? 0.0 : D[i - r0];
}

void trtri_leaves_f64(hipStream_t s, double* X, int64_t N, const double* Dinv, int64_t c0, int64_t ncols, int clear) {
    if (ncols <= 0) return;
    hipLaunchKernelGGL(k_trtri_leaves, dim3((unsigned)ncols), dim3(256), 0, s, X, N, Dinv, c0, clear);
}

// zero above the 64x64 diagonal blocks of X (N x N, ld N)
__global__ __launch_bounds__(256) void k_clear_upper(double* __restrict__ X, int64_t N) {
    const int64_t j = 64 + blockIdx.x, r0 = j / 64 * 64;
    for (int64_t i = threadIdx.x; i < r0; i += 256) X[i + j * N] = 0.0;
}

void clear_upper_f64(hipStream_t s, double* X, int64_t N) {
    if (N <= 64) return;
    hipLaunchKernelGGL(k_clear_upper, dim3((unsigned)(N - 64)), dim3(256), 0, s, X, N);
}

__global__ void k_fill(double* p, int64_t n, double v) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}

void fill_f64(hipStream_t s, double* p, int64_t n, double v) {
    if (n <= 0) return;
    hipLaunchKernelGGL(k_fill, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, p, n, v);
}

__global__ void k_scale_rows(double* __restrict__ A, int64_t ld, int64_t nrow, int64_t ncol,
                             const double* __restrict__ sv) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const int64_t j = blockIdx.y;
    if (i < nrow) A[i + j * ld] *= sv[i];
}

void scale_rows_f64(hipStream_t s, double* A, int64_t ld, int64_t nrow, int64_t ncol, const double* sv) {
    if (nrow <= 0 || ncol <= 0) return;
    hipLaunchKernelGGL(k_scale_rows, dim3((unsigned)((nrow + 255) / 256), (unsigned)ncol), dim3(256), 0, s, A,
                       ld, nrow, ncol, sv);
}

// B = I + S K S over lower tiles (S = diag(sv), identity on padding).  Optional
// outputs for the mixed-precision form: B32 = fl32(B) and dacc = the unrounded
// FP64 diagonal tiles (64x64 column-major, one per block row).
__global__ void k_form_B(const double* __restrict__ K, double* __restrict__ B, int64_t ld, int64_t n,
                         const double* __restrict__ sv, float* __restrict__ B32, double* __restrict__ dacc) {
    int64_t ti, tj;
    lower_tile(blockIdx.x, ti, tj);
    const int t = threadIdx.x, i = t & 63;
    const int64_t gi = ti * 64 + i;
    const double si = (gi < n) ? sv[gi] : 0.0;
    double* dt = (dacc && ti == tj) ? dacc + ti * 64 * 64 : nullptr;
    for (int c = t >> 6; c < 64; c += 4) {
        const int64_t gj = tj * 64 + c;
        double v;
        if (gi < n && gj < n) v = si * K[gi + gj * ld] * sv[gj] + (gi == gj ? 1.0 : 0.0);
        else v = (gi == gj) ? 1.0 : 0.0;
        B[gi + gj * ld] = v;
        if (B32) B32[gi + gj * ld] = (float)v;
        if (dt) dt[i + c * 64] = v;
    }
}

void form_B_f64(hipStream_t s, const double* K, double* B, int64_t ld, int64_t n, int64_t N, const double* sv) {
    const int64_t T = N / 64;
    hipLaunchKernelGGL(k_form_B, dim3((unsigned)(T * (T + 1) / 2)), dim3(256), 0, s, K, B, ld, n, sv, (float*)nullptr,
                       (double*)nullptr);
}

void form_B_mixed(hipStream_t s, const double* K, double* B64, float* B32, double* dacc, int64_t ld, int64_t n,
                  int64_t N, const double* sv) {
    const int64_t T = N / 64;
    hipLaunchKernelGGL(k_form_B, dim3((unsigned)(T * (T + 1) / 2)), dim3(256), 0, s, K, B64, ld, n, sv, B32, dacc);
}

// ---------------------------------------------------------------------------
// Restore a saved factor (gp_load).  In place over L (N x N, column-major): the
// n x n part holds C_chol = diag(sqrt V) chol(B)^T as saved; it becomes
// L = diag(1/sqrt V) C_chol with zeros above the diagonal, the padding becomes
// the identity, and sv[i] = 1/sqrt(V_i).  One workgroup per column.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_restore_factor(double* __restrict__ L, int64_t n, int64_t N,
                                                        const double* __restrict__ V, double* __restrict__ sv) {
    const int64_t j = blockIdx.x;
    for (int64_t i = threadIdx.x; i < N; i += 256) {
        double v;
        if (i < n && j < n) v = (i >= j) ? L[i + j * N] / sqrt(V[i]) : 0.0;
        else v = (i == j) ? 1.0 : 0.0;
        L[i + j * N] = v;
        if (j == 0 && i < n) sv[i] = 1.0 / sqrt(V[i]);
    }
}

void restore_factor_f64(hipStream_t s, double* L, int64_t n, int64_t N, const double* V, double* sv) {
    hipLaunchKernelGGL(k_restore_factor, dim3((unsigned)N), dim3(256), 0, s, L, n, N, V, sv);
}

// Inverses of the 64x64 diagonal blocks of an existing lower-triangular factor
// (what diag_finish does after the factorisation): Dinv + k*4096
// receives L_kk^-1 (column-major, ld 64, zeros above the diagonal) and
// ldiag[64k + i] = log L_ii.  Lane t forward-substitutes column t.  A pivot
// that is not positive (or NaN) sets info to its 1-based index, the lowest of them.
__global__ __launch_bounds__(64) void k_trtri_diag64(const double* __restrict__ L, int64_t ld,
                                                     double* __restrict__ Dinv, double* __restrict__ ldiag,
                                                     int* __restrict__ info) {
    __shared__ double A[64][65];  // A[col][row] = L_kk(row, col)
    __shared__ double X[64][65];  // X[col][row] = L_kk^-1(row, col)
    const int64_t k = blockIdx.x;
    const int t = threadIdx.x;
    const double* blk = L + k * 64 * (ld + 1);
    for (int c = 0; c < 64; ++c) A[c][t] = blk[t + (int64_t)c * ld];
    __syncthreads();
    for (int i = 0; i < 64; ++i) {
        double v = 0.0;
        if (i >= t) {
            double acc = (i == t) ? 1.0 : 0.0;
            for (int q = t; q < i; ++q) acc -= A[q][i] * X[t][q];
            v = acc / A[i][i];
        }
        X[t][i] = v;
    }
    __syncthreads();
    double* D = Dinv + k * 64 * 64;
    for (int c = 0; c < 64; ++c) D[t + c * 64] = X[c][t];
    const double p = A[t][t];
    ldiag[k * 64 + t] = log(p);
    const unsigned long long bad = __ballot(!(p > 0.0));
    if (t == 0 && bad) report_minor(info, (int)(k * 64 + __ffsll((long long)bad)));
}

void trtri_diag64_f64(hipStream_t s, const double* L, int64_t ld, int64_t T, double* Dinv, double* ldiag, int* info) {
    hipLaunchKernelGGL(k_trtri_diag64, dim3((unsigned)T), dim3(64), 0, s, L, ld, Dinv, ldiag, info);
}

}  // namespace gpl
