// Kernels of the FITC path (fitc_host.cpp): the per-site combination S = D + V of
// the inversion lemma, the passes over A = Lz^-1 K_zx that give alpha and the
// means, the sum of the partial Gram products, and the FITC diagonal.  Everything
// else in FITC runs on the dense kernels.
#include "gpl_internal.h"

#include <algorithm>
#include <cmath>

namespace gpl {

// i < n: S = D + V, si = 1/S (NaN for S < 0, which then fails the factorization of
// G), zs = z / S; padding (n <= i < N): zeros
__global__ void k_fitc_site(int64_t n, int64_t N, const double* __restrict__ D, const double* __restrict__ V,
                            const double* __restrict__ z, double* __restrict__ S, double* __restrict__ si,
                            double* __restrict__ zs) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= N) return;
    if (i < n) {
        const double s = D[i] + V[i];
        S[i] = s;
        si[i] = s < 0.0 ? __builtin_nan("") : 1.0 / s;
        zs[i] = z[i] / s;
    } else {
        S[i] = 0.0;
        si[i] = 0.0;
        zs[i] = 0.0;
    }
}

void fitc_site(hipStream_t s, int64_t n, int64_t N, const double* D, const double* V, const double* z, double* S,
               double* si, double* zs) {
    hipLaunchKernelGGL(k_fitc_site, dim3((unsigned)((N + 255) / 256)), dim3(256), 0, s, n, N, D, V, z, S, si, zs);
}

// W[i + j*ld] = r[i] * U[i + j*ld] over nrow x ncol (one workgroup per column)
__global__ __launch_bounds__(256) void k_scale_rows_copy(const double* __restrict__ U, int64_t ld, int64_t nrow,
                                                         const double* __restrict__ r, double* __restrict__ W) {
    const int64_t j = blockIdx.x;
    for (int64_t i = threadIdx.x; i < nrow; i += 256) W[i + j * ld] = r[i] * U[i + j * ld];
}

void scale_rows_copy_f64(hipStream_t s, const double* U, int64_t ld, int64_t nrow, int64_t ncol, const double* r,
                         double* W) {
    hipLaunchKernelGGL(k_scale_rows_copy, dim3((unsigned)ncol), dim3(256), 0, s, U, ld, nrow, r, W);
}

// G = I + sum of the P partial products, lower 64x64 tiles (sixteen workgroups per
// tile, so that few tiles with many parts still spread over the chip), in order of p
__global__ __launch_bounds__(256) void k_fitc_gram_sum(const double* __restrict__ parts, int P, int64_t Mz,
                                                       double* __restrict__ G) {
    int64_t tj = 0, ti = blockIdx.x >> 4;  // column by column
    for (int64_t T = Mz / 64; ti >= T - tj; ++tj) ti -= T - tj;
    ti += tj;
    const int e = (blockIdx.x & 15) * 256 + threadIdx.x;
    const int64_t i = ti * 64 + (e & 63), j = tj * 64 + (e >> 6);
    const double* q = parts + i + j * Mz;
    double acc = 0.0;
#pragma unroll 8
    for (int p = 0; p < P; ++p) acc += q[(int64_t)p * Mz * Mz];
    G[i + j * Mz] = (i == j) ? 1.0 + acc : acc;
}

void fitc_gram_sum(hipStream_t s, const double* parts, int P, int64_t Mz, double* G) {
    const int64_t T = Mz / 64;
    hipLaunchKernelGGL(k_fitc_gram_sum, dim3((unsigned)(T * (T + 1) / 2 * 16)), dim3(256), 0, s, parts, P, Mz, G);
}

// ---------------------------------------------------------------------------
// Passes over A = Lz^-1 K_zx (Mz x N, a column per training point), memory bound.
// A wave takes one column at a time, 2 R rows per lane held in registers, so that
// a pass that needs a column's dot product and then the column again reads it once:
//   k_fitc_pass<R, true>:  alpha_j = zs_j - (a_j . q) / S_j and out = sum alpha_j a_j
//   k_fitc_pass<R, false>: out = sum coef_j a_j
//   k_fitc_dot: alpha_j as above (MODE 0), or fmean_j = a_j . w + D_j alpha_j (MODE 1)
// With more than 1024 rows the first form runs as the other two, the second on
// ranges of 1024 rows.  Sums of a workgroup's columns go to `part`, and a small
// kernel adds those in a fixed order.
// ---------------------------------------------------------------------------
__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

template <int R, bool DOT>
__global__ __launch_bounds__(256) void k_fitc_pass(const double* __restrict__ A, int64_t Mz, int64_t n, int64_t N,
                                                   int64_t cols, const double* __restrict__ q,
                                                   const double* __restrict__ zs, const double* __restrict__ S,
                                                   double* __restrict__ coef, double* __restrict__ part) {
    __shared__ double2 red[3][64 * R];
    constexpr int U = R >= 4 ? 2 : 4;  // columns in flight
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int64_t row0 = (int64_t)blockIdx.y * 128 * R + 2 * lane;
    double2 acc[R], qv[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        acc[r] = make_double2(0.0, 0.0);
        const int64_t i = row0 + 128 * r;
        qv[r] = (DOT && i < Mz) ? *reinterpret_cast<const double2*>(q + i) : make_double2(0.0, 0.0);
    }
    const int64_t j0 = (int64_t)blockIdx.x * cols, j1 = j0 + cols < n ? j0 + cols : n;
    for (int64_t j = j0 + w; j < j1; j += 4 * U) {
        double2 a[U][R];
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int r = 0; r < R; ++r) {
                const int64_t i = row0 + 128 * r;
                a[u][r] = (j + 4 * u < j1 && i < Mz) ? *reinterpret_cast<const double2*>(A + i + (j + 4 * u) * Mz)
                                                     : make_double2(0.0, 0.0);
            }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int64_t ju = j + 4 * u;
            if (ju >= j1) break;
            double c;
            if (DOT) {
                double d = 0.0;
#pragma unroll
                for (int r = 0; r < R; ++r) d += a[u][r].x * qv[r].x + a[u][r].y * qv[r].y;
                c = zs[ju] - wave_sum(d) / S[ju];
                if (lane == 0) coef[ju] = c;
            } else {
                c = coef[ju];
            }
#pragma unroll
            for (int r = 0; r < R; ++r) {
                acc[r].x += c * a[u][r].x;
                acc[r].y += c * a[u][r].y;
            }
        }
    }
    if (DOT && blockIdx.x == 0)
        for (int64_t j = n + threadIdx.x; j < N; j += 256) coef[j] = 0.0;
    if (w > 0)
#pragma unroll
        for (int r = 0; r < R; ++r) red[w - 1][64 * r + lane] = acc[r];
    __syncthreads();
    if (w > 0) return;
#pragma unroll
    for (int r = 0; r < R; ++r) {
        for (int v = 0; v < 3; ++v) {
            acc[r].x += red[v][64 * r + lane].x;
            acc[r].y += red[v][64 * r + lane].y;
        }
        const int64_t i = row0 + 128 * r;
        if (i < Mz) *reinterpret_cast<double2*>(part + (int64_t)blockIdx.x * Mz + i) = acc[r];
    }
}

// out[i] = sum_p part[i + p * Mz], 16 rows per workgroup, 16 threads per row
__global__ __launch_bounds__(256) void k_fitc_sum(const double* __restrict__ part, int P, int64_t Mz,
                                                  double* __restrict__ out) {
    __shared__ double red[16][17];
    const int r = threadIdx.x & 15, g = threadIdx.x >> 4;
    const int64_t i = (int64_t)blockIdx.x * 16 + r;
    double acc = 0.0;
#pragma unroll 8
    for (int p = g; p < P; p += 16) acc += part[i + (int64_t)p * Mz];
    red[g][r] = acc;
    __syncthreads();
    if (g > 0) return;
    for (int k = 1; k < 16; ++k) acc += red[k][r];
    out[i] = acc;
}

template <int MODE>
__global__ __launch_bounds__(256) void k_fitc_dot(const double* __restrict__ A, int64_t Mz, int64_t n, int64_t N,
                                                  const double* __restrict__ v, const double* __restrict__ p,
                                                  const double* __restrict__ q, double* __restrict__ out) {
    const int lane = threadIdx.x & 63;
    const int64_t j = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (j >= N) return;
    if (j >= n) {
        if (lane == 0) out[j] = 0.0;
        return;
    }
    double d0 = 0.0, d1 = 0.0;
#pragma unroll 4
    for (int64_t i = 2 * lane; i < Mz; i += 128) {
        const double2 a = *reinterpret_cast<const double2*>(A + i + j * Mz);
        const double2 b = *reinterpret_cast<const double2*>(v + i);
        d0 += a.x * b.x;
        d1 += a.y * b.y;
    }
    const double d = wave_sum(d0 + d1);
    if (lane == 0) out[j] = MODE == 0 ? p[j] - d / q[j] : d + p[j] * q[j];
}

// two workgroups per CU, or 16 columns each
int fitc_pass_parts(int64_t n) { return (int)std::max<int64_t>(1, std::min<int64_t>(512, n / 16)); }

template <bool DOT>
static void fitc_pass(hipStream_t s, const double* A, int64_t Mz, int64_t n, int64_t N, const double* q,
                      const double* zs, const double* S, double* coef, double* part, double* out) {
    const int G = fitc_pass_parts(n);
    const int64_t cols = (n + G - 1) / G;
#define GPL_FP(R)                                                                                                 \
    hipLaunchKernelGGL((k_fitc_pass<R, DOT>), dim3((unsigned)G, (unsigned)((Mz + 128 * R - 1) / (128 * R))),      \
                       dim3(256), 0, s, A, Mz, n, N, cols, q, zs, S, coef, part)
    if (Mz <= 128) GPL_FP(1);
    else if (Mz <= 256) GPL_FP(2);
    else if (Mz <= 512) GPL_FP(4);
    else GPL_FP(8);
#undef GPL_FP
    hipLaunchKernelGGL(k_fitc_sum, dim3((unsigned)(Mz / 16)), dim3(256), 0, s, part, G, Mz, out);
}

// out = sum_{j < n} coef_j a_j
void fitc_combine(hipStream_t s, const double* A, int64_t Mz, int64_t n, const double* coef, double* part,
                  double* out) {
    fitc_pass<false>(s, A, Mz, n, n, nullptr, nullptr, nullptr, const_cast<double*>(coef), part, out);
}

// alpha_j = zs_j - (a_j . q) / S_j (R/linear_algebra.R inv_lemma_solve, vector rhs; padding: 0), out = A alpha
void fitc_alpha_pass(hipStream_t s, const double* A, int64_t Mz, int64_t n, int64_t N, const double* q,
                     const double* zs, const double* S, double* alpha, double* part, double* out) {
    if (Mz <= 1024) {
        fitc_pass<true>(s, A, Mz, n, N, q, zs, S, alpha, part, out);
        return;
    }
    hipLaunchKernelGGL(k_fitc_dot<0>, dim3((unsigned)((N + 3) / 4)), dim3(256), 0, s, A, Mz, n, N, q, zs, S, alpha);
    fitc_combine(s, A, Mz, n, alpha, part, out);
}

// fmean_j = a_j . w + D_j alpha_j; padding: 0
void fitc_mean(hipStream_t s, const double* A, int64_t Mz, int64_t n, int64_t N, const double* w, const double* D,
               const double* alpha, double* fmean) {
    hipLaunchKernelGGL(k_fitc_dot<1>, dim3((unsigned)((N + 3) / 4)), dim3(256), 0, s, A, Mz, n, N, w, D, alpha, fmean);
}

// out[j] = sum_i A[i + j*ld] B[i + j*ld], i < nrow (one wavefront per column, fixed order)
__global__ __launch_bounds__(64) void k_coldot(const double* __restrict__ A, const double* __restrict__ B, int64_t ld,
                                               int64_t nrow, double* __restrict__ out) {
    const int64_t j = blockIdx.x;
    const int l = threadIdx.x;
    double acc = 0.0;
    for (int64_t i = l; i < nrow; i += 64) acc += A[i + j * ld] * B[i + j * ld];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) acc += __shfl_xor(acc, o, 64);
    if (l == 0) out[j] = acc;
}

void coldot_f64(hipStream_t s, const double* A, const double* B, int64_t ld, int64_t nrow, int64_t ncol, double* out) {
    if (ncol <= 0) return;
    hipLaunchKernelGGL(k_coldot, dim3((unsigned)ncol), dim3(64), 0, s, A, B, ld, nrow, out);
}

// FITC diagonal (R/gp_fit.R:107-108): D = (k(x_i, x_i) + jitter) - cs_i for
// i < n, 0 on padding
__global__ void k_fitc_diag(int64_t n, int64_t N, const double* __restrict__ kd, const double* __restrict__ cs,
                            double jitter, double* __restrict__ D) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= N) return;
    D[i] = (i < n) ? (kd[i] + jitter) - cs[i] : 0.0;
}

void fitc_diag(hipStream_t s, int64_t n, int64_t N, const double* kd, const double* cs, double jitter, double* D) {
    hipLaunchKernelGGL(k_fitc_diag, dim3((unsigned)((N + 255) / 256)), dim3(256), 0, s, n, N, kd, cs, jitter, D);
}

// out[i] = log a[i], i < n
__global__ void k_vec_log(int64_t n, const double* __restrict__ a, double* __restrict__ out) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) out[i] = log(a[i]);
}

void vec_log(hipStream_t s, int64_t n, const double* a, double* out) {
    if (n <= 0) return;
    hipLaunchKernelGGL(k_vec_log, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, n, a, out);
}

// B (ncol x nrow, ld ldb) = A^T for A (nrow x ncol, ld lda); both dimensions
// multiples of 64.  64x64 tiles through LDS so reads and writes are coalesced.
__global__ __launch_bounds__(256) void k_transpose64(const double* __restrict__ A, int64_t lda, int64_t tiles_r,
                                                     double* __restrict__ B, int64_t ldb) {
    __shared__ double t[64][65];
    const int64_t ti = blockIdx.x % tiles_r, tj = blockIdx.x / tiles_r;
    const int e = threadIdx.x & 63, p = threadIdx.x >> 6;
    const double* a = A + ti * 64 + tj * 64 * lda;
    for (int c = p; c < 64; c += 4) t[c][e] = a[e + (int64_t)c * lda];  // t[col][row]
    __syncthreads();
    double* b = B + tj * 64 + ti * 64 * ldb;
    for (int c = p; c < 64; c += 4) b[e + (int64_t)c * ldb] = t[e][c];  // B(tj*64+e, ti*64+c) = A(ti*64+c, tj*64+e)
}

void transpose_f64(hipStream_t s, const double* A, int64_t lda, int64_t nrow, int64_t ncol, double* B, int64_t ldb) {
    const int64_t tr = nrow / 64, tc = ncol / 64;
    if (tr <= 0 || tc <= 0) return;
    hipLaunchKernelGGL(k_transpose64, dim3((unsigned)(tr * tc)), dim3(256), 0, s, A, lda, tr, B, ldb);
}

// C[i + i*ld] += v[i] + jitter for i < n; the padded diagonal (n <= i < N) becomes 1
__global__ void k_add_diag(double* __restrict__ C, int64_t ld, int64_t n, int64_t N, const double* __restrict__ v,
                           double jitter) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= N) return;
    if (i < n) C[i + i * ld] += v[i] + jitter;
    else C[i + i * ld] = 1.0;
}

void add_diag_f64(hipStream_t s, double* C, int64_t ld, int64_t n, int64_t N, const double* v, double jitter) {
    hipLaunchKernelGGL(k_add_diag, dim3((unsigned)((N + 255) / 256)), dim3(256), 0, s, C, ld, n, N, v, jitter);
}

// EP posterior variance of FITC (R/ep.R:170-174 through the inversion lemma):
// fvar = V [K_f C^-1]_ii = V (q/S + D (1/S - q/S^2)), q_i = |Lc^-1 u_i|^2
__global__ void k_fitc_ep_var(int64_t n, const double* __restrict__ V, const double* __restrict__ S,
                              const double* __restrict__ D, const double* __restrict__ q, double* __restrict__ fvar) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const double si = S[i], qi = q[i];
    fvar[i] = V[i] * (qi / si + D[i] * (1.0 / si - qi / (si * si)));
}

void fitc_ep_var(hipStream_t s, int64_t n, const double* V, const double* S, const double* D, const double* q,
                 double* fvar) {
    hipLaunchKernelGGL(k_fitc_ep_var, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, n, V, S, D, q, fvar);
}

// Training-input variance (R/gp_pred.R:270-285): prior - (t1 + 2 Dt q/S + Dt^2 (1/S - q/S^2)),
// t1 = (A^T M A)_ii = |a_i|^2 - q_i, the three terms diag1 + diag2 + diag3 of the reference
__global__ void k_fitc_train_var(int64_t n, const double* __restrict__ prior, const double* __restrict__ t1,
                                 const double* __restrict__ Dt, const double* __restrict__ q,
                                 const double* __restrict__ S, double* __restrict__ out) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const double si = S[i], qi = q[i], d = Dt[i];
    out[i] = prior[i] - (t1[i] + 2.0 * d * qi / si + d * d * (1.0 / si - qi / (si * si)));
}

void fitc_train_var(hipStream_t s, int64_t n, const double* prior, const double* t1, const double* Dt,
                    const double* q, const double* S, double* out) {
    hipLaunchKernelGGL(k_fitc_train_var, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, n, prior, t1, Dt, q, S,
                       out);
}

}  // namespace gpl
