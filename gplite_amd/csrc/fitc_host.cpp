// FITC (method_fitc) on the device, in whitened form: A = Lz^-1 K_zx (m x n,
// Kz = Lz Lz^T) stays resident, and every Newton step reduces to one product
// A S^-1 A^T on MFMA, an m x m Cholesky and three passes over A (kernels of their
// own: fitc.hip).  With G = I + A S^-1 A^T the reference's Kz + K_zx S^-1 K_xz is
// Lz G Lz^T: its leading minors have the same signs, its log-determinant is
// log|Kz| + log|G|, and its inverse between K_xz and K_zx is G^-1 between A^T and A.
// The rows of K_xz themselves are only needed while A is formed, a block of
// columns at a time.  (Both orientations of K_xz resident, a scaled copy and six
// passes took 16.2 ms of kernels at n = 131072, m = 1024 and 3.1 GB; now 1.5 GB.)
//
// Reference: R/gp_fit.R:101-123 (fit_laplace.method_fitc),
// R/laplace.R:122-180 (laplace_iter.method_fitc, log-concave branch),
// R/laplace.R:300-322 (laplace.method_fitc), R/linear_algebra.R:3-172
// (inv_lemma_get / inv_lemma_solve), R/gp_pred.R:234-290
// (gp_pred_post.method_fitc).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <string>
#include <vector>

#include "gplite_amd.h"
#include "host_common.h"

using namespace gpl;

namespace {

enum {
    F_PROG, F_X, F_F, F_ZX, F_FZ, F_Y, F_TR, F_OFF,
    F_LZ, F_DINVZ, F_LDZ, F_XZ,  // Kz -> its factor Lz, diagonal inverses, log pivots, Lz^-1
    F_A, F_W,                    // A = Lz^-1 K_zx (Mz x N), a block of columns (of K_zx, of Lc^-1 A)
    F_G, F_DINVG, F_LDG, F_XG,   // G = I + A S^-1 A^T -> its factor Lc, Lc^-1
    F_WZ,                        // w = A alpha = Lz^-1 K_zx alpha
    F_D, F_Z, F_V, F_SV, F_S, F_SI, F_ZS, F_ALPHA, F_FMEAN, F_FOLD, F_V1, F_V2, F_V3, F_V4,
    F_FVAR, F_FVOLD, F_ZOLD, F_POLD, F_CAVM, F_CAVV, F_LOGZS, F_TERM, F_GH,  // EP state
    F_Q1, F_Q2, F_SCAL, F_INFO, F_SPLIT, F_PART,
    F_COUNT
};

}  // namespace

struct gpl_fitc {
    gpl_ctx* ctx = nullptr;
    int64_t n = 0, N = 0, m = 0, Mz = 0, ncols = 0;
    DevProg prog{};
    gpl_lik lik{};
    gpl_opts opts{};
    bool has_trials = false, has_offset = false;
    double logZ = 0;
    int32_t iters = 0;
    DevBuf b[F_COUNT];
    ~gpl_fitc() {
        for (auto& x : b) x.free_();
    }
    double* d(int i) const { return b[i].as<double>(); }
};

#define FENSURE(fm, idx, bytes)                                                               \
    do {                                                                                      \
        if (!(fm)->b[idx].ensure(bytes, (fm)->ctx->blocks)) return fail(GPL_ERR_OOM, "device allocation failed"); \
    } while (0)

// Partial products of A S^-1 A^T over column ranges, summed in a fixed order: as
// many as fill the chip with 64x64 output tiles four times over (2048 of them), at
// least 256 columns each.  n = 131072, products and sum, in 7 / 15 / 30 / 64 parts, us:
// m = 1024 2797 / 2668 / 2683 / 2723 (15 are taken), m = 512 749 / 964 / 843 / 736 (56:
// 744), m = 128 630 / 306 / 165 / 90 (64).
static int64_t fitc_part_cols(const gpl_fitc* f) {
    const int64_t T = f->Mz / 64, tiles = T * (T + 1) / 2;
    const int64_t P = std::max<int64_t>(1, std::min<int64_t>({2048 / tiles, 64, f->N / 256}));
    return pad64((f->N + P - 1) / P);
}
static int fitc_parts(const gpl_fitc* f) {
    const int64_t kp = fitc_part_cols(f);
    return (int)((f->N + kp - 1) / kp);
}

// Columns of K_zx (of Lc^-1 A) formed at a time: 2^25 elements, four blocks at
// m = 1024, n = 131072
static int64_t fitc_block_cols(const gpl_fitc* f) {
    return std::max<int64_t>(64, std::min<int64_t>(f->N, ((int64_t)1 << 25) / f->Mz / 64 * 64));
}

static int fitc_alloc(gpl_fitc* f) {
    const int64_t N = f->N, Mz = f->Mz;
    const size_t vN = (size_t)N * 8, vM = (size_t)Mz * 8, mm = (size_t)Mz * Mz * 8;
    FENSURE(f, F_PROG, sizeof(DevProg));
    FENSURE(f, F_X, (size_t)f->n * std::max<int64_t>(f->ncols, 1) * 8);
    FENSURE(f, F_ZX, (size_t)f->m * std::max<int64_t>(f->ncols, 1) * 8);
    FENSURE(f, F_F, (size_t)N * MAX_FEAT * 8);
    FENSURE(f, F_FZ, (size_t)Mz * MAX_FEAT * 8);
    for (int i : {F_LZ, F_XZ, F_G, F_XG}) FENSURE(f, i, mm);
    for (int i : {F_DINVZ, F_DINVG}) FENSURE(f, i, (size_t)Mz * 64 * 8);
    for (int i : {F_LDZ, F_LDG, F_WZ, F_Q1, F_Q2}) FENSURE(f, i, vM);
    FENSURE(f, F_A, (size_t)N * Mz * 8);
    FENSURE(f, F_W, (size_t)fitc_block_cols(f) * Mz * 8);
    for (int i : {F_Y, F_TR, F_OFF, F_D, F_Z, F_V, F_SV, F_S, F_SI, F_ZS, F_ALPHA, F_FMEAN, F_FOLD, F_V1, F_V2, F_V3,
                  F_V4, F_FVAR, F_FVOLD, F_ZOLD, F_POLD, F_CAVM, F_CAVV, F_LOGZS, F_TERM})
        FENSURE(f, i, vN);
    FENSURE(f, F_GH, 64 * 8);
    FENSURE(f, F_SCAL, 64 * 8);
    FENSURE(f, F_INFO, 64);
    FENSURE(f, F_SPLIT, fitc_parts(f) * mm);
    FENSURE(f, F_PART, fitc_pass_parts(f->n) * vM);
    return GPL_OK;
}

static int fitc_upload(gpl_fitc* f, int idx, const double* h) {
    hipStream_t s = f->ctx->stream;
    fill_f64(s, f->d(idx), f->N, 0.0);
    if (h) HIP_TRY(upload(f->ctx, s, f->d(idx), h, f->n * 8));
    return GPL_OK;
}

static int fitc_scalars(gpl_fitc* f, double* out, int k, int* flags) {
    hipStream_t s = f->ctx->stream;
    double* st = f->ctx->stage;
    HIP_TRY(hipMemcpyAsync(st, f->d(F_SCAL), k * 8, hipMemcpyDeviceToHost, s));
    HIP_TRY(hipMemcpyAsync(st + k, f->b[F_INFO].p, 8, hipMemcpyDeviceToHost, s));
    HIP_TRY(hipStreamSynchronize(s));
    memcpy(out, st, k * 8);
    memcpy(flags, st + k, 8);
    return GPL_OK;
}

// One inversion-lemma solve for the current sites: S = D + V, G = I + A S^-1 A^T
// and its factor Lc, alpha = C^-1 z, w = A alpha and the posterior mean K_f alpha
// into F_FMEAN (R/laplace.R:134-141, R/ep.R:166-176).  With `inverse` also Lc^-1,
// its leading half beside the factor.  flags[0] receives G's failing minor.
static void fitc_lemma_step(gpl_fitc* f, int* flags, bool inverse) {
    gpl_ctx* c = f->ctx;
    hipStream_t s = c->stream;
    const int64_t n = f->n, N = f->N, Mz = f->Mz;
    const double* A = f->d(F_A);
    fitc_site(s, n, N, f->d(F_D), f->d(F_V), f->d(F_Z), f->d(F_S), f->d(F_SI), f->d(F_ZS));
    {
        Prof p(c, "fitc_syrk", (double)Mz * Mz * N, 8.0 * N * Mz);
        const int P = fitc_parts(f);
        gemm_gram_f64(s, Mz, N, A, Mz, f->d(F_SI), P, fitc_part_cols(f), f->d(F_SPLIT), Mz, Mz * Mz);
        fitc_gram_sum(s, f->d(F_SPLIT), P, Mz, f->d(F_G));
    }
    {
        Prof p(c, "fitc_pass", 0, 8.0 * N * Mz);
        fitc_combine(s, A, Mz, n, f->d(F_ZS), f->d(F_PART), f->d(F_Q1));
    }
    potrf_blocked(c, f->d(F_G), Mz, f->d(F_DINVG), f->d(F_LDG), flags, inverse ? f->d(F_XG) : nullptr, nullptr,
                  f->d(F_Q1));
    trsv_back(c, s, f->d(F_G), Mz, f->d(F_DINVG), Mz, f->d(F_Q1), f->d(F_Q2), flags);
    Prof pv(c, "fitc_pass", 0, 16.0 * N * Mz);
    fitc_alpha_pass(s, A, Mz, n, N, f->d(F_Q2), f->d(F_ZS), f->d(F_S), f->d(F_ALPHA), f->d(F_PART), f->d(F_WZ));
    fitc_mean(s, A, Mz, n, N, f->d(F_WZ), f->d(F_D), f->d(F_ALPHA), f->d(F_FMEAN));
}

// q_i = |Lc^-1 a_i|^2 for the current G (into `out`), through F_W
static void fitc_q(gpl_fitc* f, double* out) {
    hipStream_t s = f->ctx->stream;
    const int64_t N = f->N, Mz = f->Mz, nb = fitc_block_cols(f);
    Prof p(f->ctx, "fitc_q", (double)Mz * Mz * N, 16.0 * N * Mz);
    for (int64_t c0 = 0; c0 < N; c0 += nb) {
        const int64_t w = std::min(nb, N - c0);
        gemm2_f64(s, 0, 0, Mz, w, Mz, 1.0, f->d(F_XG), Mz, f->d(F_A) + c0 * Mz, Mz, 0.0, f->d(F_W), Mz, 3);
        colsumsq_f64(s, f->d(F_W), Mz, Mz, std::min(w, f->n - c0), out + c0, 0);
    }
}

// Damped parallel EP over the FITC prior: ep.method_fitc (R/ep.R:332-370; its
// tolerance is 1e-3) around the log-concave branch of ep_iter.method_fitc
// (R/ep.R:148-185,271-278).
static int fitc_ep_loop(gpl_fitc* f, const double* tr, const double* off) {
    gpl_ctx* c = f->ctx;
    hipStream_t s = c->stream;
    const int64_t n = f->n, N = f->N, Mz = f->Mz;
    const int q = f->opts.quad_order > 0 ? f->opts.quad_order : 11;
    if (q > 32) return fail(GPL_ERR_ARG, "quad_order must be <= 32");
    std::vector<double> gx, gw;
    gauss_hermite(q, gx, gw);
    HIP_TRY(hipMemcpyAsync(f->d(F_GH), gx.data(), q * 8, hipMemcpyHostToDevice, s));
    HIP_TRY(hipMemcpyAsync(f->d(F_GH) + 32, gw.data(), q * 8, hipMemcpyHostToDevice, s));
    // P_old = 0, z_old = 0, fmean_old = 0, fvar_old = diag K + jitter (R/gp_fit.R:171, R/ep.R:339)
    fill_f64(s, f->d(F_POLD), N, 0.0);
    fill_f64(s, f->d(F_ZOLD), N, 0.0);
    fill_f64(s, f->d(F_FOLD), N, 0.0);
    fill_f64(s, f->d(F_V3), N, 0.0);
    launch_build_diag(s, f->b[F_PROG].as<DevProg>(), f->prog, f->d(F_F), N, f->d(F_F), N, n, f->d(F_V2));
    fitc_diag(s, n, N, f->d(F_V2), f->d(F_V3), f->opts.jitter, f->d(F_FVOLD));
    const int maxiter = f->opts.maxiter > 0 ? f->opts.maxiter : 100;
    const double tol = 1e-3, damping = f->opts.damping;
    const double dmin = f->opts.damping_min > 0 ? f->opts.damping_min : 0.1;
    double damp = damping, diff_old = INFINITY, diff_new = INFINITY;
    bool quad_ok = true;
    int* flags = f->b[F_INFO].as<int>();
    int fl[2];
    double sc[8];
    int it;
    for (it = 1; it <= maxiter; ++it) {
        HIP_TRY(hipMemsetAsync(flags, 0, 8, s));
        ep_sites(s, f->lik.kind, f->lik.link, lik_par(f->lik), n, f->d(F_FOLD), f->d(F_FVOLD), f->d(F_ZOLD), f->d(F_POLD), f->d(F_Y),
                 tr, off, q, f->d(F_GH), f->d(F_GH) + 32, damp, f->d(F_Z), f->d(F_V), f->d(F_SV), f->d(F_LOGZS),
                 f->d(F_CAVM), f->d(F_CAVV), flags + 1);
        HIP_TRY(hipMemcpyAsync(fl, flags, 8, hipMemcpyDeviceToHost, s));
        HIP_TRY(hipStreamSynchronize(s));
        if (fl[1] & 2) {
            f->logZ = -INFINITY;
            f->iters = it;
            return fail(GPL_ERR_NAN, "NaN in EP site parameters (R/ep.R:163-165 returns log_evidence = -Inf)");
        }
        if (fl[1] & 4) {
            f->logZ = -INFINITY;
            return fail(GPL_ERR_UNSUPPORTED, "EP site variance <= 0: R/ep.R:186-270 is not on the device path");
        }
        if (fl[1] & 1) quad_ok = false;
        fitc_lemma_step(f, flags, true);
        fitc_q(f, f->d(F_V1));
        fitc_ep_var(s, n, f->d(F_V), f->d(F_S), f->d(F_D), f->d(F_V1), f->d(F_FVAR));
        // per-site evidence terms (the binv argument only feeds an unused output here)
        ep_post(s, n, f->d(F_V), f->d(F_Z), f->d(F_V1), f->d(F_CAVM), f->d(F_CAVV), f->d(F_LOGZS), f->d(F_V4),
                f->d(F_TERM));
        double* scd = f->d(F_SCAL);
        reduce_sum(s, f->d(F_TERM), n, scd + 0);
        reduce_dot(s, f->d(F_Z), f->d(F_ALPHA), n, scd + 1);
        vec_log(s, n, f->d(F_V), f->d(F_V3));
        reduce_sum(s, f->d(F_V3), n, scd + 2);
        vec_log(s, n, f->d(F_S), f->d(F_V4));
        reduce_sum(s, f->d(F_V4), n, scd + 3);
        reduce_sum(s, f->d(F_LDG), Mz, scd + 4);
        reduce_maxabsdiff(s, f->d(F_FOLD), f->d(F_FMEAN), n, scd + 5);
        int r = fitc_scalars(f, sc, 6, fl);
        if (r) return r;
        if (fl[0] == kPanelWaitTimeout) return wait_timeout_fail();
        if (fl[0] > 0) {
            set_minor(fl[0]);
            return fail(GPL_ERR_NOT_PD, "inversion lemma: the leading minor of order " + std::to_string(fl[0]) +
                                            " of Kz + K_zx S^-1 K_xz is not positive");
        }
        // log Z_EP (R/ep.R:179-181); the site terms carry -1/2 log V, added back here
        const double logdet = sc[3] + 2.0 * sc[4];
        f->logZ = sc[0] + 0.5 * sc[2] - 0.5 * logdet - 0.5 * sc[1];
        diff_new = sc[5];
        if (diff_new > diff_old) {
            damp = damp * damping;
            continue;
        }
        damp = std::max(damp, dmin);
        HIP_TRY(hipMemcpyAsync(f->d(F_FOLD), f->d(F_FMEAN), N * 8, hipMemcpyDeviceToDevice, s));
        HIP_TRY(hipMemcpyAsync(f->d(F_FVOLD), f->d(F_FVAR), N * 8, hipMemcpyDeviceToDevice, s));
        HIP_TRY(hipMemcpyAsync(f->d(F_ZOLD), f->d(F_Z), N * 8, hipMemcpyDeviceToDevice, s));
        vec_recip(s, n, f->d(F_V), f->d(F_POLD));
        diff_old = diff_new;
        if (diff_new < tol) break;
    }
    if (it > maxiter) it = maxiter;
    f->iters = it;
    if (!quad_ok) f->logZ = -INFINITY;
    if (maxiter > 1 && it == maxiter) {  // R/ep.R:362-365
        f->logZ = -INFINITY;
        fail(GPL_ERR_NOCONV, "Maximum number of iterations in EP reached, max delta f = " + std::to_string(diff_new));
        return GPL_ERR_NOCONV;
    }
    return GPL_OK;
}

static int fitc_run(gpl_fitc* f) {
    gpl_ctx* c = f->ctx;
    hipStream_t s = c->stream;
    const int64_t n = f->n, N = f->N, m = f->m, Mz = f->Mz;
    const DevProg* pd = f->b[F_PROG].as<DevProg>();
    const double jitter = f->opts.jitter;
    int* flags = f->b[F_INFO].as<int>();
    int fl[2] = {0, 0};
    // Kz = K(z, z) + jitter I (padding: identity), its factor Lz and Lz^-1
    launch_build_sym_f64(s, pd, f->prog, f->d(F_FZ), m, Mz, jitter, 0, 1.0, nullptr, f->d(F_LZ), Mz);
    HIP_TRY(hipMemsetAsync(flags, 0, 8, s));
    potrf_blocked(c, f->d(F_LZ), Mz, f->d(F_DINVZ), f->d(F_LDZ), flags, f->d(F_XZ));
    double sc[8];
    int r = fitc_scalars(f, sc, 1, fl);
    if (r) return r;
    if (fl[0] == kPanelWaitTimeout) return wait_timeout_fail();
    if (fl[0] > 0) {
        set_minor(fl[0]);
        return fail(GPL_ERR_NOT_PD, "Kz: the leading minor of order " + std::to_string(fl[0]) + " is not positive");
    }
    // A = Lz^-1 K_zx (zero outside m x n), a block of K_zx's columns at a time;
    // D = diag K + jitter - colSums(A^2)  (R/gp_fit.R:107-108)
    {
        Prof p(c, "fitc_whiten", (double)Mz * Mz * N, 32.0 * N * Mz);
        const int64_t nb = fitc_block_cols(f);
        for (int64_t c0 = 0; c0 < N; c0 += nb) {
            const int64_t w = std::min(nb, N - c0);
            double* A = f->d(F_A) + c0 * Mz;
            launch_build_cross(s, pd, f->prog, f->d(F_FZ), Mz, m, Mz, f->d(F_F) + c0, N, std::min(w, n - c0), w,
                               f->d(F_W), Mz);
            gemm2_f64(s, 0, 0, Mz, w, Mz, 1.0, f->d(F_XZ), Mz, f->d(F_W), Mz, 0.0, A, Mz, 3);
        }
        colsumsq_f64(s, f->d(F_A), Mz, Mz, n, f->d(F_V1), 0);
    }
    launch_build_diag(s, pd, f->prog, f->d(F_F), N, f->d(F_F), N, n, f->d(F_V2));
    fitc_diag(s, n, N, f->d(F_V2), f->d(F_V1), jitter, f->d(F_D));

    const double* tr = f->has_trials ? f->d(F_TR) : nullptr;
    const double* off = f->has_offset ? f->d(F_OFF) : nullptr;
    if (f->opts.approx == GPL_APPROX_EP) {
        r = fitc_ep_loop(f, tr, off);
        if (r && r != GPL_ERR_NOCONV) return r;
        HIP_TRY(hipStreamSynchronize(s));
        return r;
    }
    const bool gauss = f->lik.kind == GPL_LIK_GAUSSIAN;
    const int maxiter = gauss ? 1 : (f->opts.maxiter > 0 ? f->opts.maxiter : 30);  // R/laplace.R:303-305
    double log_post_old = -INFINITY, diff = INFINITY;
    fill_f64(s, f->d(F_FOLD), N, 0.0);
    int it;
    for (it = 1; it <= maxiter; ++it) {
        HIP_TRY(hipMemsetAsync(flags, 0, 8, s));
        if (gauss)
            lik_pseudodata_la(s, GPL_LIK_GAUSSIAN, 0, f->lik.sigma, n, nullptr, f->d(F_Y), nullptr, nullptr,
                              f->d(F_Z), f->d(F_V), f->d(F_SV), flags + 1);
        else
            lik_pseudodata_la(s, f->lik.kind, f->lik.link, lik_par(f->lik), n, f->d(F_FOLD), f->d(F_Y), tr, off, f->d(F_Z),
                              f->d(F_V), f->d(F_SV), flags + 1, (f->opts.flags & GPL_FLAG_ANALYTIC_W) ? 1 : 0);
        // inversion lemma for C = K_xz Kz^-1 K_zx + S, S = D + V (R/linear_algebra.R:3-47)
        fitc_lemma_step(f, flags, gauss);
        // log evidence (R/laplace.R:143-151): logdet C - log|V| from the lemma
        lik_loglik(s, f->lik.kind, f->lik.link, lik_par(f->lik), n, f->d(F_FMEAN), f->d(F_Y), tr, off,
                   f->d(F_V3));
        double* scd = f->d(F_SCAL);
        reduce_sum(s, f->d(F_V3), n, scd + 0);
        reduce_dot(s, f->d(F_FMEAN), f->d(F_ALPHA), n, scd + 1);
        vec_log(s, n, f->d(F_V), f->d(F_V3));
        reduce_sum(s, f->d(F_V3), n, scd + 2);
        vec_log(s, n, f->d(F_S), f->d(F_V4));
        reduce_sum(s, f->d(F_V4), n, scd + 3);
        reduce_sum(s, f->d(F_LDG), Mz, scd + 4);
        r = fitc_scalars(f, sc, 5, fl);
        if (r) return r;
        if (fl[1] & 6) {
            f->logZ = -INFINITY;
            return fail((fl[1] & 2) ? GPL_ERR_NAN : GPL_ERR_UNSUPPORTED,
                        (fl[1] & 2) ? "NaN in Laplace pseudo-data"
                                    : "non-log-concave pseudo-variance (V <= 0): R/laplace.R:155-235 is not on "
                                      "the device path");
        }
        if (fl[0] == kPanelWaitTimeout) return wait_timeout_fail();
        if (fl[0] > 0) {
            set_minor(fl[0]);
            return fail(GPL_ERR_NOT_PD, "inversion lemma: the leading minor of order " + std::to_string(fl[0]) +
                                            " of Kz + K_zx S^-1 K_xz is not positive");
        }
        const double logdet = sc[3] + 2.0 * sc[4];
        const double log_post = sc[0] - 0.5 * sc[1];
        f->logZ = log_post + 0.5 * (sc[2] - logdet);
        HIP_TRY(hipMemcpyAsync(f->d(F_FOLD), f->d(F_FMEAN), N * 8, hipMemcpyDeviceToDevice, s));
        diff = log_post - log_post_old;
        log_post_old = log_post;
        if (std::fabs(diff) < f->opts.tol) break;
    }
    if (it > maxiter) it = maxiter;
    f->iters = it;
    // prediction state: w (from the last step) and Lc^-1
    if (!gauss) trtri_blocked(c, f->d(F_G), f->d(F_DINVG), Mz, f->d(F_XG));
    HIP_TRY(hipStreamSynchronize(s));
    if (maxiter > 1 && it == maxiter) {  // R/laplace.R:318-320 warns whenever the cap is reached
        fail(GPL_ERR_NOCONV, "Maximum number of iterations in Laplace reached, delta log post = " +
                                 std::to_string(diff));
        return GPL_ERR_NOCONV;
    }
    return GPL_OK;
}

extern "C" int gpl_fitc_fit(gpl_ctx* c, const gpl_cf_term* terms, int32_t nterms, const double* x, int64_t n,
                            int64_t ncols, const double* z, int64_t m, const double* y, const double* trials,
                            const double* offset, const gpl_lik* lik, const gpl_opts* opts, gpl_fitc** out,
                            double* log_evidence) {
    if (!c || !x || !z || !y || !lik || !out) return fail(GPL_ERR_ARG, "NULL argument");
    if (n < 1 || m < 1 || ncols < 0) return fail(GPL_ERR_ARG, "n and m must be >= 1");
    gpl_opts o;
    if (opts) o = *opts;
    else gpl_opts_default(&o);
    if (lik->kind == GPL_LIK_GAUSSIAN && o.approx == GPL_APPROX_EP)
        return fail(GPL_ERR_ARG, "approx_ep disabled for lik_gaussian");  // R/gp.R:54-56
    if (o.precision != GPL_PREC_FP64) return fail(GPL_ERR_UNSUPPORTED, "FITC runs in FP64");
    if (lik->kind == GPL_LIK_GAUSSIAN && !(lik->sigma > 0)) return fail(GPL_ERR_ARG, "sigma must be positive");
    if ((o.flags & GPL_FLAG_ANALYTIC_W) && lik->kind == GPL_LIK_BETABINOM)
        return fail(GPL_ERR_UNSUPPORTED, "the exact curvature is provided for the logit, probit and log links "
                                         "(not the beta-binomial likelihood)");
    DevProg P;
    int r = prepare_prog(terms, nterms, ncols, P);
    if (r) return r;
    std::lock_guard<std::mutex> lk(c->mu);
    HIP_TRY(hipSetDevice(c->device));
    gpl_fitc* f = new gpl_fitc();
    f->ctx = c;
    f->n = n;
    f->N = pad64(n);
    f->m = m;
    f->Mz = pad64(m);
    f->ncols = ncols;
    f->prog = P;
    f->lik = *lik;
    f->opts = o;
    f->has_trials = trials != nullptr;
    f->has_offset = offset != nullptr;
    r = fitc_alloc(f);
    hipStream_t s = c->stream;
    auto setup = [&]() -> int {
        HIP_TRY(hipMemcpyAsync(f->b[F_PROG].p, &f->prog, sizeof(DevProg), hipMemcpyHostToDevice, s));
        if (n * ncols > 0) HIP_TRY(upload(c, s, f->d(F_X), x, n * ncols * 8));
        if (m * ncols > 0) HIP_TRY(upload(c, s, f->d(F_ZX), z, m * ncols * 8));
        const DevProg* pd = f->b[F_PROG].as<DevProg>();
        launch_features(s, f->d(F_X), n, n, (int)ncols, pd, f->prog, f->d(F_F), f->N);
        launch_features(s, f->d(F_ZX), m, m, (int)ncols, pd, f->prog, f->d(F_FZ), f->Mz);
        int q = fitc_upload(f, F_Y, y);
        if (!q) q = fitc_upload(f, F_TR, trials);
        if (!q) q = fitc_upload(f, F_OFF, offset);
        return q;
    };
    if (!r) r = setup();
    if (!r) r = fitc_run(f);
    if (r && r != GPL_ERR_NOCONV) {
        const double lz = f->logZ;
        delete f;
        if (log_evidence) *log_evidence = (r == GPL_ERR_NAN) ? -INFINITY : lz;
        return r;
    }
    *out = f;
    if (log_evidence) *log_evidence = f->logZ;
    return r;
}

extern "C" int gpl_fitc_pred(gpl_fitc* f, const double* xt, int64_t mt, int32_t want_var, double* mean,
                             double* var) {
    if (!f || (!xt && mt > 0) || !mean || (want_var && !var)) return fail(GPL_ERR_ARG, "NULL argument");
    if (mt <= 0) return GPL_OK;
    gpl_ctx* c = f->ctx;
    std::lock_guard<std::mutex> lk(c->mu);
    HIP_TRY(hipSetDevice(c->device));
    hipStream_t s = c->stream;
    const int64_t m = f->m, Mz = f->Mz, Mt = pad64(mt);
    const DevProg* pd = f->b[F_PROG].as<DevProg>();
    double* xtd = (double*)c->buf(10, (size_t)mt * std::max<int64_t>(f->ncols, 1) * 8);
    double* Ft = (double*)c->buf(11, (size_t)Mt * MAX_FEAT * 8);
    double* KzT = (double*)c->buf(12, (size_t)Mz * Mt * 8);
    double* A2 = (double*)c->buf(13, (size_t)Mz * Mt * 8);
    double* Yv = (double*)c->buf(14, (size_t)Mz * Mt * 8);
    double* vb = (double*)c->buf(15, (size_t)Mt * 6 * 8);
    if (!xtd || !Ft || !KzT || !A2 || !Yv || !vb) return fail(GPL_ERR_OOM, "device allocation failed");
    if (mt * f->ncols > 0) HIP_TRY(hipMemcpyAsync(xtd, xt, mt * f->ncols * 8, hipMemcpyHostToDevice, s));
    launch_features(s, xtd, mt, mt, (int)f->ncols, pd, f->prog, Ft, Mt);
    launch_build_cross(s, pd, f->prog, f->d(F_FZ), Mz, m, Mz, Ft, Mt, mt, Mt, KzT, Mz);
    // A_t = Lz^-1 K_zt (Kt_aux2); mean = A_t^T w
    gemm2_f64(s, 0, 0, Mz, Mt, Mz, 1.0, f->d(F_XZ), Mz, KzT, Mz, 0.0, A2, Mz, 3);
    gemv_t_f64(s, A2, Mz, Mz, mt, f->d(F_WZ), vb);
    if (want_var) {
        // prior_var = colSums(K_zt * Kz^-1 K_zt) + Dt with Dt = diag K_tt - colSums(A_t^2) is
        // diag K_tt, and var_reduction = colSums(A_t * (M A_t)), M = A C^-1 A^T = I - G^-1, is
        // colSums(A_t^2) - colSums((Lc^-1 A_t)^2)  (R/gp_pred.R:244-246,271,278-280)
        double* c2 = vb + Mt;
        double* kd = vb + 2 * Mt;
        double* q = vb + 3 * Mt;
        double* red = vb + 4 * Mt;
        colsumsq_f64(s, A2, Mz, Mz, mt, c2, 0);
        launch_build_diag(s, pd, f->prog, Ft, Mt, Ft, Mt, mt, kd);
        vec_axpby(s, mt, 1.0, kd, -1.0, c2, c2);
        gemm2_f64(s, 0, 0, Mz, Mt, Mz, 1.0, f->d(F_XG), Mz, A2, Mz, 0.0, Yv, Mz, 3);
        colsumsq_f64(s, Yv, Mz, Mz, mt, q, 0);
        vec_axpby(s, mt, 1.0, c2, 1.0, q, red);
        HIP_TRY(read_back(c, var, red, mt * 8));
    }
    HIP_TRY(read_back(c, mean, vb, mt * 8));
    return GPL_OK;
}

// gp_draw_analytic.method_fitc with marginal = FALSE (R/gp_draw.R:126-140):
// mean + chol(cov + jitter I) z, cov = A_t^T A_t + diag(Dt) - A_t^T M A_t
// (R/gp_pred.R:258-268, train = FALSE), = (Lc^-1 A_t)^T (Lc^-1 A_t) + diag(Dt).
extern "C" int gpl_fitc_draw(gpl_fitc* f, const double* xt, int64_t mt, double jitter, const double* z,
                             int64_t draws, double* out) {
    if (!f || !xt || !z || !out || mt < 1 || draws < 1) return fail(GPL_ERR_ARG, "bad argument");
    gpl_ctx* c = f->ctx;
    std::lock_guard<std::mutex> lk(c->mu);
    HIP_TRY(hipSetDevice(c->device));
    hipStream_t s = c->stream;
    const int64_t m = f->m, Mz = f->Mz, Mt = pad64(mt), Dp = pad64(draws);
    const DevProg* pd = f->b[F_PROG].as<DevProg>();
    double* xtd = (double*)c->buf(10, (size_t)mt * std::max<int64_t>(f->ncols, 1) * 8);
    double* Ft = (double*)c->buf(11, (size_t)Mt * MAX_FEAT * 8);
    double* KzT = (double*)c->buf(12, (size_t)Mz * Mt * 8);
    double* A2 = (double*)c->buf(13, (size_t)Mz * Mt * 8);
    double* Yv = (double*)c->buf(14, (size_t)Mz * Mt * 8);
    double* vb = (double*)c->buf(15, (size_t)Mt * 6 * 8);
    double* Cv = (double*)c->buf(16, (size_t)Mt * Mt * 8);
    double* Dv = (double*)c->buf(17, (size_t)Mt * 64 * 8 + (size_t)Mt * 8 + 64);
    double* Zd = (double*)c->buf(18, (size_t)Mt * Dp * 8);
    double* Wd = (double*)c->buf(19, (size_t)Mt * Dp * 8);
    if (!xtd || !Ft || !KzT || !A2 || !Yv || !vb || !Cv || !Dv || !Zd || !Wd)
        return fail(GPL_ERR_OOM, "device allocation failed");
    double* ld = Dv + Mt * 64;
    int* info = (int*)(ld + Mt);
    if (mt * f->ncols > 0) HIP_TRY(hipMemcpyAsync(xtd, xt, mt * f->ncols * 8, hipMemcpyHostToDevice, s));
    launch_features(s, xtd, mt, mt, (int)f->ncols, pd, f->prog, Ft, Mt);
    launch_build_cross(s, pd, f->prog, f->d(F_FZ), Mz, m, Mz, Ft, Mt, mt, Mt, KzT, Mz);
    gemm2_f64(s, 0, 0, Mz, Mt, Mz, 1.0, f->d(F_XZ), Mz, KzT, Mz, 0.0, A2, Mz, 3);
    gemv_t_f64(s, A2, Mz, Mz, mt, f->d(F_WZ), vb);
    // Dt = diag K_tt - colSums(A_t^2)
    double* dt = vb + Mt;
    colsumsq_f64(s, A2, Mz, Mz, mt, dt, 0);
    launch_build_diag(s, pd, f->prog, Ft, Mt, Ft, Mt, mt, vb + 2 * Mt);
    vec_axpby(s, mt, 1.0, vb + 2 * Mt, -1.0, dt, dt);
    // lower tiles of the product, then the diagonal terms
    gemm2_f64(s, 0, 0, Mz, Mt, Mz, 1.0, f->d(F_XG), Mz, A2, Mz, 0.0, Yv, Mz, 3);
    gemm2_f64(s, 1, 0, Mt, Mt, Mz, 1.0, Yv, Mz, Yv, Mz, 0.0, Cv, Mt, 1);
    add_diag_f64(s, Cv, Mt, mt, Mt, dt, jitter);
    HIP_TRY(hipMemsetAsync(info, 0, 64, s));
    potrf_blocked(c, Cv, Mt, Dv, ld, info);
    int inf = 0;
    HIP_TRY(hipMemcpyAsync(&inf, info, 4, hipMemcpyDeviceToHost, s));
    fill_f64(s, Zd, Mt * Dp, 0.0);
    HIP_TRY(upload_2d(c, s, Zd, Mt, z, mt, draws, 20));
    gemm2_f64(s, 0, 0, Mt, Dp, Mt, 1.0, Cv, Mt, Zd, Mt, 0.0, Wd, Mt, 3);
    std::vector<double> mean(mt);
    HIP_TRY(hipMemcpyAsync(mean.data(), vb, mt * 8, hipMemcpyDeviceToHost, s));
    HIP_TRY(download_2d(c, s, out, Wd, Mt, mt, draws, 21));
    HIP_TRY(hipStreamSynchronize(s));
    if (inf > 0) {
        set_minor(inf);
        return fail(GPL_ERR_NOT_PD, "predictive covariance: the leading minor of order " + std::to_string(inf) +
                                        " is not positive (raise jitter)");
    }
    for (int64_t j = 0; j < draws; ++j)
        for (int64_t i = 0; i < mt; ++i) out[i + j * mt] += mean[i];
    return GPL_OK;
}

// Predictive variance at the training inputs with the FITC diagonal
// (gp_pred_post.method_fitc, train = TRUE: R/gp_pred.R:270-285), the input of
// loo_posteriors.approx_laplace (R/gp_loo.R:120-130).  With A = Lz^-1 K_zx,
// Dt = diag K - colSums(A^2) and q_i = |Lc^-1 a_i|^2 the reference's three terms
// are (A^T M A)_ii, 2 Dt_i q_i / S_i and Dt_i^2 [C^-1]_ii.
extern "C" int gpl_fitc_train_var(gpl_fitc* f, double* out) {
    if (!f || !out) return fail(GPL_ERR_ARG, "NULL argument");
    gpl_ctx* c = f->ctx;
    std::lock_guard<std::mutex> lk(c->mu);
    HIP_TRY(hipSetDevice(c->device));
    hipStream_t s = c->stream;
    const int64_t n = f->n, N = f->N, Mz = f->Mz;
    double* v = (double*)c->buf(24, (size_t)N * 6 * 8);
    if (!v) return fail(GPL_ERR_OOM, "device allocation failed");
    double *c2 = v, *kd = v + N, *t1 = v + 2 * N, *q = v + 3 * N, *res = v + 4 * N;
    colsumsq_f64(s, f->d(F_A), Mz, Mz, n, c2, 0);
    launch_build_diag(s, f->b[F_PROG].as<DevProg>(), f->prog, f->d(F_F), N, f->d(F_F), N, n, kd);
    fitc_q(f, q);
    vec_axpby(s, n, 1.0, c2, -1.0, q, t1);
    vec_axpby(s, n, 1.0, kd, -1.0, c2, c2);  // Dt
    fitc_train_var(s, n, kd, t1, c2, q, f->d(F_S), res);
    HIP_TRY(hipMemcpyAsync(out, res, n * 8, hipMemcpyDeviceToHost, s));
    HIP_TRY(hipStreamSynchronize(s));
    return GPL_OK;
}

extern "C" int gpl_fitc_vector(gpl_fitc* f, int32_t which, double* out) {
    if (!f || !out) return fail(GPL_ERR_ARG, "NULL argument");
    int idx;
    switch (which) {
        case GPL_VEC_FMEAN: idx = F_FMEAN; break;
        case GPL_VEC_ALPHA: idx = F_ALPHA; break;
        case GPL_VEC_Z: idx = F_Z; break;
        case GPL_VEC_V: idx = F_V; break;
        case GPL_VEC_FVAR: idx = F_FVAR; break;
        case GPL_VEC_CAVITY_MEAN: idx = F_CAVM; break;
        case GPL_VEC_CAVITY_VAR: idx = F_CAVV; break;
        case 7: idx = F_D; break;
        default: return fail(GPL_ERR_ARG, "unknown FITC vector");
    }
    std::lock_guard<std::mutex> lk(f->ctx->mu);
    HIP_TRY(hipSetDevice(f->ctx->device));
    HIP_TRY(read_back(f->ctx, out, f->d(idx), f->n * 8));
    return GPL_OK;
}

extern "C" int gpl_fitc_info(gpl_fitc* f, int64_t* n, int64_t* m, int32_t* iters, double* log_evidence) {
    if (!f) return fail(GPL_ERR_ARG, "NULL model");
    if (n) *n = f->n;
    if (m) *m = f->m;
    if (iters) *iters = f->iters;
    if (log_evidence) *log_evidence = f->logZ;
    return GPL_OK;
}

extern "C" void gpl_fitc_free(gpl_fitc* f) {
    if (!f) return;
    gpl_ctx* c = f->ctx;
    hipSetDevice(c->device);
    for (hipStream_t st : {c->stream, c->side, c->aux}) hipStreamSynchronize(st);
    for (auto& x : f->b) x.give(c->blocks);
    c->blocks->age();
    delete f;
}
