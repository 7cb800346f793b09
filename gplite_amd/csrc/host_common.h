// Host-side pieces shared by the C-ABI translation units: device context,
// per-kernel-class event profiling, device buffers and error reporting.
#pragma once

#include <hip/hip_runtime.h>
#include <rocprofiler-sdk-roctx/roctx.h>

#include <algorithm>
#include <cstring>
#include <map>
#include <mutex>
#include <string>
#include <vector>

#include "gpl_internal.h"

namespace gpl {

int fail(int code, const std::string& msg);
void set_minor(int64_t minor);

#define HIP_TRY(expr)                                                                              \
    do {                                                                                           \
        hipError_t e_ = (expr);                                                                    \
        if (e_ != hipSuccess)                                                                      \
            return ::gpl::fail(GPL_ERR_HIP, std::string(#expr) + ": " + hipGetErrorString(e_));   \
    } while (0)

int prepare_prog(const gpl_cf_term* terms, int32_t nterms, int64_t ncols, DevProg& P);
// Blocked FP64 Cholesky of the N x N lower tiles of L in place (Dinv: the 64x64
// diagonal-block inverses, ldiag: log L_ii, info: first failing row + 1) and the
// triangular inverse X = L^-1 by recursive doubling (all tiles written; T, Tm: N x N
// scratch for its products, which otherwise lie above X's diagonal and are cleared
// at the end); potrf_blocked with X forms both, the inverse's front half beside the
// factor's last panels, and with rhs overwrites that vector (N rows) with L^-1 rhs
void potrf_blocked(gpl_ctx* c, double* L, int64_t N, double* Dinv, double* ldiag, int* info, double* X = nullptr,
                   double* Tm = nullptr, double* rhs = nullptr);
void trtri_blocked(gpl_ctx* c, const double* L, const double* Dinv, int64_t N, double* X, double* T = nullptr);
// L^T x = b with one vector in one launch (trsv_lower_f64's arguments, b left
// unchanged).  info receives kPanelWaitTimeout if a device wait times out.  With `scaled` also scaled =
// scale .* x (n entries, zero on the padding) unless *gate (if any) flags NaN or
// V <= 0.
void trsv_back(gpl_ctx* c, hipStream_t s, const double* L, int64_t ld, const double* Dinv, int64_t N, const double* b,
               double* x, int* info, const double* scale = nullptr, int64_t n = 0, double* scaled = nullptr,
               const int* gate = nullptr);
// L Y = diag(sv) B in place for M right-hand sides, of which the first mt are not
// padding (sv: the first n rows, or null): the forward solve of a prediction, in
// launches of at most kTrsmFlags blocks.  info receives kPanelWaitTimeout if a device
// wait times out.
void trsm_forward(gpl_ctx* c, hipStream_t s, const double* L, int64_t ld, const double* Dinv, int64_t N, double* B,
                int64_t ldb, int64_t M, int64_t mt, const double* sv, int64_t n, int* info);
// the error reported for an info word of kPanelWaitTimeout
int wait_timeout_fail();
// probabilists' Gauss-Hermite nodes and weights normalised to sum 1 (R/quadrature.R:1-44)
void gauss_hermite(int q, std::vector<double>& x, std::vector<double>& w);
// Device buffers of one prediction launch over M = pad64(mt) test points (see
// pred_bufs_bytes); when given to pred_on they replace the context's own scratch.
struct PredBufs {
    double *xt, *Ft, *KtT, *v, *A2;
    bool staged = false;  // the test inputs are already in xt (leading dimension mt)
};
// Bytes of the PredBufs for a model of padded size N with ncols input columns and
// M test-point rows, each part aligned to 256 bytes; carve them out of `base`.
size_t pred_bufs_bytes(int64_t N, int64_t ncols, int64_t M);
PredBufs pred_bufs_carve(void* base, int64_t N, int64_t ncols, int64_t M);
// padded size and input columns of a fitted model, and the context that owns it
void model_dims(const gpl_model* m, int64_t* N, int64_t* ncols);
gpl_ctx* model_ctx(const gpl_model* m);
// device address of gpl_pred_noalloc's scratch array on `device` (current), once
int noalloc_init(int device);
// terms/nsel (optional): predict with the model's terms terms[0..nsel) only (cfind);
// pb (optional): caller-provided device buffers instead of the context's scratch
int pred_on(gpl_ctx* c, gpl_model* m, const double* xt, int64_t mt, int32_t want_var, double* mean, double* var,
            const int32_t* terms = nullptr, int32_t nsel = 0, const PredBufs* pb = nullptr);

}  // namespace gpl

using gpl::fail;

inline int64_t pad64(int64_t n) { return (n + 63) / 64 * 64; }

// the likelihood's parameter the device kernels take: Gaussian sigma, beta-binomial phi
inline double lik_par(const gpl_lik& l) {
    return l.kind == GPL_LIK_GAUSSIAN ? l.sigma : (l.kind == GPL_LIK_BETABINOM ? l.phi : 0.0);
}

// ---------------------------------------------------------------------------
// context, profiling
// ---------------------------------------------------------------------------
struct ProfRec {
    int cls;
    hipEvent_t a, b;
    double flops, bytes;
};

struct ProfClass {
    std::string name;
    double ms = 0, flops = 0, bytes = 0;
    int64_t launches = 0;
};

// Device blocks above kMin bytes that freed models leave for the next one: such a
// block costs 13 us to allocate and 15 us to free, 45 and 280 us from 256 MB up
// (smaller ones come out of the runtime's own suballocator in under 1 us), which
// was 1.5 of the 13.5 ms of a fit and gradient at n = 8192.  Bounded: the pools of
// all contexts on a device hold at most 1/32 of its memory together, and a block that
// none of the last kKeep frees of a model has led to a use of is given back.  A block
// enters only after its streams were waited for.  Any allocation of the library that
// fails empties the pools of all contexts of the process and is tried again; other
// allocators' programs call gpl_release_memory.
struct BlockPool {
    static constexpr size_t kMin = (size_t)1 << 20;
    static constexpr unsigned kKeep = 16;
    struct Block {
        void* p;
        size_t sz;
        unsigned born;
    };
    std::mutex mu;
    std::vector<Block> blocks;
    const int device;
    const size_t cap;    // of the device's pools together (0: this one keeps nothing)
    unsigned frees = 0;  // models freed so far
    BlockPool(int dev, size_t cap_bytes);
    ~BlockPool();
    bool reserve(size_t sz);  // room for sz more bytes under the cap
    void drop(size_t i);      // frees a block (mu is held)
    void* take(size_t bytes, size_t* sz);  // the smallest block of bytes .. 1.25 bytes, or nullptr
    void put(void* p, size_t sz);          // keeps or frees it
    void age();                            // a model was freed
    void clear();
};
constexpr int kMaxDevices = 64;
hipError_t dev_malloc(void** p, size_t bytes);  // hipMalloc; when that fails, once more with empty pools

struct gpl_ctx {
    int device = 0;
    hipStream_t stream = nullptr;
    hipStream_t side = nullptr;  // look-ahead panel work (default priority, like the main stream)
    hipStream_t aux = nullptr;   // the front half of L^-1 beside the Cholesky's last panels
    hipEvent_t ev_h = nullptr, ev_t = nullptr, ev_h2 = nullptr;
    hipEvent_t ev_a = nullptr, ev_p = nullptr, ev_d = nullptr;
    // flags and ticket counter of the single-launch panel factorisation
    // (kPanelSyncWords words, zero at creation), its launch epoch and tickets handed out so far,
    // and the polls after which one of its waits gives up (2^20; the
    // environment variable GPL_PANEL_WAIT_POLLS overrides it, which tests use to
    // reach the timeout path)
    unsigned* psync = nullptr;
    double* dpub = nullptr;  // its published diagonal blocks (kPanelMaxBlocks 64x64 blocks)
    unsigned pepoch = 0, pbase = 0;
    // the single-launch triangular solves with one or a few vectors: their ticket word,
    // and the two arrays that the launches publish in by turns (every launch clears what the last one left)
    unsigned* tticket = nullptr;
    unsigned tbase = 0;
    double* tpub[2] = {nullptr, nullptr};
    int64_t tdirty[2] = {0, 0};  // blocks of each that are not cleared
    int tcur = 0;
    // and of the solve with many right-hand sides (kTrsmFlags + 1 words), with an
    // info word for its time-outs
    unsigned* msync = nullptr;
    unsigned mbase = 0;
    int* minfo = nullptr;
    unsigned* fin = nullptr;  // counter of the step-ending kernels' workgroups (zero between launches)
    // pinned host memory: results on their way to the caller (`stage`), inputs on
    // theirs to the device (`up`, filled from upos; a call that needs it from the
    // start again waits for the stream)
    static constexpr int64_t kStage = 1 << 17;
    double* stage = nullptr;
    char* up = nullptr;
    size_t upos = 0;
    BlockPool* blocks = nullptr;  // device blocks of freed models
    unsigned pwait = 1u << 20;
    bool prof = false;
    std::vector<ProfRec> pending;
    std::vector<hipEvent_t> pool;
    std::vector<ProfClass> classes;
    std::map<std::string, int> cls_index;
    std::vector<void*> scratch;
    std::vector<size_t> scratch_sz;
    std::mutex mu;

    // the array that a launch of nblocks blocks publishes in, and the other, of which
    // it clears the first `nreset` blocks
    void next_pub(int64_t nblocks, double** pub, double** reset, int64_t* nreset) {
        *pub = tpub[tcur];
        *reset = tpub[1 - tcur];
        *nreset = tdirty[1 - tcur];
        tdirty[tcur] = nblocks;
        tdirty[1 - tcur] = 0;
        tcur = 1 - tcur;
    }
    hipEvent_t ev() {
        if (!pool.empty()) {
            hipEvent_t e = pool.back();
            pool.pop_back();
            return e;
        }
        hipEvent_t e;
        hipEventCreate(&e);
        return e;
    }
    void resolve() {
        if (pending.empty()) return;
        hipEventSynchronize(pending.back().b);
        for (auto& r : pending) {
            float ms = 0;
            hipEventElapsedTime(&ms, r.a, r.b);
            auto& c = classes[r.cls];
            c.ms += ms;
            c.launches += 1;
            c.flops += r.flops;
            c.bytes += r.bytes;
            pool.push_back(r.a);
            pool.push_back(r.b);
        }
        pending.clear();
    }
    int cls(const char* name) {
        auto it = cls_index.find(name);
        if (it != cls_index.end()) return it->second;
        int id = (int)classes.size();
        classes.push_back(ProfClass{name});
        cls_index[name] = id;
        return id;
    }
    void* buf(int slot, size_t bytes) {
        if ((int)scratch.size() <= slot) {
            scratch.resize(slot + 1, nullptr);
            scratch_sz.resize(slot + 1, 0);
        }
        if (scratch_sz[slot] < bytes) {
            if (scratch[slot]) hipFree(scratch[slot]);
            scratch[slot] = nullptr;
            scratch_sz[slot] = 0;
            if (dev_malloc(&scratch[slot], bytes) != hipSuccess) return nullptr;
            scratch_sz[slot] = bytes;
        }
        return scratch[slot];
    }
};

// Column-major host matrix (rows x cols, leading dimension rows) to a device
// matrix of leading dimension dld, and back.  The host side goes through one
// contiguous copy into a staging buffer (context slot `slot`): a pageable 2D
// copy with short rows is carried out row by row.
inline hipError_t upload_2d(gpl_ctx* c, hipStream_t s, double* dst, int64_t dld, const double* src, int64_t rows,
                            int64_t cols, int slot) {
    double* st = (double*)c->buf(slot, (size_t)rows * cols * 8);
    if (!st) return hipErrorOutOfMemory;
    hipError_t e = hipMemcpyAsync(st, src, (size_t)rows * cols * 8, hipMemcpyHostToDevice, s);
    if (e != hipSuccess) return e;
    return hipMemcpy2DAsync(dst, dld * 8, st, rows * 8, rows * 8, cols, hipMemcpyDeviceToDevice, s);
}

inline hipError_t download_2d(gpl_ctx* c, hipStream_t s, double* dst, const double* src, int64_t sld, int64_t rows,
                              int64_t cols, int slot) {
    double* st = (double*)c->buf(slot, (size_t)rows * cols * 8);
    if (!st) return hipErrorOutOfMemory;
    hipError_t e = hipMemcpy2DAsync(st, rows * 8, src, sld * 8, rows * 8, cols, hipMemcpyDeviceToDevice, s);
    if (e != hipSuccess) return e;
    return hipMemcpyAsync(dst, st, (size_t)rows * cols * 8, hipMemcpyDeviceToHost, s);
}

// Host to device through pinned memory (pageable copies of 64 KB .. 1 MB run at
// 2.5 GB/s: 100 us for 256 KB), in pieces; small and very large ones directly.
// The source may be reused at once.
inline hipError_t upload(gpl_ctx* c, hipStream_t s, void* dst, const void* src, size_t bytes) {
    constexpr size_t kUp = gpl_ctx::kStage * 8;
    if (bytes <= 16384 || bytes > 4 * kUp) return hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, s);
    for (size_t o = 0; o < bytes;) {
        if (c->upos >= kUp) {
            hipError_t e = hipStreamSynchronize(c->stream);
            if (e == hipSuccess && s != c->stream) e = hipStreamSynchronize(s);
            if (e != hipSuccess) return e;
            c->upos = 0;
        }
        const size_t m = std::min({bytes - o, kUp - c->upos, kUp / 4});
        memcpy(c->up + c->upos, (const char*)src + o, m);
        hipError_t e = hipMemcpyAsync((char*)dst + o, c->up + c->upos, m, hipMemcpyHostToDevice, s);
        if (e != hipSuccess) return e;
        c->upos += (m + 255) / 256 * 256;
        o += m;
    }
    return hipSuccess;
}

// Device to host on the context's stream, waiting for it: through the pinned block
// (13 us against 20 for a vector of n = 500, 90 against 410 for one of n = 131072),
// very large ones directly.
inline hipError_t read_back(gpl_ctx* c, void* dst, const void* src, size_t bytes) {
    constexpr size_t kSt = gpl_ctx::kStage * 8;
    if (bytes > 2 * kSt) {
        hipError_t e = hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, c->stream);
        return e == hipSuccess ? hipStreamSynchronize(c->stream) : e;
    }
    for (size_t o = 0; o < bytes; o += kSt) {
        const size_t m = std::min(bytes - o, kSt);
        hipError_t e = hipMemcpyAsync(c->stage, (const char*)src + o, m, hipMemcpyDeviceToHost, c->stream);
        if (e == hipSuccess) e = hipStreamSynchronize(c->stream);
        if (e != hipSuccess) return e;
        memcpy((char*)dst + o, c->stage, m);
    }
    return hipSuccess;
}

// A ROCTX range over one phase of a call (fit, gradient, prediction, batched
// pass, serving job), shown by rocprofv3 --marker-trace beside the kernels.
struct Range {
    explicit Range(const char* name) { roctxRangePushA(name); }
    ~Range() { roctxRangePop(); }
    Range(const Range&) = delete;
    Range& operator=(const Range&) = delete;
};

// Times one launch group on the library stream when profiling is on.
struct Prof {
    gpl_ctx* c;
    ProfRec r;
    bool on;
    hipStream_t st;
    Prof(gpl_ctx* ctx, const char* name, double flops, double bytes, hipStream_t stream = nullptr)
        : c(ctx), on(ctx->prof), st(stream ? stream : ctx->stream) {
        if (!on) return;
        r.cls = c->cls(name);
        r.a = c->ev();
        r.b = c->ev();
        r.flops = flops;
        r.bytes = bytes;
        hipEventRecord(r.a, st);
    }
    ~Prof() {
        if (!on) return;
        hipEventRecord(r.b, st);
        c->pending.push_back(r);
        if (c->pending.size() > 8192) c->resolve();
    }
};

// ---------------------------------------------------------------------------
// model
// ---------------------------------------------------------------------------
struct DevBuf {
    void* p = nullptr;
    size_t sz = 0;
    void free_() {
        if (p) hipFree(p);
        p = nullptr;
        sz = 0;
    }
    bool ensure(size_t bytes, BlockPool* pool = nullptr) {
        if (sz >= bytes && p) return true;
        free_();
        if (bytes == 0) bytes = 8;
        if (pool && (p = pool->take(bytes, &sz))) return true;
        if (dev_malloc(&p, bytes) != hipSuccess) {
            p = nullptr;
            return false;
        }
        sz = bytes;
        return true;
    }
    // The streams that used the block have been waited for.
    void give(BlockPool* pool) {
        if (p) pool->put(p, sz);
        p = nullptr;
        sz = 0;
    }
    template <typename T>
    T* as() const { return reinterpret_cast<T*>(p); }
};

