// C ABI of libdagtm_gpu: context, data movement, and the host-side control
// of one DA-GTM iteration and of the annealing loop.  Kernels live in
// dg_fp64.hip, dg_mixed.hip and dg_mstep.hip.
#include <hip/hip_runtime.h>

#include <cfloat>
#include <cmath>
#include <cstring>
#include <algorithm>
#include <array>
#include <atomic>
#include <chrono>
#include <cstdio>
#include <cstdlib>
#include <functional>
#include <map>
#include <memory>
#include <mutex>
#include <new>
#include <string>
#include <thread>
#include <vector>

#include "dg_internal.h"

#ifndef DG_VERSION_STRING
#define DG_VERSION_STRING "dagtm_gpu gfx950"
#endif

int dg_fail(dg_ctx *ctx, int code, const std::string &msg) {
    if (ctx) ctx->err = msg;
    return code;
}

int dg_hip_check(dg_ctx *ctx, hipError_t e, const char *what) {
    if (ctx) ctx->err = std::string(what) + ": " + hipGetErrorString(e);
    return DG_EHIP;
}

namespace {

template <typename T>
int dalloc(dg_ctx *c, T **p, size_t count) {
    *p = nullptr;
    if (count == 0) count = 1;
    hipError_t e = hipMalloc((void **)p, count * sizeof(T));
    if (e != hipSuccess) {
        *p = nullptr;
        (void)hipGetLastError();
        return dg_fail(c, DG_ENOMEM, std::string("hipMalloc failed: ") + hipGetErrorString(e));
    }
    return DG_OK;
}

template <typename T>
void dfree(T *&p) {
    if (p) (void)hipFree((void *)p);
    p = nullptr;
}

// Runs fn(t) for t = 0 .. nth - 1 on up to nth threads; a thread that cannot
// be started runs its share on the calling thread.  fn must not throw.
template <class F>
void run_threads(unsigned nth, F &&fn) {
    std::vector<std::thread> pool;
    pool.reserve(nth);
    unsigned started = 1;
    try {
        for (; started < nth; ++started) pool.emplace_back(fn, started);
    } catch (...) {
    }
    fn(0u);
    for (unsigned t = started; t < nth; ++t) fn(t);
    for (auto &th : pool) th.join();
}

// A device buffer freed when it goes out of scope (error and exception paths).
struct DevBuf {
    double *p = nullptr;
    ~DevBuf() { dfree(p); }
};

// Device state whose size depends on K: basis, centres, per-centre
// statistics and the partial sums of their reductions.
void free_kstate(dg_ctx *c) {
    dfree(c->FI); dfree(c->Y64); dfree(c->yy); dfree(c->G); dfree(c->Gm); dfree(c->RT);
    dfree(c->partRT); dfree(c->partG); dfree(c->partAB);
}

void free_problem(dg_ctx *c) {
    free_kstate(c);
    dfree(c->T64); dfree(c->tt); dfree(c->W); dfree(c->A); dfree(c->A0); dfree(c->Bm);
    dfree(c->pm); dfree(c->pl); dfree(c->logg); dfree(c->logh);
    dg_mixed_free(c);
    dfree(c->perm);
    dfree(c->p1start);
    c->loaded = false;
    c->have_estep = false;
    c->have_w = false;
}

// Allocates the K-dependent state for c->K (c->N, c->D, c->M1 set); Y64 and
// Gm start at zero.
int alloc_kstate(dg_ctx *c) {
    const long N = c->N, K = c->K;
    const int D = c->D, M1 = c->M1;
    const size_t ld = (size_t)c->ldt;
    // N chunks of E-pass 2: enough (centre tile x chunk) workgroups to fill
    // 256 CUs several times, each chunk at least one 64-point tile.
    const long tiles = (N + 63) / 64;
    const long ktiles = (K + 63) / 64;
    long nc = (1024 + ktiles - 1) / ktiles;
    if (nc > tiles) nc = tiles;
    if (nc < 1) nc = 1;
    c->NC = (int)nc;
    // A/B reduction: at most 64 chunks of centres, at least 64 centres each
    long nch = (K + 63) / 64;
    if (nch > 64) nch = 64;
    c->nchAB = (int)(nch < 1 ? 1 : nch);
    c->partRT_len = std::max({(size_t)c->NC * K * D, dg_pass1_part(N),
                              dg_map_part(N, c->K) + (size_t)3 * (K + N)});
    int rc;
    if ((rc = dalloc(c, &c->FI, (size_t)K * M1)) || (rc = dalloc(c, &c->Y64, (size_t)K * ld)) ||
        (rc = dalloc(c, &c->yy, K)) || (rc = dalloc(c, &c->G, K)) || (rc = dalloc(c, &c->Gm, K)) ||
        (rc = dalloc(c, &c->RT, (size_t)K * D)) ||
        (rc = dalloc(c, &c->partRT, c->partRT_len)) ||
        (rc = dalloc(c, &c->partG, (size_t)c->NC * K + (size_t)3 * dg_pass1_wgs(N))) ||
        (rc = dalloc(c, &c->partAB, std::max((size_t)c->nchAB * ((size_t)M1 * M1 + (size_t)M1 * D),
                                             (size_t)2 * bk_cdiv(K, kBCentres)))))
        return rc;
    c->partLog64 = c->partG + (size_t)c->NC * K;
    DG_HIP(c, hipMemsetAsync(c->Y64, 0, (size_t)K * ld * sizeof(double), c->stream));
    DG_HIP(c, hipMemsetAsync(c->Gm, 0, (size_t)K * sizeof(double), c->stream));
    return DG_OK;
}

// Rows cross between host and device as one block each way: a strided copy
// of pageable host memory goes row by row, at 6 to 9 microseconds a row (10^6
// rows of 166 doubles up: 9.4 s, as one block 0.2 s; 8000 rows of 166 down:
// 53 ms, as one block 1 ms).

// Host rows (stride lds) -> device rows (stride ldd >= cols, zero padding).  The
// host block -- (rows - 1) lds + cols doubles, nothing past the last row's data
// -- is repacked on the device; `scratch` (room doubles) is used for it where it
// is large enough.
int upload_rows(dg_ctx *c, double *dst, int ldd, const double *src, long lds, long rows,
                int cols, double *scratch = nullptr, size_t room = 0) {
    const size_t n = (size_t)(rows - 1) * lds + cols;
    if (lds == cols && ldd == cols) {
        DG_HIP(c, hipMemcpyAsync(dst, src, n * sizeof(double), hipMemcpyHostToDevice, c->stream));
        return DG_OK;
    }
    DevBuf tmp;
    int rc;
    if (room < n) {
        if ((rc = dalloc(c, &tmp.p, n))) return rc;
        scratch = tmp.p;
    }
    DG_HIP(c, hipMemcpyAsync(scratch, src, n * sizeof(double), hipMemcpyHostToDevice, c->stream));
    if ((rc = dg_pad_rows(c, scratch, rows, cols, lds, ldd, dst))) return rc;
    // a block of its own is freed on return: wait for the repack that reads it
    if (tmp.p) DG_HIP(c, hipStreamSynchronize(c->stream));
    return DG_OK;
}

// Dense device rows -> host rows (stride ldd >= cols); what lies between the
// host's rows is not touched.  Returns when the rows are there.
int download_rows(dg_ctx *c, double *dst, long ldd, const double *src, long rows, long cols) {
    const size_t row = (size_t)cols * sizeof(double);
    if (ldd == cols) {
        DG_HIP(c, hipMemcpyAsync(dst, src, (size_t)rows * row, hipMemcpyDeviceToHost, c->stream));
        DG_HIP(c, hipStreamSynchronize(c->stream));
        return DG_OK;
    }
    // padded host rows: through a host block of at most 32 MB (or one row)
    const long step = std::max(1L, std::min(rows, (long)((32u << 20) / row)));
    double *block = static_cast<double *>(std::malloc((size_t)step * row));
    if (!block) return dg_fail(c, DG_ENOMEM, "host allocation");
    hipError_t e = hipSuccess;
    for (long r0 = 0; r0 < rows && e == hipSuccess; r0 += step) {
        const long n = std::min(step, rows - r0);
        e = hipMemcpyAsync(block, src + r0 * cols, (size_t)n * row, hipMemcpyDeviceToHost, c->stream);
        if (e == hipSuccess) e = hipStreamSynchronize(c->stream);
        for (long r = 0; r < n && e == hipSuccess; ++r)
            std::memcpy(dst + (r0 + r) * ldd, block + r * cols, row);
    }
    std::free(block);
    return e == hipSuccess ? DG_OK : dg_hip_check(c, e, "copy to the host");
}

// the step's kernels leave their scalars in h_scal themselves
int sync_step(dg_ctx *c) {
    DG_HIP(c, hipStreamSynchronize(c->stream));
    return DG_OK;
}

int sync_scalars(dg_ctx *c) {
    DG_HIP(c, hipMemcpyAsync(c->h_scal, c->scal, kScalCount * sizeof(double),
                             hipMemcpyDeviceToHost, c->stream));
    DG_HIP(c, hipStreamSynchronize(c->stream));
    return DG_OK;
}

int select_device(dg_ctx *c) {
    DG_HIP(c, hipSetDevice(c->device));
    return DG_OK;
}

// Quality of mpicomm.c:463-500: [N((D/2) log(beta/2pi) - log K) + w * sum] / N
double quality(long N, int K, int D, double beta, double sum, double w) {
    double q = N * ((D / 2.0) * log(beta / (2.0 * M_PI)) - log((double)K));
    q += w * sum;
    return q / (double)N;
}

// ---- tuned pass-2 chunk counts ------------------------------------------
// A text table, one line per shape: "<precision> <D> <K> <nbits(N)> <NC>"
// (the last line for a shape wins), named by the DG_TUNE_FILE environment
// variable and written by dg_tune.  Shared by every context of the process.
std::mutex g_tune_mu;
std::string g_tune_path;
std::map<std::array<long, 4>, int> g_tune;

std::array<long, 4> tune_key(const dg_ctx *c) {
    long nb = 0;
    while (nb < 62 && (1L << nb) < c->N) ++nb;
    return {(long)c->cfg.precision, (long)c->D, (long)c->K, nb};
}

// caller holds g_tune_mu
void tune_load(const std::string &path) {
    if (path == g_tune_path) return;
    g_tune.clear();
    g_tune_path = path;
    FILE *f = std::fopen(path.c_str(), "r");
    if (!f) return;
    long p, d, k, nb, nc;
    while (std::fscanf(f, "%ld %ld %ld %ld %ld", &p, &d, &k, &nb, &nc) == 5)
        g_tune[{p, d, k, nb}] = (int)nc;
    std::fclose(f);
}

int tune_find(const dg_ctx *c) {
    const char *path = std::getenv("DG_TUNE_FILE");
    if (!path || !*path) return 0;
    std::lock_guard<std::mutex> lk(g_tune_mu);
    tune_load(path);
    auto it = g_tune.find(tune_key(c));
    return it == g_tune.end() ? 0 : it->second;
}

// ---- dg_map_noalloc's scratch ---------------------------------------------
// A file-scope device array: every GPU the library runs on holds its own copy
// (16 MiB) until the process ends.  Its device address is looked up once per
// device (hipGetSymbolAddress with that device current) and kept; host code
// uses only that address, never the array's name.
constexpr size_t kMapScratchDoubles = (size_t)1 << 21;
__device__ __align__(256) double scratch[kMapScratchDoubles];

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
double *g_scratch_ptr[kMaxDevices] = {};
bool g_scratch_done[kMaxDevices] = {};

// The calling thread has `device` current.  Returns this device's scratch
// address, or nullptr when the lookup failed (reported by dg_map_noalloc).
double *scratch_for_device(int device) {
    if (device < 0 || device >= kMaxDevices) return nullptr;
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if (!g_scratch_done[device]) {
        void *ptr = nullptr;
        if (hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)) == hipSuccess) {
            g_scratch_ptr[device] = static_cast<double *>(ptr);
        } else {
            (void)hipGetLastError();
            g_scratch_ptr[device] = nullptr;
        }
        g_scratch_done[device] = true;
    }
    return g_scratch_ptr[device];
}

}  // namespace

extern "C" {

const char *dg_version(void) { return DG_VERSION_STRING; }

const char *dg_last_error(const dg_ctx *ctx) {
    if (!ctx) return "null context";
    return ctx->err.c_str();
}

int dg_create(const dg_config *cfg, dg_ctx **out) {
    if (!out) return DG_EINVAL;
    *out = nullptr;
    dg_config def{0, DG_FP64, 0.0};
    const dg_config &cf = cfg ? *cfg : def;
    if (cf.precision != DG_FP64 && cf.precision != DG_MIXED && cf.precision != DG_MIXED_R1)
        return DG_EINVAL;
    if (cf.lambda < 0.0) return DG_EINVAL;
    dg_ctx *c = new (std::nothrow) dg_ctx();
    if (!c) return DG_ENOMEM;
    c->cfg = cf;
    c->device = cf.device;
    int ndev = 0;
    hipError_t e = hipGetDeviceCount(&ndev);
    if (e != hipSuccess || ndev <= 0 || cf.device < 0 || cf.device >= ndev) {
        delete c;
        (void)hipGetLastError();
        return DG_EHIP;
    }
    int rc = DG_OK;
    if ((rc = select_device(c)) != DG_OK) { delete c; return rc; }
    if (hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking) != hipSuccess) {
        delete c;
        return DG_EHIP;
    }
    for (auto &ev : c->ev)
        if (hipEventCreate(&ev) != hipSuccess) { dg_destroy(c); return DG_EHIP; }
    if (dalloc(c, &c->scal, kScalCount) != DG_OK ||
        hipHostMalloc((void **)&c->h_scal, kScalCount * sizeof(double), hipHostMallocDefault) !=
            hipSuccess ||
        hipHostGetDevicePointer((void **)&c->m_scal, c->h_scal, 0) != hipSuccess) {
        dg_destroy(c);
        return DG_ENOMEM;
    }
    std::memset(c->h_scal, 0, kScalCount * sizeof(double));
    c->map_scratch = scratch_for_device(c->device);
    *out = c;
    return DG_OK;
}

int dg_destroy(dg_ctx *c) {
    if (!c) return DG_OK;
    (void)hipSetDevice(c->device);
    if (c->stream) (void)hipStreamSynchronize(c->stream);
    free_problem(c);
    dfree(c->scal);
    if (c->h_scal) (void)hipHostFree(c->h_scal);
    for (auto &ev : c->ev)
        if (ev) (void)hipEventDestroy(ev);
    if (c->stream) (void)hipStreamDestroy(c->stream);
    delete c;
    return DG_OK;
}

int dg_upload(dg_ctx *c, const double *T, long N, int D, long ldT, const double *FI, int K,
              int M1, long ldFI, const double *Y, long ldY, double beta) {
    if (!c) return DG_EINVAL;
    if (!T || !FI || !Y || N < 1 || D < 1 || K < 1 || M1 < 1 || ldT < D || ldFI < M1 || ldY < D ||
        !(beta > 0.0))
        return dg_fail(c, DG_EINVAL, "dg_upload: bad shape, stride or beta");
    if (D > 192) return dg_fail(c, DG_EINVAL, "dg_upload: D > 192 is not supported");
    if (M1 > 2048) return dg_fail(c, DG_EINVAL, "dg_upload: M+1 > 2048 is not supported");
    int rc;
    if ((rc = select_device(c)) != DG_OK) return rc;
    free_problem(c);
    c->N = N; c->D = D; c->K = K; c->M1 = M1; c->beta = beta;
    c->ldt = ((D + 15) / 16) * 16;
    const size_t ld = (size_t)c->ldt;
    if ((rc = dalloc(c, &c->T64, (size_t)N * ld)) || (rc = dalloc(c, &c->tt, N)) ||
        (rc = dalloc(c, &c->W, (size_t)M1 * D)) || (rc = dalloc(c, &c->A, (size_t)M1 * M1)) ||
        (rc = dalloc(c, &c->A0, (size_t)M1 * M1)) || (rc = dalloc(c, &c->Bm, (size_t)M1 * D)) ||
        (rc = dalloc(c, &c->pm, N)) || (rc = dalloc(c, &c->pl, N)) ||
        (rc = dalloc(c, &c->logg, N)) || (rc = dalloc(c, &c->logh, N)) ||
        (rc = alloc_kstate(c))) {
        free_problem(c);
        return rc;
    }
    if ((rc = upload_rows(c, c->T64, (int)ld, T, ldT, N, D)) ||
        (rc = upload_rows(c, c->FI, M1, FI, ldFI, K, M1, c->partRT, c->partRT_len)) ||
        (rc = upload_rows(c, c->Y64, (int)ld, Y, ldY, K, D, c->partRT, c->partRT_len))) {
        free_problem(c);
        return rc;
    }
    if ((rc = dg_rownorms(c, c->T64, N, c->ldt, D, c->tt))) return rc;
    if ((rc = dg_rownorms(c, c->Y64, K, c->ldt, D, c->yy))) return rc;
    // sum_n |t_n|^2 for the closed-form beta update
    if ((rc = dg_sum_into(c, c->tt, N, kScalBetaSum)) || (rc = sync_scalars(c))) return rc;
    c->sum_tt = c->h_scal[kScalBetaSum];
    c->loaded = true;
    if (c->mixed()) {
        c->nc_override = tune_find(c);
        if ((rc = dg_mixed_prepare_t(c)) || (rc = dg_mixed_prepare_y(c)) ||
            (rc = dg_mixed_order(c)))
            return rc;
    }
    DG_HIP(c, hipStreamSynchronize(c->stream));
    return DG_OK;
}

int dg_set_state(dg_ctx *c, const double *Y, long ldY, double beta) {
    if (!c) return DG_EINVAL;
    if (!c->loaded) return dg_fail(c, DG_ESTATE, "dg_set_state before dg_upload");
    if (!Y || ldY < c->D || !(beta > 0.0)) return dg_fail(c, DG_EINVAL, "dg_set_state: bad args");
    int rc;
    if ((rc = select_device(c))) return rc;
    if ((rc = upload_rows(c, c->Y64, c->ldt, Y, ldY, c->K, c->D, c->partRT, c->partRT_len))) return rc;
    if ((rc = dg_rownorms(c, c->Y64, c->K, c->ldt, c->D, c->yy))) return rc;
    DG_HIP(c, hipMemsetAsync(c->Gm, 0, (size_t)c->K * sizeof(double), c->stream));
    c->beta = beta;
    c->have_w = false;
    c->have_estep = false;
    if (c->mixed() && (rc = dg_mixed_prepare_y(c))) return rc;
    DG_HIP(c, hipStreamSynchronize(c->stream));
    return DG_OK;
}

int dg_estep(dg_ctx *c, int isDA, double temp, dg_estep_out *out) {
    if (!c) return DG_EINVAL;
    if (!c->loaded) return dg_fail(c, DG_ESTATE, "dg_estep before dg_upload");
    if (isDA && !(temp > 0.0)) return dg_fail(c, DG_EINVAL, "dg_estep: temp must be > 0");
    int rc;
    if ((rc = select_device(c))) return rc;
    c->fp64_due = c->fp64_norm = false;
    if (c->mixed()) rc = dg_estep_mixed(c, isDA, temp);
    else rc = dg_estep_fp64(c, isDA, temp);
    if (rc) return rc;
    if (c->timing) DG_HIP(c, hipEventRecord(c->ev[3], c->stream));
    if ((rc = sync_step(c))) return rc;
    if (c->timing) {
        float a = 0, b = 0, d = 0;
        (void)hipEventElapsedTime(&a, c->ev[0], c->ev[1]);
        (void)hipEventElapsedTime(&b, c->ev[1], c->ev[2]);
        (void)hipEventElapsedTime(&d, c->ev[2], c->ev[3]);
        c->t_ms[0] = a; c->t_ms[1] = b; c->t_ms[2] = d;
    }
    c->have_estep = true;
    c->last_isDA = isDA != 0;
    c->last_temp = isDA ? temp : 1.0;
    const double sg = c->h_scal[kScalSumLogG], sh = c->h_scal[kScalSumLogH];
    if (out) {
        out->llh = quality(c->N, c->K, c->D, c->beta, sg, 1.0);
        out->nfree = isDA ? quality(c->N, c->K, c->D, c->beta, sh, temp) : -out->llh;
        out->nzero = (long)c->h_scal[kScalNZero];
    }
    return DG_OK;
}

// The FP64 outputs of a mixed context (dg_map, dg_next_ctemp, dg_resp_dense)
// leave G and R T in FP64 for what reads them next, as the rest of their state:
// computed here, when something does, from the normalisers where one of them made
// those.
static int due_stats(dg_ctx *c) {
    if (!c->fp64_due) return DG_OK;
    const int rc = c->fp64_norm ? dg_stats_fp64(c, c->last_isDA, c->last_temp)
                                : dg_estep_fp64(c, c->last_isDA, c->last_temp);
    if (rc) return rc;
    c->fp64_due = false;
    c->fp64_norm = c->mixed();
    return DG_OK;
}

// the FP64 normalisers of a mixed context's E-step
static int fp64_normalisers(dg_ctx *c) {
    const int rc = dg_pass1_fp64(c, c->last_isDA, c->last_temp);
    c->fp64_norm = rc == DG_OK;
    return rc;
}

int dg_mstep(dg_ctx *c, double *beta_out) {
    if (!c) return DG_EINVAL;
    if (!c->loaded || !c->have_estep) return dg_fail(c, DG_ESTATE, "dg_mstep needs a dg_estep first");
    int rc;
    if ((rc = select_device(c)) || (rc = due_stats(c))) return rc;
    if (c->timing) DG_HIP(c, hipEventRecord(c->ev[4], c->stream));
    if ((rc = dg_mstep_run(c, 0.0))) return rc;
    if (c->timing) DG_HIP(c, hipEventRecord(c->ev[5], c->stream));
    if ((rc = sync_step(c))) return rc;
    if (c->h_scal[kScalSolveOK] != 1.0 && c->M1 > 126) {
        // a non-positive pivot: retry with a jitter of 1e-13 tr(A) / n, growing
        // x10 per retry, at most 8 retries (the policy of the one-kernel
        // factorisation that M + 1 <= 126 uses)
        if ((rc = dg_mstep_trace(c)) || (rc = sync_scalars(c))) return rc;
        double jit = 1e-13 * c->h_scal[kScalJitter] / c->M1;
        for (int attempt = 1; attempt <= 8; ++attempt, jit *= 10.0) {
            if ((rc = dg_mstep_run(c, jit)) || (rc = sync_step(c))) return rc;
            if (c->h_scal[kScalSolveOK] == 1.0) break;
        }
    }
    if (c->timing) {
        float a = 0;
        (void)hipEventElapsedTime(&a, c->ev[4], c->ev[5]);
        c->t_ms[3] = a;
    }
    c->have_estep = false;
    if (c->h_scal[kScalSolveOK] != 1.0)
        return dg_fail(c, DG_ESOLVE, "M-step Cholesky failed after jitter retries");
    c->have_w = true;
    const double s = c->sum_tt + c->h_scal[kScalBetaSum];
    c->beta = ((double)c->N * c->D) / s;
    if (c->mixed() && (rc = dg_mixed_prepare_y(c, true))) return rc;
    if (beta_out) *beta_out = c->beta;
    return DG_OK;
}

namespace {
// dg_anneal's steps for dg_anneal_ctl: the context's own E-step, M-step and
// critical temperatures, and the progress callback with the current beta.
struct AnnealSteps {
    dg_ctx *c;
    dg_iter_cb cb;
    void *user;
};
int st_estep(void *u, int isDA, double temp, double *llh, double *nfree) {
    dg_estep_out eo;
    const int rc = dg_estep(static_cast<AnnealSteps *>(u)->c, isDA, temp, &eo);
    *llh = eo.llh; *nfree = eo.nfree;
    return rc;
}
int st_mstep(void *u) { return dg_mstep(static_cast<AnnealSteps *>(u)->c, nullptr); }
int st_ctemp(void *u, double temp, double eps, double *ct) {
    return dg_next_ctemp(static_cast<AnnealSteps *>(u)->c, temp, eps, nullptr, ct, nullptr);
}
int st_iter(void *u, int nloop, int lloop, double temp, double nfree, double llh, double diff) {
    const AnnealSteps *a = static_cast<AnnealSteps *>(u);
    if (a->cb) a->cb(a->user, nloop, lloop, temp, nfree, llh, diff, a->c->beta);
    return DG_OK;
}
}  // namespace

int dg_anneal(dg_ctx *c, const dg_anneal_params *p, dg_anneal_result *res, dg_iter_cb cb,
              void *user) {
    if (!c || !p || !res) return DG_EINVAL;
    if (!c->loaded) return dg_fail(c, DG_ESTATE, "dg_anneal before dg_upload");
    if (p->schedule != DG_SCHED_EXP && p->schedule != DG_SCHED_LINEAR &&
        p->schedule != DG_SCHED_AUTO)
        return dg_fail(c, DG_EINVAL, "dg_anneal: unknown schedule");
    AnnealSteps steps{c, cb, user};
    const dg_anneal_ops ops{st_estep, st_mstep, st_ctemp, st_iter, nullptr};
    const int rc = dg_anneal_ctl(p, nullptr, &ops, &steps, res);
    res->beta = c->beta;
    return rc;
}

int dg_tune(dg_ctx *c, const char *table_path, int *nc_out) {
    if (!c) return DG_EINVAL;
    if (!c->loaded) return dg_fail(c, DG_ESTATE, "dg_tune before dg_upload");
    if (nc_out) *nc_out = 0;
    if (!c->mixed()) return DG_OK;             // the FP64 path has no tuned choice
    int rc;
    if ((rc = select_device(c))) return rc;
    long lo = 0, hi = 0;
    const long heur = dg_mixed_nc_limits(c, &lo, &hi);
    std::vector<long> cand;
    for (long v : {heur, heur / 2, heur / 4, heur / 8, heur / 16, lo, 2 * heur}) {
        v = std::max(lo, std::min(hi, (v + 7) / 8 * 8));
        if (std::find(cand.begin(), cand.end(), v) == cand.end()) cand.push_back(v);
    }
    // time three DA E-steps at temperature 2 (three exponentials per
    // element) per candidate, after one untimed step
    using clk = std::chrono::steady_clock;
    long best = heur;
    double best_ms = HUGE_VAL;
    for (long nc : cand) {
        c->nc_override = (int)nc;
        if ((rc = dg_mixed_prepare_t(c)) || (rc = dg_mixed_prepare_y(c))) return rc;
        if ((rc = dg_estep(c, 1, 2.0, nullptr))) return rc;
        double ms = HUGE_VAL;
        for (int r = 0; r < 3; ++r) {
            const auto t0 = clk::now();
            if ((rc = dg_estep(c, 1, 2.0, nullptr))) return rc;
            ms = std::min(ms, std::chrono::duration<double, std::milli>(clk::now() - t0).count());
        }
        if (ms < best_ms) { best_ms = ms; best = nc; }
    }
    c->nc_override = (int)best;
    if ((rc = dg_mixed_prepare_t(c)) || (rc = dg_mixed_prepare_y(c))) return rc;
    c->have_estep = false;
    if (nc_out) *nc_out = (int)best;
    if (table_path && *table_path) {
        std::lock_guard<std::mutex> lk(g_tune_mu);
        FILE *f = std::fopen(table_path, "a");
        if (!f) return dg_fail(c, DG_EINVAL, std::string("dg_tune: cannot write ") + table_path);
        const auto k = tune_key(c);
        std::fprintf(f, "%ld %ld %ld %ld %ld\n", k[0], k[1], k[2], k[3], best);
        std::fclose(f);
        if (g_tune_path == table_path) g_tune[k] = (int)best;
    }
    return DG_OK;
}

int dg_set_basis(dg_ctx *c, const double *FI, int K, int M1, long ldFI, const double *W, long ldW) {
    if (!c) return DG_EINVAL;
    if (!c->loaded) return dg_fail(c, DG_ESTATE, "dg_set_basis before dg_upload");
    if (!FI || K < 1 || M1 != c->M1 || ldFI < M1 || (W && ldW < c->D))
        return dg_fail(c, DG_EINVAL, "dg_set_basis: bad shape or stride (M+1 must not change)");
    if (!W && !c->have_w)
        return dg_fail(c, DG_ESTATE, "dg_set_basis: no M-step since the last upload; pass W");
    int rc;
    if ((rc = select_device(c))) return rc;
    DG_HIP(c, hipStreamSynchronize(c->stream));
    free_kstate(c);
    c->K = K;
    c->have_estep = false;
    if ((rc = alloc_kstate(c))) { free_problem(c); return rc; }
    if ((rc = upload_rows(c, c->FI, M1, FI, ldFI, K, M1))) return rc;
    if (W && (rc = upload_rows(c, c->W, c->D, W, ldW, M1, c->D))) return rc;
    c->have_w = true;
    if ((rc = dg_centres_from_w(c))) return rc;
    // the mixed path's operand layout and chunking depend on K: rebuild it
    // from the resident FP64 data
    if (c->mixed()) c->nc_override = tune_find(c);
    if (c->mixed() &&
        ((rc = dg_mixed_prepare_t(c)) || (rc = dg_mixed_prepare_y(c))))
        return rc;
    DG_HIP(c, hipStreamSynchronize(c->stream));
    return DG_OK;
}

static int next_ctemp_impl(dg_ctx *c, double temp, double eps, const double *gg,
                           double *ctemp_max, double *ctemp_k);

int dg_next_ctemp(dg_ctx *c, double temp, double eps, const double *gg, double *ctemp_max,
                  double *ctemp_k) {
    if (!c) return DG_EINVAL;
    try {
        return next_ctemp_impl(c, temp, eps, gg, ctemp_max, ctemp_k);
    } catch (...) {
        return dg_fail(c, DG_ENOMEM, "dg_next_ctemp: host allocation failed");
    }
}

static int next_ctemp_impl(dg_ctx *c, double temp, double eps, const double *gg,
                           double *ctemp_max, double *ctemp_k) {
    if (!c->loaded || !c->have_estep)
        return dg_fail(c, DG_ESTATE, "dg_next_ctemp needs a dg_estep at the current state");
    if (!ctemp_max || !std::isfinite(temp) || !std::isfinite(eps))
        return dg_fail(c, DG_EINVAL, "dg_next_ctemp: bad args");
    int rc;
    if ((rc = select_device(c))) return rc;
    // R in FP64: the mixed path refreshes the FP64 per-point normalisers
    c->fp64_due = c->mixed();
    if (c->mixed() && (rc = fp64_normalisers(c))) return rc;
    const int K = c->K;
    std::vector<double> g(K), ck(K);
    if (gg) {
        std::copy(gg, gg + K, g.begin());
    } else {
        DG_HIP(c, hipMemcpyAsync(g.data(), c->Gm, (size_t)K * sizeof(double),
                                 hipMemcpyDeviceToHost, c->stream));
        DG_HIP(c, hipStreamSynchronize(c->stream));
    }
    // per centre: eig(H) of mpicomm.c:599-626 with H = [[2S1 - S2, -S2], [-S2, 2S1 - S2]]
    // is eig(2 S1) together with eig(2 S1 - 2 S2) (H is block-symmetric).  The
    // kernel scales each matrix by its size (mpicomm.c:617-628 does below a weight
    // of 1e-250).
    const DgCtempPlan p = dg_ctemp_plan(c);
    std::vector<double> lim((size_t)2 * K), val((size_t)2 * K);
    for (int k0 = 0; k0 < K; k0 += p.KB) {
        const int kb = std::min(p.KB, K - k0);
        for (int i = 0; i < kb; ++i) {
            lim[(size_t)2 * k0 + i] = (temp - eps) * g[k0 + i] * 2.0 / c->beta;
            lim[(size_t)2 * k0 + kb + i] = g[k0 + i] == 0.0 ? 0.0 : 1.0;
        }
    }
    DevBuf buf;
    if ((rc = dalloc(c, &buf.p, p.buf_len() + (size_t)4 * K))) return rc;
    double *dLim = buf.p + p.buf_len(), *dVal = dLim + (size_t)2 * K;
    DG_HIP(c, hipMemcpyAsync(dLim, lim.data(), (size_t)2 * K * sizeof(double), hipMemcpyHostToDevice,
                             c->stream));
    for (int k0 = 0; k0 < K; k0 += p.KB)
        if ((rc = dg_ctemp_fp64(c, k0, std::min(p.KB, K - k0), p, dLim, buf.p, dVal))) return rc;
    DG_HIP(c, hipMemcpyAsync(val.data(), dVal, (size_t)2 * K * sizeof(double), hipMemcpyDeviceToHost,
                             c->stream));
    DG_HIP(c, hipStreamSynchronize(c->stream));
    for (int k = 0; k < K; ++k) {
        const double a = val[(size_t)2 * k], b = val[(size_t)2 * k + 1];
        if (g[k] != 0.0 && (std::isnan(a) || std::isnan(b)))
            return dg_fail(c, DG_ESOLVE, "dg_next_ctemp: no eigenvalues (data not finite)");
        ck[k] = g[k] == 0.0 ? HUGE_VAL : c->beta / 2.0 / g[k] * std::max(a, b);
    }
    double cmax = -HUGE_VAL;
    for (int k = 0; k < K; ++k) cmax = std::max(cmax, ck[k]);
    *ctemp_max = cmax;
    if (ctemp_k) std::copy(ck.begin(), ck.end(), ctemp_k);
    return DG_OK;
}

constexpr int kMaxBatchWorkers = 4;

static int batch_anneal_impl(const dg_config *cfg, int workers, const dg_batch_item *items,
                             int n, dg_anneal_result *res, int *status, double *phase_ms);

int dg_batch_anneal(const dg_config *cfg, int workers, const dg_batch_item *items, int n,
                    dg_anneal_result *res, int *status, double *phase_ms) {
    try {
        return batch_anneal_impl(cfg, workers, items, n, res, status, phase_ms);
    } catch (...) {
        return DG_ENOMEM;
    }
}

static int batch_anneal_impl(const dg_config *cfg, int workers, const dg_batch_item *items,
                             int n, dg_anneal_result *res, int *status, double *phase_ms) {
    if (!cfg || n < 0 || (n > 0 && (!items || !res || !status))) return DG_EINVAL;
    if (phase_ms) phase_ms[0] = phase_ms[1] = 0.0;
    if (n == 0) return DG_OK;
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || cfg->device < 0 || cfg->device >= ndev) {
        (void)hipGetLastError();
        return DG_EHIP;
    }
    // workers 0 / -1: the batched launch sequence (with / without hipGraph
    // capture) on this thread, for the mixed precisions; otherwise host
    // workers, at most kMaxBatchWorkers: one per hardware queue of the
    // process (HIP's default of four)
    const bool batched = workers <= 0 && cfg->precision != DG_FP64;
    const bool graphs = workers == 0;
    if (batched || workers <= 0 || workers > kMaxBatchWorkers) workers = kMaxBatchWorkers;
    workers = batched ? 1 : std::min(workers, n);
    // largest work first, so the tail of the queue holds the short items
    std::vector<int> order(n);
    for (int i = 0; i < n; ++i) order[i] = i;
    std::stable_sort(order.begin(), order.end(), [&](int a, int b) {
        return (double)items[a].K * items[a].N * items[a].D >
               (double)items[b].K * items[b].N * items[b].D;
    });
    for (int i = 0; i < n; ++i) { status[i] = DG_EHIP; std::memset(&res[i], 0, sizeof(res[i])); }
    std::vector<dg_ctx *> ctx(n, nullptr);
    auto run_pool = [&](const std::function<void(int)> &job) {
        std::atomic<int> next{0};
        run_threads((unsigned)workers, [&](unsigned) noexcept {
            for (int j; (j = next.fetch_add(1)) < n;) {
                try {
                    job(order[j]);
                } catch (...) {
                    status[order[j]] = DG_ENOMEM;
                }
            }
        });
    };
    using clk = std::chrono::steady_clock;
    // phase 1: one context per instance, data resident on the device, on the
    // calling thread: every device allocation and free of the batch happens
    // here or after phase 2, never while workers launch
    const auto t0 = clk::now();
    for (int j = 0; j < n; ++j) {
        const int i = order[j];
        const dg_batch_item &it = items[i];
        try {
            int rc = dg_create(cfg, &ctx[i]);
            if (!rc) rc = dg_upload(ctx[i], it.T, it.N, it.D, it.ldT, it.FI, it.K, it.M1, it.ldFI,
                                    it.Y0, it.ldY0, it.beta0);
            status[i] = rc;
        } catch (...) {
            status[i] = DG_ENOMEM;
        }
    }
    // phase 2: the annealing runs, concurrently on the workers' host threads,
    // or all instances' steps as batched launches
    const auto t1 = clk::now();
    int brc = DG_OK;
    if (batched) {
        std::vector<int> ok;
        for (int i = 0; i < n; ++i)
            if (status[i] == DG_OK) ok.push_back(i);
        std::vector<dg_ctx *> cs;
        std::vector<dg_anneal_params> ps;
        std::vector<dg_anneal_result> rs(ok.size());
        std::vector<int> st(ok.size(), DG_OK);
        for (int i : ok) { cs.push_back(ctx[i]); ps.push_back(items[i].params); }
        if (!ok.empty() && (brc = select_device(ctx[ok[0]])) == DG_OK)
            brc = dg_batch_run_mixed(cs, ps.data(), rs.data(), st.data(), graphs);
        for (size_t j = 0; j < ok.size(); ++j) {
            res[ok[j]] = rs[j];
            status[ok[j]] = brc ? brc : st[j];
        }
    } else {
        run_pool([&](int i) {
            if (status[i] != DG_OK) return;
            status[i] = dg_anneal(ctx[i], &items[i].params, &res[i], nullptr, nullptr);
        });
    }
    const auto t2 = clk::now();
    for (int i = 0; i < n; ++i) {
        const dg_batch_item &it = items[i];
        if (status[i] == DG_OK && (it.W || it.Y))
            status[i] = dg_download(ctx[i], it.W, it.ldW, it.Y, it.ldY, nullptr);
        if (ctx[i]) dg_destroy(ctx[i]);
    }
    if (phase_ms) {
        phase_ms[0] = std::chrono::duration<double, std::milli>(t1 - t0).count();
        phase_ms[1] = std::chrono::duration<double, std::milli>(t2 - t1).count();
    }
    return brc == DG_EHIP ? DG_EHIP : DG_OK;
}

int dg_map(dg_ctx *c, const double *X, int L, long ldX, double *M, long ldM) {
    if (!c) return DG_EINVAL;
    if (!c->loaded) return dg_fail(c, DG_ESTATE, "dg_map before dg_upload");
    if (!X || !M || L < 1 || L > 3 || ldX < L || ldM < L) return dg_fail(c, DG_EINVAL, "dg_map: bad args");
    int rc;
    if ((rc = select_device(c))) return rc;
    if (!c->have_estep) {
        dg_estep_out eo;
        if ((rc = dg_estep(c, c->last_isDA, c->last_temp, &eo))) return rc;
    }
    c->fp64_due = c->mixed();
    // a centre's coordinates may be a few doubles of a much longer row
    std::unique_ptr<double[]> packed;
    if (ldX != L) {
        packed.reset(new (std::nothrow) double[(size_t)c->K * L]);
        if (!packed) return dg_fail(c, DG_ENOMEM, "host allocation");
        for (int k = 0; k < c->K; ++k)
            std::memcpy(&packed[(size_t)k * L], X + (size_t)k * ldX, (size_t)L * sizeof(double));
        X = packed.get();
    }
    // the coordinates and the projection behind the projection's sums
    double *dX = c->partRT + dg_map_part(c->N, c->K), *dM = dX + (size_t)c->K * L;
    if ((rc = upload_rows(c, dX, L, X, L, c->K, L)) || (rc = dg_map_fp64(c, dX, L, dM))) return rc;
    return download_rows(c, M, ldM, dM, c->N, L);
}

int dg_map_noalloc(dg_ctx *c, const double *X, int L, long ldX, double *M, long ldM) {
    if (!c) return DG_EINVAL;
    if (!c->loaded) return dg_fail(c, DG_ESTATE, "dg_map_noalloc before dg_upload");
    if (!X || !M || L < 1 || L > 3 || ldX < L || ldM < L)
        return dg_fail(c, DG_EINVAL, "dg_map_noalloc: bad args");
    if (((size_t)c->K + (size_t)c->N) * (size_t)L > kMapScratchDoubles)
        return dg_fail(c, DG_EINVAL,
                       "dg_map_noalloc: (K + N) * L exceeds the scratch maximum of 2^21 "
                       "doubles (use dg_map)");
    if (!c->map_scratch)
        return dg_fail(c, DG_EHIP, "dg_map_noalloc: no scratch address for this device");
    int rc;
    if ((rc = select_device(c))) return rc;
    // the steps below launch kernels on buffers the context already owns
    if (!c->have_estep) {
        dg_estep_out eo;
        if ((rc = dg_estep(c, c->last_isDA, c->last_temp, &eo))) return rc;
    }
    c->fp64_due = c->mixed();
    double *dX = c->map_scratch;                       // K x L
    double *dM = c->map_scratch + (size_t)c->K * L;    // N x L
    const size_t row = (size_t)L * sizeof(double);
    if (ldX == L)
        DG_HIP(c, hipMemcpyAsync(dX, X, (size_t)c->K * row, hipMemcpyHostToDevice, c->stream));
    else
        DG_HIP(c, hipMemcpy2DAsync(dX, row, X, (size_t)ldX * sizeof(double), row, (size_t)c->K,
                                   hipMemcpyHostToDevice, c->stream));
    if ((rc = dg_map_fp64(c, dX, L, dM))) return rc;
    return download_rows(c, M, ldM, dM, c->N, L);
}

int dg_resp_dense(dg_ctx *c, double *R, long ldR) {
    if (!c) return DG_EINVAL;
    if (!c->loaded || !c->have_estep) return dg_fail(c, DG_ESTATE, "dg_resp_dense needs a dg_estep");
    if (!R || ldR < c->N) return dg_fail(c, DG_EINVAL, "dg_resp_dense: bad args");
    int rc;
    if ((rc = select_device(c))) return rc;
    c->fp64_due = c->mixed();
    if (c->mixed() && (rc = fp64_normalisers(c))) return rc;
    DevBuf own;
    double *dR = c->partRT;
    if ((size_t)c->K * c->N > c->partRT_len) {
        if ((rc = dalloc(c, &own.p, (size_t)c->K * c->N))) return rc;
        dR = own.p;
    }
    if ((rc = dg_resp_dense_fp64(c, dR, c->N))) return rc;
    return download_rows(c, R, ldR, dR, c->K, c->N);
}

int dg_download(dg_ctx *c, double *W, long ldW, double *Y, long ldY, double *beta) {
    if (!c) return DG_EINVAL;
    if (!c->loaded) return dg_fail(c, DG_ESTATE, "dg_download before dg_upload");
    int rc;
    if ((rc = select_device(c))) return rc;
    if (W) {
        if (ldW < c->D) return dg_fail(c, DG_EINVAL, "dg_download: ldW < D");
        if ((rc = download_rows(c, W, ldW, c->W, c->M1, c->D))) return rc;
    }
    if (Y) {
        if (ldY < c->D) return dg_fail(c, DG_EINVAL, "dg_download: ldY < D");
        const double *src = c->Y64;
        if (c->ldt != c->D) {                      // its rows without their padding
            if ((rc = dg_pad_rows(c, c->Y64, c->K, c->D, c->ldt, c->D, c->partRT))) return rc;
            src = c->partRT;
        }
        if ((rc = download_rows(c, Y, ldY, src, c->K, c->D))) return rc;
    }
    DG_HIP(c, hipStreamSynchronize(c->stream));
    if (beta) *beta = c->beta;
    return DG_OK;
}

int dg_get_stats(dg_ctx *c, double *G, double *RT, long ldRT) {
    if (!c) return DG_EINVAL;
    if (!c->loaded || !c->have_estep) return dg_fail(c, DG_ESTATE, "dg_get_stats needs a dg_estep");
    int rc;
    if ((rc = select_device(c)) || (rc = due_stats(c))) return rc;
    if (G)
        DG_HIP(c, hipMemcpyAsync(G, c->G, (size_t)c->K * sizeof(double), hipMemcpyDeviceToHost,
                                 c->stream));
    if (RT) {
        if (ldRT < c->D) return dg_fail(c, DG_EINVAL, "dg_get_stats: ldRT < D");
        if ((rc = download_rows(c, RT, ldRT, c->RT, c->K, c->D))) return rc;
    }
    DG_HIP(c, hipStreamSynchronize(c->stream));
    return DG_OK;
}

int dg_device_peaks(dg_ctx *c, double *mfma_f16_tflops, double *exp_per_s, double *fp64_tflops) {
    if (!c) return DG_EINVAL;
    int rc;
    if ((rc = select_device(c))) return rc;
    int cus = 0;
    DG_HIP(c, hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, c->device));
    double m = 0, e = 0, f = 0;
    // eight 4-wave workgroups per CU: eight waves per SIMD
    if ((rc = dg_peaks_run(c, 8 * std::max(cus, 1), &m, &e, &f))) return rc;
    if (mfma_f16_tflops) *mfma_f16_tflops = m;
    if (exp_per_s) *exp_per_s = e;
    if (fp64_tflops) *fp64_tflops = f;
    return DG_OK;
}

int dg_pass2_blocks(dg_ctx *c, long *visited, long *total) {
    if (!c || !visited || !total) return DG_EINVAL;
    if (!c->mixed() || !c->have_estep)
        return dg_fail(c, DG_ESTATE, "dg_pass2_blocks: no mixed-precision E-step yet");
    int rc;
    if ((rc = select_device(c))) return rc;
    return dg_mixed_pass2_blocks(c, visited, total);
}

int dg_set_timing(dg_ctx *c, int on) {
    if (!c) return DG_EINVAL;
    c->timing = on ? 1 : 0;
    return DG_OK;
}

int dg_get_timing(dg_ctx *c, double t[4]) {
    if (!c || !t) return DG_EINVAL;
    for (int i = 0; i < 4; ++i) t[i] = c->t_ms[i];
    return DG_OK;
}

}  // extern "C"
