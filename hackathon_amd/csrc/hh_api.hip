// C-ABI layer of the MI355X compact-Helmholtz library (include/hh_solver.h).
//
// Contexts own the stream, the per-length twiddle tables, the dense DST
// matrices of non power-of-two sizes and a growable scratch buffer.  Plans
// own the device copies of the O(N) stencil coefficient vectors and the
// eigenvalues 2cos(k pi/(N+1)); they replace the reference's LU() factors.
#include <hip/hip_runtime.h>
#include <rocprofiler-sdk-roctx/roctx.h>

#include <cmath>
#include <complex>
#include <cstdarg>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <string>
#include <vector>

#include "../../include/hh_solver.h"
#include "hh_internal.h"

using cd = std::complex<double>;

static thread_local std::string g_err;

// Workspace of hh_solve_noalloc, for callers that cannot allocate (code under
// HIP graph capture, tight serving loops, harnesses that forbid hipMalloc):
// one array per device, held until the process ends.  In host code the
// array's name is a host-side stand-in: its device address is looked up once
// per device at context creation (hipGetSymbolAddress) and only that address
// is ever passed to kernels.
#define HH_NOALLOC_BYTES ((size_t)128 << 20)
static __device__ __align__(256) unsigned char noalloc_scratch[HH_NOALLOC_BYTES];
static std::mutex g_noalloc_mu;
static std::map<int, std::pair<void *, hipError_t>> g_noalloc;   // device -> (address, lookup status)

static int fail(int code, const char *fmt, ...) __attribute__((format(printf, 2, 3)));
static int fail(int code, const char *fmt, ...) {
    char buf[512];
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(buf, sizeof buf, fmt, ap);
    va_end(ap);
    g_err = buf;
    return code;
}

#define HIPCHK(call)                                                                               \
    do {                                                                                           \
        hipError_t e_ = (call);                                                                    \
        if (e_ != hipSuccess)                                                                      \
            return fail(HH_ERR_DEVICE, "%s failed: %s (%s:%d)", #call, hipGetErrorString(e_),     \
                        __FILE__, __LINE__);                                                       \
    } while (0)

constexpr size_t STAGE_LEAST = (size_t)256 << 10, STAGE_MOST = (size_t)8 << 20;

struct hh_context {
    int device = 0;
    hipStream_t own = nullptr, stream = nullptr;
    std::map<int, void *> tw64, tw32;   // twiddles by FFT length
    std::map<int, void *> S64, S32;     // dense DST matrices by N
    std::map<int, void *> th64, th32;   // half-length transform tables by N+1
    int dst_algo = -1;                  // -1 auto; bit 0: odd extension (else (N+1)-point), bit 1: 64-thread blocks
    void *scratch = nullptr;
    size_t scratch_bytes = 0;
    double *d_norm = nullptr;           // per-block norms, then the residuals' maxima (zero between solves)
    // their two results, in host memory that the kernels write (copied from the
    // device they cost a refinement 28 us more per sweep)
    double *h_norm = nullptr;
    // pinned memory from which the device reads a plan's operator tables (from
    // STAGE_LEAST up to STAGE_MOST), and the event of its last reader
    void *stage = nullptr;
    size_t stage_bytes = 0;
    hipEvent_t staged = nullptr;
    void *residual_slots() const { return d_norm + 2 * hh::NORM_BLOCKS; }
    size_t budget = 0, in_use = 0;
    void *noalloc_ws = nullptr;         // this device's noalloc_scratch (device address)
    hipError_t noalloc_status = hipSuccess;
    bool no_alloc = false;              // inside hh_solve_noalloc: allocations are refused
    std::mutex mu;
    // kernel timing (hh_context_enable_timing)
    struct Rec { hipEvent_t a, b; int cat; double bytes; };
    bool timing = false;
    std::vector<Rec> recs;
    std::vector<hipEvent_t> pool;
    double acc_ms[5] = {0, 0, 0, 0, 0}, acc_bytes[5] = {0, 0, 0, 0, 0};
    long acc_n[5] = {0, 0, 0, 0, 0};
};

// Records a pair of events around the launches in its scope when timing is on.
// Phase ranges for rocprofv3 --marker-trace (the reference's NVTX ranges,
// 2D_Program/solver_functions/cuda_helper.h:13-25 around the phases of
// solver.c:16-92): one roctx range per kernel pass, named by category, and
// one per solve; they cost a call each when no profiler listens.
static const char *const kPhaseName[] = {"hh:dst", "hh:dst_dense", "hh:tridiagonal", "hh:residual_update",
                                         "hh:rhs"};
struct Range {
    explicit Range(const char *name) { roctxRangePushA(name); }
    ~Range() { roctxRangePop(); }
};

struct TimeScope {
    hh_context *c;
    hh_context::Rec r;
    bool on;
    Range range;
    TimeScope(hh_context *ctx, int cat, double bytes)
        : c(ctx), on(ctx->timing && !ctx->no_alloc), range(kPhaseName[cat]) {
        if (!on) return;
        r.cat = cat;
        r.bytes = bytes;
        r.a = take();
        r.b = take();
        (void)hipEventRecord(r.a, c->stream);
    }
    hipEvent_t take() {
        if (!c->pool.empty()) { hipEvent_t e = c->pool.back(); c->pool.pop_back(); return e; }
        hipEvent_t e = nullptr;
        (void)hipEventCreate(&e);
        return e;
    }
    ~TimeScope() {
        if (!on) return;
        (void)hipEventRecord(r.b, c->stream);
        c->recs.push_back(r);
    }
};

struct hh_plan {
    hh_context *ctx = nullptr;
    int dim = 2, Nx = 0, Ny = 0, Nz = 1, prec = HH_PREC_F64;
    int nop = 1;                                 // operators (one per right-hand side b % nop)
    void *coef64 = nullptr, *coef32 = nullptr;   // [op][q][6] or [op][q][12]
    double *lamx = nullptr, *lamy = nullptr;
    std::vector<cd> hcoef;                       // host copy of the band table
    // real parts of the table, same order (read as (re c_2i, re c_2i+1) pairs by
    // the real-band tridiagonal kernels), FP64 and FP32
    void *coefr64 = nullptr, *coefr32 = nullptr;
    int real_op = 0;                             // every coefficient of the current operators real
    int real_mode = -1;                          // -1: real-band kernels when real_op; 0: complex-band always
    int cap_nop = 1;                             // operator slots allocated on the device
    double tol = 1e-12;
    int max_iter = 6;
    int tri_W = 0, tri_mm = 0;                   // tuned tridiagonal block shape (0 = heuristic)
    int tri_nr = 1;                              // right-hand sides per thread of the tuned shape
    // 2D spectrum layout: 0 row-major (default: measured fastest for the whole
    // solve, 1753 us against 1761-1844 us for tiles of 4..32 modes at N=1023,
    // 64 right-hand sides), -1 tiles of the block width, else the tile width
    int tile_w = 0;
    int last_sweeps = 0;
    double last_rel = 0;
    // eigenvalues 2cos(k pi/(N+1)) (host copies of lamx / lamy)
    std::vector<double> hlamx, hlamy;
    // near-resonant modes of the current operators and their reference-order
    // factors (hh_modes.hip), with their device copies
    double kappa_flag = hh::HH_KAPPA_FLAG;
    hh::ModeSet ms;
    int2 *d_ent = nullptr;                       // [op][nfx] (mode, entry)
    std::vector<int2> hent;
    uint32_t *d_bits = nullptr;
    void *d_facc = nullptr, *d_facr = nullptr;
    size_t cap_ent = 0, cap_bits = 0, cap_facc = 0, cap_facr = 0;
    // the operators before the present ones: a replacement that fails goes back to them
    std::vector<cd> prev_coef;
    hh::ModeSet prev_ms;
    int lost = 0;                                // the device tables of neither could be made
    // Generation: bumped whenever a change would invalidate a recorded graph
    // (device tables reallocated, band kind, operator count, near-resonant mode
    // counts or launch shapes changed); graphs record it at capture and refuse to replay a newer plan.
    long gen = 0;
};

// ------------------------------------------------------------------ helpers
static int dev_alloc(hh_context *c, void **p, size_t bytes) {
    if (c->no_alloc)
        return fail(HH_ERR_UNSUPPORTED, "hh_solve_noalloc: a table of %zu bytes is missing (create the plan with the "
                                        "context's current DST algorithm, or solve once with hh_solve first)", bytes);
    if (c->budget && c->in_use + bytes > c->budget)
        return fail(HH_ERR_NOMEM, "allocation of %zu bytes exceeds the memory budget (%zu of %zu in use)", bytes,
                    c->in_use, c->budget);
    hipError_t e = hipMalloc(p, bytes ? bytes : 16);
    if (e != hipSuccess) {
        (void)hipGetLastError();   // a caller that goes on without it must not find the error at its next launch
        return fail(HH_ERR_NOMEM, "hipMalloc(%zu) failed: %s", bytes, hipGetErrorString(e));
    }
    c->in_use += bytes;
    return HH_OK;
}

static void dev_free(hh_context *c, void *p, size_t bytes) {
    if (!p) return;
    (void)hipFree(p);
    c->in_use -= bytes < c->in_use ? bytes : c->in_use;
}

static int ensure_scratch(hh_context *c, size_t bytes) {
    if (c->scratch_bytes >= bytes) return HH_OK;
    if (c->scratch) {
        HIPCHK(hipStreamSynchronize(c->stream));
        dev_free(c, c->scratch, c->scratch_bytes);
        c->scratch = nullptr;
        c->scratch_bytes = 0;
    }
    int rc = dev_alloc(c, &c->scratch, bytes);
    if (rc) return rc;
    c->scratch_bytes = bytes;
    return HH_OK;
}

static int set_device(hh_context *c) {
    HIPCHK(hipSetDevice(c->device));
    return HH_OK;
}

// e^{-2 pi i q/L}, q < L, with exact argument reduction to the first octant
static void twiddles(int L, std::vector<cd> &out) {
    out.resize(L);
    for (int q = 0; q < L; q++) {
        long double a = -2.0L * 3.14159265358979323846264338327950288L * (long double)q / (long double)L;
        out[q] = cd((double)cosl(a), (double)sinl(a));
    }
}

static int get_twiddles(hh_context *c, int N, int f32, void **out) {
    int L = 2 * (N + 1);
    auto &m = f32 ? c->tw32 : c->tw64;
    auto it = m.find(L);
    if (it != m.end()) { *out = it->second; return HH_OK; }
    std::vector<cd> tw;
    twiddles(L, tw);
    void *d = nullptr;
    size_t bytes = (size_t)L * (f32 ? 8 : 16);
    int rc = dev_alloc(c, &d, bytes);
    if (rc) return rc;
    if (f32) {
        std::vector<float> h(2 * L);
        for (int q = 0; q < L; q++) { h[2 * q] = (float)tw[q].real(); h[2 * q + 1] = (float)tw[q].imag(); }
        HIPCHK(hipMemcpy(d, h.data(), bytes, hipMemcpyHostToDevice));
    } else {
        HIPCHK(hipMemcpy(d, tw.data(), bytes, hipMemcpyHostToDevice));
    }
    m[L] = d;
    *out = d;
    return HH_OK;
}

// Tables of the dense DST, from sqrt(2/(N+1)) sin(pi q/(N+1)) with the angle
// reduced exactly in integers, q = (n+1)(k+1) mod 2(N+1): its odd outputs
// k = 2c and its even ones k = 2c+1 on the first half of the line, each padded
// to half_dst_rows x half_dst_cols; the middle point of an odd N meets itself
// in x_j + x_{M-j} and enters at half weight.
static int get_dst_matrix(hh_context *c, int N, int f32, void **out) {
    auto &m = f32 ? c->S32 : c->S64;
    auto it = m.find(N);
    if (it != m.end()) { *out = it->second; return HH_OK; }
    const long M2 = 2L * (N + 1), HP = hh::half_dst_rows(N), WP = hh::half_dst_cols(N), H = (N + 1) / 2;
    const double s = std::sqrt(2.0 / (N + 1));
    std::vector<double> sine(M2), S((size_t)2 * HP * WP, 0.0);
    for (long q = 0; q < M2; q++)
        sine[q] = s * (double)sinl(3.14159265358979323846264338327950288L * (long double)q / (long double)(N + 1));
    for (int par = 0; par < 2; par++)
        for (long n = 0; n < (par == 0 ? H : N / 2); n++)
            for (long k = par; k < N; k += 2)
                S[(par * HP + n) * WP + k / 2] = sine[((n + 1) * (k + 1)) % M2] * (2 * n + 1 == N ? 0.5 : 1.0);
    void *d = nullptr;
    size_t bytes = S.size() * (f32 ? 4 : 8);
    int rc = dev_alloc(c, &d, bytes);
    if (rc) return rc;
    if (f32) {
        std::vector<float> h(S.begin(), S.end());
        HIPCHK(hipMemcpy(d, h.data(), bytes, hipMemcpyHostToDevice));
    } else {
        HIPCHK(hipMemcpy(d, S.data(), bytes, hipMemcpyHostToDevice));
    }
    m[N] = d;
    *out = d;
    return HH_OK;
}

// Table of the half-length transform: M = N+1 twiddles e^{-2 pi i q/M}, then
// the M reals sin(pi j/M) (packed into (M+1)/2 complex slots).
static int get_half_table(hh_context *c, int N, int f32, void **out) {
    const int M = N + 1;
    auto &m = f32 ? c->th32 : c->th64;
    auto it = m.find(M);
    if (it != m.end()) { *out = it->second; return HH_OK; }
    std::vector<cd> tw;
    twiddles(M, tw);
    const int ns = (M + 1) / 2;
    std::vector<double> h(2 * ((size_t)M + ns), 0.0);
    for (int q = 0; q < M; q++) { h[2 * q] = tw[q].real(); h[2 * q + 1] = tw[q].imag(); }
    for (int j = 0; j < M; j++)
        h[2 * (size_t)M + j] = (double)sinl(3.14159265358979323846264338327950288L * (long double)j / (long double)M);
    size_t n = h.size();
    void *d = nullptr;
    int rc = dev_alloc(c, &d, n * (f32 ? 4 : 8));
    if (rc) return rc;
    if (f32) {
        std::vector<float> hf(h.begin(), h.end());
        HIPCHK(hipMemcpy(d, hf.data(), n * 4, hipMemcpyHostToDevice));
    } else {
        HIPCHK(hipMemcpy(d, h.data(), n * 8, hipMemcpyHostToDevice));
    }
    m[M] = d;
    *out = d;
    return HH_OK;
}

// DST variant for lines of length N.  Automatic choice: the half-length
// transform at every power-of-two N+1: 20-45% faster than the odd extension
// above N+1 = 1024 (503 against 636 us for 1 GB of rows at N+1 = 2048, 566
// against 1055 at 4096), and accurate to 7e-15 relative per transform at
// N+1 = 4096; its error is correlated across the spectrum (prefix sums of
// transform values), so a transform and its inverse give 7e-14 there
// against 5e-16 for the odd extension, far inside a solve's 1e-12.
static int dst_algo_for(const hh_context *c, int N) {
    if (c->dst_algo >= 0) return c->dst_algo;
    return 0;
}

// Block size of the automatic choice (the blocks compute the same bits): 64,
// 256 or 512 threads, by the number nb of 256-thread blocks the lines fill.
//
// Rows (microseconds per pass, 64 against 256 threads): small one-wave blocks
// spread a small grid over four times as many CUs and wait for no other wave
// at their barriers: 6.0 against 9.4 (63 x 63, nb = 1), 7.8 against 10.0 (255
// rows of 255 x 6, nb = 96), 8.9 against 10.8 (511 x 511 x 2, nb = 128); their
// smaller LDS lets more of them share a CU in a large one: 47 against 82
// (63 x 63 x 2048), 40 against 43 (255 x 127 x 200), 99 against 109 (255^3),
// 414 against 460 (1023 x 1023 x 64).  Where one 256-thread block falls on
// each CU the larger block is better from N+1 = 128 on: 14 against 17.5 (1023
// rows of 1023), 11.0 against 12.8 (127 x 127 x 64), with a tie at both ends
// of the range taken (191 and 319 blocks).  In FP32 a 256-thread block's LDS
// is already half as large and above N+1 = 128 only the small grids gain:
// 8.4 against 9.4 (255 x 255 x 8, nb = 128), but 136 against 116 (255^3).
//
// Strided lines: the block's width is its segment of a row, so 64 threads pay
// only where the grid leaves half of the CUs idle and a segment is still 16
// lines or more (N+1 <= 64): 9.0 against 11.6 (63^3, nb = 63) but 15.8 against
// 13.4 at nb = 200.  FP32 takes 512 threads at N+1 = 256 (57 against 76 per
// 255^3 pass; in FP64 such a tile leaves one block per CU and it is slower),
// and at 128 where the wide tiles fill the chip once (17.2 against 19.3 at
// 255 x 127 x 63; 14.2 against 12.4 with half of the CUs idle, 35 against 31
// in two rounds at 255 x 127 x 200).
static int dst_algo_lines(const hh_context *c, const hh::Lines &ln, int tc) {
    const int algo = dst_algo_for(c, ln.N), M = ln.N + 1;
    if (c->dst_algo >= 0 || ln.in_tw || ln.out_tw) return algo;   // mode-tiled rows: a block's lines share segments
    const long per = M > 16 ? std::max(1, 4096 / M) : 256;   // lines of a 256-thread block
    if (ln.elem_stride == 1) {
        const long nb = (ln.ncols * ln.nplanes + per - 1) / per;
        if (M <= 64) return algo | 2;
        if (tc) return M <= 128 || nb <= 192 ? algo | 2 : algo;
        return nb > 192 && nb < 320 ? algo : algo | 2;
    }
    const long nb = (ln.ncols + per - 1) / per * ln.nplanes;
    if (M <= 64) return nb < 128 ? algo | 2 : algo;
    if (tc && (M == 256 || (M == 128 && nb > 448 && nb <= 1024))) return algo | 4;
    return algo;
}

// One DST pass over lines; in-place when the FFT path applies.
static int dst_pass(hh_context *c, const hh::Lines &ln0, int ti, int tc, int to, const void *in, void *out,
                    double acc = 0) {
    hh::Lines ln = ln0;
    ln.acc = acc;
    void *tw = nullptr, *S = nullptr;
    int rc;
    const int algo = dst_algo_lines(c, ln, tc);
    if (hh::fft_supported(ln.N))
        rc = (algo & 1) == 0 ? get_half_table(c, ln.N, tc, &tw) : get_twiddles(c, ln.N, tc, &tw);
    else rc = get_dst_matrix(c, ln.N, tc, &S);
    if (rc) return rc;
    const double elems = (double)ln.N * ln.ncols * ln.nplanes;
    TimeScope ts(c, tw ? 0 : 1, elems * ((ti ? 8 : 16) + (to ? 8 : 16) * (acc != 0 ? 2 : 1)));
    hh::DstTypes ty{ti, tc, to};
    ty.algo = algo;
    hipError_t e = hh::launch_dst(ln, ty, in, out, tw, S, c->stream);
    if (e != hipSuccess) return fail(HH_ERR_DEVICE, "DST launch (N=%d) failed: %s", ln.N, hipGetErrorString(e));
    return HH_OK;
}

static hh::Lines rows_lines(int N, long nrows) {
    hh::Lines l;
    l.N = N; l.ncols = nrows; l.nplanes = 1; l.plane_stride = (long)N * nrows; l.col_stride = N; l.elem_stride = 1;
    return l;
}

static hh::Lines cols_lines(int Nx, int Ny, long nplanes) {
    hh::Lines l;
    l.N = Ny; l.ncols = Nx; l.nplanes = nplanes; l.plane_stride = (long)Nx * Ny; l.col_stride = 1; l.elem_stride = Nx;
    return l;
}

static bool plan_all_fft(const hh_plan *p) {
    return hh::fft_supported(p->Nx) && (p->dim == 2 || hh::fft_supported(p->Ny));
}

// ------------------------------------------------------------------ errors
extern "C" const char *hh_last_error(void) { return g_err.c_str(); }

extern "C" const char *hh_status_string(int s) {
    switch (s) {
    case HH_OK: return "ok";
    case HH_ERR_ARG: return "invalid argument";
    case HH_ERR_DEVICE: return "device error";
    case HH_ERR_NOMEM: return "out of device memory";
    case HH_ERR_UNSUPPORTED: return "unsupported shape";
    case HH_ERR_SINGULAR: return "singular mode";
    default: return "unknown status";
    }
}

// ------------------------------------------------------------------ context
extern "C" int hh_context_create(int device, hh_context **out) {
    if (!out) return fail(HH_ERR_ARG, "hh_context_create: null output pointer");
    int n = 0;
    hipError_t e = hipGetDeviceCount(&n);
    if (e != hipSuccess || n == 0) return fail(HH_ERR_DEVICE, "no HIP device available (%s)", hipGetErrorString(e));
    if (device < 0 || device >= n) return fail(HH_ERR_ARG, "device %d out of range (%d devices)", device, n);
    hh_context *c = new hh_context();
    c->device = device;
    HIPCHK(hipSetDevice(device));
    e = hipStreamCreateWithFlags(&c->own, hipStreamNonBlocking);
    if (e != hipSuccess) { delete c; return fail(HH_ERR_DEVICE, "stream creation failed: %s", hipGetErrorString(e)); }
    c->stream = c->own;
    {
        // the static workspace of hh_solve_noalloc: its address on this device,
        // looked up once per device with the device current
        std::lock_guard<std::mutex> lk(g_noalloc_mu);
        auto it = g_noalloc.find(device);
        if (it == g_noalloc.end()) {
            void *ptr = nullptr;
            const hipError_t se = hipGetSymbolAddress(&ptr, HIP_SYMBOL(noalloc_scratch));
            it = g_noalloc.emplace(device, std::make_pair(se == hipSuccess ? ptr : nullptr, se)).first;
        }
        c->noalloc_ws = it->second.first;
        c->noalloc_status = it->second.second;
    }
    const std::vector<double> zeros(2 * hh::NORM_SLOTS, 0.0);
    if (hipMalloc((void **)&c->d_norm, 2 * (hh::NORM_BLOCKS + hh::NORM_SLOTS) * sizeof(double)) != hipSuccess ||
        hipMemcpy(c->residual_slots(), zeros.data(), zeros.size() * sizeof(double), hipMemcpyHostToDevice) != hipSuccess ||
        hipHostMalloc((void **)&c->h_norm, 2 * sizeof(double), hipHostMallocDefault) != hipSuccess ||
        hipEventCreateWithFlags(&c->staged, hipEventDisableTiming) != hipSuccess) {
        (void)hipHostFree(c->h_norm);
        (void)hipFree(c->d_norm);
        (void)hipStreamDestroy(c->own);
        delete c;
        return fail(HH_ERR_NOMEM, "norm buffer allocation failed");
    }
    *out = c;
    return HH_OK;
}

extern "C" int hh_context_destroy(hh_context *c) {
    if (!c) return HH_OK;
    (void)hipSetDevice(c->device);
    (void)hipStreamSynchronize(c->stream);
    for (auto &kv : c->tw64) (void)hipFree(kv.second);
    for (auto &kv : c->tw32) (void)hipFree(kv.second);
    for (auto &kv : c->S64) (void)hipFree(kv.second);
    for (auto &kv : c->S32) (void)hipFree(kv.second);
    for (auto &kv : c->th64) (void)hipFree(kv.second);
    for (auto &kv : c->th32) (void)hipFree(kv.second);
    if (c->scratch) (void)hipFree(c->scratch);
    for (auto &r : c->recs) { (void)hipEventDestroy(r.a); (void)hipEventDestroy(r.b); }
    for (auto e : c->pool) (void)hipEventDestroy(e);
    (void)hipFree(c->d_norm);
    (void)hipHostFree(c->h_norm);
    (void)hipEventSynchronize(c->staged);
    (void)hipHostFree(c->stage);
    (void)hipEventDestroy(c->staged);
    (void)hipStreamDestroy(c->own);
    delete c;
    return HH_OK;
}

extern "C" int hh_context_set_stream(hh_context *c, void *stream) {
    if (!c) return fail(HH_ERR_ARG, "null context");
    // NULL is the HIP default (null) stream, which orders against the work
    // of callers (e.g. PyTorch's default stream) that use it
    const hipStream_t next = (hipStream_t)stream;
    if (next == c->stream) return HH_OK;
    // Replaced operators' tables may still be on their way on the stream before:
    // the next one waits for them, or the host where it is being recorded (a
    // wait for work outside it would end the recording).
    int rc = set_device(c);
    if (rc) return rc;
    hipStreamCaptureStatus recording = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(next, &recording) == hipSuccess && recording == hipStreamCaptureStatusNone) {
        HIPCHK(hipStreamWaitEvent(next, c->staged, 0));
    } else {
        (void)hipGetLastError();
        hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
        HIPCHK(hipThreadExchangeStreamCaptureMode(&mode));
        const hipError_t e = hipEventSynchronize(c->staged);
        HIPCHK(hipThreadExchangeStreamCaptureMode(&mode));
        HIPCHK(e);
    }
    c->stream = next;
    return HH_OK;
}

extern "C" void *hh_context_get_stream(hh_context *c) { return c ? (void *)c->stream : nullptr; }

extern "C" int hh_context_synchronize(hh_context *c) {
    if (!c) return fail(HH_ERR_ARG, "null context");
    HIPCHK(hipStreamSynchronize(c->stream));
    return HH_OK;
}

extern "C" int hh_context_set_memory_budget(hh_context *c, size_t bytes) {
    if (!c) return fail(HH_ERR_ARG, "null context");
    c->budget = bytes;
    return HH_OK;
}

extern "C" size_t hh_context_bytes_in_use(const hh_context *c) { return c ? c->in_use : 0; }

static int collect_timing(hh_context *c) {
    if (c->recs.empty()) return HH_OK;
    HIPCHK(hipStreamSynchronize(c->stream));
    for (auto &r : c->recs) {
        float ms = 0;
        HIPCHK(hipEventElapsedTime(&ms, r.a, r.b));
        c->acc_ms[r.cat] += ms;
        c->acc_bytes[r.cat] += r.bytes;
        c->acc_n[r.cat] += 1;
        c->pool.push_back(r.a);
        c->pool.push_back(r.b);
    }
    c->recs.clear();
    return HH_OK;
}

extern "C" int hh_context_set_dst_algorithm(hh_context *c, int algo) {
    if (!c) return fail(HH_ERR_ARG, "null context");
    if (algo < -1 || algo > 15) return fail(HH_ERR_ARG, "DST algorithm must be -1..15 (got %d)", algo);
    std::lock_guard<std::mutex> lk(c->mu);
    c->dst_algo = algo;
    return HH_OK;
}

extern "C" int hh_context_enable_timing(hh_context *c, int on) {
    if (!c) return fail(HH_ERR_ARG, "null context");
    std::lock_guard<std::mutex> lk(c->mu);
    c->timing = on != 0;
    return HH_OK;
}

extern "C" int hh_context_read_timing(hh_context *c, double ms[5], long launches[5], double bytes[5]) {
    if (!c) return fail(HH_ERR_ARG, "null context");
    std::lock_guard<std::mutex> lk(c->mu);
    int rc = collect_timing(c);
    if (rc) return rc;
    for (int k = 0; k < 5; k++) {
        if (ms) ms[k] = c->acc_ms[k];
        if (launches) launches[k] = c->acc_n[k];
        if (bytes) bytes[k] = c->acc_bytes[k];
    }
    return HH_OK;
}

extern "C" int hh_context_reset_timing(hh_context *c) {
    if (!c) return fail(HH_ERR_ARG, "null context");
    std::lock_guard<std::mutex> lk(c->mu);
    int rc = collect_timing(c);
    for (int k = 0; k < 5; k++) { c->acc_ms[k] = 0; c->acc_bytes[k] = 0; c->acc_n[k] = 0; }
    return rc;
}

// ------------------------------------------------------------------ coefficients
static inline cd ld(const double *p, long i) { return p ? cd(p[2 * i], p[2 * i + 1]) : cd(0, 0); }
static inline void st(double *p, long i, cd v) { p[2 * i] = v.real(); p[2 * i + 1] = v.imag(); }

extern "C" int hh_coefficients2d(int order, int Nx, int Ny, double hx, double hy, const double *k2e,
                                 const double *k2y, const double *k2yy, double *bp, double *ap, double *b, double *a,
                                 double *bm, double *am) {
    if (Nx < 1 || Ny < 1 || !k2e || !bp || !ap || !b || !a || !bm || !am)
        return fail(HH_ERR_ARG, "hh_coefficients2d: bad arguments");
    if (order != 2 && order != 4 && order != 6) return fail(HH_ERR_ARG, "order must be 2, 4 or 6 (got %d)", order);
    const double hy2 = hy * hy, hy3 = hy2 * hy, hy4 = hy2 * hy2, Ryx = hy * hy / hx / hx;
    for (int j = 0; j < Ny; j++) {
        cd k2 = ld(k2e, j + 1), k2p = ld(k2e, j + 2), k2m = ld(k2e, j);
        if (order == 6) {                                   // coefficients.c:44-61
            cd ky2 = ld(k2y, j), kyy = ld(k2yy, j);
            st(ap, j, 2.0 / 3.0 + hy2 * k2p / 90.0 + hy3 * ky2 * (hy2 * k2p / 6.0 + 2.0 / 3.0) / 20.0);
            st(bp, j, 1.0 / 6.0 + hy2 * k2p / 90.0 + hy3 * ky2 / 120.0);
            st(a, j, -10.0 / 3.0 + 41.0 * hy2 * k2 / 45.0 - hy4 * k2 * k2 / 20.0 + hy4 * kyy / 20.0);
            st(b, j, 2.0 / 3.0 + hy2 * k2 / 90.0);
            st(am, j, 2.0 / 3.0 + hy2 * k2m / 90.0 - hy3 * ky2 * (hy2 * k2m / 6.0 + 2.0 / 3.0) / 20.0);
            st(bm, j, 1.0 / 6.0 + hy2 * k2m / 90.0 - hy3 * ky2 / 120.0);
        } else if (order == 4) {                            // coefficients.c:25-42
            st(bp, j, cd(Ryx / 12.0 + 1.0 / 12.0));
            st(ap, j, 5.0 / 6.0 - Ryx / 6.0 + hy2 * k2p / 12.0);
            st(b, j, Ryx * (5.0 / 6.0) - 1.0 / 6.0 + hy2 * k2 / 12.0);
            st(a, j, -Ryx * (5.0 / 3.0) - 5.0 / 3.0 + 2.0 * hy2 * k2 / 3.0);
            st(bm, j, cd(Ryx / 12.0 + 1.0 / 12.0));
            st(am, j, 5.0 / 6.0 - Ryx / 6.0 + hy2 * k2m / 12.0);
        } else {                                            // coefficients.c:9-23
            st(bp, j, cd(0));
            st(ap, j, cd(1));
            st(b, j, cd(Ryx));
            st(a, j, -2.0 * Ryx - 2.0 + k2 * hy2);
            st(bm, j, cd(0));
            st(am, j, cd(1));
        }
    }
    return HH_OK;
}

// compact (1, diag, 1) solve of a complex vector (4th_order_partials.c:322-336)
static void compact_line(std::vector<cd> &v, double diag) {
    int n = (int)v.size();
    std::vector<double> U(n);
    U[0] = diag;
    for (int j = 1; j < n; j++) U[j] = diag - 1.0 / U[j - 1];
    for (int j = 1; j < n; j++) v[j] = v[j] - (1.0 / U[j - 1]) * v[j - 1];
    v[n - 1] = v[n - 1] / U[n - 1];
    for (int j = n - 2; j >= 0; j--) v[j] = (v[j] - v[j + 1]) / U[j];
}

extern "C" int hh_coefficients3d(int order, int Nx, int Ny, int Nz, double hx, double hy, double hz,
                                 const double *k2e, const double *k2d, double *const coef[12]) {
    if (Nx < 1 || Ny < 1 || Nz < 1 || !k2e || !coef) return fail(HH_ERR_ARG, "hh_coefficients3d: bad arguments");
    for (int q = 0; q < 12; q++)
        if (!coef[q]) return fail(HH_ERR_ARG, "hh_coefficients3d: null coefficient array %d", q);
    if (order != 2 && order != 4 && order != 6) return fail(HH_ERR_ARG, "order must be 2, 4 or 6 (got %d)", order);
    double *A = coef[0], *B = coef[1], *C = coef[2], *D = coef[3], *Ap = coef[4], *Bp = coef[5], *Cp = coef[6],
           *Dp = coef[7], *Am = coef[8], *Bm = coef[9], *Cm = coef[10], *Dm = coef[11];
    const double Rzx = hz * hz / hx / hx, Rzy = hz * hz / hy / hy, h2 = hz * hz;
    std::vector<cd> k2(Nz + 2);
    for (int l = 0; l < Nz + 2; l++) k2[l] = ld(k2e, l);
    if (order == 6) {                                       // coefficients.c:67-103
        std::vector<cd> kp(Nz), kpp(Nz);
        for (int l = 0; l < Nz; l++) {
            kp[l] = 3.0 * (k2[l + 2] - k2[l]) / hz;
            kpp[l] = 12.0 * (k2[l] - 2.0 * k2[l + 1] + k2[l + 2]) / hz / hz;
        }
        kp[0] -= ld(k2d, 0); kp[Nz - 1] -= ld(k2d, 1);
        kpp[0] -= ld(k2d, 2); kpp[Nz - 1] -= ld(k2d, 3);
        compact_line(kp, 4.0);
        compact_line(kpp, 10.0);
        for (int i = 0; i < Nz; i++) {
            st(A, i, 1.0 / 10.0 + h2 * k2[i + 1] / 90.0);
            st(B, i, 7.0 / 15.0 - h2 * k2[i + 1] / 90.0);
            st(C, i, 7.0 / 15.0 - h2 * k2[i + 1] / 90.0);
            st(D, i, -64.0 / 15.0 + 14.0 * h2 * k2[i + 1] / 15.0 - h2 * h2 * k2[i + 1] * k2[i + 1] / 20.0 +
                         h2 * h2 * kpp[i] / 20.0);
            st(Ap, i, cd(1.0 / 30.0));
            st(Bp, i, 1.0 / 10.0 + h2 * k2[i + 2] / 90.0 + (kp[i] * h2 * hz / 120.0));
            st(Cp, i, 1.0 / 10.0 + h2 * k2[i + 2] / 90.0 + (kp[i] * h2 * hz / 120.0));
            st(Dp, i, 7.0 / 15.0 - h2 * k2[i + 2] / 90.0 + (kp[i] * h2 * hz / 20.0) * (1.0 / 3.0 + k2[i + 2] * h2 / 6.0));
            st(Am, i, cd(1.0 / 30.0));
            st(Bm, i, 1.0 / 10.0 + h2 * k2[i] / 90.0 - (kp[i] * h2 * hz / 120.0));
            st(Cm, i, 1.0 / 10.0 + h2 * k2[i] / 90.0 - (kp[i] * h2 * hz / 120.0));
            st(Dm, i, 7.0 / 15.0 - h2 * k2[i] / 90.0 - (kp[i] * h2 * hz / 20.0) * (1.0 / 3.0 + k2[i] * h2 / 6.0));
        }
    } else if (order == 4) {                                // coefficients.c:35-65
        for (int i = 0; i < Nz; i++) {
            st(A, i, cd((1.0 / 12.0) * (Rzx + Rzy)));
            st(B, i, (1.0 / 6.0) * (4.0 * Rzx - Rzy - 1.0 + 0.5 * h2 * k2[i + 1]));
            st(C, i, (1.0 / 6.0) * (4.0 * Rzy - Rzx - 1.0 + 0.5 * h2 * k2[i + 1]));
            st(D, i, -4.0 * (1.0 + Rzx + Rzy) / 3.0 + 0.5 * h2 * k2[i + 1]);
            st(Ap, i, cd(0));
            st(Bp, i, cd((1.0 / 12.0) * (1.0 + Rzx)));
            st(Cp, i, cd((1.0 / 12.0) * (1.0 + Rzy)));
            st(Dp, i, 1.0 - (1.0 / 6.0) * (2.0 + Rzx + Rzy) + (1.0 / 12.0) * h2 * k2[i + 2]);
            st(Am, i, cd(0));
            st(Bm, i, cd((1.0 / 12.0) * (1.0 + Rzx)));
            st(Cm, i, cd((1.0 / 12.0) * (1.0 + Rzy)));
            st(Dm, i, 1.0 - (1.0 / 6.0) * (2.0 + Rzx + Rzy) + (1.0 / 12.0) * h2 * k2[i]);
        }
    } else {                                                // coefficients.c:7-33
        for (int i = 0; i < Nz; i++) {
            st(A, i, cd(0)); st(B, i, cd(Rzx)); st(C, i, cd(Rzy));
            st(D, i, -2.0 * (Rzx + Rzy + 1.0) + h2 * k2[i + 1]);
            st(Ap, i, cd(0)); st(Bp, i, cd(0)); st(Cp, i, cd(0)); st(Dp, i, cd(1));
            st(Am, i, cd(0)); st(Bm, i, cd(0)); st(Cm, i, cd(0)); st(Dm, i, cd(1));
        }
    }
    return HH_OK;
}

// ------------------------------------------------------------------ Robin closure
// Boundary condition du/dn + alpha u = g on the first (lo) or last (hi) row of
// the tridiagonal axis, the row itself lying on the boundary.  The central
// difference (u_1 - u_{-1}) / 2h places a ghost row u_{-1} = u_1 - 2h alpha u_0
// + 2h g outside the grid; substituting it into the boundary row's stencil
// M u_{-1} + C u_0 + P u_1 = F_0 gives (C - 2h alpha M) u_0 + (P + M) u_1 =
// F_0 - 2h M g (mirrored on the hi side).  M, C and P are the same
// combinations of the DST-direction neighbour sums in every row, so the fold
// is band-wise on the coefficient vectors, and the DST still diagonalises
// the folded operator.  corr receives -2h M g (the row of F to add).
// bands: pointers to nb centre, nb plus and nb minus vectors, in that order.
static void robin_fold(int n, double h, cd alpha, bool lo, double *const *ctr, double *const *pls,
                       double *const *mns, int nb, cd *orig) {
    const int r = lo ? 0 : n - 1;
    for (int q = 0; q < nb; q++) {
        const cd m = ld(mns[q], r), p = ld(pls[q], r), c = ld(ctr[q], r);
        const cd out = lo ? m : p;             // band that reached the ghost row
        orig[q] = out;
        st(ctr[q], r, c - 2.0 * h * alpha * out);
        if (lo) { st(pls[q], r, p + m); st(mns[q], r, cd(0)); }
        else    { st(mns[q], r, m + p); st(pls[q], r, cd(0)); }
    }
}

extern "C" int hh_robin2d(int Nx, int Ny, double h, const double *alpha_lo, const double *g_lo,
                          const double *alpha_hi, const double *g_hi, double *const coef[6], double *corr_lo,
                          double *corr_hi) {
    if (Nx < 1 || Ny < 2 || !(h > 0) || !coef) return fail(HH_ERR_ARG, "hh_robin2d: bad arguments");
    for (int q = 0; q < 6; q++)
        if (!coef[q]) return fail(HH_ERR_ARG, "hh_robin2d: null coefficient array %d", q);
    // [bp, ap, b, a, bm, am]: centre (b, a), plus (bp, ap), minus (bm, am); per band the x-operator
    // is (first) * (u_{i-1} + u_{i+1}) + (second) * u_i
    double *ctr[2] = {coef[2], coef[3]}, *pls[2] = {coef[0], coef[1]}, *mns[2] = {coef[4], coef[5]};
    for (int side = 0; side < 2; side++) {
        const double *al = side == 0 ? alpha_lo : alpha_hi, *g = side == 0 ? g_lo : g_hi;
        double *corr = side == 0 ? corr_lo : corr_hi;
        if (!al) continue;
        cd o[2];
        robin_fold(Ny, h, cd(al[0], al[1]), side == 0, ctr, pls, mns, 2, o);
        if (!corr) continue;
        for (int i = 0; i < Nx; i++) {
            const cd nb = (i > 0 ? ld(g, i - 1) : cd(0)) + (i + 1 < Nx ? ld(g, i + 1) : cd(0));
            st(corr, i, -2.0 * h * (o[0] * nb + o[1] * ld(g, i)));
        }
    }
    return HH_OK;
}

extern "C" int hh_robin3d(int Nx, int Ny, int Nz, double h, const double *alpha_lo, const double *g_lo,
                          const double *alpha_hi, const double *g_hi, double *const coef[12], double *corr_lo,
                          double *corr_hi) {
    if (Nx < 1 || Ny < 1 || Nz < 2 || !(h > 0) || !coef) return fail(HH_ERR_ARG, "hh_robin3d: bad arguments");
    for (int q = 0; q < 12; q++)
        if (!coef[q]) return fail(HH_ERR_ARG, "hh_robin3d: null coefficient array %d", q);
    // [a, b, c, d | ap..dp | am..dm]: per band the (x, y)-operator is a * (diagonal neighbours)
    // + b * (x neighbours) + c * (y neighbours) + d * u
    double *ctr[4] = {coef[0], coef[1], coef[2], coef[3]}, *pls[4] = {coef[4], coef[5], coef[6], coef[7]},
           *mns[4] = {coef[8], coef[9], coef[10], coef[11]};
    auto G = [&](const double *g, int i, int j) {
        return (i >= 0 && i < Nx && j >= 0 && j < Ny) ? ld(g, i + (long)j * Nx) : cd(0);
    };
    for (int side = 0; side < 2; side++) {
        const double *al = side == 0 ? alpha_lo : alpha_hi, *g = side == 0 ? g_lo : g_hi;
        double *corr = side == 0 ? corr_lo : corr_hi;
        if (!al) continue;
        cd o[4];
        robin_fold(Nz, h, cd(al[0], al[1]), side == 0, ctr, pls, mns, 4, o);
        if (!corr) continue;
        for (int j = 0; j < Ny; j++)
            for (int i = 0; i < Nx; i++) {
                const cd dg = G(g, i - 1, j - 1) + G(g, i + 1, j - 1) + G(g, i - 1, j + 1) + G(g, i + 1, j + 1);
                const cd xg = G(g, i - 1, j) + G(g, i + 1, j), yg = G(g, i, j - 1) + G(g, i, j + 1);
                st(corr, i + (long)j * Nx, -2.0 * h * (o[0] * dg + o[1] * xg + o[2] * yg + o[3] * G(g, i, j)));
            }
    }
    return HH_OK;
}

// ------------------------------------------------------------------ plans
// Device band-table order from the caller's operator vectors.
// 2D: input [op][bp, ap, b, a, bm, am][Ny] -> table [op][q](bm, am, b, a, bp, ap);
// 3D: input [op][a..dm][Nz] -> table [op][l][12].
static void build_table(int dim, int n, int nop, const double *coef, std::vector<cd> &tab) {
    if (dim == 2) {
        static const int src[6] = {4, 5, 2, 3, 0, 1};
        tab.resize(6 * (size_t)n * nop);
        for (int o = 0; o < nop; o++)
            for (int q = 0; q < n; q++)
                for (int t = 0; t < 6; t++)
                    tab[((size_t)o * n + q) * 6 + t] = ld(coef, ((size_t)o * 6 + src[t]) * n + q);
    } else {
        tab.resize(12 * (size_t)n * nop);
        for (int o = 0; o < nop; o++)
            for (int l = 0; l < n; l++)
                for (int q = 0; q < 12; q++)
                    tab[((size_t)o * n + l) * 12 + q] = ld(coef, ((size_t)o * 12 + q) * n + l);
    }
}

static bool table_real(const std::vector<cd> &tab) {
    for (const cd &v : tab)
        if (v.imag() != 0.0) return false;
    return true;
}

static void classify(hh_plan *p, int nop) {
    hh::classify_modes(p->dim, p->Nx, p->Ny, p->Nz, nop, p->hcoef.data(), p->hlamx.data(), p->hlamy.data(),
                       p->real_op != 0, p->kappa_flag, p->ms);
}

static void fill_table(hh_plan *p, int nop, const double *coef) {
    build_table(p->dim, p->dim == 2 ? p->Ny : p->Nz, nop, coef, p->hcoef);
    p->real_op = table_real(p->hcoef);
    classify(p, nop);
}

// eigenvalues 2cos(k pi/(N+1)), k = 1..N (LU.c:12-14)
static void eigenvalues(int N, std::vector<double> &v) {
    v.resize(N);
    for (int k = 0; k < N; k++) v[k] = 2.0 * std::cos((k + 1) * M_PI / (N + 1));
}

// Device array holding at least `bytes`; a new allocation bumps the plan's
// generation (recorded graphs hold the old address).
static int ensure_dev(hh_plan *p, void **ptr, size_t *cap, size_t bytes) {
    if (*ptr && bytes <= *cap) return HH_OK;
    hh_context *c = p->ctx;
    const size_t old = *ptr ? *cap : 0;
    if (*ptr) {
        HIPCHK(hipStreamSynchronize(c->stream));
        dev_free(c, *ptr, *cap);
        *ptr = nullptr;
        *cap = 0;
    }
    // grow by at least half again (a serving loop's operators flag a few
    // modes more or fewer from batch to batch: reallocate seldom, since a
    // free waits for the stream)
    size_t b = bytes ? bytes : 16;
    if (old) b = std::max(b, old + old / 2);
    int rc = dev_alloc(c, ptr, b);
    if (rc) return rc;
    *cap = b;
    p->gen++;
    return HH_OK;
}

// Staging memory for `bytes`, up to STAGE_MOST: pinning is slow (94 MiB for the
// factors of every mode of 127^3: 20 ms of 45, in pieces 25).  Where that much
// cannot be had, the one there stays or a smaller one does.
static int grow_stage(hh_context *c, size_t bytes) {
    if (bytes <= c->stage_bytes || c->stage_bytes >= STAGE_MOST) return HH_OK;
    size_t want = std::min(std::max((bytes + bytes / 2 + 15) / 16 * 16, STAGE_LEAST), STAGE_MOST);
    void *more = nullptr;
    while (hipHostMalloc(&more, want, hipHostMallocDefault) != hipSuccess) {
        (void)hipGetLastError();
        if (c->stage) return HH_OK;
        if (want <= 4096) return fail(HH_ERR_NOMEM, "pinned allocation of %zu bytes failed", want);
        want = want / 32 * 16;
    }
    (void)hipEventSynchronize(c->staged);
    (void)hipHostFree(c->stage);
    c->stage = more;
    c->stage_bytes = want;
    return HH_OK;
}

// The device tables of the plan's operators (nop of them in hcoef and ms) from
// the host's, stream-ordered after the work already queued; the context's lock
// is held.
static int upload_tables(hh_plan *p) {
    hh_context *c = p->ctx;
    const hh::ModeSet &m = p->ms;
    const size_t ne = m.fmode.size(), nf = ne * m.n * 4;
    int rc;
    // one row of nfx entries per operator, padded with (-1, 0)
    p->hent.assign((size_t)m.nop * m.nfx, make_int2(-1, 0));
    for (int o = 0; o < m.nop; o++)
        for (int e = m.foff[o]; e < m.foff[o + 1]; e++) p->hent[(size_t)o * m.nfx + e - m.foff[o]] = make_int2(m.fmode[e], e);
    if ((rc = ensure_dev(p, (void **)&p->d_ent, &p->cap_ent, p->hent.size() * sizeof(int2)))) return rc;
    if ((rc = ensure_dev(p, (void **)&p->d_bits, &p->cap_bits, m.bits.size() * sizeof(uint32_t)))) return rc;
    if ((rc = ensure_dev(p, &p->d_facc, &p->cap_facc, nf * sizeof(cd)))) return rc;
    if ((rc = ensure_dev(p, &p->d_facr, &p->cap_facr, (p->real_op ? nf : 0) * sizeof(double)))) return rc;
    // bands, factors, entries and bits go through the staging memory in turn, as
    // much at a time as it holds
    const size_t fac = p->real_op ? sizeof(double) : sizeof(cd), unit[4] = {sizeof(cd), fac, sizeof(int2), sizeof(uint32_t)};
    const void *src[4] = {p->hcoef.data(), p->real_op ? (const void *)m.facr.data() : (const void *)m.facc.data(),
                          p->hent.data(), m.bits.data()};
    const size_t len[4] = {p->hcoef.size(), nf, p->hent.size(), m.bits.size()};
    size_t total = 0, done[4] = {};
    for (int k = 0; k < 4; k++) total += (len[k] * unit[k] + 15) / 16 * 16;
    if ((rc = grow_stage(c, total))) return rc;
    for (bool more = true; more;) {
        HIPCHK(hipEventSynchronize(c->staged));
        size_t at[4], n[4], used = 0;
        for (int k = 0; k < 4; k++) {
            at[k] = used;
            n[k] = std::min(len[k] - done[k], (c->stage_bytes - used) / unit[k]);
            if (n[k]) memcpy((char *)c->stage + used, (const char *)src[k] + done[k] * unit[k], n[k] * unit[k]);
            used += (n[k] * unit[k] + 15) / 16 * 16;
        }
        const char *base = (const char *)c->stage;
        hh::OperatorTables t;
        t.ncoef = (long)n[0];
        t.coef = (const double2 *)(base + at[0]);
        t.coef64 = (double2 *)p->coef64 + done[0]; t.coef32 = (float2 *)p->coef32 + done[0];
        t.coefr64 = (double *)p->coefr64 + done[0]; t.coefr32 = (float *)p->coefr32 + done[0];
        t.n = m.n; t.nent = (long)ne;
        t.fac0 = (long)done[1]; t.nfac = (long)n[1];
        (p->real_op ? (const void *&)t.facr : (const void *&)t.facc) = base + at[1];
        t.outr = (double *)p->d_facr; t.outc = (double2 *)p->d_facc;
        t.nslot = (long)n[2]; t.ent = (const int2 *)(base + at[2]); t.outent = p->d_ent + done[2];
        t.nbits = (long)n[3]; t.bits = (const uint32_t *)(base + at[3]); t.outbits = p->d_bits + done[3];
        const hipError_t e = hh::launch_operator_tables(t, c->stream);
        if (e != hipSuccess) return fail(HH_ERR_DEVICE, "operator tables: launch failed: %s", hipGetErrorString(e));
        HIPCHK(hipEventRecord(c->staged, c->stream));
        more = false;
        for (int k = 0; k < 4; k++) {
            done[k] += n[k];
            more = more || done[k] < len[k];
        }
    }
    return HH_OK;
}

// The plan's operators become the nop of coef or, with coef null, are classified
// again, for the threshold kappa; the context's lock is held.  When the new
// tables do not fit (memory budget), the plan stays as it was: its mode tables
// get their old sizes and contents back, after what the new ones took is freed.
static int replace_operators(hh_plan *p, int nop, const double *coef, double kappa) {
    hh_context *c = p->ctx;
    int rc = set_device(c);
    if (rc) return rc;
    HIPCHK(hipStreamSynchronize(c->stream));   // replaced tables may be reallocated
    struct Dev { void **ptr; size_t *cap, was; };
    Dev dev[4] = {{(void **)&p->d_ent, &p->cap_ent, p->cap_ent}, {(void **)&p->d_bits, &p->cap_bits, p->cap_bits},
                  {&p->d_facc, &p->cap_facc, p->cap_facc}, {&p->d_facr, &p->cap_facr, p->cap_facr}};
    const int old_real = p->real_op;
    const double old_kappa = p->kappa_flag;
    std::swap(p->ms, p->prev_ms);
    p->kappa_flag = kappa;
    if (coef) {
        p->hcoef.swap(p->prev_coef);
        fill_table(p, nop, coef);
    } else {
        classify(p, nop);
    }
    rc = upload_tables(p);   // solves queued before this call still read the old ones
    if (rc == HH_OK) {
        const hh::ModeSet &was = p->prev_ms, &now = p->ms;
        // the sum over all operators is the factors' row length
        if (p->real_op != old_real || now.nfx != was.nfx || now.fmode.size() != was.fmode.size() || nop != p->nop)
            p->gen++;
        p->nop = nop;
        p->lost = 0;
        if (was.facr.size() + 2 * was.facc.size() > ((size_t)1 << 20)) p->prev_ms = hh::ModeSet();   // 8 MiB
        return HH_OK;
    }
    const std::string why = g_err;
    std::swap(p->ms, p->prev_ms);
    if (coef) p->hcoef.swap(p->prev_coef);
    p->real_op = old_real;
    p->kappa_flag = old_kappa;
    for (Dev &d : dev)
        if (*d.ptr && *d.cap != d.was) {
            dev_free(c, *d.ptr, *d.cap);
            *d.ptr = nullptr;
            *d.cap = 0;
        }
    int back = HH_OK;
    for (Dev &d : dev)
        if (back == HH_OK) back = ensure_dev(p, d.ptr, d.cap, d.was);
    if (back == HH_OK) back = upload_tables(p);
    if (back != HH_OK) {
        p->lost = 1;
        p->gen++;
    }
    g_err = why;
    return rc;
}

static int upload_plan(hh_plan *p, int ncoef, int n) {
    hh_context *c = p->ctx;
    size_t b64 = (size_t)ncoef * n * p->nop * 16, b32 = (size_t)ncoef * n * p->nop * 8;
    int rc = dev_alloc(c, &p->coef64, b64);
    if (rc) return rc;
    rc = dev_alloc(c, &p->coef32, b32);
    if (rc) return rc;
    if ((rc = dev_alloc(c, &p->coefr64, b64 / 2))) return rc;
    if ((rc = dev_alloc(c, &p->coefr32, b32 / 2))) return rc;
    const std::vector<double> &lx = p->hlamx, &ly = p->hlamy;
    rc = dev_alloc(c, (void **)&p->lamx, lx.size() * 8);
    if (rc) return rc;
    HIPCHK(hipMemcpy(p->lamx, lx.data(), lx.size() * 8, hipMemcpyHostToDevice));
    if (p->dim == 3) {
        rc = dev_alloc(c, (void **)&p->lamy, ly.size() * 8);
        if (rc) return rc;
        HIPCHK(hipMemcpy(p->lamy, ly.data(), ly.size() * 8, hipMemcpyHostToDevice));
    }
    std::lock_guard<std::mutex> lk(c->mu);
    if ((rc = upload_tables(p))) return rc;
    HIPCHK(hipStreamSynchronize(c->stream));
    return HH_OK;
}

// ------------------------------------------------------------------ host-only mode classification
extern "C" int hh_operator_modes(int dim, int Nx, int Ny, int Nz, const double *coef, double kappa, int *nflagged,
                                 int *modes, int cap, int *singular, double *kappa_worst) {
    if ((dim != 2 && dim != 3) || Nx < 2 || Ny < 2 || (dim == 3 && Nz < 2) || !coef || !(kappa >= 0) ||
        (cap > 0 && !modes))
        return fail(HH_ERR_ARG, "hh_operator_modes: bad arguments");
    std::vector<cd> tab;
    build_table(dim, dim == 2 ? Ny : Nz, 1, coef, tab);
    std::vector<double> lx, ly;
    eigenvalues(Nx, lx);
    if (dim == 3) eigenvalues(Ny, ly);
    hh::ModeSet ms;
    hh::classify_modes(dim, Nx, Ny, Nz, 1, tab.data(), lx.data(), ly.data(), table_real(tab), kappa, ms);
    if (nflagged) *nflagged = (int)ms.fmode.size();
    for (int i = 0; i < (int)ms.fmode.size() && i < cap; i++) modes[i] = ms.fmode[i];
    if (singular) *singular = ms.singular[0];
    if (kappa_worst) *kappa_worst = ms.kappa_worst[0];
    return HH_OK;
}

extern "C" int hh_operator_mode_factors(int dim, int Nx, int Ny, int Nz, const double *coef, int mode,
                                        double *factors) {
    const long nmodes = dim == 2 ? Nx : (long)Nx * Ny;
    if ((dim != 2 && dim != 3) || Nx < 2 || Ny < 2 || (dim == 3 && Nz < 2) || !coef || !factors || mode < 0 ||
        mode >= nmodes)
        return fail(HH_ERR_ARG, "hh_operator_mode_factors: bad arguments");
    const int n = dim == 2 ? Ny : Nz;
    std::vector<cd> tab;
    build_table(dim, n, 1, coef, tab);
    std::vector<double> lx, ly;
    eigenvalues(Nx, lx);
    if (dim == 3) eigenvalues(Ny, ly);
    // classify with kappa = 0: every mode flagged, entry index = mode index
    hh::ModeSet ms;
    const bool real = table_real(tab);
    hh::classify_modes(dim, Nx, Ny, Nz, 1, tab.data(), lx.data(), ly.data(), real, 0.0, ms);
    const size_t at = (size_t)mode * n * 4;
    auto f = [&](long i) { return real ? cd(ms.facr[at + i]) : ms.facc[at + i]; };
    for (long q = 0; q < n; q++) {   // (L, R, Up) of each row
        const cd v[3] = {f(4 * q), f(4 * q + 2), f(4 * q + 3)};
        for (int k = 0; k < 3; k++) {
            factors[2 * (3 * q + k)] = v[k].real();
            factors[2 * (3 * q + k) + 1] = v[k].imag();
        }
    }
    return ms.singular[0] ? fail(HH_ERR_SINGULAR, "operator is singular to working precision") : HH_OK;
}

static int prepare_tables(hh_plan *p);

static int plan_check_dims(int dim, int Nx, int Ny, int Nz) {
    if (Nx < 2 || Ny < 2 || (dim == 3 && Nz < 2))
        return fail(HH_ERR_ARG, "grid sizes must be at least 2 (got %d x %d x %d)", Nx, Ny, Nz);
    long big = 1L << 30;
    if ((long)Nx * Ny * (dim == 3 ? Nz : 1) > 64 * big) return fail(HH_ERR_UNSUPPORTED, "grid too large");
    int sys = dim == 2 ? Ny : Nz;
    if (sys > 8192) return fail(HH_ERR_UNSUPPORTED, "system length %d above 8192", sys);
    return HH_OK;
}

extern "C" int hh_plan2d_create(hh_context *ctx, int Nx, int Ny, const double *bp, const double *ap,
                                const double *b, const double *a, const double *bm, const double *am, int precision,
                                hh_plan **out) {
    if (!ctx || !out || !bp || !ap || !b || !a || !bm || !am) return fail(HH_ERR_ARG, "hh_plan2d_create: null argument");
    if (Ny < 1) return fail(HH_ERR_ARG, "grid sizes must be at least 2 (got %d x %d)", Nx, Ny);
    const double *v[6] = {bp, ap, b, a, bm, am};
    std::vector<double> packed(2 * 6 * (size_t)Ny);
    for (int q = 0; q < 6; q++) memcpy(packed.data() + 2 * (size_t)q * Ny, v[q], 16 * (size_t)Ny);
    return hh_plan2d_create_multi(ctx, Nx, Ny, 1, packed.data(), precision, out);
}

extern "C" int hh_plan2d_create_multi(hh_context *ctx, int Nx, int Ny, int nop, const double *coef, int precision,
                                      hh_plan **out) {
    if (!ctx || !out || !coef) return fail(HH_ERR_ARG, "hh_plan2d_create_multi: null argument");
    if (nop < 1) return fail(HH_ERR_ARG, "number of operators must be >= 1 (got %d)", nop);
    if (precision != HH_PREC_F64 && precision != HH_PREC_MIXED) return fail(HH_ERR_ARG, "unknown precision %d", precision);
    int rc = plan_check_dims(2, Nx, Ny, 1);
    if (rc) return rc;
    if ((rc = set_device(ctx))) return rc;
    hh_plan *p = new hh_plan();
    p->ctx = ctx; p->dim = 2; p->Nx = Nx; p->Ny = Ny; p->Nz = 1; p->prec = precision; p->nop = nop;
    p->cap_nop = nop;
    eigenvalues(Nx, p->hlamx);
    fill_table(p, nop, coef);
    if ((rc = upload_plan(p, 6, Ny))) { hh_plan_destroy(p); return rc; }
    // the transform tables the plan's solves read: a solve then allocates nothing but workspace
    if ((rc = prepare_tables(p))) { hh_plan_destroy(p); return rc; }
    *out = p;
    return HH_OK;
}

extern "C" int hh_plan3d_create(hh_context *ctx, int Nx, int Ny, int Nz, const double *const coef[12], int precision,
                                hh_plan **out) {
    if (!ctx || !out || !coef) return fail(HH_ERR_ARG, "hh_plan3d_create: null argument");
    for (int q = 0; q < 12; q++)
        if (!coef[q]) return fail(HH_ERR_ARG, "hh_plan3d_create: null coefficient array %d", q);
    if (Nz < 1) return fail(HH_ERR_ARG, "grid sizes must be at least 2 (got Nz = %d)", Nz);
    std::vector<double> packed(2 * 12 * (size_t)Nz);
    for (int q = 0; q < 12; q++) memcpy(packed.data() + 2 * (size_t)q * Nz, coef[q], 16 * (size_t)Nz);
    return hh_plan3d_create_multi(ctx, Nx, Ny, Nz, 1, packed.data(), precision, out);
}

extern "C" int hh_plan3d_create_multi(hh_context *ctx, int Nx, int Ny, int Nz, int nop, const double *coef,
                                      int precision, hh_plan **out) {
    if (!ctx || !out || !coef) return fail(HH_ERR_ARG, "hh_plan3d_create_multi: null argument");
    if (nop < 1) return fail(HH_ERR_ARG, "number of operators must be >= 1 (got %d)", nop);
    if (precision != HH_PREC_F64 && precision != HH_PREC_MIXED) return fail(HH_ERR_ARG, "unknown precision %d", precision);
    int rc = plan_check_dims(3, Nx, Ny, Nz);
    if (rc) return rc;
    if ((rc = set_device(ctx))) return rc;
    hh_plan *p = new hh_plan();
    p->ctx = ctx; p->dim = 3; p->Nx = Nx; p->Ny = Ny; p->Nz = Nz; p->prec = precision; p->nop = nop;
    p->cap_nop = nop;
    eigenvalues(Nx, p->hlamx);
    eigenvalues(Ny, p->hlamy);
    fill_table(p, nop, coef);
    if ((rc = upload_plan(p, 12, Nz))) { hh_plan_destroy(p); return rc; }
    // the transform tables the plan's solves read: a solve then allocates nothing but workspace
    if ((rc = prepare_tables(p))) { hh_plan_destroy(p); return rc; }
    *out = p;
    return HH_OK;
}

extern "C" int hh_plan_num_operators(const hh_plan *p) { return p ? p->nop : 0; }

extern "C" int hh_plan_destroy(hh_plan *p) {
    if (!p) return HH_OK;
    hh_context *c = p->ctx;
    int nc = p->dim == 2 ? 6 : 12, n = p->dim == 2 ? p->Ny : p->Nz;
    (void)hipStreamSynchronize(c->stream);
    dev_free(c, p->coef64, (size_t)nc * n * p->cap_nop * 16);
    dev_free(c, p->coef32, (size_t)nc * n * p->cap_nop * 8);
    dev_free(c, p->coefr64, (size_t)nc * n * p->cap_nop * 8);
    dev_free(c, p->coefr32, (size_t)nc * n * p->cap_nop * 4);
    dev_free(c, p->lamx, (size_t)p->Nx * 8);
    if (p->lamy) dev_free(c, p->lamy, (size_t)p->Ny * 8);
    dev_free(c, p->d_ent, p->cap_ent);
    dev_free(c, p->d_bits, p->cap_bits);
    dev_free(c, p->d_facc, p->cap_facc);
    dev_free(c, p->d_facr, p->cap_facr);
    delete p;
    return HH_OK;
}

extern "C" hh_context *hh_plan_context(const hh_plan *p) { return p ? p->ctx : nullptr; }

extern "C" int hh_plan_dims(const hh_plan *p, int dims[3]) {
    if (!p || !dims) return fail(HH_ERR_ARG, "hh_plan_dims: null argument");
    dims[0] = p->Nx; dims[1] = p->Ny; dims[2] = p->Nz;
    return p->dim;
}

extern "C" long hh_plan_field_size(const hh_plan *p) {
    return p ? (long)p->Nx * p->Ny * (p->dim == 3 ? p->Nz : 1) : 0;
}

extern "C" size_t hh_plan_workspace_bytes(const hh_plan *p, int batch) {
    if (!p || batch < 1) return 0;
    size_t f = (size_t)hh_plan_field_size(p) * batch;
    size_t ws = 0;
    if (!plan_all_fft(p)) ws += f * 16;      // ping-pong buffer of the dense DST path
    else if (p->dim == 2 && p->tile_w != 0) ws += f * (p->prec == HH_PREC_MIXED ? 8 : 16);   // mode-tiled spectrum
    if (p->prec == HH_PREC_MIXED) ws += f * 8;   // FP32 correction
    return ws;
}

extern "C" int hh_plan_set_refine(hh_plan *p, double tol, int max_iter) {
    if (!p || tol < 0 || max_iter < 0) return fail(HH_ERR_ARG, "hh_plan_set_refine: bad arguments");
    p->gen++;
    p->tol = tol;
    p->max_iter = max_iter;
    return HH_OK;
}

extern "C" int hh_plan_set_tri_shape(hh_plan *p, int W, int rows_per_thread, int rhs_per_thread) {
    if (!p) return fail(HH_ERR_ARG, "null plan");
    p->gen++;
    if (W == 0 && rows_per_thread == 0) { p->tri_W = p->tri_mm = 0; p->tri_nr = 1; return HH_OK; }
    int n = p->dim == 2 ? p->Ny : p->Nz;
    if (W < 1 || W > 64 || (rows_per_thread != 4 && rows_per_thread != 8 && rows_per_thread != 16) ||
        (rhs_per_thread != 1 && rhs_per_thread != 2 && rhs_per_thread != 4))
        return fail(HH_ERR_ARG, "tridiagonal shape W=%d rows=%d rhs=%d not available", W, rows_per_thread,
                    rhs_per_thread);
    int P = (n + rows_per_thread - 1) / rows_per_thread;
    if (P > n / 2) P = n / 2;
    if (P < 1 || W * P > 1024 || (n + P - 1) / P > rows_per_thread)
        return fail(HH_ERR_UNSUPPORTED, "tridiagonal shape W=%d rows=%d does not fit n=%d", W, rows_per_thread, n);
    // the reduced system's two PCR buffers (A, C and the FP64 right-hand sides; A and C real for the
    // real-band kernel of real operators, complex otherwise) must fit the 160 KiB of LDS.  A shape that
    // fits only real bands is replaced by the built-in one while the operators are complex.
    if (hh::tri_lds_bytes(hh_plan_is_real_operator(p) ? 8 : 16, 16, P, W, rhs_per_thread) > (size_t)160 * 1024)
        return fail(HH_ERR_UNSUPPORTED, "tridiagonal shape W=%d rows=%d rhs=%d needs more LDS than a CU has", W,
                    rows_per_thread, rhs_per_thread);
    p->tri_W = W;
    p->tri_mm = rows_per_thread;
    p->tri_nr = rhs_per_thread;
    return HH_OK;
}

extern "C" int hh_plan_set_real_operator(hh_plan *p, int mode) {
    if (!p) return fail(HH_ERR_ARG, "null plan");
    p->gen++;
    if (mode < -1 || mode > 0) return fail(HH_ERR_ARG, "real-operator mode must be -1 (automatic) or 0 (complex bands)");
    p->real_mode = mode;
    return HH_OK;
}

extern "C" int hh_plan_is_real_operator(const hh_plan *p) { return p && p->real_op && p->real_mode != 0; }

extern "C" int hh_plan_set_tile_width(hh_plan *p, int tw) {
    if (!p) return fail(HH_ERR_ARG, "null plan");
    p->gen++;
    if (tw != -1 && (tw < 0 || tw > 64 || (tw & (tw - 1))))
        return fail(HH_ERR_ARG, "tile width must be -1, 0 or a power of two up to 64 (got %d)", tw);
    p->tile_w = tw;
    return HH_OK;
}

// Shape of `rows` rows per thread and about `threads` threads per block:
// W the largest power of two with W P <= threads, up to 16 (at least wmin,
// which may be more), and no more than the modes need.
static void shape_for(int n, long nmodes, int rows, int threads, int wmin, hh::TriHelm &t) {
    int P = (n + rows - 1) / rows;
    if (P > n / 2) P = n / 2;
    if (P < 1) P = 1;
    int w = 1;
    while (w * 2 * P <= threads && w * 2 <= 16) w *= 2;
    if (w < wmin) w = wmin;
    while (w > 1 && w / 2 >= nmodes) w /= 2;
    t.W = w; t.P = P; t.mmax = rows;
}

// Built-in block shape of the mode solves (W, P, rows and right-hand sides
// per thread) for FP64 or FP32 elimination; per_op: right-hand sides per
// operator in the batch.  Measured on MI355X (order-6 operators
// with k^2 = 2500 or 2500 + 50i, row-major spectrum; microseconds of the
// mode pass of one solve, near-resonant modes included; in brackets the
// former rule of 256-thread blocks, 16 rows per thread above n = 512):
//   real bands, FP64
//     2D  n <= 512: 16 rows, 2 rhs, ~512 threads: 127 x 256: 53.9 (60.0),
//         255 x 64: 59.2 (66.3), 511 x 64: 184 (216);
//         n <= 1024: 16 rows, 2 rhs, W = 4, and 8 above n = 768 from 1024
//         blocks of 8 on (against 8 rows, 1 rhs, W = 4, one band per mode):
//         255 x 520 x 1: 19 (24), 1023 x 520 x 40: 152 (263), 511 x 640 x 8:
//         28 (37), 255 x 768 x 64: 145 (164), 1023 x 850 x 16: 109 (135), 1023
//         x 1: 37 (44), x 12: 103 (100), x 64: 527 (551), with k varying 601
//         (769); W = 8 below 1024 blocks or 768 rows: 1023 x 520 x 16: 95 (W =
//         4: 64), 1023 x 1023 x 6: 60 (51); W = 4 above: 255 x 1000 x 64: 189
//         (W = 8: 145);
//         above: 16 rows, 2 rhs, 512 threads: 2047 x 16: 848 (983)
//     3D  n <= 64, or n <= 128 and at most 1024 modes: 8 rows, 2 rhs, 128 threads
//         (16 rows, W = 8: 20 x 20 x 65 x 2: 10.0 (9.6), 31 x 31 x 65 x 2: 10.2
//         (10.3), 40 x 40 x 128 x 2: 11.1 (11.4));
//         n <= 128: 16 rows, 2 rhs, W = 8, and 32 from 1024 blocks of 16 on
//         (against 8 rows, 128 threads): 52 x 52 x 100: 9.5 (10.3), x 8: 17.5
//         (21.9), 125^3: 17 (22), x 2: 23 (30), x 4: 43 (49), 127^3 x 8: 99
//         (124), 255 x 255 x 100: 43 (49); 40 x 40 x 65 x 2: 10.5 (10.2);
//         above: 16 rows, 256 threads: 255^3 x 1: 187 (212)
//   complex bands, FP64
//         n <= 512: 8 rows, 2 rhs, 256 threads: 2D 127: 67 (75), 255: 79
//         (86), 511: 240 (265); 3D 127^3 x 8: 169 (228);
//         n <= 768: 8 rows, 1 rhs (2 would round differently than a solve of
//         one), W = 4 up to 800 blocks, 2 from there (k varying with y and
//         absorbing, against W = 4 with 16 rows): 255 x 520 x 2: 54 (65), x 32:
//         97 (110), 511 x 640 x 3: 56 (69), x 12: 74 (89), x 64: 355 (431),
//         400 x 700 x 6, 600 blocks: 60, W = 2: 66 (65), 100 x 700 x 40, 1000
//         blocks: 67, W = 4: 81 (69);
//         above: 16 rows, 1 rhs, W >= 4: 2047 x 16: 1292 (1321); 8 rows there
//         are better and worse by turns: 1023 x 40: 689 (737), 300 x 1000 x 16:
//         93 (89)
//   real bands, 2D, FP32 elimination: 16 rows, 512 threads: 1023 x 64:
//         449 (506), 2047 x 16: 609 (733), 511: 131 (133), 255: 51 (53)
// and the former rule elsewhere (within 2% of the best shape measured).
// Two right-hand sides per thread need two per operator in the batch.
static void builtin_tri_shape(const hh_plan *p, bool f32, long per_op, bool real, hh::TriHelm &t) {
    const int n = p->dim == 2 ? p->Ny : p->Nz;
    const long nmodes = p->dim == 2 ? p->Nx : (long)p->Nx * p->Ny;
    hh::tri_shape(n, nmodes, &t.W, &t.P, &t.mmax);
    t.nr = 1;
    if (n <= 16) return;
    int nr = 1;
    const long blocks16 = (nmodes + 15) / 16 * p->nop * ((per_op + 1) / 2);
    if (!f32 && real && p->dim == 2) {
        if (n <= 512) { shape_for(n, nmodes, 16, 512, 1, t); nr = 2; }
        else if (n <= 1024) {
            const long blocks = (nmodes + 7) / 8 * p->nop * ((per_op + 1) / 2);
            const int w = n <= 768 || blocks < 1024 ? 4 : 8;
            shape_for(n, nmodes, 16, w * ((n + 15) / 16), w, t);
            nr = 2;
        }
        else { shape_for(n, nmodes, 16, 512, 1, t); nr = 2; }
    } else if (!f32 && real) {
        if (n <= 64 || (n <= 128 && nmodes <= 1024)) { shape_for(n, nmodes, 8, 128, 1, t); nr = 2; }
        else if (n <= 128) {
            const int w = blocks16 < 1024 ? 8 : 32;
            shape_for(n, nmodes, 16, w * ((n + 15) / 16), w, t);
            nr = 2;
        } else { shape_for(n, nmodes, 16, 256, 1, t); nr = 2; }
    } else if (!f32) {
        if (n <= 512) { shape_for(n, nmodes, 8, 256, 1, t); nr = 2; }
        else if (n <= 768) {
            const long blocks = (nmodes + 3) / 4 * p->nop * per_op;
            const int w = blocks < 800 ? 4 : 2;
            shape_for(n, nmodes, 8, w * ((n + 7) / 8), w, t);
        } else shape_for(n, nmodes, 16, 256, 4, t);
    } else if (real && p->dim == 2) {
        shape_for(n, nmodes, 16, 512, 1, t);
    }
    // Long complex systems: four modes' reduced systems pass a CU's LDS above
    // n = 3408 and a block's 1024 threads above 4096 (refused there before); one
    // mode's fits up to the longest system, 8192 rows (98 KB).
    const size_t op = (real ? 8 : 16) / (f32 ? 2 : 1), cx = f32 ? 8 : 16, lds = 160 * 1024;
    while (t.W > 1 && (t.W * t.P > 1024 || hh::tri_lds_bytes(op, cx, t.P, t.W, 1) > lds)) t.W /= 2;
    if (nr == 2 && per_op >= 2 && hh::tri_lds_bytes(op, cx, t.P, t.W, 2) <= lds) t.nr = 2;
}

extern "C" int hh_plan_get_tri_shape(const hh_plan *p, int *W, int *P, int *rows_per_thread, int *rhs_per_thread) {
    if (!p) return fail(HH_ERR_ARG, "null plan");
    hh::TriHelm t;
    int n = p->dim == 2 ? p->Ny : p->Nz;
    // the shape of the solve's elimination (mixed precision: FP32), for a
    // batch of two or more right-hand sides per operator
    builtin_tri_shape(p, p->prec == HH_PREC_MIXED, 2, p->real_op && p->real_mode != 0, t);
    if (p->tri_W > 0) {   // the tuned shape, where its reduced system fits the LDS (as in solve_core)
        const bool mixed = p->prec == HH_PREC_MIXED, real = p->real_op && p->real_mode != 0;
        const int nr = mixed ? 1 : p->tri_nr;
        int P2 = (n + p->tri_mm - 1) / p->tri_mm;
        if (P2 > n / 2) P2 = n / 2;
        if (hh::tri_lds_bytes((real ? 8 : 16) / (mixed ? 2 : 1), mixed ? 8 : 16, P2, p->tri_W, nr) <=
            (size_t)160 * 1024) {
            t.W = p->tri_W;
            t.mmax = p->tri_mm;
            t.nr = nr;
            t.P = P2;
        }
    }
    if (W) *W = t.W;
    if (P) *P = t.P;
    if (rows_per_thread) *rows_per_thread = t.mmax;
    if (rhs_per_thread) *rhs_per_thread = t.nr;
    return HH_OK;
}

extern "C" int hh_plan_set_resonance_threshold(hh_plan *p, double kappa) {
    if (!p || !(kappa >= 0)) return fail(HH_ERR_ARG, "hh_plan_set_resonance_threshold: bad arguments");
    std::lock_guard<std::mutex> lk(p->ctx->mu);
    return replace_operators(p, p->nop, nullptr, kappa);
}

extern "C" int hh_plan_mode_info(const hh_plan *p, int op, int *flagged, int *singular, double *kappa) {
    if (!p || op < 0 || op >= p->nop) return fail(HH_ERR_ARG, "hh_plan_mode_info: bad arguments");
    if (flagged) *flagged = p->ms.foff[op + 1] - p->ms.foff[op];
    if (singular) *singular = p->ms.singular[op];
    if (kappa) *kappa = p->ms.kappa_worst[op];
    return HH_OK;
}

extern "C" int hh_plan_flagged_modes(const hh_plan *p, int op, int *modes, int cap) {
    if (!p || op < 0 || op >= p->nop || (cap > 0 && !modes)) return fail(HH_ERR_ARG, "hh_plan_flagged_modes: bad arguments");
    const int n = p->ms.foff[op + 1] - p->ms.foff[op];
    for (int i = 0; i < n && i < cap; i++) modes[i] = p->ms.fmode[p->ms.foff[op] + i];
    return n;
}

extern "C" int hh_plan_last_refine(const hh_plan *p, int *sweeps, double *rel) {
    if (!p) return fail(HH_ERR_ARG, "null plan");
    if (sweeps) *sweeps = p->last_sweeps;
    if (rel) *rel = p->last_rel;
    return HH_OK;
}

// ------------------------------------------------------------------ solve
// Transform-solve-transform on one buffer.  Types: ti input, tc compute /
// intermediate storage, to output (0 = FP64, 1 = FP32).  tri_comp is the
// arithmetic of the tridiagonal elimination.
// acc != 0: sol += acc A^{-1} rhs, the last pass accumulating into the FP64
// sol (rhs is then consumed: it may serve as scratch).
// op >= 0: the batch is one right-hand side, of operator op.
static int solve_core(hh_plan *p, int ti, int tc, int to, int tri_comp, const void *rhs, void *sol, void *ws,
                      int batch, double acc = 0, int op = -1) {
    hh_context *c = p->ctx;
    const int Nx = p->Nx, Ny = p->Ny, Nz = p->Nz;
    int rc;
    hh::TriHelm t;
    t.dim = p->dim; t.Nx = Nx; t.Ny = Ny; t.Nz = Nz;
    t.field = hh_plan_field_size(p);
    t.batch = batch;
    t.coef = tri_comp == 0 ? p->coef64 : p->coef32;
    t.real = p->real_op && p->real_mode != 0;
    t.coefr = tri_comp == 0 ? p->coefr64 : p->coefr32;
    t.nop = op < 0 ? p->nop : 1;
    t.uni = p->d_bits;
    t.cstride = p->dim == 2 ? 6L * Ny : 12L * Nz;
    t.lamx = p->lamx; t.lamy = p->lamy;
    int n = p->dim == 2 ? Ny : Nz;
    const long per_op = (batch + t.nop - 1) / t.nop;
    builtin_tri_shape(p, tri_comp == 1, per_op, t.real, t);
    if (p->tri_W > 0 && p->tri_mm > 0) {   // shape chosen by the autotuner
        const int nr = tri_comp == 0 ? p->tri_nr : 1;
        int P = (n + p->tri_mm - 1) / p->tri_mm;
        if (P > n / 2) P = n / 2;
        const size_t op = (t.real ? 8 : 16) / (tri_comp == 0 ? 1 : 2), cx = tri_comp == 0 ? 16 : 8;
        if (hh::tri_lds_bytes(op, cx, P, p->tri_W, nr) <= (size_t)160 * 1024) {
            t.W = p->tri_W;
            t.mmax = p->tri_mm;
            t.nr = nr;
            t.P = P;
        }
    }
    // near-resonant modes: reference-order substitution from the host's
    // factors (FP64 arithmetic), beside the partitioned elimination of the rest
    t.nfx = p->ms.nfx;
    if (t.nfx > 0) {
        t.fbits = p->d_bits + p->nop;
        t.fwords = p->ms.words;
        t.ent = p->d_ent;
        t.fac = t.real ? p->d_facr : p->d_facc;
        t.nent = (long)p->ms.fmode.size();
    }
    if (op > 0) {   // the operator's own tables; its factors are indexed through ent
        const size_t cb = tri_comp == 0 ? 16 : 8;
        t.coef = (const char *)t.coef + op * t.cstride * cb;
        t.coefr = (const char *)t.coefr + op * t.cstride * (cb / 2);
        t.uni += op;
        if (t.nfx > 0) {
            t.fbits += (size_t)op * t.fwords;
            t.ent += (size_t)op * t.nfx;
        }
    }
    auto tri = [&](void *buf) -> int {
        TimeScope ts(c, 2, (double)t.field * batch * (tc ? 16 : 32));
        hipError_t e = hh::launch_tri_helm(t, hh::DstTypes{tc, tri_comp, tc}, buf, buf, c->stream);
        if (e != hipSuccess) return fail(HH_ERR_DEVICE, "tridiagonal launch failed: %s", hipGetErrorString(e));
        return HH_OK;
    };
    const bool fft = plan_all_fft(p);
    if (p->dim == 2) {
        // FFT path: the forward row DST writes the spectrum mode-tiled into
        // ws (tiles of W modes, the tridiagonal block width), the mode solves
        // run there in place, the inverse row DST reads it back row-major
        // into sol.  Dense path: ws is a plain row-major intermediate.
        hh::Lines lx = rows_lines(Nx, (long)Ny * batch);
        const int tw = p->tile_w < 0 ? t.W : p->tile_w;
        if (fft && tw > 0) {
            if (!ws || ws == rhs || ws == sol) return fail(HH_ERR_ARG, "internal: missing workspace");
            // tiles hold whole blocks: the built-in W (a power of two) is cut
            // to a narrower tile; a shape set by hand must fit as given
            if (p->tri_W == 0 && t.W > tw) t.W = tw;
            t.tiled = tw;
            hh::Lines fwd = lx, inv = lx;
            fwd.out_tw = tw; fwd.ny = Ny; fwd.field = t.field;
            inv.in_tw = tw; inv.ny = Ny; inv.field = t.field;
            if ((rc = dst_pass(c, fwd, ti, tc, tc, rhs, ws))) return rc;
            if ((rc = tri(ws))) return rc;
            return dst_pass(c, inv, tc, tc, to, ws, sol, acc);
        }
        // row-major spectrum: in sol (in place) on the FFT path, in ws otherwise
        void *mid = fft ? (tc == to && acc == 0 ? sol : ws) : ws;
        if (!mid) return fail(HH_ERR_ARG, "internal: missing workspace");
        if ((rc = dst_pass(c, lx, ti, tc, tc, rhs, mid))) return rc;
        if ((rc = tri(mid))) return rc;
        return dst_pass(c, lx, tc, tc, to, mid, sol, acc);
    }
    if (acc != 0 && (to != 0 || ti != tc)) return fail(HH_ERR_UNSUPPORTED, "internal: accumulating solve types");
    hh::Lines lx = rows_lines(Nx, (long)Ny * Nz * batch);
    hh::Lines ly = cols_lines(Nx, Ny, (long)Nz * batch);
    // FFT passes start where the pass before ended: y backwards before the mode
    // solves, x after them (255^3: 525 -> 514 us; smaller fields fit the cache either way)
    hh::Lines lyr = ly, lxr = lx;
    lyr.reverse = lxr.reverse = 1;
    if (fft && tc == to && acc == 0) {
        if ((rc = dst_pass(c, lx, ti, tc, tc, rhs, sol))) return rc;
        if ((rc = dst_pass(c, lyr, tc, tc, tc, sol, sol))) return rc;
        if ((rc = tri(sol))) return rc;
        if ((rc = dst_pass(c, ly, tc, tc, tc, sol, sol))) return rc;
        return dst_pass(c, lxr, tc, tc, to, sol, sol);
    }
    if (!ws) return fail(HH_ERR_ARG, "internal: missing workspace");
    if (fft) {   // intermediate precision differs from the output: keep it in ws
        if ((rc = dst_pass(c, lx, ti, tc, tc, rhs, ws))) return rc;
        if ((rc = dst_pass(c, lyr, tc, tc, tc, ws, ws))) return rc;
        if ((rc = tri(ws))) return rc;
        if ((rc = dst_pass(c, ly, tc, tc, tc, ws, ws))) return rc;
        return dst_pass(c, lxr, tc, tc, to, ws, sol, acc);
    }
    // dense 3D path: ping-pong between ws and a second buffer holding the
    // intermediate in the compute type: sol (no smaller than the compute
    // type), or, when sol is accumulated into, the consumed rhs
    if (tc == 0 && to == 1) return fail(HH_ERR_UNSUPPORTED, "internal: FP64 intermediate in an FP32 output");
    void *mid = acc != 0 ? const_cast<void *>(rhs) : sol;
    if (mid == ws) return fail(HH_ERR_ARG, "internal: workspace aliases the intermediate");
    if ((rc = dst_pass(c, lx, ti, tc, tc, rhs, ws))) return rc;
    if ((rc = dst_pass(c, ly, tc, tc, tc, ws, mid))) return rc;
    if ((rc = tri(mid))) return rc;
    if ((rc = dst_pass(c, ly, tc, tc, tc, mid, ws))) return rc;
    return dst_pass(c, lx, tc, tc, to, ws, sol, acc);
}

static int read_norms(hh_context *c, double out[2]) {
    HIPCHK(hipStreamSynchronize(c->stream));
    out[0] = c->h_norm[0];
    out[1] = c->h_norm[1];
    return HH_OK;
}

// norms (FP32 results): norms[0..1] = max |res| and max |F|, waited for.
static int residual_into(hh_plan *p, const void *u, const void *F, void *res, int res_f32, int batch,
                         double *norms = nullptr) {
    TimeScope ts(p->ctx, 3, (double)hh_plan_field_size(p) * batch * (32 + (res_f32 ? 8 : 16)));
    hh_context *c = p->ctx;
    void *slots = norms ? c->residual_slots() : nullptr;
    hipError_t e;
    if (p->dim == 2)
        e = hh::launch_residual2d(p->Nx, p->Ny, batch, p->coef64, p->nop, u, F, res, res_f32, slots, c->stream);
    else
        e = hh::launch_residual3d(p->Nx, p->Ny, p->Nz, batch, p->coef64, p->nop, u, F, res, res_f32, slots, c->stream);
    if (e == hipSuccess && norms) e = hh::launch_residual_norms(slots, c->h_norm, c->stream);
    if (e != hipSuccess) return fail(HH_ERR_DEVICE, "residual launch failed: %s", hipGetErrorString(e));
    return norms ? read_norms(c, norms) : HH_OK;
}

static int norms_sync(hh_context *c, long n, const void *x, const void *y, double out[2], bool l2 = false) {
    hipError_t e = hh::launch_norms(n, x, y, c->d_norm, c->h_norm, c->stream, l2);
    if (e != hipSuccess) return fail(HH_ERR_DEVICE, "norm launch failed: %s", hipGetErrorString(e));
    return read_norms(c, out);
}

// HH_ERR_SINGULAR when an operator that right-hand sides 0..batch-1 use is
// singular to working precision; HH_ERR_NOMEM when a failed replacement of the
// operators left the plan without device tables.
static int check_operators(const hh_plan *p, int batch) {
    if (p->lost) return fail(HH_ERR_NOMEM, "the plan lost its operators' tables when replacing them failed; set them again");
    const int used = batch < p->nop ? batch : p->nop;
    for (int o = 0; o < used; o++)
        if (p->ms.singular[o])
            return fail(HH_ERR_SINGULAR, "operator %d is singular to working precision (a mode's condition "
                                         "estimate %.3g exceeds %.0e): k^2 is at or next to an eigenvalue",
                        o, p->ms.kappa_worst[o], hh::HH_SINGULAR_KAPPA);
    return HH_OK;
}

// hh_solve with the context lock held.
// A solve on workspace `scratch` (hh_plan_workspace_bytes(p, batch) bytes:
// the context's scratch, a graph's own workspace or the caller's).
static int solve_ws(hh_plan *p, const void *rhs, void *sol, int batch, void *scratch) {
    hh_context *c = p->ctx;
    int rc;
    const long n = hh_plan_field_size(p) * batch;
    if (p->prec == HH_PREC_F64) {
        void *ws = (plan_all_fft(p) && (p->dim == 3 || p->tile_w == 0)) ? nullptr : scratch;
        return solve_core(p, 0, 0, 0, 0, rhs, sol, ws, batch);
    }
    // mixed: FP32 transforms, storage and elimination of the well-separated
    // modes, FP64 substitution of the near-resonant ones, FP64 residual and
    // update; the correction lives in FP32 scratch, followed (2D) by the
    // FP32 mode-tiled spectrum of the solves
    // (or, with a dense DST, the FP32 intermediate of its out-of-place passes)
    void *dlt = scratch;
    const bool own_ws = !plan_all_fft(p) || (p->dim == 2 && p->tile_w != 0);
    void *tws = own_ws ? (void *)((char *)scratch + (size_t)n * 8) : dlt;
    if (rhs == sol) return fail(HH_ERR_ARG, "mixed precision solve needs d_sol != d_rhs");
    if ((rc = solve_core(p, 0, 1, 0, 1, rhs, sol, tws, batch))) return rc;   // u0 = A32^{-1} F
    if (p->tol == 0) {
        // fixed number of sweeps: no norms, no host synchronisation, so the
        // whole solve can be recorded into a HIP graph
        // (each sweep: r = A u - F, then u -= A32^{-1} r with the update
        // applied by the last DST pass as it stores)
        for (int it = 0; it < p->max_iter; it++) {
            if ((rc = residual_into(p, sol, rhs, dlt, 1, batch))) return rc;
            if ((rc = solve_core(p, 1, 1, 0, 1, dlt, sol, tws, batch, -1.0))) return rc;
        }
        p->last_sweeps = p->max_iter;
        p->last_rel = -1.0;
        return HH_OK;
    }
    int sweeps = 0;
    double rel = 0;
    for (;;) {
        // r = A u - F with FP64 arithmetic, stored in FP32 (its norm only
        // needs a few digits; the correction it drives is an FP32 solve)
        double nrf[2];   // max |r|, max |F|
        if ((rc = residual_into(p, sol, rhs, dlt, 1, batch, nrf))) return rc;
        rel = nrf[0] / (nrf[1] > 0 ? nrf[1] : 1.0);
        if (rel <= p->tol || sweeps >= p->max_iter) break;
        if ((rc = solve_core(p, 1, 1, 0, 1, dlt, sol, tws, batch, -1.0))) return rc;   // u -= A32^{-1} r
        sweeps++;
    }
    p->last_sweeps = sweeps;
    p->last_rel = rel;
    return HH_OK;
}

static int solve_locked(hh_plan *p, const void *rhs, void *sol, int batch) {
    hh_context *c = p->ctx;
    int rc = check_operators(p, batch);
    if (rc) return rc;
    if ((rc = set_device(c))) return rc;
    size_t ws_bytes = hh_plan_workspace_bytes(p, batch);
    if (ws_bytes && (rc = ensure_scratch(c, ws_bytes))) return rc;
    return solve_ws(p, rhs, sol, batch, c->scratch);
}

// One right-hand side of a batch whose right-hand side b uses operator b, FP64:
// the same bits as in the batch.
int hh::solve_one(hh_plan *p, int op, const void *rhs, void *sol) {
    if (!p || !rhs || !sol || op < 0 || op >= p->nop || p->prec != HH_PREC_F64)
        return fail(HH_ERR_ARG, "internal: bad single solve");
    hh_context *c = p->ctx;
    std::lock_guard<std::mutex> lk(c->mu);
    if (p->lost) return check_operators(p, 1);
    if (p->ms.singular[op]) return fail(HH_ERR_SINGULAR, "operator %d is singular to working precision", op);
    int rc = set_device(c);
    if (rc) return rc;
    const size_t ws_bytes = hh_plan_workspace_bytes(p, 1);
    if (ws_bytes && (rc = ensure_scratch(c, ws_bytes))) return rc;
    void *ws = (plan_all_fft(p) && (p->dim == 3 || p->tile_w == 0)) ? nullptr : c->scratch;
    return solve_core(p, 0, 0, 0, 0, rhs, sol, ws, 1, 0, op);
}

extern "C" int hh_solve_noalloc(hh_plan *p, const void *rhs, void *sol, int batch) {
    if (!p || !rhs || !sol) return fail(HH_ERR_ARG, "hh_solve_noalloc: null argument");
    if (batch < 1) return fail(HH_ERR_ARG, "hh_solve_noalloc: batch must be >= 1 (got %d)", batch);
    hh_context *c = p->ctx;
    std::lock_guard<std::mutex> lk(c->mu);
    int rc = check_operators(p, batch);
    if (rc) return rc;
    if ((rc = set_device(c))) return rc;
    if (!c->noalloc_ws)
        return fail(HH_ERR_DEVICE, "hh_solve_noalloc: no address for the static workspace on device %d: %s", c->device,
                    hipGetErrorString(c->noalloc_status));
    const size_t ws = hh_plan_workspace_bytes(p, batch);
    if (ws > HH_NOALLOC_BYTES)
        return fail(HH_ERR_UNSUPPORTED, "hh_solve_noalloc: the solve needs %zu bytes of workspace, above the %zu of "
                                        "its static workspace (use hh_solve, or a smaller batch)",
                    ws, HH_NOALLOC_BYTES);
    c->no_alloc = true;
    Range range("hh_solve_noalloc");
    rc = solve_ws(p, rhs, sol, batch, c->noalloc_ws);
    c->no_alloc = false;
    return rc;
}

extern "C" int hh_solve(hh_plan *p, const void *rhs, void *sol, int batch) {
    if (!p || !rhs || !sol) return fail(HH_ERR_ARG, "hh_solve: null argument");
    if (batch < 1) return fail(HH_ERR_ARG, "hh_solve: batch must be >= 1 (got %d)", batch);
    std::lock_guard<std::mutex> lk(p->ctx->mu);
    Range range("hh_solve");
    return solve_locked(p, rhs, sol, batch);
}

// ------------------------------------------------------------------ graphs
struct hh_graph {
    hh_context *ctx = nullptr;
    hipGraph_t graph = nullptr;
    hipGraphExec_t exec = nullptr;
    int nodes = 0;
    // the graph's own workspace: later solves on the context may grow (and
    // move) the context's scratch, never this
    void *ws = nullptr;
    size_t ws_bytes = 0;
    // plans and their generations at capture: a plan changed since (tables
    // reallocated, band kind, operator count or shapes) refuses the replay
    std::vector<std::pair<hh_plan *, long>> plans;
};

// Builds every table a plan's solves read (twiddles or DST matrices) so
// that recording a solve needs no allocation or synchronous copy.
static int prepare_tables(hh_plan *p) {
    hh_context *c = p->ctx;
    const int tc = p->prec == HH_PREC_F64 ? 0 : 1;
    const int lens[2] = {p->Nx, p->dim == 3 ? p->Ny : 0};
    for (int N : lens) {
        if (N <= 0) continue;
        void *t = nullptr;
        int rc;
        if (hh::fft_supported(N))
            rc = (dst_algo_for(c, N) & 1) == 0 ? get_half_table(c, N, tc, &t) : get_twiddles(c, N, tc, &t);
        else rc = get_dst_matrix(c, N, tc, &t);
        if (rc) return rc;
    }
    return HH_OK;
}

// Branch (0 or 1) of each solve of a graph.  Solves that touch no buffer of one
// another are independent and run on two parallel branches, so that the
// launches and latencies of small grids lie beside a large one's memory
// traffic: each solve goes to the branch with less work so far, largest
// first.  63 .. 2047 squared x 6: 890 -> 810 us; 300, 511, 1023 squared x 2: 160 ->
// 111.  As soon as one solve's result is another's input or result, all keep the
// caller's order on one branch.
//
// Short lists keep one branch too.  Two solves whose lighter one is short lose
// (63, 100 squared: 36 -> 44; 255, 300 squared x 3, 3 MB: 68 and 67).  Of three
// and more, one branch takes about 15 us a solve and 3.5 us a MB, two take at
// least 45 us and 9 a solve, whatever its size; the line lies where these meet.
// Below it, one and two branches: 3 x 63 squared 54 and 69 to 76 us; 40, 63, 100
// squared 47 and 74; 5 x 63 squared 86 and 100; 4 x 100 squared x 8 71 and 79;
// 3 x 255 squared 68 and 72.  Above: 8 x 127 squared 148 and 125; 3 x 300 squared
// x 2 95 and 77; 80, 255, 640 squared 106 and 81.  Of 130 lists two were up to 14
// us slower than one above the line (6 x 100 squared x 2) and up to 10 us faster
// below it (6 x 127 squared).
//
// one_workspace: every solve that needs one on the same branch.
static std::vector<int> graph_branches(int nsolves, hh_plan *const *plans, void *const *d_rhs, void *const *d_sol,
                                       const int *batch, bool one_workspace) {
    std::vector<int> branch(nsolves, 0);
    std::vector<size_t> bytes(nsolves);
    for (int i = 0; i < nsolves; i++) bytes[i] = (size_t)hh_plan_field_size(plans[i]) * batch[i] * 16;
    auto meet = [&](const void *a, size_t na, const void *b, size_t nb) {
        return (const char *)a < (const char *)b + nb && (const char *)b < (const char *)a + na;
    };
    for (int i = 0; i < nsolves; i++)
        for (int j = 0; j < nsolves; j++)
            if (j != i && (meet(d_sol[i], bytes[i], d_rhs[j], bytes[j]) || meet(d_sol[i], bytes[i], d_sol[j], bytes[j])))
                return branch;
    std::vector<int> by(nsolves);
    for (int i = 0; i < nsolves; i++) by[i] = i;
    std::stable_sort(by.begin(), by.end(), [&](int a, int b) { return bytes[a] > bytes[b]; });
    size_t load[2] = {0, 0};
    auto bound = [&](int i) { return one_workspace && hh_plan_workspace_bytes(plans[i], batch[i]) > 0; };
    for (int i : by)
        if (bound(i)) load[0] += bytes[i];
    for (int i : by) {
        if (bound(i)) continue;
        branch[i] = load[1] < load[0];
        load[branch[i]] += bytes[i];
    }
    const size_t mib = (size_t)1 << 20;
    const bool few = nsolves == 2 ? std::min(load[0], load[1]) < 4 * mib : load[0] + load[1] + nsolves * (mib + 3 * mib / 4) < 12 * mib;
    if (few) branch.assign(nsolves, 0);
    return branch;
}

extern "C" int hh_graph_create(hh_context *c, int nsolves, hh_plan *const *plans, void *const *d_rhs,
                               void *const *d_sol, const int *batch, hh_graph **out) {
    if (!c || !out || nsolves < 1 || !plans || !d_rhs || !d_sol || !batch)
        return fail(HH_ERR_ARG, "hh_graph_create: bad arguments");
    std::lock_guard<std::mutex> lk(c->mu);
    int rc = set_device(c);
    if (rc) return rc;
    size_t part[2] = {0, 0};   // workspace of each branch
    for (int i = 0; i < nsolves; i++) {
        hh_plan *p = plans[i];
        if (!p || !d_rhs[i] || !d_sol[i] || batch[i] < 1) return fail(HH_ERR_ARG, "hh_graph_create: bad solve %d", i);
        if (p->ctx != c) return fail(HH_ERR_ARG, "hh_graph_create: plan %d belongs to another context", i);
        if (p->prec == HH_PREC_MIXED && p->tol != 0)
            return fail(HH_ERR_UNSUPPORTED, "hh_graph_create: mixed-precision plan %d needs fixed sweeps "
                                            "(hh_plan_set_refine(plan, 0, sweeps))", i);
        if ((rc = check_operators(p, batch[i]))) return rc;
        if ((rc = prepare_tables(p))) return rc;
    }
    // Under a memory budget a graph takes no more than its solves would one after
    // the other: what a second workspace took would be refused to a later solve.
    std::vector<int> branch = graph_branches(nsolves, plans, d_rhs, d_sol, batch, c->budget > 0);
    auto workspace = [&]() {
        part[0] = part[1] = 0;
        for (int i = 0; i < nsolves; i++)
            part[branch[i]] = std::max(part[branch[i]], hh_plan_workspace_bytes(plans[i], batch[i]));
        if (part[1] > 0) part[0] = (part[0] + 255) & ~(size_t)255;
        return part[0] + part[1];
    };
    size_t ws = workspace();
    void *gws = nullptr;
    if (ws && (rc = dev_alloc(c, &gws, ws))) {   // no room for two: one branch, one workspace
        if (part[0] == 0 || part[1] == 0) return rc;
        branch.assign(nsolves, 0);
        ws = workspace();
        if ((rc = dev_alloc(c, &gws, ws))) return rc;
    }
    auto drop_ws = [&]() { if (gws) dev_free(c, gws, ws); };
    if (hipStreamSynchronize(c->stream) != hipSuccess) {
        drop_ws();
        return fail(HH_ERR_DEVICE, "hh_graph_create: stream synchronisation failed");
    }
    hipStream_t cap = nullptr, side = nullptr;
    hipEvent_t fork = nullptr, join = nullptr;
    const bool two = std::count(branch.begin(), branch.end(), 1) > 0;
    hipError_t e = hipStreamCreateWithFlags(&cap, hipStreamNonBlocking);
    if (e == hipSuccess && two) e = hipStreamCreateWithFlags(&side, hipStreamNonBlocking);
    if (e == hipSuccess && two) e = hipEventCreateWithFlags(&fork, hipEventDisableTiming);
    if (e == hipSuccess && two) e = hipEventCreateWithFlags(&join, hipEventDisableTiming);
    auto drop_streams = [&]() {
        if (fork) (void)hipEventDestroy(fork);
        if (join) (void)hipEventDestroy(join);
        if (side) (void)hipStreamDestroy(side);
        if (cap) (void)hipStreamDestroy(cap);
    };
    if (e != hipSuccess) {
        drop_streams();
        drop_ws();
        return fail(HH_ERR_DEVICE, "hh_graph_create: %s", hipGetErrorString(e));
    }
    hipStream_t saved = c->stream;
    const bool timing = c->timing;
    c->stream = cap;
    c->timing = false;
    hipGraph_t g = nullptr;
    e = hipStreamBeginCapture(cap, hipStreamCaptureModeThreadLocal);
    if (e == hipSuccess) {
        if (two) e = hipEventRecord(fork, cap);
        if (two && e == hipSuccess) e = hipStreamWaitEvent(side, fork, 0);
        if (e != hipSuccess) rc = fail(HH_ERR_DEVICE, "graph capture failed: %s", hipGetErrorString(e));
        for (int i = 0; i < nsolves && rc == HH_OK; i++) {
            c->stream = branch[i] ? side : cap;
            rc = solve_ws(plans[i], d_rhs[i], d_sol[i], batch[i], (char *)gws + (branch[i] ? part[0] : 0));
        }
        hipError_t e2 = two ? hipEventRecord(join, side) : hipSuccess;
        if (two && e2 == hipSuccess) e2 = hipStreamWaitEvent(cap, join, 0);
        hipError_t e3 = hipStreamEndCapture(cap, &g);
        if (e2 == hipSuccess) e2 = e3;
        if (rc == HH_OK && e2 != hipSuccess) rc = fail(HH_ERR_DEVICE, "graph capture failed: %s", hipGetErrorString(e2));
    } else {
        rc = fail(HH_ERR_DEVICE, "hipStreamBeginCapture failed: %s", hipGetErrorString(e));
    }
    c->stream = saved;
    c->timing = timing;
    drop_streams();
    if (rc) {
        if (g) (void)hipGraphDestroy(g);
        drop_ws();
        return rc;
    }
    hipGraphExec_t x = nullptr;
    e = hipGraphInstantiate(&x, g, nullptr, nullptr, 0);
    if (e != hipSuccess) {
        (void)hipGraphDestroy(g);
        drop_ws();
        return fail(HH_ERR_DEVICE, "hipGraphInstantiate failed: %s", hipGetErrorString(e));
    }
    hh_graph *G = new hh_graph();
    G->ctx = c;
    G->graph = g;
    G->exec = x;
    G->ws = gws;
    G->ws_bytes = ws;
    for (int i = 0; i < nsolves; i++) G->plans.emplace_back(plans[i], plans[i]->gen);
    size_t nn = 0;
    if (hipGraphGetNodes(g, nullptr, &nn) == hipSuccess) G->nodes = (int)nn;
    *out = G;
    return HH_OK;
}

extern "C" int hh_graph_launch(hh_graph *G) {
    if (!G) return fail(HH_ERR_ARG, "hh_graph_launch: null graph");
    hh_context *c = G->ctx;
    std::lock_guard<std::mutex> lk(c->mu);
    int rc = set_device(c);
    if (rc) return rc;
    for (const auto &pg : G->plans)
        if (pg.first->gen != pg.second)
            return fail(HH_ERR_ARG, "hh_graph_launch: a plan of the graph changed since it was recorded "
                                    "(tables reallocated, band kind, operator count or shapes); record it again");
    Range range("hh_graph_launch");
    HIPCHK(hipGraphLaunch(G->exec, c->stream));
    return HH_OK;
}

extern "C" int hh_graph_num_nodes(const hh_graph *G) { return G ? G->nodes : 0; }

extern "C" int hh_graph_destroy(hh_graph *G) {
    if (!G) return HH_OK;
    (void)hipStreamSynchronize(G->ctx->stream);
    if (G->exec) (void)hipGraphExecDestroy(G->exec);
    if (G->graph) (void)hipGraphDestroy(G->graph);
    if (G->ws) dev_free(G->ctx, G->ws, G->ws_bytes);
    delete G;
    return HH_OK;
}

extern "C" int hh_plan_set_operators(hh_plan *p, int nop, const double *coef) {
    if (!p || !coef) return fail(HH_ERR_ARG, "hh_plan_set_operators: null argument");
    if (nop < 1 || nop > p->cap_nop)
        return fail(HH_ERR_ARG, "hh_plan_set_operators: %d operators, the plan holds at most %d", nop, p->cap_nop);
    std::lock_guard<std::mutex> lk(p->ctx->mu);
    return replace_operators(p, nop, coef, p->kappa_flag);
}

extern "C" int hh_solve_host(hh_plan *p, const double *h_rhs, double *h_sol, int batch) {
    if (!p || !h_rhs || !h_sol) return fail(HH_ERR_ARG, "hh_solve_host: null argument");
    if (batch < 1) return fail(HH_ERR_ARG, "hh_solve_host: batch must be >= 1 (got %d)", batch);
    hh_context *c = p->ctx;
    int rc = set_device(c);
    if (rc) return rc;
    size_t bytes = (size_t)hh_plan_field_size(p) * batch * 16;
    void *d_rhs = nullptr, *d_sol = nullptr;
    if ((rc = dev_alloc(c, &d_rhs, bytes))) return rc;
    if ((rc = dev_alloc(c, &d_sol, bytes))) { dev_free(c, d_rhs, bytes); return rc; }
    hipError_t e = hipMemcpyAsync(d_rhs, h_rhs, bytes, hipMemcpyHostToDevice, c->stream);
    if (e == hipSuccess) {
        rc = hh_solve(p, d_rhs, d_sol, batch);
        if (rc == HH_OK) {
            e = hipMemcpyAsync(h_sol, d_sol, bytes, hipMemcpyDeviceToHost, c->stream);
            if (e == hipSuccess) e = hipStreamSynchronize(c->stream);
        }
    }
    (void)hipStreamSynchronize(c->stream);
    dev_free(c, d_rhs, bytes);
    dev_free(c, d_sol, bytes);
    if (rc) return rc;
    if (e != hipSuccess) return fail(HH_ERR_DEVICE, "host transfer failed: %s", hipGetErrorString(e));
    return HH_OK;
}

extern "C" int hh_residual(hh_plan *p, const void *d_sol, const void *d_rhs, void *d_res, int batch) {
    if (!p || !d_sol || !d_rhs || !d_res) return fail(HH_ERR_ARG, "hh_residual: null argument");
    if (batch < 1) return fail(HH_ERR_ARG, "hh_residual: batch must be >= 1");
    int rc = set_device(p->ctx);
    if (rc) return rc;
    return residual_into(p, d_sol, d_rhs, d_res, 0, batch);
}

extern "C" int hh_dst_rows(hh_context *c, int N, long nrows, const void *in, void *out) {
    if (!c || !in || !out || N < 1 || nrows < 0) return fail(HH_ERR_ARG, "hh_dst_rows: bad arguments");
    if (nrows == 0) return HH_OK;
    if (!hh::fft_supported(N) && N > 4096)
        return fail(HH_ERR_UNSUPPORTED, "DST length %d too large for the dense path", N);
    std::lock_guard<std::mutex> lk(c->mu);
    int rc = set_device(c);
    if (rc) return rc;
    hh::Lines l = rows_lines(N, nrows);
    if (!hh::fft_supported(N) && in == out) {   // dense path is out of place
        if ((rc = ensure_scratch(c, (size_t)N * nrows * 16))) return rc;
        HIPCHK(hipMemcpyAsync(c->scratch, in, (size_t)N * nrows * 16, hipMemcpyDeviceToDevice, c->stream));
        return dst_pass(c, l, 0, 0, 0, c->scratch, out);
    }
    return dst_pass(c, l, 0, 0, 0, in, out);
}

extern "C" int hh_dst2d_layers(hh_context *c, int Nx, int Ny, long nlayers, const void *in, void *out) {
    if (!c || !in || !out || Nx < 1 || Ny < 1 || nlayers < 0) return fail(HH_ERR_ARG, "hh_dst2d_layers: bad arguments");
    if (nlayers == 0) return HH_OK;
    std::lock_guard<std::mutex> lk(c->mu);
    int rc = set_device(c);
    if (rc) return rc;
    hh::Lines lx = rows_lines(Nx, (long)Ny * nlayers), ly = cols_lines(Nx, Ny, nlayers);
    bool fx = hh::fft_supported(Nx), fy = hh::fft_supported(Ny);
    size_t bytes = (size_t)Nx * Ny * nlayers * 16;
    if (fx && fy) {
        if ((rc = dst_pass(c, lx, 0, 0, 0, in, out))) return rc;
        return dst_pass(c, ly, 0, 0, 0, out, out);
    }
    if ((rc = ensure_scratch(c, bytes))) return rc;
    if ((rc = dst_pass(c, lx, 0, 0, 0, in, c->scratch))) return rc;
    return dst_pass(c, ly, 0, 0, 0, c->scratch, out);
}

// compact (k^2)_y (2D_Program/partial_derivatives/4th_order_first_derivative.c:4-34)
static void k2_y_compact(int Ny, double hy, const double *k2e, const double *k2yb, std::vector<cd> &k2y) {
    k2y.resize(Ny);
    for (int j = 0; j < Ny; j++) k2y[j] = 3.0 * (ld(k2e, j + 2) - ld(k2e, j)) / hy;
    k2y[0] -= ld(k2yb, 0);
    k2y[Ny - 1] -= ld(k2yb, 1);
    compact_line(k2y, 4.0);
}

extern "C" int hh_rhs2d(hh_plan *p, int order, double hx, double hy, const void *f_e, const void *u_e,
                        const void *fy_b, const void *fxx_b, const void *fyy_b, const double *k2e, const double *k2yb,
                        void *F, int batch) {
    if (!p || p->dim != 2 || !f_e || !u_e || !k2e || !F || batch < 1) return fail(HH_ERR_ARG, "hh_rhs2d: bad arguments");
    if (order != 2 && order != 4 && order != 6) return fail(HH_ERR_ARG, "order must be 2, 4 or 6 (got %d)", order);
    if (order == 6 && (!fy_b || !fxx_b || !fyy_b)) return fail(HH_ERR_ARG, "hh_rhs2d: sixth order needs boundary data");
    hh_context *c = p->ctx;
    std::lock_guard<std::mutex> lk(c->mu);
    int rc = set_device(c);
    if (rc) return rc;
    const int Nx = p->Nx, Ny = p->Ny;
    // per-row k^2 and compact (k^2)_y
    const int nop = p->nop;
    size_t tbytes = (size_t)2 * Ny * nop * 16;
    if ((rc = ensure_scratch(c, tbytes))) return rc;
    // tables [op][j]: k^2 at the interior rows, then compact (k^2)_y
    std::vector<cd> tab(2 * (size_t)Ny * nop);
    std::vector<cd> k2y;
    int k2y_nonzero = 0;
    for (int o = 0; o < nop; o++) {
        const double *ke = k2e + 2 * (size_t)o * (Ny + 2);
        if (order == 6) k2_y_compact(Ny, hy, ke, k2yb ? k2yb + 4 * (size_t)o : nullptr, k2y);
        for (int j = 0; j < Ny; j++) {
            tab[(size_t)o * Ny + j] = ld(ke, j + 1);
            tab[(size_t)(nop + o) * Ny + j] = order == 6 ? k2y[j] : cd(0);
            if (order == 6 && k2y[j] != cd(0)) k2y_nonzero = 1;
        }
    }
    char *tb = (char *)c->scratch;
    HIPCHK(hipMemcpyAsync(tb, tab.data(), tbytes, hipMemcpyHostToDevice, c->stream));
    hh::Rhs2D r;
    r.order = order; r.Nx = Nx; r.Ny = Ny; r.batch = batch; r.hx = hx; r.hy = hy;
    r.k2y_nonzero = k2y_nonzero;
    r.f_e = f_e; r.u_e = u_e; r.fy_b = fy_b; r.fxx_b = fxx_b; r.fyy_b = fyy_b;
    r.k2c = tb; r.k2y = tb + (size_t)Ny * nop * 16; r.coef = p->coef64; r.nop = nop;
    TimeScope ts(c, 4, (double)Nx * Ny * batch * 32);
    hipError_t e = hh::launch_rhs2d(r, F, c->stream);
    if (e != hipSuccess) return fail(HH_ERR_DEVICE, "rhs2d launch failed: %s", hipGetErrorString(e));
    // the host table must outlive the asynchronous copy
    HIPCHK(hipStreamSynchronize(c->stream));
    return HH_OK;
}

extern "C" int hh_rhs3d(hh_plan *p, int order, double hx, double hy, double hz, const void *f_e, const void *u_e,
                        const void *fxx_f, const void *fyy_f, const void *fzz_f, const double *k2e, const double *k2d,
                        void *F, int batch) {
    if (!p || p->dim != 3 || !f_e || !u_e || !k2e || !F || batch < 1) return fail(HH_ERR_ARG, "hh_rhs3d: bad arguments");
    if (order != 2 && order != 4 && order != 6) return fail(HH_ERR_ARG, "order must be 2, 4 or 6 (got %d)", order);
    if (order == 6 && (!fxx_f || !fyy_f || !fzz_f)) return fail(HH_ERR_ARG, "hh_rhs3d: sixth order needs face data");
    hh_context *c = p->ctx;
    std::lock_guard<std::mutex> lk(c->mu);
    int rc = set_device(c);
    if (rc) return rc;
    const int Nx = p->Nx, Ny = p->Ny, Nz = p->Nz;
    size_t wbytes = order == 6 ? (size_t)Nx * Ny * Nz * batch * 16 : 0;
    const int nop = p->nop;
    size_t tbytes = (size_t)(2 * Nz + 2) * nop * 16;
    if ((rc = ensure_scratch(c, wbytes + tbytes))) return rc;
    // tables [op]: k^2 on the extended z grid, then compact (k^2)_z
    // (derivative_kz_4th_order, 4th_order_partials.c:296-340)
    std::vector<cd> tab((2 * (size_t)Nz + 2) * nop);
    std::vector<cd> kz(Nz);
    for (int o = 0; o < nop; o++) {
        const double *ke = k2e + 2 * (size_t)o * (Nz + 2);
        const double *kd = k2d ? k2d + 8 * (size_t)o : nullptr;
        for (int l = 0; l < Nz + 2; l++) tab[(size_t)o * (Nz + 2) + l] = ld(ke, l);
        for (int l = 0; l < Nz; l++) kz[l] = 3.0 * (ld(ke, l + 2) - ld(ke, l)) / hz;
        kz[0] -= ld(kd, 0);
        kz[Nz - 1] -= ld(kd, 1);
        compact_line(kz, 4.0);
        for (int l = 0; l < Nz; l++) tab[(size_t)nop * (Nz + 2) + (size_t)o * Nz + l] = kz[l];
    }
    char *tb = (char *)c->scratch + wbytes;
    HIPCHK(hipMemcpyAsync(tb, tab.data(), tbytes, hipMemcpyHostToDevice, c->stream));
    hh::Rhs3D r;
    r.order = order; r.Nx = Nx; r.Ny = Ny; r.Nz = Nz; r.batch = batch; r.hx = hx; r.hy = hy; r.hz = hz;
    r.f_e = f_e; r.u_e = u_e; r.fxx_f = fxx_f; r.fyy_f = fyy_f; r.fzz_f = fzz_f;
    r.k2e = tb; r.kz = tb + (size_t)(Nz + 2) * nop * 16; r.coef = p->coef64; r.nop = nop; r.work = c->scratch;
    TimeScope ts(c, 4, (double)Nx * Ny * Nz * batch * 32);
    hipError_t e = hh::launch_rhs3d(r, F, c->stream);
    if (e != hipSuccess) return fail(HH_ERR_DEVICE, "rhs3d launch failed: %s", hipGetErrorString(e));
    HIPCHK(hipStreamSynchronize(c->stream));
    return HH_OK;
}

extern "C" int hh_norms(hh_context *c, long n, const void *x, const void *y, double out[2]) {
    if (!c || !out || n < 0 || (n > 0 && !x)) return fail(HH_ERR_ARG, "hh_norms: bad arguments");
    if (n == 0) { out[0] = out[1] = 0.0; return HH_OK; }   // norms of an empty vector (x may be null)
    std::lock_guard<std::mutex> lk(c->mu);
    int rc = set_device(c);
    if (rc) return rc;
    return norms_sync(c, n, x, y, out);
}

extern "C" int hh_norms_l2(hh_context *c, long n, const void *x, const void *y, double out[2]) {
    if (!c || !out || n < 0 || (n > 0 && !x)) return fail(HH_ERR_ARG, "hh_norms_l2: bad arguments");
    if (n == 0) { out[0] = out[1] = 0.0; return HH_OK; }   // norms of an empty vector (x may be null)
    std::lock_guard<std::mutex> lk(c->mu);
    int rc = set_device(c);
    if (rc) return rc;
    return norms_sync(c, n, x, y, out, true);
}
