// C ABI of libwiremom: context, geometry, fill, LU, sweeps and the drop-in
// entry points with the reference program's names.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <memory>
#include <string>
#include <unordered_map>
#include <vector>

#include "wm_front.h"
#include "wm_gmres.h"
#include "wm_internal.h"

namespace wm {

static thread_local char g_err[1024] = "";

void set_error(const char *fmt, ...)
{
    va_list ap;
    va_start(ap, fmt);
    std::vsnprintf(g_err, sizeof g_err, fmt, ap);
    va_end(ap);
}

int DevBuf::ensure(size_t need)
{
    if (bytes >= need && ptr) return WM_OK;
    if (ptr) {
        (void)hipDeviceSynchronize();
        (void)hipFree(ptr);
        ptr = nullptr;
        bytes = 0;
    }
    const size_t sz = std::max(need, (size_t)4096);
    if (hipMalloc(&ptr, sz) != hipSuccess) {
        ptr = nullptr;
        set_error("device allocation of %zu bytes failed", sz);
        return WM_ERR_NOMEM;
    }
    bytes = sz;
    return WM_OK;
}

void DevBuf::release()
{
    if (ptr) (void)hipFree(ptr);
    ptr = nullptr;
    bytes = 0;
}

int copy_h2d(void *dst, const void *src, size_t bytes, hipStream_t s)
{
    WM_HIP_TRY(hipStreamSynchronize(s));
    WM_HIP_TRY(hipMemcpy(dst, src, bytes, hipMemcpyHostToDevice));
    return WM_OK;
}

int copy_d2h(void *dst, const void *src, size_t bytes, hipStream_t s)
{
    WM_HIP_TRY(hipStreamSynchronize(s));
    WM_HIP_TRY(hipMemcpy(dst, src, bytes, hipMemcpyDeviceToHost));
    return WM_OK;
}

// Rows of `cols` 16-byte words from one pitch to another.
__global__ void k_repitch(uint4 *dst, size_t dpitch, const uint4 *src, size_t spitch, size_t cols, size_t rows)
{
    const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t < cols * rows) dst[t / cols * dpitch + t % cols] = src[t / cols * spitch + t % cols];
}

// A matrix between the host (rows without gaps) and a pitched device array.
// hipMemcpy2D moves pageable rows one by one, 9 us each whatever their length
// (1023 rows of 16 KB: 9.3 ms); here whole chunks of rows cross in one copy each
// and a kernel gives them their pitch: 1.9 ms.  False: not a case of this.
static bool copy2d_staged(void *dst, size_t dpitch, const void *src, size_t spitch, size_t width, size_t height,
                          hipStream_t s, bool to_device, int *rc)
{
    constexpr size_t kChunk = (size_t)64 << 20;  // staging bytes
    const size_t hpitch = to_device ? spitch : dpitch, pitch = to_device ? dpitch : spitch;
    const uintptr_t dev = (uintptr_t)(to_device ? dst : src);
    if (height < 2 || hpitch != width || width == 0 || width % 16 != 0 || pitch % 16 != 0 || dev % 16 != 0) return false;
    const size_t rows = std::max<size_t>(1, std::min(height, kChunk / width));
    void *stage = nullptr;
    if (hipMalloc(&stage, rows * width) != hipSuccess) {
        (void)hipGetLastError();
        return false;
    }
    auto run = [&]() -> int {
        for (size_t r = 0; r < height; r += rows) {
            const size_t k = std::min(rows, height - r), words = k * width / 16;
            const dim3 grid((unsigned)((words + 255) / 256));
            if (to_device) {
                WM_HIP_TRY(hipMemcpyAsync(stage, (const char *)src + r * width, k * width, hipMemcpyHostToDevice, s));
                hipLaunchKernelGGL(k_repitch, grid, dim3(256), 0, s, (uint4 *)((char *)dst + r * pitch), pitch / 16,
                                   (const uint4 *)stage, width / 16, width / 16, k);
            } else {
                hipLaunchKernelGGL(k_repitch, grid, dim3(256), 0, s, (uint4 *)stage, width / 16,
                                   (const uint4 *)((const char *)src + r * pitch), pitch / 16, width / 16, k);
                WM_HIP_TRY(hipMemcpyAsync((char *)dst + r * width, stage, k * width, hipMemcpyDeviceToHost, s));
            }
            WM_HIP_TRY(hipGetLastError());
            WM_HIP_TRY(hipStreamSynchronize(s));
        }
        return WM_OK;
    };
    *rc = run();
    (void)hipFree(stage);
    return true;
}

int copy2d_h2d(void *dst, size_t dpitch, const void *src, size_t spitch, size_t width, size_t height, hipStream_t s)
{
    WM_HIP_TRY(hipStreamSynchronize(s));
    int rc = WM_OK;
    if (copy2d_staged(dst, dpitch, src, spitch, width, height, s, true, &rc)) return rc;
    WM_HIP_TRY(hipMemcpy2D(dst, dpitch, src, spitch, width, height, hipMemcpyHostToDevice));
    return WM_OK;
}

int copy2d_d2h(void *dst, size_t dpitch, const void *src, size_t spitch, size_t width, size_t height, hipStream_t s)
{
    WM_HIP_TRY(hipStreamSynchronize(s));
    int rc = WM_OK;
    if (copy2d_staged(dst, dpitch, src, spitch, width, height, s, false, &rc)) return rc;
    WM_HIP_TRY(hipMemcpy2D(dst, dpitch, src, spitch, width, height, hipMemcpyDeviceToHost));
    return WM_OK;
}

static hipEvent_t prof_event(wm_ctx *ctx)
{
    if (!ctx->prof.pool.empty()) {
        hipEvent_t e = ctx->prof.pool.back();
        ctx->prof.pool.pop_back();
        return e;
    }
    hipEvent_t e = nullptr;
    (void)hipEventCreate(&e);
    return e;
}

void prof_begin(wm_ctx *ctx, int k, hipStream_t s)
{
    if (!ctx->prof.on) return;
    ProfRec r;
    r.a = prof_event(ctx);
    r.b = nullptr;
    r.flops = r.bytes = 0;
    (void)hipEventRecord(r.a, s);
    ctx->prof.rec[k].push_back(r);
}

void prof_end(wm_ctx *ctx, int k, hipStream_t s, double flops, double bytes)
{
    if (!ctx->prof.on || ctx->prof.rec[k].empty()) return;
    ProfRec &r = ctx->prof.rec[k].back();
    r.b = prof_event(ctx);
    r.flops = flops;
    r.bytes = bytes;
    (void)hipEventRecord(r.b, s);
}

int check_device_error(wm_ctx *ctx, hipStream_t s)
{
    int h = 0;
    WM_TRY(copy_d2h(&h, ctx->d_err, sizeof(int), s));
    if (h != 0) {
        const int zero = 0;
        (void)hipMemcpy(ctx->d_err, &zero, sizeof(int), hipMemcpyHostToDevice);
        set_error("a bounded device-side wait expired (code %d)", h);
        return WM_ERR_SPIN;
    }
    return WM_OK;
}

}  // namespace wm

using namespace wm;

namespace {

constexpr double kPi = 3.14159265358979323846;
constexpr double kCspeed = 2.99792448E+8;  // "wersja referencyjna/Wire_MoM.cu":5

double wavenumber(float freq_mhz)  // Wire_MoM.cu:338-340 (frequency in MHz, float32)
{
    const double ambda = kCspeed / (double)freq_mhz * 1E-6;
    return (kPi + kPi) / ambda;
}

int round_up(int v, int m) { return (v + m - 1) / m * m; }

// Smith (1962) complex division.
wm_c128 cdiv(wm_c128 a, wm_c128 b)
{
    wm_c128 q;
    if (std::fabs(b.re) >= std::fabs(b.im)) {
        const double t = b.im / b.re, d = b.re + b.im * t;
        q.re = (a.re + a.im * t) / d;
        q.im = (a.im - a.re * t) / d;
    } else {
        const double t = b.re / b.im, d = b.im + b.re * t;
        q.re = (a.re * t + a.im) / d;
        q.im = (a.im * t - a.re) / d;
    }
    return q;
}

__global__ void k_pad_identity(double2 *A, int lda, int64_t stride, int n0, int n)
{
    // sets rows/columns n0..n-1 of an n x n matrix to the identity
    const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int b = blockIdx.y;
    const int64_t total = (int64_t)n * n;
    if (idx >= total) return;
    const int i = (int)(idx % n), j = (int)(idx / n);
    if (i < n0 && j < n0) return;
    A[(size_t)b * stride + i + (size_t)j * lda] = make_double2(i == j ? 1.0 : 0.0, 0.0);
}

__global__ void k_add_diag_list(double2 *A, int lda, const int *idx, const double2 *val, int n)
{
    // A[i][i] += val for the listed (distinct) indices
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= n) return;
    const size_t o = (size_t)idx[t] * lda + idx[t];
    double2 a = A[o];
    a.x += val[t].x;
    a.y += val[t].y;
    A[o] = a;
}

__global__ void k_zero_c128(double2 *p, int64_t n)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = make_double2(0.0, 0.0);
}

std::mutex g_default_mu;
wm_ctx *g_default_ctx = nullptr;

wm_ctx *default_ctx()
{
    std::lock_guard<std::mutex> lk(g_default_mu);
    if (!g_default_ctx) {
        int dev = 0;
        if (const char *e = std::getenv("WM_DEVICE")) dev = std::atoi(e);
        if (wm_init(dev, &g_default_ctx) != WM_OK) {
            std::fprintf(stderr, "libwiremom: %s\n", wm_last_error());
            g_default_ctx = nullptr;
        }
    }
    return g_default_ctx;
}

struct DevMem {
    void *p = nullptr;
    ~DevMem()
    {
        if (p) (void)hipFree(p);
    }
    int alloc(size_t bytes)
    {
        if (hipMalloc(&p, bytes) != hipSuccess) {
            p = nullptr;
            set_error("device allocation of %zu bytes failed", bytes);
            return WM_ERR_NOMEM;
        }
        return WM_OK;
    }
};

}  // namespace

namespace {

// Value of "key": <int> in a JSON line, or false.
bool json_int(const char *line, const char *key, long *out)
{
    char pat[64];
    std::snprintf(pat, sizeof pat, "\"%s\":", key);
    const char *p = std::strstr(line, pat);
    if (!p) return false;
    p += std::strlen(pat);
    char *end = nullptr;
    const long v = std::strtol(p, &end, 10);
    if (end == p) return false;
    *out = v;
    return true;
}

// Value of "key": "<string>" in a JSON line, or empty.
std::string json_str(const char *line, const char *key)
{
    char pat[64];
    std::snprintf(pat, sizeof pat, "\"%s\":", key);
    const char *p = std::strstr(line, pat);
    if (!p) return std::string();
    p += std::strlen(pat);
    while (*p == ' ') ++p;
    if (*p != '"') return std::string();
    const char *q = std::strchr(++p, '"');
    return q ? std::string(p, q) : std::string();
}

}  // namespace

extern "C" {

const char *wm_last_error(void) { return g_err; }
const char *wm_version(void) { return "libwiremom 0.1 (gfx950)"; }

int wm_init(int device, wm_ctx **out)
{
    if (!out) { set_error("wm_init: null out"); return WM_ERR_ARG; }
    int ndev = 0;
    WM_HIP_TRY(hipGetDeviceCount(&ndev));
    if (device < 0 || device >= ndev) {
        set_error("wm_init: device %d not present (%d devices)", device, ndev);
        return WM_ERR_ARG;
    }
    WM_HIP_TRY(hipSetDevice(device));
    auto *c = new wm_ctx();
    c->device = device;
    hipDeviceProp_t p;
    WM_HIP_TRY(hipGetDeviceProperties(&p, device));
    c->num_cu = p.multiProcessorCount;
    c->hbm_bytes = p.totalGlobalMem;
    c->max_lds = p.sharedMemPerBlock;
    std::snprintf(c->name, sizeof c->name, "%s (%s)", p.name, p.gcnArchName);
    std::snprintf(c->arch, sizeof c->arch, "%s", p.gcnArchName);
    if (char *colon = std::strchr(c->arch, ':')) *colon = 0;  // "gfx950:sramecc+:xnack-" -> "gfx950"
    WM_HIP_TRY(hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking));
    WM_HIP_TRY(hipMalloc(&c->d_sync, sizeof(int) * wm_ctx::kSyncCap));
    WM_HIP_TRY(hipMalloc(&c->d_err, sizeof(int)));
    WM_HIP_TRY(hipMalloc(&c->d_tag, sizeof(uint32_t)));
    WM_HIP_TRY(hipMemset(c->d_tag, 0, sizeof(uint32_t)));
    WM_HIP_TRY(hipMemset(c->d_sync, 0, sizeof(int) * wm_ctx::kSyncCap));
    WM_HIP_TRY(hipMemset(c->d_err, 0, sizeof(int)));
    WM_TRY(noalloc_init(device));
    WM_TRY(panel_gate_join(c));
    *out = c;
    return WM_OK;
}

int wm_shutdown(wm_ctx *c)
{
    if (!c) return WM_OK;
    (void)hipSetDevice(c->device);
    (void)hipStreamSynchronize(c->stream);
    if (c->aux) (void)hipStreamSynchronize(c->aux);
    if (c->lu_side) (void)hipStreamSynchronize(c->lu_side);
    panel_gate_leave(c);
    drop_graphs(c);
    c->ws_info.release();
    c->ws_fill.release();
    c->ws_fill2.release();
    c->ws_lu.release();
    c->ws_solve.release();
    c->ws_perm.release();
    c->ws_resid.release();
    c->ws_sweep.release();
    c->ws_group.release();
    c->ws_dinv.release();
    c->ws_dinv_idx.release();
    (void)hipFree(c->d_sync);
    (void)hipFree(c->d_err);
    (void)hipFree(c->d_tag);
    for (auto e : c->aux_ev)
        if (e) (void)hipEventDestroy(e);
    if (c->aux) (void)hipStreamDestroy(c->aux);
    for (auto e : c->lu_ev)
        if (e) (void)hipEventDestroy(e);
    if (c->lu_side) (void)hipStreamDestroy(c->lu_side);
    if (c->lu_done) (void)hipEventDestroy(c->lu_done);
    (void)hipStreamDestroy(c->stream);
    if (c == g_default_ctx) g_default_ctx = nullptr;
    delete c;
    return WM_OK;
}

// FP64 factorization kernels are "panel", "swap_trsm", "gemm"; complex64 ones carry "_f32".
static const char *kClassNames[K_NCLASS] = {"fill", "panel", "swap_trsm", "gemm", "trsv", "resid",
                                            "panel_f32", "swap_trsm_f32", "gemm_f32", "gemm_bf16x3"};

int wm_prof_enable(wm_ctx *c, int on)
{
    if (!c) return WM_ERR_ARG;
    std::lock_guard<std::recursive_mutex> lk(c->mu);
    WM_HIP_TRY(hipStreamSynchronize(c->stream));
    for (auto &v : c->prof.rec) {
        for (auto &r : v) {
            if (r.a) c->prof.pool.push_back(r.a);
            if (r.b) c->prof.pool.push_back(r.b);
        }
        v.clear();
    }
    c->prof.on = on != 0;
    return WM_OK;
}

int wm_prof_get(wm_ctx *c, const char *kernel, double *ms, int64_t *launches, double *flops, double *bytes)
{
    if (!c || !kernel) return WM_ERR_ARG;
    std::lock_guard<std::recursive_mutex> lk(c->mu);
    WM_HIP_TRY(hipStreamSynchronize(c->stream));
    for (int k = 0; k < K_NCLASS; ++k) {
        if (std::strcmp(kernel, kClassNames[k]) != 0) continue;
        double t = 0, f = 0, b = 0;
        int64_t n = 0;
        for (auto &r : c->prof.rec[k]) {
            if (!r.b) continue;
            float e = 0;
            WM_HIP_TRY(hipEventElapsedTime(&e, r.a, r.b));
            t += e;
            f += r.flops;
            b += r.bytes;
            ++n;
        }
        if (ms) *ms = t;
        if (launches) *launches = n;
        if (flops) *flops = f;
        if (bytes) *bytes = b;
        return WM_OK;
    }
    set_error("wm_prof_get: unknown kernel class %s", kernel);
    return WM_ERR_ARG;
}

int wm_sync(wm_ctx *c)
{
    if (!c) return WM_ERR_ARG;
    WM_HIP_TRY(hipStreamSynchronize(c->stream));
    return check_device_error(c, c->stream);
}

int wm_device_info(wm_ctx *c, char *name, int name_len, int *num_cu, size_t *hbm)
{
    if (!c) return WM_ERR_ARG;
    if (name && name_len > 0) std::snprintf(name, name_len, "%s", c->name);
    if (num_cu) *num_cu = c->num_cu;
    if (hbm) *hbm = c->hbm_bytes;
    return WM_OK;
}

int wm_dev_alloc(wm_ctx *c, size_t bytes, void **ptr)
{
    if (!c || !ptr) return WM_ERR_ARG;
    (void)hipSetDevice(c->device);
    if (hipMalloc(ptr, bytes) != hipSuccess) {
        *ptr = nullptr;
        set_error("wm_dev_alloc: %zu bytes failed", bytes);
        return WM_ERR_NOMEM;
    }
    return WM_OK;
}

int wm_dev_free(wm_ctx *c, void *ptr)
{
    if (!c) return WM_ERR_ARG;
    WM_HIP_TRY(hipStreamSynchronize(c->stream));
    if (ptr) WM_HIP_TRY(hipFree(ptr));
    return WM_OK;
}

int wm_memcpy_h2d(wm_ctx *c, void *dst, const void *src, size_t bytes)
{
    if (!c) return WM_ERR_ARG;
    return copy_h2d(dst, src, bytes, c->stream);
}

int wm_memcpy_d2h(wm_ctx *c, void *dst, const void *src, size_t bytes)
{
    if (!c) return WM_ERR_ARG;
    return copy_d2h(dst, src, bytes, c->stream);
}

int wm_memcpy_d2d(wm_ctx *c, void *dst, const void *src, size_t bytes)
{
    if (!c) return WM_ERR_ARG;
    (void)hipSetDevice(c->device);
    WM_HIP_TRY(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToDevice, c->stream));
    WM_HIP_TRY(hipStreamSynchronize(c->stream));
    return WM_OK;
}

// ---- geometry -------------------------------------------------------------------
namespace {

// The fill's row tables (wm_geom): rows 0..ld-1 cut into runs of at most 64 rows
// with at most 64 distinct observation points (equal coordinates and segment key).
struct FillRows {
    std::vector<int> wrow, pkey, slots;
    std::vector<double> pts;
};

void fill_rows(const std::vector<double> &obs, const std::vector<int> &okey, int nkeys, int npls, int ld, FillRows &t)
{
    struct Pt {
        double r[3];
        int key;
    };
    std::vector<Pt> cur;
    t.slots.assign(ld, 0);
    t.wrow.assign(1, 0);
    auto point = [&](int m, int h) {
        Pt p;
        for (int d = 0; d < 3; ++d) p.r[d] = obs[(size_t)(6 * h + d) * ld + m];
        p.key = okey[(size_t)h * ld + m];
        return p;
    };
    // where a key's point lies in the run, as far as cur agrees; two points with one key
    // (rows whose peak is not a node of their segment) are searched for
    std::vector<int> at(nkeys, -1);
    auto same = [&](const Pt &q, const Pt &p) { return q.key == p.key && std::memcmp(q.r, p.r, sizeof p.r) == 0; };
    auto find = [&](const Pt &p) {
        const int a = at[p.key];
        if (a < 0 || a >= (int)cur.size() || cur[a].key != p.key) return -1;
        if (same(cur[a], p)) return a;
        for (int i = (int)cur.size() - 1; i >= 0; --i)
            if (same(cur[i], p)) return i;
        return -1;
    };
    auto close = [&](int row_end) {
        const size_t w = t.wrow.size() - 1;
        t.pts.resize((w + 1) * 3 * 64);
        t.pkey.resize((w + 1) * 64);
        for (int l = 0; l < 64; ++l) {  // lanes without a point repeat one, with no segment's key
            const bool own = l < (int)cur.size();
            const Pt p = own ? cur[l] : cur.empty() ? point(0, 0) : cur[0];
            for (int d = 0; d < 3; ++d) t.pts[(w * 3 + d) * 64 + l] = p.r[d];
            t.pkey[w * 64 + l] = own ? p.key : -1;
        }
        t.wrow.push_back(row_end);
        cur.clear();
    };
    for (int m = 0; m < ld; ++m) {
        int slot[2] = {0, 0};
        for (int pass = 0; pass < 2; ++pass) {  // pass 1: the row opens a new run
            const size_t had = cur.size();
            if (m < npls)
                for (int h = 0; h < 2; ++h) {
                    const Pt p = point(m, h);
                    slot[h] = find(p);
                    if (slot[h] < 0) {
                        at[p.key] = slot[h] = (int)cur.size();
                        cur.push_back(p);
                    }
                }
            if (cur.size() <= 64 && m - t.wrow.back() < 64) break;
            cur.resize(had);
            close(m);
        }
        t.slots[m] = slot[0] | slot[1] << 8;
    }
    close(ld);
}

}  // namespace

int wm_geom_create(wm_ctx *c, const float *x, const float *y, const float *z, const float *rad, const int *ipc,
                   const int *ips, const int *ise, int nsmax, int npls, wm_geom **out)
{
    return wm_geom_create_env(c, x, y, z, rad, ipc, ips, ise, nsmax, npls, 1, 1.f, 1.f, 1.f, 1.f, out);
}

int wm_geom_create_env(wm_ctx *c, const float *x, const float *y, const float *z, const float *rad, const int *ipc,
                       const int *ips, const int *ise, int nsmax, int npls, int ienv, float sgnx, float sgny,
                       float sgnz, float sgnenv, wm_geom **out)
{
    if (!c || !x || !y || !z || !rad || !ipc || !ips || !ise || !out || npls <= 0 || nsmax < npls) {
        set_error("wm_geom_create: bad arguments");
        return WM_ERR_ARG;
    }
    if (ienv != 1 && ienv != 2) {
        set_error("wm_geom_create: ienv must be 1 (free space) or 2 (PEC ground), got %d", ienv);
        return WM_ERR_ARG;
    }
    std::lock_guard<std::recursive_mutex> lk(c->mu);
    (void)hipSetDevice(c->device);
    const int ld = round_up(npls, 128);
    std::vector<double> obs((size_t)12 * ld, 0.0), src((size_t)16 * ld, 0.0), img;
    std::vector<int> okey((size_t)2 * ld, -1), skey((size_t)4 * ld, -2), ikey;
    const bool pec = ienv == 2;
    if (pec) {
        img.assign((size_t)16 * ld, 0.0);
        ikey.assign((size_t)2 * ld, -3);
    }
    const double sg[3] = {(double)sgnx, (double)sgny, (double)sgnz};
    std::unordered_map<long long, int> keys;  // unordered node pair -> segment key
    keys.reserve((size_t)2 * npls);
    auto seg_key = [&](int s) {
        const int a = ise[s - 1], b = ise[s - 1 + nsmax];
        const long long k = (long long)std::min(a, b) << 32 | (unsigned)std::max(a, b);
        auto it = keys.find(k);
        if (it != keys.end()) return it->second;
        const int id = (int)keys.size();
        keys.emplace(k, id);
        return id;
    };
    auto node = [&](int id, double r[3]) { r[0] = x[id - 1]; r[1] = y[id - 1]; r[2] = z[id - 1]; };
    for (int p = 0; p < npls; ++p) {
        const int mp = std::abs(ipc[p]);
        const int s1 = ips[p], s2 = ips[p + nsmax];
        if (mp < 1 || s1 < 1 || s2 < 1 || s1 > nsmax || s2 > nsmax) {
            set_error("wm_geom_create: basis %d has invalid topology", p);
            return WM_ERR_GEOMETRY;
        }
        double P[3], F1[3], F2[3];
        node(mp, P);
        node(ise[s1 - 1], F1);             // first node of segment s1
        node(ise[s2 - 1 + nsmax], F2);     // second node of segment s2
        for (int d = 0; d < 3; ++d) {
            const double rc1 = 0.5 * (P[d] + F1[d]);
            const double rc2 = 0.5 * (F2[d] + P[d]);
            obs[(size_t)d * ld + p] = rc1;
            obs[(size_t)(3 + d) * ld + p] = P[d] - rc1;
            obs[(size_t)(6 + d) * ld + p] = rc2;
            obs[(size_t)(9 + d) * ld + p] = rc2 - P[d];
        }
        const int k1 = seg_key(s1), k2 = seg_key(s2);
        okey[p] = k1;
        okey[ld + p] = k2;
        skey[4 * p] = k1;
        skey[4 * p + 1] = k2;
        // source half 1: first node of s1 -> peak; half 2: peak -> second node of s2
        double *r = &src[(size_t)p * 16];
        const double *A[2] = {F1, P}, *B[2] = {P, F2};
        const int segs[2] = {s1, s2};
        for (int g = 0; g < 2; ++g) {
            const double rdx = B[g][0] - A[g][0], rdy = B[g][1] - A[g][1], rdz = B[g][2] - A[g][2];
            const double dl = std::sqrt(rdx * rdx + rdy * rdy + rdz * rdz);
            if (!(dl > 0.0) || !(rad[segs[g] - 1] > 0.f)) {
                set_error("wm_geom_create: basis %d half %d has zero length or radius", p, g + 1);
                return WM_ERR_GEOMETRY;
            }
            r[8 * g + 0] = A[g][0]; r[8 * g + 1] = A[g][1]; r[8 * g + 2] = A[g][2];
            r[8 * g + 3] = rdx / dl; r[8 * g + 4] = rdy / dl; r[8 * g + 5] = rdz / dl;
            r[8 * g + 6] = dl;
            r[8 * g + 7] = (double)rad[segs[g] - 1];
            if (pec) {
                // image half (cwire1_im / cwire2_im, "wersja referencyjna/Zmatrix.cpp":342-446,
                // 559-663): coordinates scaled by the signs, so the start point and the unit
                // vector flip in the mirrored axes and dl stays; the self rule applies to it
                // when both nodes of its segment lie in the plane (Zmatrix.cpp:384)
                double *q = &img[(size_t)p * 16];
                for (int d = 0; d < 3; ++d) {
                    q[8 * g + d] = sg[d] * r[8 * g + d];
                    q[8 * g + 3 + d] = sg[d] * r[8 * g + 3 + d];
                }
                q[8 * g + 6] = r[8 * g + 6];
                q[8 * g + 7] = r[8 * g + 7];
                const int s = segs[g], na = ise[s - 1], nb = ise[s - 1 + nsmax];
                if ((double)z[na - 1] < 1.e-6 && (double)z[nb - 1] < 1.e-6) ikey[2 * p + g] = skey[4 * p + g];
            }
        }
    }
    for (int p = npls; p < ld; ++p) {  // padding: finite dummy data, overwritten by the identity
        double *r = &src[(size_t)p * 16];
        for (int g = 0; g < 2; ++g) { r[8 * g + 3] = 1.0; r[8 * g + 6] = 1.0; r[8 * g + 7] = 1.0; }
        if (pec) {
            double *q = &img[(size_t)p * 16];
            for (int g = 0; g < 2; ++g) { q[8 * g + 3] = 1.0; q[8 * g + 6] = 1.0; q[8 * g + 7] = 1.0; }
        }
        for (int d = 0; d < 12; ++d) obs[(size_t)d * ld + p] = 1.0e3;
    }
    // first halves that are not the previous basis's second half (same record,
    // key and image): along a wire the fill evaluates each segment once
    for (int p = 0; p < ld; ++p) {
        bool same = p > 0 && p < npls && skey[4 * p] == skey[4 * (p - 1) + 1] &&
                    std::memcmp(&src[(size_t)p * 16], &src[(size_t)(p - 1) * 16 + 8], 8 * sizeof(double)) == 0;
        if (pec && same)
            same = ikey[2 * p] == ikey[2 * (p - 1) + 1] &&
                   std::memcmp(&img[(size_t)p * 16], &img[(size_t)(p - 1) * 16 + 8], 8 * sizeof(double)) == 0;
        skey[4 * p + 2] = same ? 0 : 1;
        skey[4 * p + 3] = 0;
    }
    FillRows fr;
    fill_rows(obs, okey, (int)keys.size(), npls, ld, fr);
    // diameter of the structure (with its image over the PEC ground): the
    // bounding-box diagonal of every source half
    double lo[3] = {HUGE_VAL, HUGE_VAL, HUGE_VAL}, hi[3] = {-HUGE_VAL, -HUGE_VAL, -HUGE_VAL};
    for (int p = 0; p < npls; ++p)
        for (int h = 0; h < (pec ? 4 : 2); ++h) {
            const double *r8 = (h < 2 ? &src[(size_t)p * 16] : &img[(size_t)p * 16]) + 8 * (h & 1);
            for (int d = 0; d < 3; ++d)
                for (int e = 0; e < 2; ++e) {
                    const double v = r8[d] + (e ? r8[6] * r8[3 + d] : 0.0);
                    lo[d] = std::min(lo[d], v);
                    hi[d] = std::max(hi[d], v);
                }
        }
    double diam = 0.0;
    for (int d = 0; d < 3 && npls > 0; ++d) diam += (hi[d] - lo[d]) * (hi[d] - lo[d]);
    auto *g = new wm_geom();
    g->ctx = c;
    g->npls = npls;
    g->ld = ld;
    g->diam = std::sqrt(diam);
    g->h_src = src;
    g->ienv = ienv;
    g->sgnenv = (double)sgnenv;
    std::unique_ptr<wm_geom, int (*)(wm_geom *)> guard(g, wm_geom_destroy);
    g->nwaves = (int)fr.wrow.size() - 1;
    // One allocation, and the small tables in one copy: an allocation and a copy per
    // table cost 116 us for a dipole of 15 unknowns and 672 for 3000 over ground,
    // this 63 and 320 (the latter with segment keys hashed and points looked up by key).
    struct Table {
        void **dev;
        const void *host;
        size_t bytes, off;
    };
    size_t total = 0;
    auto table = [&](auto *&dev, const auto &v) {
        const Table t{(void **)&dev, v.data(), v.size() * sizeof(v[0]), total};
        total += (t.bytes + 255) & ~(size_t)255;
        return t;
    };
    std::vector<Table> small, large;
    small.push_back(table(g->d_wrow, fr.wrow));
    small.push_back(table(g->d_slots, fr.slots));
    small.push_back(table(g->d_pkey, fr.pkey));
    small.push_back(table(g->d_src_key, skey));
    if (pec) small.push_back(table(g->d_img_key, ikey));
    small.push_back(table(g->d_pts, fr.pts));
    const size_t small_b = total;
    large.push_back(table(g->d_obs, obs));
    large.push_back(table(g->d_src, src));
    if (pec) large.push_back(table(g->d_img, img));
    if (hipMalloc(&g->d_tables, total) != hipSuccess) {
        (void)hipGetLastError();
        g->d_tables = nullptr;
        set_error("wm_geom_create: device allocation failed");
        return WM_ERR_NOMEM;
    }
    std::vector<char> stage(small_b);
    for (const Table &t : small) std::memcpy(stage.data() + t.off, t.host, t.bytes);
    WM_HIP_TRY(hipMemcpy(g->d_tables, stage.data(), small_b, hipMemcpyHostToDevice));
    for (const Table &t : large)
        WM_HIP_TRY(hipMemcpy((char *)g->d_tables + t.off, t.host, t.bytes, hipMemcpyHostToDevice));
    for (const auto *l : {&small, &large})
        for (const Table &t : *l) *t.dev = (char *)g->d_tables + t.off;
    (void)guard.release();
    *out = g;
    return WM_OK;
}

int wm_geom_load(wm_ctx *c, const char *geo_path, const char *wirefile, wm_geom **out)
{
    return wm_geom_load_env(c, geo_path, wirefile, 1, out);
}

int wm_geom_load_env(wm_ctx *c, const char *geo_path, const char *wirefile, int ienv, wm_geom **out)
{
    if (ienv != 1 && ienv != 2) {
        set_error("wm_geom_load: ienv must be 1 (free space) or 2 (PEC ground), got %d", ienv);
        return WM_ERR_ARG;
    }
    GeoInput gi;
    int rc = geo_read(geo_path, gi);
    if (rc != WM_OK) {
        set_error("wm_geom_load: cannot read %s", geo_path ? geo_path : "(null)");
        return rc;
    }
    Topology t;
    std::string text;
    const bool want = wirefile && wirefile[0];
    rc = configwire_build(gi, ienv, kNsmax, kNwmax, t, want ? &text : nullptr);
    if (rc != WM_OK) {
        set_error("wm_geom_load: segmentation of %s failed (capacity or topology)", geo_path);
        return rc;
    }
    if (want) {
        FILE *f = std::fopen(wirefile, "wb");
        if (!f) { set_error("cannot write %s", wirefile); return WM_ERR_IO; }
        std::fwrite(text.data(), 1, text.size(), f);
        std::fclose(f);
    }
    // the reference's signs for its two environments ("wersja referencyjna/Wire_MoM.cu":107-122)
    const float sz = ienv == 2 ? -1.f : 1.f;
    return wm_geom_create_env(c, t.x.data(), t.y.data(), t.z.data(), t.rad.data(), t.ipc.data(), t.ips.data(),
                              t.ise.data(), t.nsmax, t.npls, ienv, 1.f, 1.f, sz, sz, out);
}

int wm_geom_destroy(wm_geom *g)
{
    if (!g) return WM_OK;
    if (g->d_tables) (void)hipFree(g->d_tables);
    delete g;
    return WM_OK;
}

int wm_geom_npls(const wm_geom *g) { return g ? g->npls : WM_ERR_ARG; }
int wm_geom_ld(const wm_geom *g) { return g ? g->ld : WM_ERR_ARG; }

// ---- fill / LU / solve on device buffers -------------------------------------------
int wm_zfill(wm_ctx *c, const wm_geom *g, int nfreq, const double *ka, wm_c128 *Z, int64_t strideZ, wm_c64 *Z32,
             int64_t strideZ32)
{
    if (!c || !g) return WM_ERR_ARG;
    std::lock_guard<std::recursive_mutex> lk(c->mu);
    (void)hipSetDevice(c->device);
    return fill_launch(c, g, nfreq, ka, Z, strideZ, Z32, strideZ32, c->stream);
}

int wm_getrf_batched(wm_ctx *c, int prec, int n, void *A, int lda, int64_t strideA, int *ipiv, int64_t strideP,
                     int batch, int *info)
{
    if (!c) return WM_ERR_ARG;
    std::lock_guard<std::recursive_mutex> lk(c->mu);
    (void)hipSetDevice(c->device);
    // info words live in a context buffer, so repeated calls on the same
    // buffers replay one captured factorization
    WM_TRY(c->ws_info.ensure(sizeof(int) * std::max(batch, 1)));
    int *dinfo = (int *)c->ws_info.ptr;
    WM_TRY(getrf_batched(c, prec, n, A, lda, strideA, ipiv, strideP, batch, dinfo, c->stream));
    std::vector<int> h(batch);
    WM_TRY(check_device_error(c, c->stream));
    WM_TRY(copy_d2h(h.data(), dinfo, sizeof(int) * batch, c->stream));
    int first = 0;
    for (int b = 0; b < batch; ++b) {
        if (info) info[b] = h[b];
        if (h[b] && !first) first = h[b];
    }
    return first;
}

// ---- factorization tuning ---------------------------------------------------------------
namespace {

// Diagonally dominant test matrices for timing: entries in [-1, 1) from a hash
// of (member, i, j), n on the diagonal; complex128 (esz 16) or complex64.
__global__ void k_tune_fill(void *A, int n, int esz, int batch)
{
    const int64_t nn = (int64_t)n * n;
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= nn * batch) return;
    const int64_t b = t / nn, r = t % nn;
    const int i = (int)(r % n), j = (int)(r / n);
    uint32_t h = (uint32_t)(b * 2654435761u) ^ (uint32_t)(i * 40503u) ^ (uint32_t)(j * 69069u + 12345u);
    h ^= h >> 15;
    h *= 0x2c1b3c6du;
    h ^= h >> 12;
    const double x = (double)(h & 0xffff) / 32768.0 - 1.0, y = (double)(h >> 16) / 32768.0 - 1.0;
    const double d = (i == j) ? (double)n : 0.0;
    if (esz == 16) ((double2 *)A)[t] = make_double2(x + d, y);
    else ((float2 *)A)[t] = make_float2((float)(x + d), (float)y);
}

int valid_block(int panels)
{
    return panels == 0 || panels == 1 || panels == 2 || panels == 4 || panels == 8 || panels == 16;
}

}  // namespace

int wm_set_graphs(wm_ctx *c, int on)
{
    if (!c) return WM_ERR_ARG;
    std::lock_guard<std::recursive_mutex> lk(c->mu);
    (void)hipSetDevice(c->device);
    (void)hipStreamSynchronize(c->stream);
    c->use_graphs = on != 0;
    if (!on) drop_graphs(c);
    return WM_OK;
}

int wm_set_fill_overlap(wm_ctx *c, int on)
{
    if (!c) return WM_ERR_ARG;
    std::lock_guard<std::recursive_mutex> lk(c->mu);
    c->overlap_fill = on != 0;
    return WM_OK;
}

int wm_set_getrf_block(wm_ctx *c, int prec, int n, int panels)
{
    if (!c || prec < 0 || prec > 2 || n <= 0 || !valid_block(panels)) {
        set_error("wm_set_getrf_block: bad arguments (panels must be 0, 1, 2, 4, 8 or 16)");
        return WM_ERR_ARG;
    }
    std::lock_guard<std::recursive_mutex> lk(c->mu);
    c->getrf_block[prec][std::min(n / 1024, wm_ctx::kTuneSizes - 1)] = panels;
    return WM_OK;
}

int wm_get_getrf_block(wm_ctx *c, int prec, int n)
{
    if (!c || prec < 0 || prec > 2 || n <= 0) return 0;
    std::lock_guard<std::recursive_mutex> lk(c->mu);
    return getrf_block(c, prec, n);
}

int wm_tune_getrf(wm_ctx *c, int prec, int n, int batch, int *best, double *ms_best)
{
    if (!c || prec < 0 || prec > 2 || n <= 0 || n % 64 != 0) {
        set_error("wm_tune_getrf: bad arguments (n must be a positive multiple of 64)");
        return WM_ERR_ARG;
    }
    std::lock_guard<std::recursive_mutex> lk(c->mu);
    (void)hipSetDevice(c->device);
    if (batch <= 0) batch = getrf_width(c, prec, n);
    const int esz = prec == WM_PREC_F64 ? 16 : 8;
    const int64_t nn = (int64_t)n * n;
    DevMem A, piv, info;
    WM_TRY(A.alloc((size_t)nn * batch * esz));
    WM_TRY(piv.alloc((size_t)n * batch * sizeof(int)));
    WM_TRY(info.alloc((size_t)batch * sizeof(int)));
    hipEvent_t e0, e1;
    WM_HIP_TRY(hipEventCreate(&e0));
    WM_HIP_TRY(hipEventCreate(&e1));
    int &slot = c->getrf_block[prec][std::min(n / 1024, wm_ctx::kTuneSizes - 1)];
    const int saved = slot;
    int bestp = 0;
    float bestms = 0.f;
    int rc = WM_OK;
    const unsigned nb = (unsigned)((nn * batch + 255) / 256);
    for (int panels : {1, 2, 4, 8, 16}) {
        if (panels > 1 && panels * 64 > n) break;
        slot = panels;
        float ms = 0.f;
        for (int rep = 0; rep < 2 && rc == WM_OK; ++rep) {  // the first run warms up
            hipLaunchKernelGGL(k_tune_fill, dim3(nb), dim3(256), 0, c->stream, A.p, n, esz, batch);
            if (hipEventRecord(e0, c->stream) != hipSuccess) rc = WM_ERR_HIP;
            if (rc == WM_OK)
                rc = getrf_batched(c, prec, n, A.p, n, nn, (int *)piv.p, n, batch, (int *)info.p, c->stream);
            if (rc == WM_OK && hipEventRecord(e1, c->stream) != hipSuccess) rc = WM_ERR_HIP;
            if (rc == WM_OK && hipEventSynchronize(e1) != hipSuccess) rc = WM_ERR_HIP;
            if (rc == WM_OK && hipEventElapsedTime(&ms, e0, e1) != hipSuccess) rc = WM_ERR_HIP;
        }
        if (rc != WM_OK) break;
        if (bestp == 0 || ms < bestms) {
            bestp = panels;
            bestms = ms;
        }
    }
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    if (rc == WM_OK) rc = check_device_error(c, c->stream);
    slot = rc == WM_OK ? bestp : saved;
    if (rc != WM_OK) return rc;
    if (best) *best = bestp;
    if (ms_best) *ms_best = bestms;
    return WM_OK;
}

int wm_set_fill_freqs(wm_ctx *c, int ienv, int n, int freqs)
{
    if (!c || (ienv != 1 && ienv != 2) || n <= 0 || freqs < 0 || freqs > 4) {
        set_error("wm_set_fill_freqs: bad arguments (ienv 1 or 2, freqs 0-4)");
        return WM_ERR_ARG;
    }
    std::lock_guard<std::recursive_mutex> lk(c->mu);
    c->fill_freqs[ienv - 1][std::min(n / 1024, wm_ctx::kTuneSizes - 1)] = freqs;
    return WM_OK;
}

int wm_get_fill_freqs(wm_ctx *c, int ienv, int n)
{
    if (!c || (ienv != 1 && ienv != 2) || n <= 0) return 0;
    std::lock_guard<std::recursive_mutex> lk(c->mu);
    return c->fill_freqs[ienv - 1][std::min(n / 1024, wm_ctx::kTuneSizes - 1)];
}

int wm_tune_fill(wm_ctx *c, const wm_geom *g, int *best, double *ms_per_freq)
{
    if (!c || !g || g->ctx != c) {
        set_error("wm_tune_fill: bad arguments");
        return WM_ERR_ARG;
    }
    std::lock_guard<std::recursive_mutex> lk(c->mu);
    (void)hipSetDevice(c->device);
    const int ld = g->ld, nf = 4;
    const int64_t nn = (int64_t)ld * ld;
    // four wavenumbers of a low-frequency sweep (the fill's cost hardly depends on k)
    double ka[nf];
    for (int f = 0; f < nf; ++f) ka[f] = wavenumber_mhz(1.0f + 2.0f * f);
    DevMem Z;
    WM_TRY(Z.alloc((size_t)nn * nf * sizeof(double2)));
    hipEvent_t e0, e1;
    WM_HIP_TRY(hipEventCreate(&e0));
    WM_HIP_TRY(hipEventCreate(&e1));
    int &slot = c->fill_freqs[g->ienv == 2 ? 1 : 0][std::min(ld / 1024, wm_ctx::kTuneSizes - 1)];
    const int saved = slot;
    int bestf = 0, rc = WM_OK;
    float bestms = 0.f;
    for (int F = 1; F <= 4 && rc == WM_OK; ++F) {
        slot = F;
        float ms = 0.f;
        for (int rep = 0; rep < 2 && rc == WM_OK; ++rep) {  // the first run warms up
            if (hipEventRecord(e0, c->stream) != hipSuccess) rc = WM_ERR_HIP;
            if (rc == WM_OK) rc = fill_launch(c, g, nf, ka, Z.p, nn, nullptr, 0, c->stream);
            if (rc == WM_OK && hipEventRecord(e1, c->stream) != hipSuccess) rc = WM_ERR_HIP;
            if (rc == WM_OK && hipEventSynchronize(e1) != hipSuccess) rc = WM_ERR_HIP;
            if (rc == WM_OK && hipEventElapsedTime(&ms, e0, e1) != hipSuccess) rc = WM_ERR_HIP;
        }
        if (rc == WM_OK && (bestf == 0 || ms < bestms)) {
            bestf = F;
            bestms = ms;
        }
    }
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    if (rc == WM_OK) rc = check_device_error(c, c->stream);
    slot = rc == WM_OK ? bestf : saved;
    if (rc != WM_OK) return rc;
    if (best) *best = bestf;
    if (ms_per_freq) *ms_per_freq = bestms / nf;
    return WM_OK;
}


int wm_tune_save(wm_ctx *c, const char *path)
{
    if (!c || !path) {
        set_error("wm_tune_save: bad arguments");
        return WM_ERR_ARG;
    }
    std::lock_guard<std::recursive_mutex> lk(c->mu);
    FILE *f = std::fopen(path, "w");
    if (!f) {
        set_error("wm_tune_save: cannot write %s", path);
        return WM_ERR_ARG;
    }
    int n = 0;
    for (int p = 0; p < 3; ++p)
        for (int sc = 0; sc < wm_ctx::kTuneSizes; ++sc)
            if (c->getrf_block[p][sc] > 0) {
                std::fprintf(f, "{\"arch\": \"%s\", \"knob\": \"getrf_block\", \"prec\": %d, \"size_class\": %d, "
                                "\"value\": %d}\n", c->arch, p, sc, c->getrf_block[p][sc]);
                ++n;
            }
    for (int e = 0; e < 2; ++e)
        for (int sc = 0; sc < wm_ctx::kTuneSizes; ++sc)
            if (c->fill_freqs[e][sc] > 0) {
                std::fprintf(f, "{\"arch\": \"%s\", \"knob\": \"fill_freqs\", \"ienv\": %d, \"size_class\": %d, "
                                "\"value\": %d}\n", c->arch, e + 1, sc, c->fill_freqs[e][sc]);
                ++n;
            }
    const bool ok = std::fclose(f) == 0;
    if (!ok) {
        set_error("wm_tune_save: write to %s failed", path);
        return WM_ERR_ARG;
    }
    return n;
}

int wm_tune_load(wm_ctx *c, const char *path)
{
    if (!c || !path) {
        set_error("wm_tune_load: bad arguments");
        return WM_ERR_ARG;
    }
    std::lock_guard<std::recursive_mutex> lk(c->mu);
    FILE *f = std::fopen(path, "r");
    if (!f) {
        set_error("wm_tune_load: cannot read %s", path);
        return WM_ERR_ARG;
    }
    char line[512];
    int applied = 0;
    while (std::fgets(line, sizeof line, f)) {
        if (json_str(line, "arch") != c->arch) continue;
        const std::string knob = json_str(line, "knob");
        long sc = -1, v = -1, k = -1;
        if (!json_int(line, "size_class", &sc) || !json_int(line, "value", &v) || sc < 0 ||
            sc >= wm_ctx::kTuneSizes)
            continue;
        if (knob == "getrf_block" && json_int(line, "prec", &k) && k >= 0 && k <= 2 && valid_block((int)v) && v > 0) {
            c->getrf_block[k][sc] = (int)v;
            ++applied;
        } else if (knob == "fill_freqs" && json_int(line, "ienv", &k) && (k == 1 || k == 2) && v >= 1 && v <= 4) {
            c->fill_freqs[k - 1][sc] = (int)v;
            ++applied;
        }
    }
    std::fclose(f);
    return applied;
}

int wm_getrs_batched(wm_ctx *c, int prec, int n, int nrhs, const void *A, int lda, int64_t strideA, const int *ipiv,
                     int64_t strideP, wm_c128 *B, int ldb, int64_t strideB, int batch)
{
    if (!c) return WM_ERR_ARG;
    std::lock_guard<std::recursive_mutex> lk(c->mu);
    (void)hipSetDevice(c->device);
    WM_TRY(getrs_batched(c, prec, n, nrhs, A, lda, strideA, ipiv, strideP, B, ldb, strideB, batch, c->stream));
    return check_device_error(c, c->stream);
}

void wm_solve_opts_default(wm_solve_opts *o)
{
    if (!o) return;
    o->prec = WM_PREC_F64;
    o->max_iter = 20;
    o->tol = 1e-12;
    o->batch = 0;
    o->hbm_fraction = 0.8;
    o->fallback_f64 = 1;
    o->size_policy = 1;
    o->cond_est = 0;
    o->recycle = 0.0;
}

}  // extern "C"

extern "C" {

namespace {

// Solves the items of one geometry (one per frequency) in batches: FP64 sweeps
// as wide as the HBM budget allows, mixed sweeps highest frequency first with
// routing (see below).
constexpr int kBlindBatch = 16;  // first batch of a mixed sweep (the top quarter of a 64-point sweep)

// Anchors of a recycled batch: f (MHz, descending) gets anchor[i], the index of
// the frequency whose factors precondition it (itself for an anchor).  The
// covering factor at f, for r: while the structure is electrically small
// (k D <= 1, D its diameter) r^(1 + log10(1 / (k D))), i.e. one more power of
// r per decade below k D = 1 (quasi-static: Z(f) ~ jwL + P/(jw), whose two
// parts the anchor's factors capture at any distance, so GMRES converges in a
// few steps however far the anchor); above, 1 + (r - 1) / (k D), where the
// resonances between an anchor and its neighbours lengthen GMRES.  It does not
// grow with f, so a frequency between an anchor and the highest frequency it
// covers is covered as well.  Greedy interval cover in log f: the anchor of
// the highest uncovered frequency is the lowest one within its factor, and it
// covers every frequency down to its own factor below.
void choose_anchors(const float *f, int cnt, double r, double diam, int *anchor)
{
    auto radius = [&](float x) {
        const double kd = wavenumber_mhz(x) * diam;
        if (kd > 1.0) return 1.0 + (r - 1.0) / kd;
        return std::pow(r, 1.0 - std::log10(std::max(kd, 1e-12)));
    };
    for (int i = 0; i < cnt;) {
        int a = i;
        while (a + 1 < cnt && (double)f[i] <= radius(f[i]) * (double)f[a + 1]) ++a;
        int k = i;
        while (k < cnt && (double)f[a] <= radius(f[a]) * (double)f[k]) anchor[k++] = a;
        i = k;
    }
}

// Recycled sweep: frequencies highest first in batches as wide as the HBM
// budget allows; in each batch the anchors of choose_anchors.
int run_sweep_recycled(wm_ctx *c, const wm_geom *g, const wm_solve_opts &o, std::vector<WorkItem> &items, int nrhs)
{
    const int nfreq = (int)items.size();
    std::stable_sort(items.begin(), items.end(), [](const WorkItem &a, const WorkItem &b) { return a.freq > b.freq; });
    int batch = o.batch;
    if (batch <= 0) {
        size_t freeb = 0, total = 0;
        if (hipMemGetInfo(&freeb, &total) != hipSuccess) freeb = c->hbm_bytes / 2;
        const double frac = o.hbm_fraction > 0 && o.hbm_fraction <= 1 ? o.hbm_fraction : 0.8;
        const size_t per = item_bytes(g->ld, nrhs, WM_PREC_F64) + gmres_bytes(g->ld, nrhs, kGmresRestart);
        batch = (int)std::max<size_t>(1, (size_t)(frac * (double)(freeb + c->ws_sweep.bytes)) / per);
        batch = std::min(batch, 128);
    }
    int status = WM_OK;
    for (int f0 = 0; f0 < nfreq;) {
        const int cnt = std::min(batch, nfreq - f0);
        WorkItem *it = items.data() + f0;
        std::vector<float> fr(cnt);
        std::vector<int> anc(cnt);
        for (int i = 0; i < cnt; ++i) fr[i] = it[i].freq;
        choose_anchors(fr.data(), cnt, o.recycle, g->diam, anc.data());
        for (int i = 0; i < cnt; ++i) it[i].anchor = anc[i];
        const int rc = solve_items(c, o, it, cnt, c->stream);
        if (rc < 0) return rc;
        if (rc != WM_OK && status == WM_OK) status = rc;
        f0 += cnt;
    }
    return status;
}

int run_sweep(wm_ctx *c, const wm_geom *g, const wm_solve_opts &o, std::vector<WorkItem> &items, int nrhs)
{
    if (o.recycle > 1.0) return run_sweep_recycled(c, g, o, items, nrhs);
    const int nfreq = (int)items.size();
    int batch = o.batch > 0 ? o.batch : auto_batch(c, g->ld, nrhs, o.prec, o.hbm_fraction);
    int status = WM_OK;
    const bool mixed = o.prec != WM_PREC_F64;
    if (mixed) {
        // Highest frequencies first: their refinement rates, recorded on the
        // geometry (cleared here), route the lower ones, whose conditioning is
        // worse, to FP64 factors when refinement cannot reach tol in max_iter.
        std::stable_sort(items.begin(), items.end(), [](const WorkItem &a, const WorkItem &b) { return a.freq > b.freq; });
        std::lock_guard<std::mutex> lk(g->rate_mu);
        g->rate_obs.clear();
    }
    int f0 = 0;
    while (f0 < nfreq) {
        int cnt = std::min(batch, nfreq - f0);
        if (mixed) {
            // Mixed sweeps go in batches at most mixed_width wide, so that each
            // batch is routed with the rates of the frequencies just above it,
            // and cut where the routed precision changes: a run of frequencies
            // that all route to FP64 factors (the lower ones once refinement
            // stops converging) goes as one batch, whose members share the
            // panel launches.
            const int w = std::min(cnt, mixed_width(c, g->ld));
            if (o.size_policy && prefer_f64(c, o.prec, g->ld, w)) {
                for (int b = f0; b < f0 + w; ++b) items[b].fprec = WM_PREC_F64;
                cnt = w;
            } else if (f0 > 0) {
                route_items(o, items.data() + f0, cnt);
                const bool f64 = items[f0].fprec == WM_PREC_F64;
                int run = 1;
                while (run < (f64 ? cnt : w) && (items[f0 + run].fprec == WM_PREC_F64) == f64) ++run;
                // a short complex64 run just above the FP64 ones joins their batch
                // when its own panel launches and refinement would cost more
                if (!f64 && run < cnt && items[f0 + run].fprec == WM_PREC_F64 && o.size_policy &&
                    join_f64(c, o.prec, g->ld, run)) {
                    for (int b = f0; b < f0 + run; ++b) items[b].fprec = WM_PREC_F64;
                    while (run < cnt && items[f0 + run].fprec == WM_PREC_F64) ++run;
                }
                cnt = run;
            } else {
                // the first batch is factored before any refinement rate of the
                // structure is known: at most kBlindBatch frequencies from the
                // top, however wide a launch is, so that frequencies far below
                // the top are not put into complex64 factors blindly
                cnt = std::min(w, kBlindBatch);
            }
        }
        const int rc = solve_items(c, o, items.data() + f0, cnt, c->stream);
        // refinement that did not converge without the FP64 fallback: the other
        // frequencies are still solved and the status is returned at the end
        if (rc < 0 && rc != WM_ERR_NOCONV) return rc;
        if (rc != WM_OK && status == WM_OK) status = rc;
        if (mixed) record_rates(items.data() + f0, cnt);
        f0 += cnt;
    }
    return status;
}

}  // namespace

// Internal test hook (not part of include/wiremom.h): the anchors of a recycled
// batch (choose_anchors) for frequencies in descending order, without a device.
extern "C" int wmx_choose_anchors(const float *f, int cnt, double r, double diam, int *anchor)
{
    if (!f || !anchor || cnt <= 0 || !(r > 1.0) || !(diam >= 0.0)) return WM_ERR_ARG;
    for (int i = 1; i < cnt; ++i)
        if (!(f[i] <= f[i - 1])) return WM_ERR_ARG;
    choose_anchors(f, cnt, r, diam, anchor);
    return WM_OK;
}

int wm_solve_sweep(wm_ctx *c, const wm_geom *g, const wm_solve_opts *opts, int nfreq, const float *freq_mhz, int nrhs,
                   const int *gaps, float ampl, float phas, wm_c128 *I, wm_c128 *zin, wm_freq_stats *st)
{
    if (!c || !g || nfreq <= 0 || !freq_mhz || nrhs <= 0 || !gaps) {
        set_error("wm_solve_sweep: bad arguments");
        return WM_ERR_ARG;
    }
    wm_solve_opts o;
    wm_solve_opts_default(&o);
    if (opts) o = *opts;
    std::lock_guard<std::recursive_mutex> lk(c->mu);
    (void)hipSetDevice(c->device);
    const int N = g->npls;
    std::vector<WorkItem> items(nfreq);
    for (int f = 0; f < nfreq; ++f) {
        WorkItem &w = items[f];
        w.g = g;
        w.freq = freq_mhz[f];
        w.nrhs = nrhs;
        w.gaps = gaps;
        w.ampl = ampl;
        w.phas = phas;
        w.I = I ? I + (size_t)f * nrhs * N : nullptr;
        w.zin = zin ? zin + (size_t)f * nrhs : nullptr;
        w.st = st ? st + f : nullptr;
    }
    return run_sweep(c, g, o, items, nrhs);
}

int wm_solve_sweep_ex(wm_ctx *c, const wm_geom *g, const wm_solve_opts *opts, int nfreq, const float *freq_mhz,
                      int nrhs, int nsrc, const wm_source *src, int npw, const wm_plane_wave *pw, int nload,
                      const wm_load *loads, wm_c128 *I, wm_c128 *zin, wm_freq_stats *st)
{
    if (!c || !g || nfreq <= 0 || !freq_mhz || nrhs <= 0 || nsrc < 0 || npw < 0 || nload < 0 || nsrc + npw == 0 ||
        (nsrc > 0 && !src) || (npw > 0 && !pw) || (nload > 0 && !loads)) {
        set_error("wm_solve_sweep_ex: bad arguments");
        return WM_ERR_ARG;
    }
    wm_solve_opts o;
    wm_solve_opts_default(&o);
    if (opts) o = *opts;
    std::lock_guard<std::recursive_mutex> lk(c->mu);
    (void)hipSetDevice(c->device);
    const int N = g->npls;
    std::vector<WorkItem> items(nfreq);
    for (int f = 0; f < nfreq; ++f) {
        WorkItem &w = items[f];
        w.g = g;
        w.freq = freq_mhz[f];
        w.nrhs = nrhs;
        w.src = src;
        w.nsrc = nsrc;
        w.pw = pw;
        w.npw = npw;
        w.loads = loads;
        w.nload = nload;
        w.I = I ? I + (size_t)f * nrhs * N : nullptr;
        w.zin = zin && nsrc > 0 ? zin + (size_t)f * nsrc : nullptr;
        w.st = st ? st + f : nullptr;
    }
    return run_sweep(c, g, o, items, nrhs);
}

// ---- drop-in entry points ------------------------------------------------------------------

void geoinp(int nnmax, int nwmax, int ntmax, int *nnod, float *xnod, float *ynod, float *znod, int *nw, int *iwn,
            float *wrad, int *nsw, int *nt, int *iwt)
{
    (void)ntmax;
    (void)iwt;
    const char *path = std::getenv("WM_GEO_PATH");
    if (!path || !path[0]) path = "dipol.geo";
    std::printf(" Nazwa pliku geo: %s\n", path);
    GeoInput g;
    if (geo_read(path, g) != WM_OK) {
        std::printf(" Nie udalo sie otworzyc pliku!\n");
        std::exit(0);
    }
    if (g.nnod > nnmax || g.nw > nwmax) {
        std::printf(" Przekroczona liczba wezlow lub drucikow w pliku geo\n");
        std::exit(0);
    }
    *nnod = g.nnod;
    *nw = g.nw;
    *nt = 0;
    for (int i = 1; i <= g.nnod; ++i) { xnod[i] = g.xnod[i]; ynod[i] = g.ynod[i]; znod[i] = g.znod[i]; }
    for (int i = 1; i <= g.nw; ++i) {
        iwn[i] = g.iwn[i];
        iwn[i + g.nw] = g.iwn[i + g.nw];
        wrad[i] = g.wrad[i];
        nsw[i] = g.nsw[i];
    }
}

void tablice(int npnt, int nseg, int nsmax, float *x, float *y, float *z, int nplsw, int *ise, int *isp, int *ips,
             int *ipc)
{
    (void)isp;
    const std::string text = tablice_text(npnt, nseg, nsmax, x, y, z, nplsw, ise, ips, ipc);
    if (FILE *f = std::fopen("tablice.txt", "wb")) {
        std::fwrite(text.data(), 1, text.size(), f);
        std::fclose(f);
    } else {
        std::fprintf(stderr, "tablice: cannot write tablice.txt\n");
    }
}

void configwire(int *npnt, int nnod, float *xnod, float *ynod, float *znod, float *x, float *y, float *z, int nw,
                int *iwn, float *wrad, int *nsw, int *ise, int *isp, int *ips, int *ipc, int *iwe, float *rad,
                int *nplsw, int *nseg, int nsmax, int nwmax, int ienv)
{
    GeoInput g;
    g.nnod = nnod;
    g.nw = nw;
    g.xnod.assign(xnod, xnod + nnod + 1);
    g.ynod.assign(ynod, ynod + nnod + 1);
    g.znod.assign(znod, znod + nnod + 1);
    g.iwn.assign(iwn, iwn + 2 * nw + 1);
    g.wrad.assign(wrad, wrad + nw + 1);
    g.nsw.assign(nsw, nsw + nw + 1);
    Topology t;
    std::string text;
    const int rc = configwire_build(g, ienv, nsmax, nwmax, t, &text);
    if (FILE *f = std::fopen("configwire.txt", "wb")) {
        std::fwrite(text.data(), 1, text.size(), f);
        std::fclose(f);
    }
    if (rc != WM_OK) {
        std::printf("\n Number of segments or basis functions exceeds the limits\n");
        std::exit(0);
    }
    *npnt = t.npnt;
    *nseg = t.nseg;
    *nplsw = t.npls;
    std::memcpy(x, t.x.data(), sizeof(float) * nsmax);
    std::memcpy(y, t.y.data(), sizeof(float) * nsmax);
    std::memcpy(z, t.z.data(), sizeof(float) * nsmax);
    std::memcpy(rad, t.rad.data(), sizeof(float) * nsmax);
    std::memcpy(ipc, t.ipc.data(), sizeof(int) * nsmax);
    std::memcpy(ise, t.ise.data(), sizeof(int) * 2 * nsmax);
    std::memcpy(isp, t.isp.data(), sizeof(int) * 2 * nsmax);
    std::memcpy(ips, t.ips.data(), sizeof(int) * 2 * nsmax);
    std::memcpy(iwe, t.iwe.data(), sizeof(int) * 2 * nsmax);
}

void config(int *npnt, int nnod, float *xnod, float *ynod, float *znod, float *x, float *y, float *z, int nw, int *iwn,
            float *wrad, int *nsw, int *ise, int *isp, int *ips, int *ipc, int *iwe, float *rad, int *npls, int *nplsw,
            int *nseg, int nsmax, int nwmax, int ienv)
{
    configwire(npnt, nnod, xnod, ynod, znod, x, y, z, nw, iwn, wrad, nsw, ise, isp, ips, ipc, iwe, rad, nplsw, nseg,
               nsmax, nwmax, ienv);
    *npls = *nplsw;
}

static int fill_to_host(wm_c128 *cz, float *x, float *y, float *z, float *rad, int *ipc, int *ips, int *ise,
                        int nsmax, double ka, int npls, int ienv, float sgnx, float sgny, float sgnz, float sgnenv)
{
    wm_ctx *c = default_ctx();
    if (!c) return WM_ERR_HIP;
    std::lock_guard<std::recursive_mutex> lk(c->mu);
    wm_geom *g = nullptr;
    WM_TRY(wm_geom_create_env(c, x, y, z, rad, ipc, ips, ise, nsmax, npls, ienv, sgnx, sgny, sgnz, sgnenv, &g));
    std::unique_ptr<wm_geom, int (*)(wm_geom *)> guard(g, wm_geom_destroy);
    DevMem Zd;
    WM_TRY(Zd.alloc((size_t)g->ld * g->ld * sizeof(double2)));
    WM_TRY(fill_launch(c, g, 1, &ka, Zd.p, 0, nullptr, 0, c->stream));
    return copy2d_d2h(cz, (size_t)npls * sizeof(wm_c128), Zd.p, (size_t)g->ld * sizeof(double2),
                      (size_t)npls * sizeof(wm_c128), npls, c->stream);
}

void zmatrix(wm_c128 *cz, float *x, float *y, float *z, int *ipc, int *ips, int *ise, float *rad, int npls, double ka,
             int nsmax, int ienv, float sgnx, float sgny, float sgnz, float sgnenv)
{
    if (fill_to_host(cz, x, y, z, rad, ipc, ips, ise, nsmax, ka, npls, ienv, sgnx, sgny, sgnz, sgnenv) != WM_OK)
        std::fprintf(stderr, "zmatrix: %s\n", wm_last_error());
}

void zmatrix_gpu(wm_c128 *cz_h, float *x_h, float *y_h, float *z_h, float *rad_h, int *ipc_h, int *ips_h, int *ise_h,
                 int nsmax, double ka, int npls, int ienv, float sgnx, float sgny, float sgnz, float sgnenv)
{
    if (fill_to_host(cz_h, x_h, y_h, z_h, rad_h, ipc_h, ips_h, ise_h, nsmax, ka, npls, ienv, sgnx, sgny, sgnz,
                     sgnenv) != WM_OK)
        std::fprintf(stderr, "zmatrix_gpu: %s\n", wm_last_error());
}

void zmatrix_gpu_rank(wm_c128 *cz_h, float *x_h, float *y_h, float *z_h, float *rad_h, int *ipc_h, int *ips_h,
                      int *ise_h, int nsmax, double ka, int npls, int ienv, float sgnx, float sgny, float sgnz,
                      float sgnenv, int rank)
{
    (void)rank;
    zmatrix_gpu(cz_h, x_h, y_h, z_h, rad_h, ipc_h, ips_h, ise_h, nsmax, ka, npls, ienv, sgnx, sgny, sgnz, sgnenv);
}

static int lu_solve_host(int n, int nrhs, wm_c128 *ci, const wm_c128 *cz)
{
    wm_ctx *c = default_ctx();
    if (!c) return WM_ERR_HIP;
    std::lock_guard<std::recursive_mutex> lk(c->mu);
    const int ld = round_up(n, 128);
    const hipStream_t s = c->stream;
    DevMem A, B, P, Inf;
    WM_TRY(A.alloc((size_t)ld * ld * sizeof(double2)));
    WM_TRY(B.alloc((size_t)ld * nrhs * sizeof(double2)));
    WM_TRY(P.alloc((size_t)ld * sizeof(int)));
    WM_TRY(Inf.alloc(sizeof(int)));
    WM_TRY(copy2d_h2d(A.p, (size_t)ld * sizeof(double2), cz, (size_t)n * sizeof(wm_c128),
                      (size_t)n * sizeof(wm_c128), n, s));
    const int64_t tot = (int64_t)ld * ld;
    hipLaunchKernelGGL(k_pad_identity, dim3((unsigned)((tot + 255) / 256), 1), dim3(256), 0, s, (double2 *)A.p, ld,
                       (int64_t)0, n, ld);
    hipLaunchKernelGGL(k_zero_c128, dim3((unsigned)((ld * nrhs + 255) / 256)), dim3(256), 0, s, (double2 *)B.p,
                       (int64_t)ld * nrhs);
    WM_TRY(copy2d_h2d(B.p, (size_t)ld * sizeof(double2), ci, (size_t)n * sizeof(wm_c128),
                      (size_t)n * sizeof(wm_c128), nrhs, s));
    WM_TRY(getrf_batched(c, WM_PREC_F64, ld, A.p, ld, tot, (int *)P.p, ld, 1, (int *)Inf.p, s));
    WM_TRY(getrs_batched(c, WM_PREC_F64, ld, nrhs, A.p, ld, tot, (int *)P.p, ld, B.p, ld, (int64_t)ld * nrhs, 1, s));
    int info = 0;
    WM_TRY(check_device_error(c, s));
    WM_TRY(copy_d2h(&info, Inf.p, sizeof(int), s));
    WM_TRY(copy2d_d2h(ci, (size_t)n * sizeof(wm_c128), B.p, (size_t)ld * sizeof(double2),
                      (size_t)n * sizeof(wm_c128), nrhs, s));
    return info;
}

void LU_cuBLAS(int n, int nrhs, wm_c128 *ci_cu, wm_c128 *cu_cu, wm_c128 *cz, int batchSize, int rank)
{
    (void)cu_cu;
    (void)rank;
    if (batchSize != 1) {
        std::fprintf(stderr, "LU_cuBLAS: batchSize must be 1\n");
        return;
    }
    const int rc = lu_solve_host(n, nrhs, ci_cu, cz);
    if (rc > 0) std::printf("FACTORIZATION ERROR\n");
    else if (rc < 0) std::fprintf(stderr, "LU_cuBLAS: %s\n", wm_last_error());
}

// One frequency of the reference's loop with Z kept on the device between the
// fill and the LU: the fill writes the padded matrix into the context's
// workspace (grown once, reused by later calls), Z goes to the caller's cz once,
// the hard-wired loads are added on the device and on the host copy alike, and
// the same device matrix is factored and solved.
static int calc_by_freq(float freq, float *x, float *y, float *z, float *rad, int *ipc, int *ips, int *ise,
                        int nsmax, int npls, int ienv, float sgnx, float sgny, float sgnz, float sgnenv, int iload,
                        float phas, int ngap, float ampl, wm_c128 *cz, wm_c128 *cu_cu, wm_c128 *ci_cu, int *info)
{
    if (npls <= 0 || ngap < 1 || ngap > npls || !cz || !cu_cu || !ci_cu) {
        set_error("CalculateByFreq: bad arguments (npls=%d, ngap=%d)", npls, ngap);
        return WM_ERR_ARG;
    }
    wm_ctx *c = default_ctx();
    if (!c) return WM_ERR_HIP;
    std::lock_guard<std::recursive_mutex> lk(c->mu);
    wm_geom *g = nullptr;
    WM_TRY(wm_geom_create_env(c, x, y, z, rad, ipc, ips, ise, nsmax, npls, ienv, sgnx, sgny, sgnz, sgnenv, &g));
    std::unique_ptr<wm_geom, int (*)(wm_geom *)> guard(g, wm_geom_destroy);
    const int ld = g->ld;
    const hipStream_t s = c->stream;
    const size_t zb = (size_t)ld * ld * sizeof(double2), vb = (size_t)ld * sizeof(double2);
    WM_TRY(c->ws_sweep.ensure(zb + vb + (size_t)ld * sizeof(int) + 256));
    double2 *Zd = (double2 *)c->ws_sweep.ptr, *Bd = (double2 *)((char *)Zd + zb);
    int *piv = (int *)((char *)Bd + vb), *dinf = (int *)((char *)piv + (size_t)ld * sizeof(int));
    const double ka = wavenumber(freq);
    WM_TRY(fill_launch(c, g, 1, &ka, Zd, 0, nullptr, 0, s));
    if (iload == 1) {  // hard-wired loads of the reference ("wersja gpu/Wire_MoM.cu":371-388)
        std::vector<int> idx;
        std::vector<double2> val;
        auto add = [&](int nl, double re, double im) {
            if (nl >= 0 && nl < npls) { idx.push_back(nl); val.push_back(make_double2(re, im)); }
        };
        for (int nl = 592 - 1; nl <= 2581 - 1; ++nl) add(nl, 1.e0, 2. * kPi * freq * 4.5);
        add(2613 - 1, 30., 0.);
        add(2582 - 1, 1.e12, 0.);
        if (!idx.empty()) {
            // indices and values staged in the right-hand-side buffer (overwritten below)
            const size_t nb = idx.size();
            WM_TRY(c->ws_solve.ensure(nb * (sizeof(int) + sizeof(double2))));
            int *di = (int *)c->ws_solve.ptr;
            double2 *dv = (double2 *)(di + nb);
            WM_TRY(copy_h2d(di, idx.data(), nb * sizeof(int), s));
            WM_TRY(copy_h2d(dv, val.data(), nb * sizeof(double2), s));
            hipLaunchKernelGGL(k_add_diag_list, dim3((unsigned)((nb + 255) / 256)), dim3(256), 0, s, Zd, ld, di, dv,
                               (int)nb);
        }
    }
    WM_TRY(copy2d_d2h(cz, (size_t)npls * sizeof(wm_c128), Zd, (size_t)ld * sizeof(double2),
                      (size_t)npls * sizeof(wm_c128), npls, s));
    for (int q = 0; q < npls; ++q) cu_cu[q] = wm_c128{0.0, 0.0};
    const double arg = kPi * phas / 180.;
    cu_cu[ngap - 1] = wm_c128{(double)ampl * std::cos(arg), (double)ampl * std::sin(arg)};
    for (int q = 0; q < npls; ++q) ci_cu[q] = cu_cu[q];
    hipLaunchKernelGGL(k_zero_c128, dim3((unsigned)((ld + 255) / 256)), dim3(256), 0, s, Bd, (int64_t)ld);
    WM_TRY(copy_h2d(Bd, ci_cu, (size_t)npls * sizeof(wm_c128), s));
    WM_TRY(getrf_batched(c, WM_PREC_F64, ld, Zd, ld, (int64_t)ld * ld, piv, ld, 1, dinf, s));
    WM_TRY(getrs_batched(c, WM_PREC_F64, ld, 1, Zd, ld, (int64_t)ld * ld, piv, ld, Bd, ld, ld, 1, s));
    WM_TRY(check_device_error(c, s));
    WM_TRY(copy_d2h(info, dinf, sizeof(int), s));
    return copy_d2h(ci_cu, Bd, (size_t)npls * sizeof(wm_c128), s);
}

void CalculateByFreq(int i, int npls, int nfreq, float freq, float *x, float *y, float *z, float *rad, int *ipc,
                     int *ips, int *ise, const int nsmax, int ienv, float sgnx, float sgny, float sgnz, float sgnenv,
                     int iload, float phas, int ngap, float ampl, wm_c128 *cz, wm_c128 *cu_cu, wm_c128 *ci_cu, int rank)
{
    (void)i;
    (void)nfreq;
    int info = 0;
    const int rc = calc_by_freq(freq, x, y, z, rad, ipc, ips, ise, nsmax, npls, ienv, sgnx, sgny, sgnz, sgnenv, iload,
                                phas, ngap, ampl, cz, cu_cu, ci_cu, &info);
    if (rc < 0) {
        std::fprintf(stderr, "CalculateByFreq: %s\n", wm_last_error());
        return;
    }
    if (info > 0) std::printf("FACTORIZATION ERROR\n");
    const wm_c128 zs = cdiv(cu_cu[ngap - 1], ci_cu[ngap - 1]);
    std::printf("\n Process - %d Freq = %.4g\t%.4g\t%.4g\n", rank, (double)freq, zs.re, zs.im);
    std::fflush(stdout);
}

}  // extern "C"
