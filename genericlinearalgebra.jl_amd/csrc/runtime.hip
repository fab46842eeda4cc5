// Handle, workspace and error reporting of libgla_hip.so.
#include <algorithm>
#include <condition_variable>
#include <cstdarg>
#include <cstring>
#include <mutex>

#include "gla_internal.hpp"

namespace gla {

namespace {
thread_local char g_err[512] = "";
}

void set_error(const char *fmt, ...)
{
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(g_err, sizeof(g_err), fmt, ap);
    va_end(ap);
}

int ensure_workspace(Handle *h, size_t bytes)
{
    if (bytes <= h->ws_bytes) return GLA_OK;
    // Round up to 64 MiB granules so that a sequence of growing calls
    // reallocates rarely.
    const size_t gran = size_t(64) << 20;
    size_t want = (bytes + gran - 1) / gran * gran;
    if (h->ws) {
        // The old buffer may still be read by queued work.
        GLA_HIP_TRY(hipDeviceSynchronize());
        GLA_HIP_TRY(hipFree(h->ws));
        h->ws = nullptr;
        h->ws_bytes = 0;
    }
    GLA_HIP_TRY(hipMalloc(&h->ws, want));
    h->ws_bytes = want;
    return GLA_OK;
}

bool capturing(hipStream_t s)
{
    hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(s, &cap) == hipSuccess && cap == hipStreamCaptureStatusNone) return false;
    (void)hipGetLastError();
    return true;
}

bool ensure_df(Handle *h, hipStream_t s, size_t bytes)
{
    // Neither the wait nor the allocation may fall into a capture, and a
    // buffer that a graph holds stays until the handle goes: then the next is
    // twice as large, so that those kept are together smaller than it.
    const bool eager = !capturing(s);
    if (bytes <= h->df_bytes) {
        h->df_captured |= !eager;
        return true;
    }
    if (!eager) return false;
    const size_t gran = size_t(16) << 20;
    size_t want = (bytes + gran - 1) / gran * gran;
    if (h->df && h->df_captured) {
        want = std::max(want, 2 * h->df_bytes);
        h->df_kept.push_back(h->df);
        h->df = nullptr;
        h->df_bytes = 0;
        h->df_captured = false;
    }
    if (h->df) {
        // the old buffer may still be read by queued work
        if (hipDeviceSynchronize() != hipSuccess || hipFree(h->df) != hipSuccess) {
            (void)hipGetLastError();
            return false;
        }
        h->df = nullptr;
        h->df_bytes = 0;
    }
    if (hipMalloc(&h->df, want) != hipSuccess) {
        (void)hipGetLastError();
        h->df = nullptr;
        return false;
    }
    h->df_bytes = want;
    return true;
}

namespace {
constexpr int kMaxDevices = 64;
constexpr int kDies = 8;                   // workgroups go to the dies in turn
struct ResidentCall {                      // the last such call of a stream
    hipEvent_t done = nullptr;
    hipStream_t s = nullptr;
    int weight = 0;
};
struct ResidentCalls {
    std::mutex lock;
    std::condition_variable turn;
    unsigned long next = 0, serving = 0;   // callers take turns in the order they come
    static constexpr int kMax = 32;
    ResidentCall call[kMax];               // those in flight, oldest first: call[0 … n)
    int n = 0;
    PanelCall *queued = nullptr;           // queued PanelCalls, linked by `link`
    int queueing = 0;                      // those not yet queued
    int panels = 0;                        // weight of both
    hipEvent_t panel_done = nullptr;       // (reused for every stream waited for)
    int mine = 0, replaces = -1;           // of the call that holds the lock: weight, its stream's entry

    void drop(int i)                       // its event goes to a later call
    {
        std::rotate(call + i, call + i + 1, call + n);
        --n;
    }
    // Drops what has finished; the weight of the rest.
    int in_flight()
    {
        int w = 0;
        for (int i = 0; i < n;) {
            if (hipEventQuery(call[i].done) == hipSuccess) {
                drop(i);
            } else {
                (void)hipGetLastError();
                w += call[i++].weight;
            }
        }
        return w;
    }
    // s waits for the oldest calls until those left weigh `room` at most.
    hipError_t make_room(hipStream_t s, int room)
    {
        hipError_t e = hipSuccess;
        int w = in_flight();
        for (int i = 0; i < n && w > room && e == hipSuccess; ++i) {
            e = hipStreamWaitEvent(s, call[i].done, 0);
            w -= call[i].weight;
        }
        return e;
    }
};
ResidentCalls g_resident[kMaxDevices];

// Another thread's capture in the global mode forbids this one event queries and
// the like; none of those made here touches a captured stream.
struct RelaxedCapture {
    hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
    RelaxedCapture() { (void)hipThreadExchangeStreamCaptureMode(&mode); }
    ~RelaxedCapture() { (void)hipThreadExchangeStreamCaptureMode(&mode); }
};

int weight_of(int64_t workgroups) { return (int)cdiv(workgroups, kDies); }
int room_of(const Handle *h) { return std::max(1, h->num_cus / kDies); }
}  // namespace

bool resident_begin(Handle *h, hipStream_t s, int64_t workgroups)
{
    if (h->device < 0 || h->device >= kMaxDevices || capturing(s)) return false;
    ResidentCalls &c = g_resident[h->device];
    const RelaxedCapture relaxed;
    const int room = room_of(h), w = std::min(room, weight_of(workgroups));
    std::unique_lock<std::mutex> lk(c.lock);
    const unsigned long mine = c.next++;
    c.turn.wait(lk, [&] {
        return c.serving == mine && (c.panels + w <= room || c.queueing == 0);
    });
    hipError_t e = hipSuccess;
    if (!c.panel_done) {
        e = hipEventCreateWithFlags(&c.panel_done, hipEventDisableTiming);
        if (e != hipSuccess) c.panel_done = nullptr;
    }
    int panels = c.panels;
    if (e == hipSuccess && panels + w > room) {
        for (const PanelCall *q = c.queued; q && e == hipSuccess; q = q->link) {
            e = hipEventRecord(c.panel_done, q->s);
            if (e == hipSuccess) e = hipStreamWaitEvent(s, c.panel_done, 0);
        }
        panels = 0;
    }
    c.mine = w;
    if (e == hipSuccess) e = c.make_room(s, room - w - panels);
    // one entry a stream: the new call follows the stream's last one (waited for
    // too, should the handle be another stream's by now), and weighs as much as
    // either until it is done
    c.replaces = -1;
    for (int i = 0; i < c.n; ++i)
        if (c.call[i].s == s) {
            if (e == hipSuccess) e = hipStreamWaitEvent(s, c.call[i].done, 0);
            c.mine = std::max(c.mine, c.call[i].weight);
            c.replaces = i;
        }
    if (c.replaces < 0 && c.n == ResidentCalls::kMax) {
        // no entry left: after all of them, and none beside it
        for (int i = 0; i < c.n && e == hipSuccess; ++i) e = hipStreamWaitEvent(s, c.call[i].done, 0);
        if (e == hipSuccess) c.n = 0;
        c.mine = room;
    } else if (c.replaces < 0 && !c.call[c.n].done && e == hipSuccess) {
        e = hipEventCreateWithFlags(&c.call[c.n].done, hipEventDisableTiming);
        if (e != hipSuccess) c.call[c.n].done = nullptr;
    }
    if (e != hipSuccess) {
        (void)hipGetLastError();
        ++c.serving;
        lk.unlock();
        c.turn.notify_all();
        return false;
    }
    lk.release();
    return true;
}

int resident_end(Handle *h, hipStream_t s)
{
    ResidentCalls &c = g_resident[h->device];
    if (c.replaces >= 0) c.drop(c.replaces);
    ResidentCall &r = c.call[c.n];
    const hipError_t e = hipEventRecord(r.done, s);
    r.s = s;
    r.weight = c.mine;
    ++c.n;
    ++c.serving;
    c.lock.unlock();
    c.turn.notify_all();
    GLA_HIP_TRY(e);
    return GLA_OK;
}

PanelCall::PanelCall(Handle *h, hipStream_t stream, int64_t workgroups) : s(stream)
{
    if (h->device < 0 || h->device >= kMaxDevices || capturing(s)) return;
    const RelaxedCapture relaxed;
    device = h->device;
    ResidentCalls &c = g_resident[device];
    weight = weight_of(workgroups);
    std::unique_lock<std::mutex> lk(c.lock);
    const unsigned long mine = c.next++;
    c.turn.wait(lk, [&] { return c.serving == mine; });
    ++c.serving;
    ++c.queueing;
    c.panels += weight;
    if (c.make_room(s, room_of(h) - c.panels) != hipSuccess) (void)hipGetLastError();
    lk.unlock();
    c.turn.notify_all();
}

void PanelCall::queued()
{
    if (device < 0) return;
    ResidentCalls &c = g_resident[device];
    {
        std::lock_guard<std::mutex> lk(c.lock);
        link = c.queued;
        c.queued = this;
        --c.queueing;
    }
    is_queued = true;
    c.turn.notify_all();
}

PanelCall::~PanelCall()
{
    if (device < 0) return;
    ResidentCalls &c = g_resident[device];
    {
        std::lock_guard<std::mutex> lk(c.lock);
        if (is_queued) {
            PanelCall **at = &c.queued;
            while (*at != this) at = &(*at)->link;
            *at = link;
        } else {
            --c.queueing;
        }
        c.panels -= weight;
    }
    c.turn.notify_all();
}

namespace {
// (Re)creates the look-ahead Cholesky's stream pair: `masked`, limited to
// every CU but the highest-numbered `reserve`, and `chain`, a non-blocking
// stream on all CUs (a CU-masked stream is created blocking, so the chain
// cannot run on the caller's stream beside it).  reserve 0 drops both.
int set_side_cu_reserve(Handle *h, int reserve)
{
    GLA_HIP_TRY(hipSetDevice(h->device));
    GLA_HIP_TRY(hipDeviceSynchronize());
    if (h->masked) { (void)hipStreamDestroy(h->masked); h->masked = nullptr; }
    if (h->chain) { (void)hipStreamDestroy(h->chain); h->chain = nullptr; }
    h->side_cu_reserve = reserve;
    if (reserve > 0) {
        const int words = (h->num_cus + 31) / 32;
        uint32_t mask[16] = {0};
        for (int c = 0; c < h->num_cus - reserve && c < 32 * 16; ++c)
            mask[c / 32] |= 1u << (c % 32);
        GLA_HIP_TRY(hipExtStreamCreateWithCUMask(&h->masked, (uint32_t)words, mask));
        GLA_HIP_TRY(hipStreamCreateWithFlags(&h->chain, hipStreamNonBlocking));
    }
    return GLA_OK;
}
}  // namespace

}  // namespace gla

extern "C" {

const char *gla_version(void) { return "gla_hip 0.1 (gfx950)"; }

const char *gla_last_error_string(void) { return gla::g_err; }

int gla_set_tuning(gla_handle_t hh, const char *key, int64_t value)
{
    auto *h = reinterpret_cast<gla::Handle *>(hh);
    if (!h) { gla::set_error("null handle"); return -1; }
    if (!key) return -2;
    if (std::strcmp(key, "chol_block") == 0) {
        if (value != 0 && value != -1 && (value < 128 || value % 128 != 0)) {
            gla::set_error("chol_block must be -1, 0 or a multiple of 128");
            return -3;
        }
        h->chol_block = value;
        return GLA_OK;
    }
    if (std::strcmp(key, "chol_df") == 0) {
        if (value < 0 || value > 8192) {
            gla::set_error("chol_df must be in [0, 8192]");
            return -3;
        }
        h->chol_df = value;
        return GLA_OK;
    }
    if (std::strcmp(key, "ldlt_block") == 0) {
        if (value < 128 || value % 128 != 0 || value > 4096) {
            gla::set_error("ldlt_block must be a multiple of 128 in [128, 4096]");
            return -3;
        }
        h->ldlt_block = value;
        return GLA_OK;
    }
    if (std::strcmp(key, "mixed_block") == 0) {
        if (value < 128 || value % 128 != 0 || value > 4096) {
            gla::set_error("mixed_block must be a multiple of 128 in [128, 4096]");
            return -3;
        }
        h->mixed_block = (int)value;
        return GLA_OK;
    }
    if (std::strcmp(key, "qr_panel") == 0) {
        if (value != 1 && value != 2) {
            gla::set_error("qr_panel must be 1 or 2");
            return -3;
        }
        h->qr_panel = (int)value;
        return GLA_OK;
    }
    if (std::strcmp(key, "qr_inner") == 0) {
        if (value != -1 && value != 0 && value != 32 && value != 64) {
            gla::set_error("qr_inner must be -1, 0, 32 or 64");
            return -3;
        }
        h->qr_inner = (int)value;
        return GLA_OK;
    }
    if (std::strcmp(key, "gemm_dl") == 0) {
        if (value < 0 || value > 3) {
            gla::set_error("gemm_dl must be 0, 1, 2 or 3");
            return -3;
        }
        gla::set_gemm_dl((int)value);
        return GLA_OK;
    }
    if (std::strcmp(key, "gemm_lds1") == 0) {
        if (value != 0 && value != 1) {
            gla::set_error("gemm_lds1 must be 0 or 1");
            return -3;
        }
        gla::set_gemm_lds1((int)value);
        return GLA_OK;
    }
    if (std::strcmp(key, "qr_hr") == 0) {
        if (value < -1) {
            gla::set_error("qr_hr must be -1, 0 or a row count");
            return -3;
        }
        h->qr_hr = value;
        return GLA_OK;
    }
    if (std::strcmp(key, "chol_psolve") == 0) {
        if (value != 0 && value != 1) {
            gla::set_error("chol_psolve must be 0 or 1");
            return -3;
        }
        h->chol_psolve = (int)value;
        return GLA_OK;
    }
    if (std::strcmp(key, "chol_syrk_late") == 0) {
        if (value != 0 && value != 1) {
            gla::set_error("chol_syrk_late must be 0 or 1");
            return -3;
        }
        h->chol_syrk_late = (int)value;
        return GLA_OK;
    }
    if (std::strcmp(key, "qr_lookahead") == 0) {
        if (value != 0 && value != 1) {
            gla::set_error("qr_lookahead must be 0 or 1");
            return -3;
        }
        h->qr_lookahead = (int)value;
        return GLA_OK;
    }
    if (std::strcmp(key, "spin_limit") == 0) {
        if (value < 1 || value > (int64_t)0x7fffffff) {
            gla::set_error("spin_limit must be in [1, 2^31)");
            return -3;
        }
        h->spin_limit = (unsigned)value;
        return GLA_OK;
    }
    if (std::strcmp(key, "side_cu_reserve") == 0) {
        if (value < 0 || value > h->num_cus / 2 || h->num_cus > 32 * 16) {
            gla::set_error("side_cu_reserve must be in [0, CUs/2]");
            return -3;
        }
        return gla::set_side_cu_reserve(h, (int)value);
    }
    if (std::strcmp(key, "qr_wait_test") == 0) {
        if (value != 0 && value != 1) {
            gla::set_error("qr_wait_test must be 0 or 1");
            return -3;
        }
        h->qr_wait_test = (int)value;
        return GLA_OK;
    }
    gla::set_error("unknown tuning key '%s'", key);
    return -2;
}

int gla_get_tuning(gla_handle_t hh, const char *key, int64_t *value)
{
    auto *h = reinterpret_cast<gla::Handle *>(hh);
    if (!h) { gla::set_error("null handle"); return -1; }
    if (!key) return -2;
    if (!value) return -3;
    const struct { const char *name; int64_t v; } knobs[] = {
        {"chol_block", h->chol_block},       {"ldlt_block", h->ldlt_block},
        {"mixed_block", h->mixed_block},     {"qr_panel", h->qr_panel},
        {"qr_inner", h->qr_inner},           {"gemm_dl", gla::get_gemm_dl()},
        {"gemm_lds1", gla::get_gemm_lds1()}, {"qr_hr", h->qr_hr},
        {"chol_syrk_late", h->chol_syrk_late}, {"qr_lookahead", h->qr_lookahead},
        {"chol_psolve", h->chol_psolve},
        {"spin_limit", (int64_t)h->spin_limit}, {"chol_df", h->chol_df}, {"side_cu_reserve", h->side_cu_reserve},
        {"qr_wait_test", h->qr_wait_test},
    };
    for (const auto &k : knobs)
        if (std::strcmp(key, k.name) == 0) { *value = k.v; return GLA_OK; }
    gla::set_error("unknown tuning knob '%s'", key);
    return -2;
}

int gla_handle_create(gla_handle_t *out)
{
    using gla::Handle;
    if (!out) return -1;
    Handle *h = new Handle();
    GLA_HIP_TRY(hipGetDevice(&h->device));
    hipDeviceProp_t prop;
    GLA_HIP_TRY(hipGetDeviceProperties(&prop, h->device));
    h->num_cus = prop.multiProcessorCount;
    GLA_HIP_TRY(hipStreamCreateWithFlags(&h->side, hipStreamNonBlocking));
    GLA_HIP_TRY(hipEventCreateWithFlags(&h->ev_fork, hipEventDisableTiming));
    GLA_HIP_TRY(hipEventCreateWithFlags(&h->ev_join, hipEventDisableTiming));
    GLA_HIP_TRY(hipEventCreateWithFlags(&h->ev_step[0], hipEventDisableTiming));
    GLA_HIP_TRY(hipEventCreateWithFlags(&h->ev_step[1], hipEventDisableTiming));
    GLA_HIP_TRY(hipMalloc(reinterpret_cast<void **>(&h->dinfo), 256));
    GLA_HIP_TRY(hipMemset(h->dinfo, 0, 256));
    GLA_HIP_TRY(hipMalloc(reinterpret_cast<void **>(&h->dbar), 4096));
    GLA_HIP_TRY(hipMemset(h->dbar, 0, 4096));
    // The trailing SYRK of the look-ahead Cholesky leaves an eighth of the
    // CUs (32 of 256) to the chain of small kernels beside it.
    if (h->num_cus <= 32 * 16) {
        const int rc = gla::set_side_cu_reserve(h, h->num_cus / 8);
        if (rc != GLA_OK) return rc;
    }
    GLA_HIP_TRY(hipDeviceSynchronize());
    *out = reinterpret_cast<gla_handle_t>(h);
    return GLA_OK;
}

int gla_handle_destroy(gla_handle_t hh)
{
    using gla::Handle;
    Handle *h = reinterpret_cast<Handle *>(hh);
    if (!h) return GLA_OK;
    GLA_HIP_TRY(hipSetDevice(h->device));
    GLA_HIP_TRY(hipDeviceSynchronize());
    if (h->ws) (void)hipFree(h->ws);
    if (h->df) (void)hipFree(h->df);
    for (void *p : h->df_kept) (void)hipFree(p);
    if (h->dinfo) (void)hipFree(h->dinfo);
    if (h->dbar) (void)hipFree(h->dbar);
    (void)hipEventDestroy(h->ev_fork);
    (void)hipEventDestroy(h->ev_join);
    (void)hipEventDestroy(h->ev_step[0]);
    (void)hipEventDestroy(h->ev_step[1]);
    (void)hipStreamDestroy(h->side);
    if (h->masked) (void)hipStreamDestroy(h->masked);
    if (h->chain) (void)hipStreamDestroy(h->chain);
    delete h;
    return GLA_OK;
}

int gla_gemm_d(gla_handle_t hh, char ta, char tb, int64_t m, int64_t n, int64_t k, double alpha,
               const double *A, int64_t lda, const double *B, int64_t ldb, double beta,
               double *C, int64_t ldc, void *stream)
{
    auto *h = reinterpret_cast<gla::Handle *>(hh);
    if (!h) return -1;
    if (m < 0) return -4;
    if (n < 0) return -5;
    if (k < 0) return -6;
    GLA_HIP_TRY(hipSetDevice(h->device));
    return gla::gemm<double>(reinterpret_cast<hipStream_t>(stream), ta, tb, 0, m, n, k, alpha, A,
                             lda, B, ldb, beta, C, ldc, 0);
}

int gla_gemm_s(gla_handle_t hh, char ta, char tb, int64_t m, int64_t n, int64_t k, float alpha,
               const float *A, int64_t lda, const float *B, int64_t ldb, float beta, float *C,
               int64_t ldc, void *stream)
{
    auto *h = reinterpret_cast<gla::Handle *>(hh);
    if (!h) return -1;
    if (m < 0) return -4;
    if (n < 0) return -5;
    if (k < 0) return -6;
    GLA_HIP_TRY(hipSetDevice(h->device));
    return gla::gemm<float>(reinterpret_cast<hipStream_t>(stream), ta, tb, 0, m, n, k, alpha, A,
                            lda, B, ldb, beta, C, ldc, 0);
}

}  // extern "C"
