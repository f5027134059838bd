// shk_context.hip -- context, errors and device memory of the shk library.
#include <algorithm>
#include <condition_variable>
#include <cstring>
#include <mutex>

#include "shk_internal.hpp"

namespace shk {

static thread_local std::string g_last_error;

void set_error(const std::string &msg) { g_last_error = msg; }

int fail(int code, const std::string &msg)
{
    g_last_error = msg;
    return code;
}

int ensure_red(shk_ctx ctx, size_t bytes)
{
    if (ctx->red.cap_bytes >= bytes) return SHK_OK;
    if (ctx->red.partials) SHK_HIP(hipFree(ctx->red.partials));
    size_t cap = bytes < (1u << 20) ? (1u << 20) : bytes;
    SHK_HIP(hipMalloc(&ctx->red.partials, cap));
    ctx->red.cap_bytes = cap;
    return SHK_OK;
}

int ensure_ws(shk_ctx ctx, size_t bytes)
{
    if (ctx->ws_cap >= bytes) return SHK_OK;
    if (ctx->ws) {
        SHK_HIP(hipStreamSynchronize(ctx->stream));
        SHK_HIP(hipFree(ctx->ws));
        ctx->ws = nullptr;
        ctx->ws_cap = 0;
    }
    hipError_t e = hipMalloc(&ctx->ws, bytes);
    if (e != hipSuccess) {
        (void)hipGetLastError();  // not left for a caller that does with less
        return fail(SHK_ERR_NOMEM, std::string("solver workspace: ") + hipGetErrorString(e));
    }
    ctx->ws_cap = bytes;
    return SHK_OK;
}

int ensure_ws2(shk_ctx ctx, size_t bytes)
{
    if (ctx->ws2_cap >= bytes) return SHK_OK;
    if (ctx->ws2) {
        SHK_HIP(hipStreamSynchronize(ctx->stream));
        SHK_HIP(hipFree(ctx->ws2));
        ctx->ws2 = nullptr;
        ctx->ws2_cap = 0;
    }
    hipError_t e = hipMalloc(&ctx->ws2, bytes);
    if (e != hipSuccess) {
        (void)hipGetLastError();
        return fail(SHK_ERR_NOMEM, std::string("refinement workspace: ") + hipGetErrorString(e));
    }
    ctx->ws2_cap = bytes;
    return SHK_OK;
}

hipError_t spare_malloc(shk_ctx ctx, void **p, size_t bytes)
{
    const hipError_t e = may_spare(ctx, bytes) ? hipMalloc(p, bytes) : hipErrorOutOfMemory;
    if (e != hipSuccess) {
        *p = nullptr;
        (void)hipGetLastError();
    }
    return e;
}

bool spare_ws2(shk_ctx ctx, size_t bytes)
{
    if (!may_spare(ctx, bytes)) return false;
    return ensure_ws2(ctx, bytes) == SHK_OK;
}

int wait_ticks(shk_ctx ctx, long long seconds, long long *ticks)
{
    int khz = 0;
    SHK_HIP(hipDeviceGetAttribute(&khz, hipDeviceAttributeWallClockRate, ctx->device));
    if (khz <= 0) khz = 100000;  // 100 MHz where none is reported
    const int64_t us = ctx->opt[SHK_OPT_WAIT_US];
    *ticks = us >= 0 ? us * khz / 1000 : (long long)khz * 1000 * seconds;
    return SHK_OK;
}

constexpr std::chrono::seconds kNoWaitsFor(60);  // 2 s of waiting in a minute, at most

bool may_wait(shk_ctx ctx)
{
    return ctx->opt[SHK_OPT_ON_CHIP] && std::chrono::steady_clock::now() >= ctx->no_waits_until;
}

void wait_ran_out(shk_ctx ctx)
{
    ctx->count[SHK_COUNT_STARTED_OVER]++;
    ctx->no_waits_until = std::chrono::steady_clock::now() + kNoWaitsFor;
}

namespace {
struct SeatQueue {
    std::mutex mu;
    std::condition_variable cv;
    uint64_t next = 0, serving = 0;  // turns given out, and whose it is
    int used = 0;
};
SeatQueue &seat_queue(int device)
{
    static SeatQueue q[64];
    return q[device & 63];
}
}  // namespace

void Seats::take(int groups)
{
    give();
    const int need = std::min((groups + kNumXcd - 1) / kNumXcd, most_);
    SeatQueue &q = seat_queue(device_);
    std::unique_lock<std::mutex> lk(q.mu);
    const uint64_t mine = q.next++;
    q.cv.wait(lk, [&]() { return q.serving == mine && q.used + need <= most_; });
    q.used += need;
    q.serving++;
    held_ = need;
    q.cv.notify_all();
}

void Seats::give()
{
    if (!held_) return;
    SeatQueue &q = seat_queue(device_);
    {
        std::lock_guard<std::mutex> lk(q.mu);
        q.used -= held_;
    }
    held_ = 0;
    q.cv.notify_all();
}

int check_device_ptr(const void *p, const char *what)
{
    if (!p) return fail(SHK_ERR_ARG, std::string("null device pointer: ") + what);
    return SHK_OK;
}

}  // namespace shk

using namespace shk;

extern "C" {

const char *shk_last_error(void) { return g_last_error.c_str(); }

const char *shk_version(void) { return "shk 0.1 (gfx950)"; }

int shk_ctx_create(int device, shk_ctx *out)
{
    SHK_CHECK(out, SHK_ERR_ARG, "shk_ctx_create: null out");
    *out = nullptr;
    int count = 0;
    hipError_t e = hipGetDeviceCount(&count);
    if (e != hipSuccess || count <= 0)
        return fail(SHK_ERR_NODEV, "shk_ctx_create: no HIP device visible");
    SHK_CHECK(device >= 0 && device < count, SHK_ERR_ARG, "shk_ctx_create: bad device index");
    SHK_HIP(hipSetDevice(device));
    hipDeviceProp_t prop;
    SHK_HIP(hipGetDeviceProperties(&prop, device));
    if (std::strncmp(prop.gcnArchName, "gfx950", 6) != 0)
        return fail(SHK_ERR_NODEV, std::string("shk_ctx_create: built for gfx950, device is ") +
                                       prop.gcnArchName);
    shk_ctx c = new shk_ctx_s();
    c->device = device;
    c->num_cus = prop.multiProcessorCount;
    std::strncpy(c->arch, prop.gcnArchName, sizeof(c->arch) - 1);
    // default priority, as every stream of this library
    if (hipStreamCreateWithFlags(&c->own, hipStreamNonBlocking) != hipSuccess) {
        delete c;
        return fail(SHK_ERR_HIP, "shk_ctx_create: hipStreamCreate failed");
    }
    c->stream = c->own;
    int st = ensure_red(c, 1u << 20);
    if (st != SHK_OK) { delete c; return st; }
    st = noalloc_scratch_init(device);
    if (st != SHK_OK) { delete c; return st; }
    SHK_HIP(hipMalloc(&c->scalars, 4096));
    SHK_HIP(hipMemset(c->scalars, 0, 4096));
    SHK_HIP(hipMalloc(&c->red.ticket, 64 * sizeof(unsigned)));
    SHK_HIP(hipMemset(c->red.ticket, 0, 64 * sizeof(unsigned)));
    c->state_bytes = 1 << 16;
    SHK_HIP(hipMalloc(&c->state, c->state_bytes));
    SHK_HIP(hipMemset(c->state, 0, c->state_bytes));
    SHK_HIP(hipHostMalloc(&c->state_host, c->state_bytes, hipHostMallocDefault));
    SHK_HIP(hipEventCreate(&c->ev0));
    SHK_HIP(hipEventCreate(&c->ev1));
    *out = c;
    return SHK_OK;
}

int shk_ctx_destroy(shk_ctx c)
{
    if (!c) return SHK_OK;
    hipSetDevice(c->device);
    hipStreamSynchronize(c->stream);
    if (c->red.partials) hipFree(c->red.partials);
    if (c->red.ticket) hipFree(c->red.ticket);
    if (c->scalars) hipFree(c->scalars);
    if (c->ws) hipFree(c->ws);
    if (c->ws2) hipFree(c->ws2);
    if (c->state) hipFree(c->state);
    if (c->state_host) hipHostFree(c->state_host);
    if (c->ev0) hipEventDestroy(c->ev0);
    if (c->ev1) hipEventDestroy(c->ev1);
    if (c->own) hipStreamDestroy(c->own);
    delete c;
    return SHK_OK;
}

int shk_ctx_set_stream(shk_ctx c, void *s)
{
    SHK_CHECK(c, SHK_ERR_ARG, "null ctx");
    SHK_HIP(hipStreamSynchronize(c->stream));
    c->stream = (hipStream_t)s;  // verbatim: NULL is the default (null) stream
    return SHK_OK;
}

int shk_ctx_synchronize(shk_ctx c)
{
    SHK_CHECK(c, SHK_ERR_ARG, "null ctx");
    SHK_HIP(hipStreamSynchronize(c->stream));
    return SHK_OK;
}

int shk_ctx_device_info(shk_ctx c, int *num_cus, int *num_xcds, char *arch, int arch_len)
{
    SHK_CHECK(c, SHK_ERR_ARG, "null ctx");
    if (num_cus) *num_cus = c->num_cus;
    if (num_xcds) *num_xcds = kNumXcd;
    if (arch && arch_len > 0) {
        std::strncpy(arch, c->arch, arch_len - 1);
        arch[arch_len - 1] = 0;
    }
    return SHK_OK;
}

int shk_ctx_set_option(shk_ctx c, int option, int64_t value)
{
    SHK_CHECK(c, SHK_ERR_ARG, "null ctx");
    bool ok = false;
    if (option == SHK_OPT_ON_CHIP) ok = value == 0 || value == 1;
    else if (option == SHK_OPT_WAIT_US) ok = value >= -1 && value <= 3600LL * 1000000;
    else if (option == SHK_OPT_BUFFER_BYTES) ok = value >= 0 && value <= INT32_MAX;
    else if (option == SHK_OPT_SPARE_BYTES) ok = value >= 0;
    else if (option == SHK_OPT_CG_ITERS) ok = value >= 1 && value <= INT32_MAX;
    SHK_CHECK(ok, SHK_ERR_ARG, "shk_ctx_set_option: unknown option or value out of range");
    c->opt[option] = value;
    c->no_waits_until = {};
    return SHK_OK;
}

int shk_ctx_counter(shk_ctx c, int counter, int64_t *value)
{
    SHK_CHECK(c && value, SHK_ERR_ARG, "shk_ctx_counter: null argument");
    SHK_CHECK(counter >= 0 && counter <= SHK_COUNT_COO_BUCKETS, SHK_ERR_ARG, "shk_ctx_counter: unknown counter");
    SHK_HIP(hipStreamSynchronize(c->stream));
    if (counter != SHK_COUNT_SOR_RESCUED) {
        *value = c->count[counter];
        return SHK_OK;
    }
    unsigned v = 0;
    SHK_HIP(hipMemcpy(&v, c->red.ticket + kRescuedSlot, sizeof(v), hipMemcpyDeviceToHost));
    *value = v;
    return SHK_OK;
}

int shk_malloc(shk_ctx c, size_t bytes, void **p)
{
    SHK_CHECK(c && p, SHK_ERR_ARG, "shk_malloc: null argument");
    *p = nullptr;
    if (bytes == 0) bytes = 16;
    hipError_t e = hipMalloc(p, bytes);
    if (e != hipSuccess) return fail(SHK_ERR_NOMEM, std::string("shk_malloc: ") + hipGetErrorString(e));
    return SHK_OK;
}

int shk_free(shk_ctx c, void *p)
{
    SHK_CHECK(c, SHK_ERR_ARG, "shk_free: null ctx");
    if (p) {
        SHK_HIP(hipStreamSynchronize(c->stream));
        SHK_HIP(hipFree(p));
    }
    return SHK_OK;
}

int shk_memcpy_h2d(shk_ctx c, void *dst, const void *src, size_t bytes)
{
    SHK_CHECK(c, SHK_ERR_ARG, "null ctx");
    if (!bytes) return SHK_OK;
    SHK_HIP(hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, c->stream));
    SHK_HIP(hipStreamSynchronize(c->stream));
    return SHK_OK;
}

int shk_memcpy_d2h(shk_ctx c, void *dst, const void *src, size_t bytes)
{
    SHK_CHECK(c, SHK_ERR_ARG, "null ctx");
    if (!bytes) return SHK_OK;
    SHK_HIP(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, c->stream));
    SHK_HIP(hipStreamSynchronize(c->stream));
    return SHK_OK;
}

int shk_memcpy_d2d(shk_ctx c, void *dst, const void *src, size_t bytes)
{
    SHK_CHECK(c, SHK_ERR_ARG, "null ctx");
    if (!bytes) return SHK_OK;
    SHK_HIP(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToDevice, c->stream));
    return SHK_OK;
}

}  // extern "C"
