// Context, memory and timing entry points of the C ABI.
#include <algorithm>
#include <cstring>

#include "vx_internal.h"

using namespace vxi;

extern "C" {

int vx_ctx_create(int device, vx_ctx **out) {
    if (!out) return VX_EINVAL;
    *out = nullptr;
    int n = 0;
    if (hipGetDeviceCount(&n) != hipSuccess || n <= device || device < 0) return VX_EHIP;
    vx_ctx *c = new vx_ctx;
    c->device = device;
    if (hipSetDevice(device) != hipSuccess || hipStreamCreate(&c->stream) != hipSuccess) {
        delete c;
        return VX_EHIP;
    }
    for (auto &e : c->ev)
        if (hipEventCreate(&e) != hipSuccess) {
            delete c;
            return VX_EHIP;
        }
    int ncu = 0;
    if (hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, device) == hipSuccess && ncu > 0)
        c->n_cu = ncu;
    // the fixed work array of vx_poisson_noalloc; on failure that entry point
    // reports the error and every other one works
    (void)vx_noalloc_scratch_init(c);
    *out = c;
    return VX_OK;
}

void vx_ctx_destroy(vx_ctx *ctx) {
    if (!ctx) return;
    (void)hipSetDevice(ctx->device);
    (void)hipStreamSynchronize(ctx->stream);
    for (auto &e : ctx->ev)
        if (e) (void)hipEventDestroy(e);
    for (auto &e : ctx->tev) (void)hipEventDestroy(e);
    if (ctx->mom_table) (void)hipFree(ctx->mom_table);
    for (double *t : ctx->mom_old) (void)hipFree(t);
    if (ctx->batch_ring && ctx->batch_ring_free) ctx->batch_ring_free(ctx->batch_ring);
    if (ctx->xev) (void)hipEventDestroy(ctx->xev);
    if (ctx->cfl_ev) (void)hipEventDestroy(ctx->cfl_ev);
    if (ctx->cfl_host) (void)hipHostFree(ctx->cfl_host);
    for (auto &e : ctx->ring_ev)
        if (e) (void)hipEventDestroy(e);
    if (ctx->ring) (void)hipHostFree(ctx->ring);
    for (auto &e : ctx->stage_ev)
        if (e) (void)hipEventDestroy(e);
    if (ctx->stage) (void)hipHostFree(ctx->stage);
    (void)hipStreamDestroy(ctx->stream);
    delete ctx;
}

const char *vx_last_error(vx_ctx *ctx) { return ctx ? ctx->err.c_str() : "null context"; }

// entry points that wait for the device or allocate cannot be recorded in a step graph
static int not_recording(vx_ctx *ctx, const char *what) {
    return ctx->capturing ? fail(ctx, VX_EINVAL, "%s while a step graph is being recorded", what) : VX_OK;
}

int vx_sync(vx_ctx *ctx) {
    if (int rc = not_recording(ctx, "sync")) return rc;
    return check_hip(ctx, hipStreamSynchronize(ctx->stream), "sync");
}

void *vx_stream(vx_ctx *ctx) { return ctx ? (void *)ctx->stream : nullptr; }

int vx_malloc(vx_ctx *ctx, size_t bytes, void **dptr) {
    if (!dptr) return fail(ctx, VX_EINVAL, "null out pointer");
    *dptr = nullptr;
    if (int rc = not_recording(ctx, "vx_malloc")) return rc;
    if (bytes == 0) return VX_OK;
    hipError_t e = hipMalloc(dptr, bytes);
    if (e != hipSuccess) return fail(ctx, VX_ENOMEM, "hipMalloc(%zu): %s", bytes, hipGetErrorString(e));
    ctx->allocs[*dptr] = bytes;
    ctx->live_bytes += bytes;
    e = hipMemsetAsync(*dptr, 0, bytes, ctx->stream);
    if (e == hipSuccess) e = hipStreamSynchronize(ctx->stream);
    return check_hip(ctx, e, "zero fill");
}

int vx_free(vx_ctx *ctx, void *dptr) {
    if (!dptr) return VX_OK;
    if (int rc = not_recording(ctx, "vx_free")) return rc;
    auto it = ctx->allocs.find(dptr);
    if (it != ctx->allocs.end()) {
        ctx->live_bytes -= it->second;
        ctx->allocs.erase(it);
    }
    (void)hipStreamSynchronize(ctx->stream);
    return check_hip(ctx, hipFree(dptr), "hipFree");
}

}  // extern "C"

// Rows of `w` doubles between a device array of `pitch` doubles a row and a
// contiguous host-visible one.
__global__ __launch_bounds__(256) void k_rows_out(const double *dev, double *host, long pitch, long w, long n) {
    const long e = blockIdx.x * 256L + threadIdx.x;
    if (e < n) host[e] = dev[(e / w) * pitch + e % w];
}
__global__ __launch_bounds__(256) void k_rows_in(double *dev, const double *host, long pitch, long w, long n) {
    const long e = blockIdx.x * 256L + threadIdx.x;
    if (e < n) dev[(e / w) * pitch + e % w] = host[e];
}

// The pinned buffers, allocated on first use (40 us), with their events on the
// context's device, whichever device the calling thread has current.
int vx_stage_init(vx_ctx *ctx) {
    if (ctx->stage) return VX_OK;
    struct Device {
        int was = -1;
        explicit Device(int d) {
            if (hipGetDevice(&was) != hipSuccess || was == d || hipSetDevice(d) != hipSuccess) was = -1;
        }
        ~Device() {
            if (was >= 0) (void)hipSetDevice(was);
        }
    } device(ctx->device);
    void *p = nullptr;
    int rc = check_hip(ctx, hipHostMalloc(&p, 2 * vx_ctx::STAGE_BYTES), "pinned staging");
    if (rc) return rc;
    for (auto &e : ctx->stage_ev)
        if (!rc && !e) rc = check_hip(ctx, hipEventCreateWithFlags(&e, hipEventDisableTiming), "staging event");
    if (rc) (void)hipHostFree(p);
    else ctx->stage = (double *)p;
    return rc;
}

// Whether n doubles at dev lie inside one allocation of the context's device, so
// that a kernel may read and write them.  Whatever else a caller passes (null, a
// count past the allocation, another device's memory) goes to HIP's own copy,
// which refuses it or knows how to reach it; a kernel would fault on it.
bool vx_device_range(const vx_ctx *ctx, const double *dev, size_t n) {
    if (!dev || (uintptr_t)dev % sizeof(double) != 0) return false;
    hipPointerAttribute_t at;
    hipDeviceptr_t base = nullptr;
    size_t size = 0;
    if (hipPointerGetAttributes(&at, dev) != hipSuccess ||
        hipMemGetAddressRange(&base, &size, (hipDeviceptr_t)dev) != hipSuccess) {
        (void)hipGetLastError();  // (an address that HIP does not know)
        return false;
    }
    const size_t off = (size_t)((const char *)dev - (const char *)base);
    return at.type == hipMemoryTypeDevice && at.device == ctx->device && off <= size &&
           n <= (size - off) / sizeof(double);
}

// Whether HIP does not know the host address: pinned memory takes HIP's own copy,
// which reaches it without a second copy on the host (1024 x 1024 doubles of a
// patch 155 us, 240 up and 360 down through the buffers).
static bool pageable(const void *host) {
    hipPointerAttribute_t at;
    if (hipPointerGetAttributes(&at, host) == hipSuccess) return at.type == hipMemoryTypeUnregistered;
    (void)hipGetLastError();
    return true;
}

// Whether there are pinned buffers to stage through; without them a copy is HIP's.
static bool stage_there(vx_ctx *ctx) {
    std::lock_guard<std::mutex> lock(ctx->stage_mu);
    return vx_stage_init(ctx) == VX_OK;
}

// h rows of w doubles between a pitched device array and pageable host memory,
// through the context's two pinned buffers: a kernel packs one (or unpacks it)
// over the link while the host copies the other.  hipMemcpy2DAsync on pageable
// memory goes row by row: 64 x 256 doubles up 600 us, down 430, 1024 x 1024 9.6 and
// 7.2 ms, 4096 x 4096 40 and 37 ms on an MI355X; these 16 and 17 us, 0.24 and 0.35
// ms, 4.7 and 4.4 ms.  Waits for the copy.
// Threads that copy at once on one context take the buffers in turn.
static int staged_rows(vx_ctx *ctx, double *dev, size_t pitch, double *host, size_t w, size_t h, bool up,
                       const char *what) {
    constexpr size_t BUF = vx_ctx::STAGE_BYTES / sizeof(double);
    std::lock_guard<std::mutex> lock(ctx->stage_mu);
    int rc = VX_OK;
    const size_t rows = BUF / w;  // (the caller checked w <= BUF)
    double *prev_host = nullptr;  // downloads: the chunk whose kernel is under way
    size_t prev_n = 0;
    int k = 0;
    for (size_t r = 0; r < h || prev_host; k++) {
        const size_t nr = r < h ? std::min(rows, h - r) : 0, n = nr * w;
        double *buf = ctx->stage + (size_t)(k & 1) * BUF;
        const unsigned grid = (unsigned)((n + 255) / 256);
        if (n && up) {
            if (k >= 2 && (rc = check_hip(ctx, hipEventSynchronize(ctx->stage_ev[k & 1]), what))) return rc;
            std::memcpy(buf, host + r * w, sizeof(double) * n);
            k_rows_in<<<grid, 256, 0, ctx->stream>>>(dev + r * pitch, buf, (long)pitch, (long)w, (long)n);
        } else if (n) {
            k_rows_out<<<grid, 256, 0, ctx->stream>>>(dev + r * pitch, buf, (long)pitch, (long)w, (long)n);
        }
        if (n && ((rc = check_launch(ctx, what)) ||
                  (rc = check_hip(ctx, hipEventRecord(ctx->stage_ev[k & 1], ctx->stream), what))))
            return rc;
        if (!up && prev_host) {
            if ((rc = check_hip(ctx, hipEventSynchronize(ctx->stage_ev[~k & 1]), what))) return rc;
            std::memcpy(prev_host, ctx->stage + (size_t)(~k & 1) * BUF, sizeof(double) * prev_n);
        }
        prev_host = !up && n ? host + r * w : nullptr;
        prev_n = n;
        r += nr;
    }
    return check_hip(ctx, hipStreamSynchronize(ctx->stream), what);
}

// A contiguous copy: HIP's own, but for downloads of whole doubles of up to 16 KB
// or from 2 MB on to pageable memory, which the staging buffers take in less time.
// us on an MI355X, HIP's / staged: downloads 4 KB 21.7 / 13.1, 16 KB 22.0 / 13.8, 24
// KB 10.3 / 13.9, 256 KB 20 / 23, 1 MB 62 / 63, 2 MB 122 / 115, 8 MB 482 / 363, 64 MB
// 3870 / 2370; uploads 4 KB 13.7 / 13.4, 64 KB 10.8 / 14.5, 1 MB 39 / 43, 64 MB
// 2360 / 2470.
static int host_copy(vx_ctx *ctx, void *dev, void *host, size_t bytes, bool up, const char *what) {
    if (bytes == 0) return vx_sync(ctx);
    const size_t n = bytes / sizeof(double);
    const bool size = bytes % sizeof(double) == 0 && (bytes <= (16 << 10) || bytes >= (2 << 20));
    if (!up && size && host && vx_device_range(ctx, (const double *)dev, n) && pageable(host) && stage_there(ctx))
        return staged_rows(ctx, (double *)dev, 1, (double *)host, 1, n, false, what);
    int rc = check_hip(ctx, up ? hipMemcpyAsync(dev, host, bytes, hipMemcpyHostToDevice, ctx->stream)
                               : hipMemcpyAsync(host, dev, bytes, hipMemcpyDeviceToHost, ctx->stream), what);
    return rc ? rc : vx_sync(ctx);
}

extern "C" {

int vx_memcpy_h2d(vx_ctx *ctx, void *dst, const void *src, size_t bytes) {
    if (int rc = not_recording(ctx, "vx_memcpy_h2d")) return rc;
    return host_copy(ctx, dst, const_cast<void *>(src), bytes, true, "h2d");
}

int vx_memcpy_d2h(vx_ctx *ctx, void *dst, const void *src, size_t bytes) {
    if (int rc = not_recording(ctx, "vx_memcpy_d2h")) return rc;
    return host_copy(ctx, const_cast<void *>(src), dst, bytes, false, "d2h");
}

int vx_memcpy_d2d(vx_ctx *ctx, void *dst, const void *src, size_t bytes) {
    return check_hip(ctx, hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToDevice, ctx->stream), "d2d");
}

__global__ void k_fill(double *dst, double v, size_t n) {
    size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x;
    size_t stride = (size_t)gridDim.x * blockDim.x;
    for (; i < n; i += stride) dst[i] = v;
}

int vx_fill(vx_ctx *ctx, double *dst, double value, size_t count) {
    if (count == 0) return VX_OK;
    size_t blocks = (count + 255) / 256;
    if (blocks > 65536) blocks = 65536;
    k_fill<<<(unsigned)blocks, 256, 0, ctx->stream>>>(dst, value, count);
    return check_launch(ctx, "fill");
}

int vx_event_record(vx_ctx *ctx, int slot) {
    if (slot < 0 || slot >= 8) return fail(ctx, VX_EINVAL, "event slot %d", slot);
    return check_hip(ctx, hipEventRecord(ctx->ev[slot], ctx->stream), "event record");
}

int vx_event_elapsed_ms(vx_ctx *ctx, int a, int b, float *ms) {
    if (a < 0 || a >= 8 || b < 0 || b >= 8 || !ms) return fail(ctx, VX_EINVAL, "event slots");
    int rc = check_hip(ctx, hipEventSynchronize(ctx->ev[b]), "event sync");
    if (rc) return rc;
    return check_hip(ctx, hipEventElapsedTime(ms, ctx->ev[a], ctx->ev[b]), "event elapsed");
}

int vx_timing_begin(vx_ctx *ctx, const char *kernel) {
    ctx->timed_kernel = kernel ? kernel : "";
    ctx->tcount = 0;
    return VX_OK;
}

int vx_timing_end(vx_ctx *ctx, double *total_ms, int *launches) {
    int rc = vx_sync(ctx);
    if (rc) return rc;
    double tot = 0.0;
    for (size_t k = 0; k < ctx->tcount; k++) {
        float ms = 0.0f;
        rc = check_hip(ctx, hipEventElapsedTime(&ms, ctx->tev[2 * k], ctx->tev[2 * k + 1]), "timing");
        if (rc) return rc;
        tot += ms;
    }
    if (total_ms) *total_ms = tot;
    if (launches) *launches = (int)ctx->tcount;
    ctx->timed_kernel.clear();
    ctx->tcount = 0;
    return VX_OK;
}

int32_t vx_plane_pitch(int32_t n_p) { return ((n_p + 4 + 7) / 8) * 8; }

size_t vx_plane_elems(int32_t n_x, int32_t n_p) {
    return (size_t)(n_x + 4) * (size_t)vx_plane_pitch(n_p);
}


int vx_graph_begin(vx_ctx *ctx) {
    if (ctx->capturing) return fail(ctx, VX_EINVAL, "a step graph is already being recorded");
    int rc = check_hip(ctx, hipStreamBeginCapture(ctx->stream, hipStreamCaptureModeThreadLocal),
                       "begin capture");
    if (rc == VX_OK) ctx->capturing = true;
    return rc;
}

int vx_graph_end(vx_ctx *ctx, vx_graph **out) {
    if (out) *out = nullptr;
    if (!ctx->capturing) return fail(ctx, VX_EINVAL, "no step graph is being recorded");
    ctx->capturing = false;
    hipGraph_t graph = nullptr;
    hipError_t e = hipStreamEndCapture(ctx->stream, &graph);
    if (e != hipSuccess || !graph) {
        if (graph) (void)hipGraphDestroy(graph);
        (void)hipGetLastError();
        return fail(ctx, VX_EHIP, "end capture: %s", hipGetErrorString(e));
    }
    if (!out) {  // discard
        (void)hipGraphDestroy(graph);
        return VX_OK;
    }
    hipGraphExec_t exec = nullptr;
    e = hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0);
    (void)hipGraphDestroy(graph);
    if (e != hipSuccess) return fail(ctx, VX_EHIP, "graph instantiate: %s", hipGetErrorString(e));
    vx_graph *g = new vx_graph;
    g->exec = exec;
    *out = g;
    return VX_OK;
}

int vx_graph_launch(vx_ctx *ctx, const vx_graph *g) {
    if (!g || !g->exec) return fail(ctx, VX_EINVAL, "null graph");
    if (int rc = not_recording(ctx, "vx_graph_launch")) return rc;
    return check_hip(ctx, hipGraphLaunch(g->exec, ctx->stream), "graph launch");
}

void vx_graph_destroy(vx_graph *g) {
    if (!g) return;
    if (g->exec) (void)hipGraphExecDestroy(g->exec);
    delete g;
}

int vx_upload_small(vx_ctx *ctx, void *dst, const void *src, size_t bytes) {
    if (bytes > (size_t)vx_ctx::RING_BYTES) return fail(ctx, VX_EINVAL, "upload of %zu bytes", bytes);
    if (int rc = not_recording(ctx, "vx_upload_small")) return rc;
    if (!ctx->ring) {
        int rc = check_hip(ctx, hipHostMalloc((void **)&ctx->ring, (size_t)vx_ctx::RING * vx_ctx::RING_BYTES),
                           "pinned ring");
        if (rc) return rc;
        for (auto &ev : ctx->ring_ev)
            if ((rc = check_hip(ctx, hipEventCreateWithFlags(&ev, hipEventDisableTiming), "ring event")))
                return rc;
    }
    const int k = ctx->ring_next;
    ctx->ring_next = (k + 1) % vx_ctx::RING;
    if (ctx->ring_pending[k]) {
        int rc = check_hip(ctx, hipEventSynchronize(ctx->ring_ev[k]), "ring slot wait");
        if (rc) return rc;
    }
    char *slot = ctx->ring + (size_t)k * vx_ctx::RING_BYTES;
    std::memcpy(slot, src, bytes);
    int rc = check_hip(ctx, hipMemcpyAsync(dst, slot, bytes, hipMemcpyHostToDevice, ctx->stream), "upload");
    if (rc) return rc;
    rc = check_hip(ctx, hipEventRecord(ctx->ring_ev[k], ctx->stream), "ring event record");
    ctx->ring_pending[k] = rc == VX_OK;
    return rc;
}


int vx_ctx_wait(vx_ctx *waiter, vx_ctx *signaller) {
    if (!waiter || !signaller) return VX_EINVAL;
    if (waiter->device != signaller->device) return fail(waiter, VX_EINVAL, "ctx wait across devices");
    if (!signaller->xev) {
        int rc = check_hip(waiter, hipEventCreateWithFlags(&signaller->xev, hipEventDisableTiming), "ctx event");
        if (rc) return rc;
    }
    int rc = check_hip(waiter, hipEventRecord(signaller->xev, signaller->stream), "ctx event record");
    if (rc) return rc;
    return check_hip(waiter, hipStreamWaitEvent(waiter->stream, signaller->xev, 0), "ctx stream wait");
}

size_t vx_ctx_live_bytes(vx_ctx *ctx) { return ctx ? ctx->live_bytes : 0; }


// Slot `slot` of a patch <-> a host array of (n_x + 2g) x (n_p + 2g) doubles,
// row-major (g = 0, 1, 2 ghost layers kept), one pass each way.
static int patch_copy(vx_ctx *ctx, const vx_patch *p, int slot, int ghosts, double *host, bool up) {
    if (!p || !host || slot < 0 || slot > 2 || ghosts < 0 || ghosts > 2 || !p->f[slot])
        return fail(ctx, VX_EINVAL, "patch copy: bad slot %d or ghosts %d", slot, ghosts);
    if (int rc = not_recording(ctx, "patch copy")) return rc;
    const size_t w = (size_t)(p->n_p + 2 * ghosts), h = (size_t)(p->n_x + 2 * ghosts);
    double *dev = p->f[slot] + (size_t)(2 - ghosts) * p->pitch + (2 - ghosts);
    const char *what = up ? "patch upload" : "patch download";
    // (an empty shape copies nothing, rows that lap over each other are HIP's to refuse too)
    const bool rows = p->n_x + 2 * ghosts > 0 && w > 0 && w <= (size_t)p->pitch && w * sizeof(double) <= vx_ctx::STAGE_BYTES;
    if (rows && vx_device_range(ctx, dev, (h - 1) * p->pitch + w) && pageable(host) && stage_there(ctx))
        return staged_rows(ctx, dev, p->pitch, host, w, h, up, what);
    hipError_t e = up ? hipMemcpy2DAsync(dev, sizeof(double) * p->pitch, host, sizeof(double) * w,
                                         sizeof(double) * w, h, hipMemcpyHostToDevice, ctx->stream)
                      : hipMemcpy2DAsync(host, sizeof(double) * w, dev, sizeof(double) * p->pitch,
                                         sizeof(double) * w, h, hipMemcpyDeviceToHost, ctx->stream);
    int rc = check_hip(ctx, e, what);
    return rc ? rc : vx_sync(ctx);
}

int vx_patch_upload(vx_ctx *ctx, const vx_patch *p, int slot, int ghosts, const double *host) {
    return patch_copy(ctx, p, slot, ghosts, const_cast<double *>(host), true);
}

int vx_patch_download(vx_ctx *ctx, const vx_patch *p, int slot, int ghosts, double *host) {
    return patch_copy(ctx, p, slot, ghosts, host, false);
}

}  // extern "C"
