// download.cpp -- a field from the device into the caller's (pageable) array.
//
// A copy straight into pageable memory runs at the pace at which one thread faults in the
// destination's fresh pages (3.7 GB/s), an FP32 field's through a temporary besides.  Here the
// device copies chunks into a ring of pinned buffers, and a few threads move them out,
// widening FP32 on the way, while the next chunks arrive.  Measured (ms, fresh destination,
// direct / 1 / 2 / 4 / 8 threads): FP64 134 MB 35.6 / 25.3 / 13.3 / 7.5 / 6.6, 8 MB 2.1 / 1.5 / 0.8 /
// 0.75 / 0.6, 2 MB 1.3 / 0.34 / 0.32 / 0.23 / 0.25; chunks of 1 and 2 MB instead of 512 KB: 134 MB
// with four threads 9.2 and 9.2.  So four threads, 512 KB chunks, two per thread.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <mutex>
#include <new>
#include <thread>

#include "imh_host.h"

namespace imh {

namespace {

constexpr size_t DL_CHUNK = 512 << 10;   // device bytes
constexpr int DL_THREADS = 4;
constexpr int DL_RING = 2 * DL_THREADS;  // buffer k % DL_RING belongs to thread k % DL_THREADS
// below, one chunk's copy costs less than the threads and events
constexpr size_t DL_MIN = 256 << 10;
constexpr int DL_DEVICES = 64;

}  // namespace

// The pinned ring of a device: made at the first large download from it, shared by its contexts
// (one download at a time: four threads move a ring's chunks at the pace of the bus), given
// back with the last context that has used it.
struct DownloadRing {
    int device = 0;
    int users = 0;               // contexts that hold it, under g_rings_mutex
    std::mutex busy;             // one download at a time
    char* buf = nullptr;
    hipEvent_t ev[DL_RING] = {};
};

static std::mutex g_rings_mutex;
static DownloadRing* g_rings[DL_DEVICES];

static void ring_free(DownloadRing* r) {
    for (hipEvent_t& e : r->ev)
        if (e) (void)hipEventDestroy(e);
    if (r->buf) (void)hipHostFree(r->buf);
    delete r;
}

void download_ring_release(DownloadRing* r) {
    if (!r) return;
    std::lock_guard<std::mutex> lock(g_rings_mutex);
    if (--r->users > 0) return;
    g_rings[r->device] = nullptr;
    ring_free(r);
}

// The ring of the context's device, which is current; nullptr: no pinned memory.
static DownloadRing* download_ring(imh_ctx* c) {
    std::lock_guard<std::mutex> lock(g_rings_mutex);
    if (c->dl_ring) return c->dl_ring;
    if (c->cfg.device < 0 || c->cfg.device >= DL_DEVICES) return nullptr;
    DownloadRing*& r = g_rings[c->cfg.device];
    if (!r) {
        r = new (std::nothrow) DownloadRing();
        hipError_t e = r ? hipHostMalloc((void**)&r->buf, DL_CHUNK * DL_RING, hipHostMallocDefault)
                         : hipErrorOutOfMemory;
        for (int i = 0; i < DL_RING && e == hipSuccess; ++i)
            e = hipEventCreateWithFlags(&r->ev[i], hipEventDisableTiming);
        if (e != hipSuccess) {
            (void)hipGetLastError();
            if (r) ring_free(r);
            return r = nullptr;
        }
        r->device = c->cfg.device;
    }
    r->users += 1;
    return c->dl_ring = r;
}

// The calling thread's current device while an object lives: events belong to the device that
// is current when they are made, and are recorded on that device's streams only.
namespace {
struct OnDevice {
    int before = -1;
    explicit OnDevice(int device) {
        if (hipGetDevice(&before) != hipSuccess || before == device ||
            hipSetDevice(device) != hipSuccess)
            before = -1;
    }
    ~OnDevice() {
        if (before >= 0) (void)hipSetDevice(before);
    }
};
}  // namespace

// n elements of esz bytes (4: float) at src into out, on the context's stream, which is idle.
// `staged` is false when the copy is left to the caller: a small field, or no pinned memory.
hipError_t download_staged(imh_ctx* c, const void* src, size_t n, size_t esz, double* out,
                           bool& staged) {
    staged = false;
    const size_t bytes = n * esz;
    if (bytes < DL_MIN) return hipSuccess;
    const OnDevice on(c->cfg.device);
    DownloadRing* r = download_ring(c);
    if (!r) return hipSuccess;
    std::lock_guard<std::mutex> lock(r->busy);
    staged = true;
    const int nchunk = int((bytes + DL_CHUNK - 1) / DL_CHUNK);
    auto issue = [&](int k) -> hipError_t {
        const size_t off = (size_t)k * DL_CHUNK, len = std::min(DL_CHUNK, bytes - off);
        hipError_t e = hipMemcpyAsync(r->buf + (k % DL_RING) * DL_CHUNK, (const char*)src + off, len,
                                      hipMemcpyDeviceToHost, c->st);
        return e == hipSuccess ? hipEventRecord(r->ev[k % DL_RING], c->st) : e;
    };
    hipError_t err[DL_THREADS] = {};
    for (int k = 0; k < DL_RING && k < nchunk; ++k)
        if ((err[0] = issue(k)) != hipSuccess) break;
    // a thread reuses a buffer only after it has moved the chunk before out of it
    auto work = [&](int w) {
        hipError_t e = hipSuccess;
        for (int k = w; k < nchunk && e == hipSuccess; k += DL_THREADS) {
            e = hipEventSynchronize(r->ev[k % DL_RING]);
            if (e != hipSuccess) break;
            const size_t off = (size_t)k * DL_CHUNK, len = std::min(DL_CHUNK, bytes - off);
            const char* b = r->buf + (k % DL_RING) * DL_CHUNK;
            if (esz == sizeof(double)) {
                memcpy((char*)out + off, b, len);
            } else {
                double* o = out + off / sizeof(float);
                const float* f = (const float*)b;
                for (size_t i = 0; i < len / sizeof(float); ++i) o[i] = f[i];
            }
            if (k + DL_RING < nchunk) e = issue(k + DL_RING);
        }
        err[w] = e;
    };
    if (err[0] == hipSuccess) {
        std::thread th[DL_THREADS];
        int started = 1;
        try {
            for (; started < DL_THREADS && started < nchunk; ++started)
                th[started] = std::thread([&, started] {
                    err[started] = hipSetDevice(c->cfg.device);
                    if (err[started] == hipSuccess) work(started);
                });
        } catch (...) {  // no more threads: their chunks below
        }
        work(0);
        for (int w = started; w < DL_THREADS && w < nchunk; ++w) work(w);
        for (int w = 1; w < started; ++w) th[w].join();
    }
    hipError_t e = hipSuccess;
    for (hipError_t x : err)
        if (e == hipSuccess) e = x;
    // an error can leave copies in flight
    if (e != hipSuccess) (void)hipStreamSynchronize(c->st);
    return e;
}

}  // namespace imh
