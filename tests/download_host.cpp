// Host program around csrc/download.cpp: the HIP calls it makes, on two devices that are host
// memory, so that what it does with devices, streams, events and pinned memory shows without a
// GPU (tests/test_download_host.py builds and runs it).
#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <thread>
#include <vector>

#include "imh_host.h"

struct ihipStream_t {
    int device;
};
struct ihipEvent_t {
    int device;
};

static thread_local int t_device = 0;
static std::atomic<long> g_pinned{0}, g_events{0}, g_fail_copy{-1};

hipError_t hipGetDevice(int* d) { return *d = t_device, hipSuccess; }
hipError_t hipSetDevice(int d) {
    if (d < 0 || d > 1) return hipErrorInvalidDevice;
    t_device = d;
    return hipSuccess;
}
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
    size_t* q = (size_t*)malloc(n + 64);
    *q = n;
    g_pinned += (long)n;
    *p = (char*)q + 64;
    return hipSuccess;
}
hipError_t hipHostFree(void* p) {
    size_t* q = (size_t*)((char*)p - 64);
    g_pinned -= (long)*q;
    free(q);
    return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
    *e = new ihipEvent_t{t_device};
    ++g_events;
    return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t e) {
    delete e;
    --g_events;
    return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
    return e->device == s->device ? hipSuccess : hipErrorInvalidHandle;
}
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) {
    if (g_fail_copy >= 0 && g_fail_copy-- == 0) return hipErrorUnknown;
    memcpy(d, s, n);
    return hipSuccess;
}

static int g_bad = 0;
#define CHECK(x)                                                   \
    do {                                                           \
        if (!(x)) {                                                \
            printf("line %d: %s\n", __LINE__, #x);                 \
            ++g_bad;                                               \
        }                                                          \
    } while (0)

struct Sim {
    imh_ctx c;
    ihipStream_t st;
    Sim(int device) : st{device} {
        c.cfg.device = device;
        c.st = &st;
    }
    ~Sim() { imh::download_ring_release(c.dl_ring); }
    // whether n elements come back whole
    template <typename T>
    bool fetch(size_t n, hipError_t* err = nullptr) {
        std::vector<T> src(n);
        for (size_t i = 0; i < n; ++i) src[i] = T(i % 16777213) + T(st.device);
        std::vector<double> out(n, -1.0);
        bool staged = false;
        const hipError_t e = imh::download_staged(&c, src.data(), n, sizeof(T), out.data(), staged);
        if (err) *err = e;
        if (e != hipSuccess || !staged) return false;
        for (size_t i = 0; i < n; ++i)
            if (out[i] != double(src[i])) return false;
        return true;
    }
};

int main() {
    const long ring = 4 << 20;
    {   // sizes around the chunk and the ring, both precisions
        Sim a(0);
        for (size_t n : {size_t(1) << 16, (size_t(1) << 16) + 1, size_t(523), size_t(1) << 20}) {
            const size_t m = n < 1000 ? (size_t(1) << 19) + n : n;
            CHECK(a.fetch<double>(m));
            CHECK(a.fetch<float>(m));
        }
        bool staged = true;
        double x[4] = {1, 2, 3, 4}, y[4];
        CHECK(imh::download_staged(&a.c, x, 4, 8, y, staged) == hipSuccess && !staged);
    }
    CHECK(g_pinned == 0 && g_events == 0);
    {   // a context of a device that is not the calling thread's
        Sim b(1);
        CHECK(hipSetDevice(0) == hipSuccess);
        CHECK(b.fetch<double>(300000));
        CHECK(t_device == 0);
    }
    {   // many contexts share one ring per device, and give it back
        std::vector<Sim*> sims;
        for (int i = 0; i < 16; ++i) sims.push_back(new Sim(i & 1));
        for (Sim* s : sims) CHECK(s->fetch<float>(200000));
        CHECK(g_pinned <= 2 * ring);
        std::vector<std::thread> th;
        std::atomic<int> good{0};
        for (Sim* s : sims)
            th.emplace_back([&good, s] { good += s->fetch<double>(700001) && s->fetch<float>(900001); });
        for (std::thread& t : th) t.join();
        CHECK(good == 16);
        for (int i = 2; i < 16; ++i) delete sims[i];
        CHECK(g_pinned <= 2 * ring && g_pinned > 0);
        CHECK(sims[0]->fetch<double>(700001));
        delete sims[0];
        delete sims[1];
    }
    CHECK(g_pinned == 0 && g_events == 0);
    {   // a failed copy is an error of that call alone
        Sim a(0);
        for (long k : {0, 3, 9, 20}) {
            hipError_t e = hipSuccess;
            g_fail_copy = k;
            CHECK(!a.fetch<double>(3000000, &e));
            CHECK(e == hipErrorUnknown);
            g_fail_copy = -1;
            CHECK(a.fetch<double>(3000000));
        }
    }
    CHECK(g_pinned == 0 && g_events == 0);
    printf(g_bad ? "FAILED\n" : "OK\n");
    return g_bad != 0;
}
