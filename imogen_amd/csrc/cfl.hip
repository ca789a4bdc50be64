// cfl.hip -- CFL timestep reduction (time/TimeManager.m:55-99) with the device-side time
// bookkeeping, and the compensated conservation totals.
//
// Two launches per time update: every block reduces |p_i/rho| + c_s, i = 1..3, over its cells
// (16-byte loads of four consecutive cells, wavefront shuffles, one LDS pass) and stores its
// three maxima; a block per simulation then reduces those, computes dt and advances time and
// iteration.  A simulation of one tile (up to 4096 cells) is finished by the first launch.
// Whether a simulation runs at all both evaluate from its time state.  dt is computed on the
// device, so an iteration needs no host round trip and can be replayed as a hipGraph.
//
// Bound by HBM on large grids, by FP64 issue on FP32 fields: one reciprocal of rho serves
// its four quotients (LMath: rounded as the divisions are).  CFL reduction, us, against one
// cell per load and three 64-bit atomics per block on the same addresses: FP64 125^3 45 -> 21,
// 512^2 25 -> 11, FP32 1024^2 37 -> 14, 192^3 78 -> 34 (141 MB).  The loop body's bookkeeping
// launches: 4 -> 1, or none up to 4096 cells.  Finding the last block by a ticket instead of a
// second launch loses (1024^2 38 us, 256^3 186: each block's release and acquire).
#include "cfl_impl.h"
#include "imh_common.h"
#include "imh_host.h"
#include "imh_kernels.h"

namespace imh {

constexpr int CFL_BS = 256;

template <typename T>
__global__ void __launch_bounds__(CFL_BS) cfl_kernel(const CflArgs<T>* args, const BatchTile* tiles,
                                                     int ntiles, int gate, int step, int count) {
    __shared__ double s_red[3][CFL_BS / 64];
    for (int r = 0;; ++r) {
        const BatchTile* tl = tiles;
        asm volatile("" : "+s"(tl));  // opaque: one copy of the body serves both forms
        int arg = 0;
        long long tile;
        if (tl) {
            const int t = xcd_round_tile(r, ntiles);
            if (t < 0) break;
            uniform_tile(tl, t, arg, tile);
        } else {
            if (r > 0 || (int)blockIdx.x >= ntiles) break;
            tile = blockIdx.x;
        }
        const CflArgs<T> a = uniform_load(&args[arg]);
        const SimParams par = uniform_load(a.par);
        const int run = cfl_runs(*a.sim, par, gate, step);
        double m[3] = {NAN, NAN, NAN};
        if (run > 0) {
            const long long c0 = tile * a.chunk;
            cfl_cells<CFL_BS>(a, c0, c0 + a.chunk < a.ncell ? c0 + a.chunk : a.ncell, m);
            block_max<CFL_BS>(m, s_red);
        }
        if (a.chunk >= a.ncell) {
            __syncthreads();  // every thread has read the time state
            if (run >= 0 && threadIdx.x == 0) cfl_finish(*a.sim, par, run, gate, step, count, m);
        } else if (run > 0 && threadIdx.x == 0) {
#pragma unroll
            for (int k = 0; k < 3; ++k) gmem(a.part)[3 * tile + k] = m[k];
        }
        __syncthreads();
    }
}

// The second launch: block s finishes simulation s (of those with several tiles).
template <typename T>
__global__ void __launch_bounds__(CFL_BS) cfl_finish_kernel(const CflArgs<T>* args, int gate,
                                                            int step, int count) {
    __shared__ double s_red[3][CFL_BS / 64];
    const CflArgs<T> a = uniform_load(&args[blockIdx.x]);
    if (a.chunk >= a.ncell) return;
    const SimParams par = uniform_load(a.par);
    const int run = cfl_runs(*a.sim, par, gate, step);
    if (run < 0) return;
    double m[3] = {NAN, NAN, NAN};
    if (run) {
        const int ntile = int((a.ncell + a.chunk - 1) / a.chunk);
        for (int t = threadIdx.x; t < ntile; t += CFL_BS)
#pragma unroll
            for (int k = 0; k < 3; ++k) m[k] = fmax(m[k], gmem(a.part)[3 * t + k]);
    }
    block_max<CFL_BS>(m, s_red);
    if (threadIdx.x == 0) cfl_finish(*a.sim, par, run, gate, step, count, m);
}

template <typename T>
hipError_t launch_cfl(const CflArgs<T>* args, const BatchTile* tiles, int ntiles, int nblocks,
                      int gate, int step, int count, hipStream_t st) {
    if (ntiles == 0) return hipSuccess;
    hipLaunchKernelGGL((cfl_kernel<T>), dim3(nblocks), dim3(CFL_BS), 0, st, args, tiles, ntiles,
                       gate, step, count);
    return hipGetLastError();
}
template <typename T>
hipError_t launch_cfl_finish(const CflArgs<T>* args, int nsims, int gate, int step, int count,
                             hipStream_t st) {
    hipLaunchKernelGGL((cfl_finish_kernel<T>), dim3(nsims), dim3(CFL_BS), 0, st, args, gate, step,
                       count);
    return hipGetLastError();
}

template hipError_t launch_cfl<double>(const CflArgs<double>*, const BatchTile*, int, int, int, int,
                                       int, hipStream_t);
template hipError_t launch_cfl<float>(const CflArgs<float>*, const BatchTile*, int, int, int, int,
                                      int, hipStream_t);
template hipError_t launch_cfl_finish<double>(const CflArgs<double>*, int, int, int, int,
                                              hipStream_t);
template hipError_t launch_cfl_finish<float>(const CflArgs<float>*, int, int, int, int, hipStream_t);

// Cells per tile: a whole simulation of up to 4096; else at most CFL_TILES tiles of a
// multiple of four cells per thread.
long long cfl_chunk(long long ncell) {
    const long long per = 4LL * CFL_BS;
    if (ncell <= 4 * per) return 4 * per;
    return per * ((ncell + per * CFL_TILES - 1) / (per * CFL_TILES));
}

// The top of the loop body on its own (direct calls of parts of it), one thread per
// simulation over an array of per-simulation pointers.
__global__ void begin_iteration_kernel(SimDev* const* sim, const SimParams* const* p, int nsims,
                                       int unconditional) {
    int s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= nsims) return;
    SimDev& d = *sim[s];
    d.active = (unconditional || running(d, *p[s])) ? 1 : 0;
}

static inline int nblk(int n) { return (n + 255) / 256; }

hipError_t launch_begin_iteration(SimDev* const* sim, const SimParams* const* p, int nsims,
                                  int unconditional, hipStream_t st) {
    hipLaunchKernelGGL(begin_iteration_kernel, dim3(nblk(nsims)), dim3(256), 0, st, sim, p, nsims,
                       unconditional);
    return hipGetLastError();
}

// ---- conservation totals -------------------------------------------------------------
// Neumaier-compensated sums; every block owns a fixed contiguous range and combines its
// 256 partials in a fixed binary tree, the block partials are combined the same way, so
// the result is independent of timing and of the device.

struct CSum {
    double s, c;
};

__device__ inline CSum csum_add(CSum a, double x) {
    double t = a.s + x;
    double e = (fabs(a.s) >= fabs(x)) ? (a.s - t) + x : (x - t) + a.s;
    return {t, a.c + e};
}

__device__ inline CSum csum_merge(CSum a, CSum b) {
    CSum r = csum_add(a, b.s);
    r.c += b.c;
    return r;
}

template <typename T>
__global__ void __launch_bounds__(256) csum_blocks_kernel(const T* x, long long n, long long chunk,
                                                          double* partials) {
    __shared__ double ss[256], sc[256];
    const long long b0 = (long long)blockIdx.x * chunk;
    long long b1 = b0 + chunk;
    if (b1 > n) b1 = n;
    CSum acc = {0.0, 0.0};
    const long long per = (chunk + 255) / 256;
    long long s0 = b0 + (long long)threadIdx.x * per;
    long long s1 = s0 + per;
    if (s1 > b1) s1 = b1;
    for (long long i = s0; i < s1; ++i) acc = csum_add(acc, double(x[i]));
    ss[threadIdx.x] = acc.s;
    sc[threadIdx.x] = acc.c;
    __syncthreads();
    for (int w = 128; w >= 1; w >>= 1) {
        if ((int)threadIdx.x < w) {
            CSum r = csum_merge({ss[threadIdx.x], sc[threadIdx.x]},
                                {ss[threadIdx.x + w], sc[threadIdx.x + w]});
            ss[threadIdx.x] = r.s;
            sc[threadIdx.x] = r.c;
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        partials[2 * blockIdx.x] = ss[0];
        partials[2 * blockIdx.x + 1] = sc[0];
    }
}

__global__ void csum_final_kernel(const double* partials, int nb, double* out) {
    if (threadIdx.x != 0 || blockIdx.x != 0) return;
    CSum acc = {0.0, 0.0};
    for (int b = 0; b < nb; ++b) acc = csum_merge(acc, {partials[2 * b], partials[2 * b + 1]});
    *out = acc.s + acc.c;
}

template <typename T>
hipError_t launch_conservation(const T* const* fields, int nfields, long long ncell,
                               double* partials, int nblocks, double* out, hipStream_t st) {
    long long chunk = (ncell + nblocks - 1) / nblocks;
    if (chunk < 1) chunk = 1;
    int nb = int((ncell + chunk - 1) / chunk);
    for (int f = 0; f < nfields; ++f) {
        hipLaunchKernelGGL((csum_blocks_kernel<T>), dim3(nb), dim3(256), 0, st, fields[f], ncell,
                           chunk, partials + (size_t)f * 2 * nblocks);
        hipLaunchKernelGGL(csum_final_kernel, dim3(1), dim3(1), 0, st,
                           partials + (size_t)f * 2 * nblocks, nb, out + f);
    }
    return hipGetLastError();
}

template hipError_t launch_conservation<double>(const double* const*, int, long long, double*, int,
                                                double*, hipStream_t);
template hipError_t launch_conservation<float>(const float* const*, int, long long, double*, int,
                                               double*, hipStream_t);

// ---- device copy probe ----------------------------------------------------------------
// A plain streaming copy (16-byte vectors, grid-stride): the reference kernel of known
// traffic for scaling HBM counters and the measured copy bandwidth beside the roofline.
__global__ void __launch_bounds__(256) copy_probe_kernel(const float4* __restrict__ src,
                                                         float4* __restrict__ dst, long long n) {
    for (long long i = (long long)blockIdx.x * 256 + threadIdx.x; i < n;
         i += (long long)gridDim.x * 256)
        dst[i] = src[i];
}

}  // namespace imh

extern "C" int imh_copy_probe(size_t bytes, int reps, double* ms_per_copy) {
    using namespace imh;
    if (bytes < 16 || reps < 1 || !ms_per_copy) return fail(IMH_EINVAL, "bad argument");
    const long long n = (long long)(bytes / 16);
    void *a = nullptr, *b = nullptr;
    hipEvent_t e0 = nullptr, e1 = nullptr;
    hipStream_t st = nullptr;
    hipError_t e = hipMalloc(&a, n * 16);
    if (e == hipSuccess) e = hipMalloc(&b, n * 16);
    if (e == hipSuccess) e = hipMemset(a, 0, n * 16);
    if (e == hipSuccess) e = hipStreamCreateWithFlags(&st, hipStreamNonBlocking);
    if (e == hipSuccess) e = hipEventCreate(&e0);
    if (e == hipSuccess) e = hipEventCreate(&e1);
    int nb = 0;
    if (e == hipSuccess) {
        hipDeviceProp_t prop;
        e = hipGetDeviceProperties(&prop, 0);
        nb = prop.multiProcessorCount * 8;
    }
    if (e == hipSuccess) {
        hipLaunchKernelGGL(copy_probe_kernel, dim3(nb), dim3(256), 0, st, (const float4*)a,
                           (float4*)b, n);  // warm-up
        e = hipEventRecord(e0, st);
    }
    for (int r = 0; r < reps && e == hipSuccess; ++r) {
        hipLaunchKernelGGL(copy_probe_kernel, dim3(nb), dim3(256), 0, st, (const float4*)a,
                           (float4*)b, n);
        e = hipGetLastError();
    }
    if (e == hipSuccess) e = hipEventRecord(e1, st);
    if (e == hipSuccess) e = hipEventSynchronize(e1);
    float ms = 0;
    if (e == hipSuccess) e = hipEventElapsedTime(&ms, e0, e1);
    if (e0) (void)hipEventDestroy(e0);
    if (e1) (void)hipEventDestroy(e1);
    if (st) (void)hipStreamDestroy(st);
    if (a) (void)hipFree(a);
    if (b) (void)hipFree(b);
    if (e != hipSuccess) return hip_fail(e, "copy probe");
    *ms_per_copy = ms / reps;
    return IMH_OK;
}
