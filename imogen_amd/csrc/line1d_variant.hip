// line1d_variant.hip -- several iterations of one 1-D simulation (grid N x 1 x 1) in one launch,
// compiled with -DIMH_LINE_ESZ=8 and -DIMH_LINE_ESZ=4.
//
// A 1-D simulation is one pencil: every launch of its iteration is one workgroup's work, and
// the iteration's time is that of its launches (time update, two fluid sweeps, with a
// magnetic field four magnet launches more).  Here one workgroup runs whole iterations back
// to back: TimeManager.update over the pencil, flux call +1, flux call -1 (flux.m:37-62 for
// X = 1, the only direction with >= 3 cells; source terms and viscosity take the launches),
// the iteration count, until `iterations` are done or the run has ended.  The bodies are
// those of the launches (cfl_impl.h, fluid_lean_body, mag_flow_body, mag_ct_body) and so are
// the results, bit for bit.  The time state lives in LDS in between: scalar loads would not
// see it change within a launch.  As few cells per thread as hold the pencil: the chain of
// one tile is all there is.  Measured, us per iteration against a
// graph of the launches: hydro FP32 257 cells 35 -> 18, FP64 1024 cells 38 -> 27; MHD FP32 1024
// cells 34, FP64 43.  Bound by the latency of the chain at two waves per SIMD.
#include "cfl_impl.h"
#include "magnet_lean_impl.h"

#include <algorithm>

namespace imh {

#if IMH_LINE_ESZ == 8
using LineT = double;
#else
using LineT = float;
#endif

namespace {

// A value that is the same for all lanes, into scalar registers.
__device__ __forceinline__ double uniform(double x) {
    typedef int I2 __attribute__((ext_vector_type(2)));
    I2 v = __builtin_bit_cast(I2, x);
    v.x = __builtin_amdgcn_readfirstlane(v.x);
    v.y = __builtin_amdgcn_readfirstlane(v.y);
    return __builtin_bit_cast(double, v);
}

template <typename T, int K, bool MHD>
__global__ void __launch_bounds__(LINE1D_BS)
line1d_kernel(const FluidArgs<T>* fa, const MagnetLeanArgs<T>* ml0, const MagnetLeanArgs<T>* ml1,
              const CflArgs<T>* ca, int mag, int iterations) {
    extern __shared__ __attribute__((aligned(16))) char line_lds[];
    __shared__ double s_red[3][LINE1D_BS / 64];
    __shared__ SimDev s_sim;
    const CflArgs<T> c = uniform_load(ca);
    const SimParams par = uniform_load(c.par);
    if (threadIdx.x == 0) s_sim = *c.sim;
    __syncthreads();
    for (int it = 0; it < iterations; ++it) {
        bool ended = false;
        for (int step = 1; step <= 2; ++step) {
            if (step == 1 || par.update_mode == 0) {
                const int gate = step == 1 ? CFL_RUNNING : CFL_ACTIVE;
                const int run = cfl_runs(s_sim, par, gate, step);
                double m[3] = {NAN, NAN, NAN};
                if (run) cfl_cells<LINE1D_BS>(c, 0, c.ncell, m);
                block_max<LINE1D_BS>(m, s_red);
                __syncthreads();  // every thread has read the time state
                if (threadIdx.x == 0) cfl_finish(s_sim, par, run, gate, step, 1, m);
                __syncthreads();
            }
            ended = !__builtin_amdgcn_readfirstlane(s_sim.active);
            if (ended) break;
            const double dt = uniform(s_sim.dt);
            // order +1: fluid, then magnet; order -1: magnet, then fluid
            for (int op = 0; op < 2; ++op) {
                if (op == step - 1) {
                    fluid_lean_body<T, LINE1D_BS, K, MHD, 0>(*fa, 0, line_lds, dt);
                    __syncthreads();
                } else if (MHD && mag) {
                    const MagnetLeanArgs<T>& ml = step == 1 ? *ml0 : *ml1;
                    T* const lds = reinterpret_cast<T*>(line_lds);
                    for (int j = 0; j < 2; ++j) {
                        mag_flow_body<T, 0, true>(ml, j, 0, lds, dt);
                        __syncthreads();
                    }
                    mag_ct_body<T, 0, true>(ml, 0, lds, dt);
                    __syncthreads();
                }
            }
        }
        if (ended) break;
    }
    __syncthreads();
    if (threadIdx.x == 0) *c.sim = s_sim;
}

}  // namespace

template <>
hipError_t launch_line1d<LineT>(const FluidArgs<LineT>* fa, const MagnetLeanArgs<LineT>* const ml[2],
                                const CflArgs<LineT>* ca, int N, bool mhd, bool mag,
                                int iterations, hipStream_t st) {
    size_t lds = (size_t)lean::lds_layout(LINE1D_BS, 1, sizeof(LineT)).total;
    if (mag) {
        const size_t m = std::max(mag_lean_lds(0, 0, N, 1, sizeof(LineT)),
                                  mag_lean_lds(1, 0, N, 1, sizeof(LineT)));
        lds = std::max(lds, m);
    }
#define IMH_LINE(K, M)                                                                      \
    if (N <= K * LINE1D_BS && mhd == M) {                                                   \
        auto* fn = line1d_kernel<LineT, K, M>;                                              \
        if (lds > 64 * 1024) {                                                              \
            hipError_t e = hipFuncSetAttribute((const void*)fn,                             \
                                               hipFuncAttributeMaxDynamicSharedMemorySize,  \
                                               150 * 1024);                                 \
            if (e != hipSuccess) return e;                                                  \
        }                                                                                   \
        hipLaunchKernelGGL(fn, dim3(1), dim3(LINE1D_BS), lds, st, fa, ml[0], ml[1], ca,     \
                           mag ? 1 : 0, iterations);                                        \
        return hipGetLastError();                                                           \
    }
    IMH_LINE(1, false) IMH_LINE(1, true) IMH_LINE(2, false) IMH_LINE(2, true)
    IMH_LINE(4, false) IMH_LINE(4, true) IMH_LINE(8, false) IMH_LINE(8, true)
#undef IMH_LINE
    return hipErrorInvalidValue;
}

}  // namespace imh
