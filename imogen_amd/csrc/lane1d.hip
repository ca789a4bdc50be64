// lane1d.hip -- one launch per batched iteration for the one-dimensional MHD simulations
// of a batch (FP32 bulk).
//
// A 1-D simulation (grid N x 1 x 1) is one pencil: every sweep of its iteration is a
// single tile, so the per-launch plan of the batch spends about a dozen grid-wide
// launches per iteration on work that one workgroup holds.  Here one workgroup runs the simulation's whole flux call (flux.m:37-62 for X = 1, the only
// direction with >= 3 cells) back to back, with workgroup barriers between the steps
// (one workgroup per simulation):
//
//   order +1: relaxingFluid(X=1); magnetFlux(X=1, I=[2 3]): advection + CT for I = 2, then
//             I = 3 (relaxingMagnet.m:15-60); updateCellCentered of mag(3) and mag(1)
//   order -1: magnetFlux(X=1, I=[3 2]); updateCellCentered of mag(2) and mag(1);
//             relaxingFluid(X=1)
//
// The bodies are those of the per-launch kernels (fluid_lean_body, mag_flow_body,
// mag_ct_body), on argument blocks whose tile is one pencil over
// the workgroup (LANE1D_BS threads of LANE1D_KMAX, 3/4, 1/2 or 1/4 of it cells each: the
// bodies are instantiated for all four, sharing their LDS, and a simulation runs the
// smallest that holds its pencil), so the results are those of the per-launch plan bit for
// bit.  The time step and the iteration count come from the batch-wide time update before.
// The state stays in the workgroup's L2 between the steps.  Bound by the latency of the longest pencils' chain (128 simulations of 256..4096
// cells: 130 us per iteration; 228 with the general fluid and magnet bodies, 181 with the lean
// fluid body alone); two waves per SIMD, as four (128 registers) spill the 8-cell body.
#include "fluid_lean_impl.h"
#include "magnet_lean_impl.h"

namespace imh {

namespace {

// The flux call of one simulation with KC cells per thread (the fluid and magnet bodies
// instantiated for that many): a short pencil does not run the longest pencil's body.
template <typename T, int KC>
__device__ __forceinline__ void lane1d_run(const Lane1dArgs<T>& a, char* s_fluid, T* s_mag) {
    double dt;
    if (!sweep_runs(a.fa, dt)) return;
    // steps 0 and 3: the fluid sweep; 1: magnetFlux(X=1, I=[2 3]) (order +1); 2:
    // magnetFlux(X=1, I=[3 2]) (order -1).  One call site per body (they are large).
    for (int step = 0; step < 4; ++step) {
        if (step == 0 || step == 3) {
            fluid_lean_body<T, LANE1D_BS, KC, true, 0>(a.fa, 0, s_fluid, dt);
        } else {
            for (int j = 0; j < 2; ++j) {
                mag_flow_body<T, 0, true>(a.ml[step - 1], j, 0, s_mag, dt);
                __syncthreads();
            }
            mag_ct_body<T, 0, true>(a.ml[step - 1], 0, s_mag, dt);
        }
        __syncthreads();
    }
}

#ifndef IMH_LANE1D_WAVES
#define IMH_LANE1D_WAVES 2
#endif
template <typename T>
__global__ void __launch_bounds__(LANE1D_BS) __attribute__((amdgpu_waves_per_eu(IMH_LANE1D_WAVES)))
lane1d_kernel(const Lane1dArgs<T>* args,
                                                           int nsims) {
    // the magnet rows of the longest pencil
    __shared__ __attribute__((aligned(16))) T s_mag[2 * mag_lean_row(true, LANE1D_NMAX)];
    __shared__ __attribute__((aligned(16))) char s_fluid[lean::lds_layout(LANE1D_BS, 1, sizeof(T)).total];
    const int s = blockIdx.x;
    if (s >= nsims) return;
    const Lane1dArgs<T>& a = args[s];
    // cells per thread of this simulation (its fluid tile's K), uniform over the block
    const int kc = __builtin_amdgcn_readfirstlane(a.fa.K);
    if (kc <= LANE1D_KMAX / 4)
        lane1d_run<T, LANE1D_KMAX / 4>(a, s_fluid, s_mag);
    else if (kc <= LANE1D_KMAX / 2)
        lane1d_run<T, LANE1D_KMAX / 2>(a, s_fluid, s_mag);
    else if (kc <= 3 * LANE1D_KMAX / 4)
        lane1d_run<T, 3 * LANE1D_KMAX / 4>(a, s_fluid, s_mag);
    else
        lane1d_run<T, LANE1D_KMAX>(a, s_fluid, s_mag);
}

}  // namespace

hipError_t launch_lane1d(const void* args, int nsims, hipStream_t st) {
    if (nsims <= 0) return hipSuccess;
    hipLaunchKernelGGL(lane1d_kernel<float>, dim3(nsims), dim3(LANE1D_BS), 0, st,
                       (const Lane1dArgs<float>*)args, nsims);
    return hipGetLastError();
}

}  // namespace imh
