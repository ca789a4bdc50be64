// One (precision, block size, KMAX) variant of the general fluid sweep; the build compiles
// this file once per entry of IMH_FLUID_VARIANTS with -DIMH_FLUID_ESZ=<4|8>
// -DIMH_FLUID_BS=<256|512> -DIMH_FLUID_KMAX=<k>.
//
// FP32 chunks of at most 4 cells fit in 128 registers without spilling: those variants
// ask the register allocator for 4 waves per SIMD (the allocator otherwise spends the
// 256 registers a 512-thread block allows, leaving 2).
#if !defined(IMH_FLUID_WAVES_PER_EU) && IMH_FLUID_ESZ == 4 && IMH_FLUID_KMAX <= 4
#define IMH_FLUID_WAVES_PER_EU 4
#endif
#include "fluid_sweep_impl.h"

namespace imh {

#if IMH_FLUID_ESZ == 8
using FluidT = double;
#else
using FluidT = float;
#endif

hipError_t IMH_FLUID_LAUNCHER(IMH_FLUID_ESZ, IMH_FLUID_BS, IMH_FLUID_KMAX)(
    const void* args, const BatchTile* tiles, int ntiles, int nblocks, bool mhd, hipStream_t st) {
    const FluidArgs<FluidT>* a = (const FluidArgs<FluidT>*)args;
    auto* fn = mhd ? fluid_sweep_batch_kernel<FluidT, IMH_FLUID_BS, IMH_FLUID_KMAX, true>
                   : fluid_sweep_batch_kernel<FluidT, IMH_FLUID_BS, IMH_FLUID_KMAX, false>;
    hipLaunchKernelGGL(fn, dim3(nblocks), dim3(IMH_FLUID_BS), 0, st, a, tiles, ntiles);
    return hipGetLastError();
}

}  // namespace imh
