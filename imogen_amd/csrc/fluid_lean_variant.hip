// One (precision, block size, cells per thread) variant of the lean fluid sweep
// (fluid_lean_impl.h); the build compiles this file once per entry of IMH_FLUID_VARIANTS
// with -DIMH_FLUID_ESZ=<4|8> -DIMH_FLUID_BS=<256|512|1024> -DIMH_FLUID_KMAX=<k>.
#ifndef IMH_LEAN_WAVES
#if IMH_FLUID_ESZ == 8
#define IMH_LEAN_WAVES (IMH_FLUID_KMAX <= 4 ? 3 : 2)
#else
#define IMH_LEAN_WAVES (IMH_FLUID_KMAX <= 4 ? 4 : 2)
#endif
#endif
#define IMH_LEAN_OCCUPANCY __attribute__((amdgpu_waves_per_eu(IMH_LEAN_WAVES)))
#include "fluid_lean_impl.h"

namespace imh {

#if IMH_FLUID_ESZ == 8
using LeanT = double;
#else
using LeanT = float;
#endif

hipError_t IMH_LEAN_LAUNCHER(IMH_FLUID_ESZ, IMH_FLUID_BS, IMH_FLUID_KMAX)(
    const void* args, const BatchTile* tiles, int ntiles, int nblocks, int d, bool mhd,
    int px, int form, hipStream_t st) {
    if (px > lean::PXMAX) return hipErrorInvalidValue;
    const FluidArgs<LeanT>* a = (const FluidArgs<LeanT>*)args;
    const size_t lds =
        (size_t)lean::lds_layout(IMH_FLUID_BS, px, IMH_FLUID_ESZ, form == LEAN_VISC).total;
#define IMH_LL(M, DD, F)                                                                    \
    if (mhd == M && d == DD && form == F) {                                                 \
        auto* fn = fluid_lean_kernel<LeanT, IMH_FLUID_BS, IMH_FLUID_KMAX, M, DD, F>;          \
        if (lds > 64 * 1024) {                                                              \
            hipError_t e = hipFuncSetAttribute((const void*)fn,                             \
                                               hipFuncAttributeMaxDynamicSharedMemorySize,  \
                                               160 * 1024);                                 \
            if (e != hipSuccess) return e;                                                  \
        }                                                                                   \
        hipLaunchKernelGGL(fn, dim3(nblocks), dim3(IMH_FLUID_BS), lds, st, a, tiles, ntiles); \
        return hipGetLastError();                                                           \
    }
#define IMH_LF(F) \
    IMH_LL(false, 0, F) IMH_LL(false, 1, F) IMH_LL(false, 2, F) IMH_LL(true, 0, F) \
    IMH_LL(true, 1, F) IMH_LL(true, 2, F)
    IMH_LF(LEAN_PLAIN) IMH_LF(LEAN_ENDS) IMH_LF(LEAN_VISC)
#undef IMH_LF
#undef IMH_LL
    return hipErrorInvalidValue;
}

}  // namespace imh
