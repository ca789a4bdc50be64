// The lean magnetic sweep (magnet_lean_impl.h) of one precision; the build compiles this
// file with -DIMH_MAG_ESZ=8 and -DIMH_MAG_ESZ=4.
#include "magnet_lean_impl.h"

namespace imh {

#if IMH_MAG_ESZ == 8
using MagLeanT = double;
#else
using MagLeanT = float;
#endif
#ifndef IMH_MLEAN_WAVES
#define IMH_MLEAN_WAVES 3
#endif

namespace {

// The advection (FLOW) of a tile, or its CT.  Advection tiles 2p and 2p + 1 are the two
// components on pencil group p (their reads of the mass and the momentum meet in one L2).
template <typename T, int D, bool FLOW, bool TRK>
__global__ void __launch_bounds__(MLEAN_BS) __attribute__((amdgpu_waves_per_eu(IMH_MLEAN_WAVES)))
magnet_lean_kernel(const MagnetLeanArgs<T>* args, const BatchTile* tiles, int ntiles) {
    extern __shared__ __attribute__((aligned(16))) unsigned char mlean_lds[];
    T* const lds = reinterpret_cast<T*>(mlean_lds);
    for (int r = 0;; ++r) {
        // opaque: one copy of the body serves both forms
        const BatchTile* tl = tiles;
        asm volatile("" : "+s"(tl));
        int arg = 0;
        long long tile;
        if (tl) {
            const int t = xcd_round_tile(r, ntiles);
            if (t < 0) break;
            uniform_tile(tl, t, arg, tile);
        } else {
            if (r > 0 || (int)blockIdx.x >= ntiles) break;
            tile = xcd_tile(blockIdx.x, ntiles);
        }
        double dt;
        if (sweep_runs(args[arg], dt)) {
            if constexpr (FLOW) mag_flow_body<T, D, TRK>(args[arg], int(tile & 1), tile >> 1, lds, dt);
            else mag_ct_body<T, D, TRK>(args[arg], tile, lds, dt);
        }
        __syncthreads();
    }
}

}  // namespace

template <>
hipError_t launch_magnet_lean<MagLeanT>(int which, const MagnetLeanArgs<MagLeanT>* args,
                                        const BatchTile* tiles, int ntiles, int nblocks, int d,
                                        bool trk, size_t lds, hipStream_t st) {
    if (ntiles == 0) return hipSuccess;
    if (lds > 150 * 1024) return hipErrorInvalidValue;
#define IMH_ML(W, DD, TK)                                                                       \
    if (which == W && d == DD && trk == TK) {                                                        \
        auto* fn = magnet_lean_kernel<MagLeanT, DD, W == 0, TK>;                            \
        if (lds > 64 * 1024) {                                                              \
            hipError_t e = hipFuncSetAttribute((const void*)fn,                             \
                                               hipFuncAttributeMaxDynamicSharedMemorySize,  \
                                               150 * 1024);                                 \
            if (e != hipSuccess) return e;                                                  \
        }                                                                                   \
        hipLaunchKernelGGL(fn, dim3(nblocks), dim3(MLEAN_BS), lds, st, args, tiles, ntiles);      \
        return hipGetLastError();                                                           \
    }
    IMH_ML(0, 0, false) IMH_ML(0, 1, false) IMH_ML(0, 2, false)
    IMH_ML(0, 0, true) IMH_ML(0, 1, true) IMH_ML(0, 2, true)
    IMH_ML(1, 0, false) IMH_ML(1, 1, false) IMH_ML(1, 2, false)
    IMH_ML(1, 0, true) IMH_ML(1, 1, true) IMH_ML(1, 2, true)
#undef IMH_ML
    return hipErrorInvalidValue;
}

}  // namespace imh
