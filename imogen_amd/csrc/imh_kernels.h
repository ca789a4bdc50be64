// imh_kernels.h -- kernel argument blocks and launcher declarations.
#pragma once

#include "imh_common.h"

namespace imh {

constexpr int MAX_FADE = 64;

// BC modes [side][dim] packed 4 bits each (kernel arguments are never indexed at run
// time: that would copy the whole argument block to scratch memory).
__host__ __device__ inline int mode_at(int packed, int side, int dim) {
    return (packed >> (4 * (3 * side + dim))) & 15;
}
inline int pack_modes(const int m[2][3]) {
    int p = 0;
    for (int s = 0; s < 2; ++s)
        for (int d = 0; d < 3; ++d) p |= (m[s][d] & 15) << (4 * (3 * s + d));
    return p;
}
__host__ __device__ inline int sel3i(int i, int a, int b, int c) {
    return i == 0 ? a : (i == 1 ? b : c);
}

// One fluid sweep of one simulation (fluid_sweep_impl.h).
template <typename T>
struct FluidArgs {
    T* q[5];                 // mass, mom(1..3), ener -- updated in place
    const T* bc[3];          // cell-centred B (MagnetArray.cellMag)
    double* edges;           // edge-tracker storage
    const long long* eoff;   // [NOBJ][2][3] offsets into edges
    // edges of flux object o (OBJ_SFR .. OBJ_FL + 4) on side s of dim d: eo[s] + o * eo_step
    long long eo[2], eo_step;
    const SimDev* sim;       // device time state (dt, active)
    int n0, n1, n2;
    int d;                   // sweep dimension 0..2
    int ndims;
    int modes;               // BC modes [side][dim], packed (mode_at)
    int active_lin;          // Edges.ACTIVE(d+1) read as a linear index
    int limiter;
    MagUse use;              // !MagnetArray.isZero per component
    double gamma, minmass, dx;
    const double* dxl;       // non-uniform DGRID{X}: spacing of cell i along d, or nullptr
    int init_edges;          // first assignment of the flux objects (first fluid sweep)
    int PX, TL, K, xmajor;   // tile: PX pencils x TL threads, K cells per thread
    long long npencil;       // pencil slots (worm_slots with a lower wormhole boundary)
    int worm;                // lower boundary along d is a wormhole: slots hold pencil pairs
    int bc_inf;
    int xcd_remap;
    int force;               // run even when the loop's running flag is off (direct calls)
    const double* fade;      // fade_shift.m coefficients (device)
    int visc_type;           // run.fluid.viscosity: 0 'empty', 1 'neumann_richtmyer'
    double visc_lin, visc_quad;  // linear / quadraticViscousStrength
};

// One entry of a batched launch: argument block `arg` (one simulation and sweep) and the
// tile (pencil group, or cell chunk) within it.  Every launcher below also takes
// tiles == nullptr: then args[0] is one simulation and ntiles its tile count.
struct BatchTile {
    int arg;
    int pad;
    long long tile;
};

// A tile-list entry read so that the compiler knows it is the same in every lane (the
// block works on one tile): the argument-block index and tile go to scalar registers,
// and the argument block's fields are then read as uniform values rather than as
// per-lane loads that each cost a memory round trip.
__device__ __forceinline__ void uniform_tile(const BatchTile* tiles, int t, int& arg,
                                             long long& tile) {
    const BatchTile bt = tiles[t];
    arg = __builtin_amdgcn_readfirstlane(bt.arg);
    const unsigned lo = __builtin_amdgcn_readfirstlane(unsigned(bt.tile & 0xffffffffll));
    const unsigned hi = __builtin_amdgcn_readfirstlane(unsigned(bt.tile >> 32));
    tile = (long long)(((unsigned long long)hi << 32) | lo);
}

// Block index -> tile index so that consecutive tiles run on the same XCD (blocks are
// dispatched round-robin over the 8 XCDs; neighbouring pencils then share an L2).  A
// bijection of 0..nblocks-1; launches of one block per tile pass their tile count.
__device__ inline long long xcd_tile(long long b, long long nblocks) {
    long long q = nblocks / 8, r = nblocks % 8;
    long long x = b % 8, t = b / 8;
    return x * q + (x < r ? x : r) + t;
}

// Schedule of a persistent launch over a tile list: the list is cut into 8 contiguous
// ranges, one per XCD (blocks are dispatched round-robin over the XCDs, block b runs on
// XCD b % 8), and the blocks of an XCD walk its range together, so tiles that neighbour
// in memory (adjacent pencils of one simulation) are in flight on the same L2.  Returns
// the tile of round r of this block, or -1 when the block is done.  A grid that is not a
// multiple of 8 falls back to the grid-stride order.
__device__ __forceinline__ int xcd_round_tile(int r, int ntiles) {
    const int G = gridDim.x, b = blockIdx.x;
    if (G % 8 != 0) {
        const int t = b + r * G;
        return t < ntiles ? t : -1;
    }
    const int x = b & 7, j = b >> 3, per = G >> 3;
    const int lo = int((long long)ntiles * x / 8);
    const int hi = int((long long)ntiles * (x + 1) / 8);
    const int t = lo + j + r * per;
    return t < hi ? t : -1;
}

// The (argument block, tile) a block works on in round t of a persistent launch; with
// tiles == nullptr the launch is one simulation, args[0], one block per tile.
__device__ inline bool next_tile(const BatchTile* tiles, int ntiles, int r, int& arg,
                                 long long& tile) {
    if (!tiles) {
        if (r > 0 || (int)blockIdx.x >= ntiles) return false;
        arg = 0;
        tile = xcd_tile(blockIdx.x, ntiles);  // neighbouring tiles on one XCD
        return true;
    }
    const int t = xcd_round_tile(r, ntiles);
    if (t < 0) return false;
    uniform_tile(tiles, t, arg, tile);
    return true;
}

// Whether the sweep of an argument block runs, and its time step (the time state is that of
// the launches before: no kernel that reads it so may change it).
template <typename A>
__device__ __forceinline__ bool sweep_runs(const A& a, double& dt) {
    const SimDev* sim = uniform_load(&a.sim);
    dt = uniform_load(&sim->dt);
    return uniform_load(&a.force) || uniform_load(&sim->active);
}

// The general form of the sweep (fluid_sweep_impl.h).
template <typename T>
hipError_t launch_fluid_batch(const FluidArgs<T>* args, const BatchTile* tiles, int ntiles,
                              int nblocks, int bs, int kmax, bool mhd, hipStream_t st);
constexpr int LEAN_PXMAX = 16;   // pencils per tile of the lean sweep
// Kernels of the lean sweep: both ends circular or constant (no ghost jobs), any ends, and any
// ends with Neumann-Richtmyer viscosity.
constexpr int LEAN_PLAIN = 0, LEAN_ENDS = 1, LEAN_VISC = 2;
__host__ __device__ constexpr bool lean_plain_end(int mode) {
    return mode == IMH_BC_CIRC || mode == IMH_BC_CONST;
}
inline int lean_form(int visc_type, int mlo, int mhi) {
    if (visc_type) return LEAN_VISC;
    return lean_plain_end(mlo) && lean_plain_end(mhi) ? LEAN_PLAIN : LEAN_ENDS;
}
// The lean form (fluid_lean_impl.h) of a sweep along d that fluid_needs_general() does not
// send to the general form; px: the most pencils a tile of the launch holds; form: lean_form.
template <typename T>
hipError_t launch_fluid_lean(const FluidArgs<T>* args, const BatchTile* tiles, int ntiles,
                             int nblocks, int bs, int kmax, int d, bool mhd, int px, int form,
                             hipStream_t st);
// The column march for sweeps along y / z with circular or constant boundaries: one
// thread per pencil, fluid_column_pencils() pencils per tile.
template <typename T>
hipError_t launch_fluid_column(const FluidArgs<T>* args, const BatchTile* tiles, int ntiles,
                               int nblocks, bool mhd, hipStream_t st);
int fluid_column_pencils();

// whether a sweep of these arguments needs the general kernel form: the first sweep of a
// simulation, a fade boundary, Caramana-Shashkov-Whalen viscosity or a spacing line
template <typename T>
inline bool fluid_needs_general(const FluidArgs<T>& a) {
    return a.init_edges || a.visc_type == 2 || a.dxl || mode_at(a.modes, 0, a.d) == IMH_BC_FADE ||
           mode_at(a.modes, 1, a.d) == IMH_BC_FADE;
}

// Compiled fluid sweep variants X(element size, block size, KMAX): FP64 keeps K <= KMAX
// cells per thread in registers with KMAX 1..4 (8 for pencils of 2049..4096 cells, with
// register spills), FP32 with 1..8.  Pencils up to BS * KMAX cells fit one block.  Each
// variant is its own translation unit.
#define IMH_FLUID_VARIANTS(X) \
    X(8, 256, 1) X(8, 256, 2) X(8, 256, 4) X(8, 512, 2) X(8, 512, 4) X(8, 512, 8) \
    X(4, 256, 2) X(4, 256, 4) X(4, 512, 4) X(4, 512, 8) X(4, 1024, 4) \
    X(4, 256, 1) X(4, 512, 2)
#define IMH_FLUID_LAUNCHER_(E, B, K) launch_fluid_v##E##_##B##_##K
#define IMH_FLUID_LAUNCHER(E, B, K) IMH_FLUID_LAUNCHER_(E, B, K)
#define IMH_FLUID_DECLARE(E, B, K)                                                         \
    hipError_t IMH_FLUID_LAUNCHER(E, B, K)(const void* args, const BatchTile* tiles, int ntiles, \
                                           int nblocks, bool mhd, hipStream_t st);
IMH_FLUID_VARIANTS(IMH_FLUID_DECLARE)
#define IMH_LEAN_LAUNCHER_(E, B, K) launch_fluid_lean_v##E##_##B##_##K
#define IMH_LEAN_LAUNCHER(E, B, K) IMH_LEAN_LAUNCHER_(E, B, K)
#define IMH_LEAN_DECLARE(E, B, K)                                                          \
    hipError_t IMH_LEAN_LAUNCHER(E, B, K)(const void* args, const BatchTile* tiles, int ntiles, \
                                          int nblocks, int d, bool mhd, int px, int form,   \
                                          hipStream_t st);
IMH_FLUID_VARIANTS(IMH_LEAN_DECLARE)
bool fluid_variant_compiled(int esz, int bs, int kmax);

// One magnetFlux sub-step (component I advected along X) of one simulation
// (magnet_sweep_impl.h).
template <typename T>
struct MagnetArgs {
    const T* rho;            // mass
    const T* mom;            // mom(X)
    T* bI;                   // mag(I), updated in place
    T* bX;                   // mag(X), updated by the CT step
    T* flux;                 // scratch: mag(I).flux(X) after the limiter
    double* edges;
    const long long* eoff;
    const SimDev* sim;
    int n0, n1, n2;
    int dX, dI;              // 0-based sweep and component dimensions
    int ndims;
    int modes;               // packed BC modes
    int active_linX, active_linI;  // Edges.ACTIVE(D) (linear index) for D = X, I
    int limiter;
    double dxX, dxI;
    const double* dxlX;      // non-uniform DGRID{X} / DGRID{I} lines, or nullptr
    const double* dxlI;
    int init_vg, init_store, init_wmag, init_flux;  // first assignments
    int PX, TL;              // tile for the pencil kernel
    long long npencil;
    int bc_inf;
    int force;
    const double* fade;
};


// One magnetFlux(X, [I1 I2]) of one simulation in the lean form (magnet_lean_impl.h): both
// components' advection, then both CT steps and the cell-centred updates.
template <typename T>
struct MagnetLeanArgs {
    const T* rho;            // mass
    const T* mom;            // mom(X)
    T* bI[2];                // mag(I1), mag(I2)
    T* bX;                   // mag(X)
    T* cI;                   // cell-centred mag(I2) and mag(X)
    T* cX;
    T* flux;                 // scratch: the limited fluxes of I1, then of I2 (ncell each)
    double* edges;
    const long long* eoff;
    const SimDev* sim;
    int n0, n1, n2;
    int dI[2];
    int ndims;
    int modes;               // packed BC modes
    int active_linX, active_linI[2];
    int limiter;
    double dxX, dxI[2];
    int PX, TL;              // tile: PX pencils x TL threads, powers of two
    long long npencil, ncell;
    int bc_inf;
    int force;
};
constexpr int MLEAN_BS = 256;
// which = 0: advection, 2 tiles (I1, I2) per pencil group; 1: CT, one.  trk: some boundary
// of the grid is transparent or a wall (magnet_lean_tracked).  lds: mag_lean_lds
// of the launch's largest tile.
template <typename T>
hipError_t launch_magnet_lean(int which, const MagnetLeanArgs<T>* args, const BatchTile* tiles,
                              int ntiles, int nblocks, int d, bool trk, size_t lds,
                              hipStream_t st);
template <>
hipError_t launch_magnet_lean<double>(int, const MagnetLeanArgs<double>*, const BatchTile*, int,
                                      int, int, bool, size_t, hipStream_t);
template <>
hipError_t launch_magnet_lean<float>(int, const MagnetLeanArgs<float>*, const BatchTile*, int, int,
                                     int, bool, size_t, hipStream_t);

// LDS of a tile.  Advection: two rows per pencil of N + 8 values (x rows padded by one value
// in four, mlean::pad); CT: one row of N.
__host__ __device__ constexpr int mag_lean_row(bool x, int N) {
    return x ? (N + 8) + ((N + 8) >> 2) + 1 : N + 8;
}
inline size_t mag_lean_lds(int which, int d, int N, int PX, size_t esz) {
    return which == 0 ? 2 * esz * PX * mag_lean_row(d == 0, N) : esz * PX * N;
}

// updateCellCentered for component k: cmag_k = 0.5*(B_k + shift_k(B_k, +1)).
template <typename T>
struct CellMagArgs {
    const T* b;
    T* cb;
    double* edges;
    const long long* eoff;
    const SimDev* sim;
    int n0, n1, n2;
    int k;                   // component (0-based) = shift dim
    int ndims;
    int modes;
    int active_lin;
    int bc_inf;
    int force;               // run even if the simulation is not active (constructor)
    const double* fade;
};


// Batched magnet kernels: which = 0 advection sub-step, 1 CT step.  kmax from
// magnet_kmax_for(N, TL); smem = sizeof(T) * 2 * PX * (N + 4) of the largest tile.
template <typename T>
hipError_t launch_magnet_batch(int which, const MagnetArgs<T>* args, const BatchTile* tiles,
                               int ntiles, int nblocks, int kmax, size_t smem, hipStream_t st);
template <typename T>
hipError_t launch_cell_centered_batch(const CellMagArgs<T>* args, const BatchTile* tiles,
                                      int ntiles, int nblocks, hipStream_t st);
int magnet_kmax_for(int N, int TL);
constexpr int MAG_PENCIL_MAX = 4096;  // magnet pencils: 256 threads x 16 cells

// The fluid sweep along pencils longer than the fused sweep's tile (fluid_long.hip):
// five launches over the cells, the pencil-wide quantities in a scratch area of
// fluid_long_bytes (U^{n+1/2}, two pencil maxima, the end ghosts).
constexpr int FLUID_LONG_GH = 8;   // ghost values per pencil and field
constexpr int FLUID_LONG_EN = 36;  // row ends per pencil and field: 3 stages x 2 rows x 6
constexpr int FLUID_LONG_VG = 11;  // viscosity ghosts per pencil
inline size_t fluid_long_align(size_t b) { return (b + 255) & ~size_t(255); }
inline size_t fluid_long_bytes(size_t esz, long long ncell, long long npencil) {
    return 6 * fluid_long_align(esz * (size_t)ncell) +
           fluid_long_align(sizeof(unsigned long long) * 2 * (size_t)npencil) +
           fluid_long_align(sizeof(double) * 5 * FLUID_LONG_GH * (size_t)npencil) +
           fluid_long_align(sizeof(double) * 5 * FLUID_LONG_EN * (size_t)npencil) +
           sizeof(double) * FLUID_LONG_VG * (size_t)npencil;
}
template <typename T>
hipError_t launch_fluid_long(const FluidArgs<T>& a, void* scratch, long long ncell, bool mhd,
                             hipStream_t st);

// One launch per batched iteration for the 1-D MHD simulations of an FP32 batch
// (lane1d.hip): one workgroup per simulation runs its fluid sweeps, magnet sub-steps and
// cell-centred updates back to back.  The argument blocks carry a tile of one pencil
// over the whole workgroup.  IMH_LANE1D_BS (a build-time knob) is the workgroup size;
// each thread holds up to 4096 / IMH_LANE1D_BS cells.
#ifndef IMH_LANE1D_BS
#define IMH_LANE1D_BS 512
#endif
constexpr int LANE1D_BS = IMH_LANE1D_BS;
constexpr int LANE1D_NMAX = 4096;
constexpr int LANE1D_KMAX = LANE1D_NMAX / LANE1D_BS;
template <typename T>
struct Lane1dArgs {
    FluidArgs<T> fa;        // the sweep along x
    MagnetLeanArgs<T> ml[2];  // magnetFlux(X=1), I = [2 3] and [3 2]
};
hipError_t launch_lane1d(const void* args, int nsims, hipStream_t st);

// CFL reduction (TimeManager.update) over one simulation.
template <typename T>
struct CflArgs {
    const T* q[5];
    const T* bc[3];
    SimDev* sim;
    const SimParams* par;
    double* part;            // the tiles' maxima, 3 * CFL_TILES
    long long ncell;
    long long chunk;         // cells per tile (cfl_chunk)
    MagUse use;
    double gamma;
};

// Several iterations of one 1-D simulation in one launch (line1d_variant.hip): time update,
// flux call and iteration count of a pencil of up to LINE1D_NMAX cells by one workgroup.  mag: the
// magnetic sweeps too, with ml[0] / ml[1] magnetFlux(X=1) for order +1 / -1.  bs * k >= N.
constexpr int LINE1D_BS = 512;
constexpr int LINE1D_NMAX = 8 * LINE1D_BS;
template <typename T>
hipError_t launch_line1d(const FluidArgs<T>* fa, const MagnetLeanArgs<T>* const ml[2],
                         const CflArgs<T>* ca, int N, bool mhd, bool mag, int iterations,
                         hipStream_t st);
template <>
hipError_t launch_line1d<double>(const FluidArgs<double>*, const MagnetLeanArgs<double>* const[2],
                                 const CflArgs<double>*, int, bool, bool, int, hipStream_t);
template <>
hipError_t launch_line1d<float>(const FluidArgs<float>*, const MagnetLeanArgs<float>* const[2],
                                const CflArgs<float>*, int, bool, bool, int, hipStream_t);

// Compiled magnet variants X(element size, KMAX): each a translation unit with the
// advection and CT kernels for pencils of up to KMAX * TL cells.
#define IMH_MAG_VARIANTS(X) \
    X(8, 1) X(8, 2) X(8, 4) X(8, 8) X(8, 16) X(4, 1) X(4, 2) X(4, 4) X(4, 8) X(4, 16)
#define IMH_MAG_LAUNCHER_(E, K) launch_magnet_v##E##_##K
#define IMH_MAG_LAUNCHER(E, K) IMH_MAG_LAUNCHER_(E, K)
#define IMH_MAG_DECLARE(E, K)                                                               \
    hipError_t IMH_MAG_LAUNCHER(E, K)(int which, const void* args, const BatchTile* tiles,  \
                                      int ntiles, int nblocks, size_t smem, hipStream_t st);
IMH_MAG_VARIANTS(IMH_MAG_DECLARE)

constexpr int CFL_TILES = 1024;  // most tiles of one simulation
// gate: whether a simulation runs: always, when TimeManager.running holds (both set its
// active flag), or by that flag.
constexpr int CFL_ALWAYS = 0, CFL_RUNNING = 1, CFL_ACTIVE = 2;
template <typename T>
hipError_t launch_cfl(const CflArgs<T>* args, const BatchTile* tiles, int ntiles, int nblocks,
                      int gate, int step, int count, hipStream_t st);
// After launch_cfl, where a simulation has several tiles (chunk < ncell).
template <typename T>
hipError_t launch_cfl_finish(const CflArgs<T>* args, int nsims, int gate, int step, int count,
                             hipStream_t st);
long long cfl_chunk(long long ncell);

// The top of the loop body on its own (cfl.hip), one thread per simulation; `sim` and `p`
// are device arrays of per-simulation pointers.
hipError_t launch_begin_iteration(SimDev* const* sim, const SimParams* const* p, int nsims,
                                  int unconditional, hipStream_t st);

// Conservation totals (Neumaier-compensated FP64, fixed-order tree).
template <typename T>
hipError_t launch_conservation(const T* const* fields, int nfields, long long ncell,
                               double* partials, int nblocks, double* out, hipStream_t st);

}  // namespace imh
