// fluid_lean_impl.h -- the fluid sweep (relaxingFluid.m:16-73, wFluidFlux.m:14-44,
// pressure.m) of the common case: no fade end, no first assignment of the flux objects, no
// Caramana-Shashkov-Whalen viscosity, uniform spacing.  fluid_sweep_impl.h holds the general
// form.
//
// A workgroup owns PX whole pencils, TL = BS / PX threads each, K consecutive cells per
// thread in registers.  What bounds a sweep here is not HBM but the latency of one tile
// (loads, two pencil-wide maxima, exchanges, boundary ghosts) at the number of tiles a CU
// holds, then FP64 issue; so the form is built around few live values, little LDS and
// few dependent steps:
//  * The flux numerators w*C are formed before the freezing speed C is known: P and u die
//    early, the predictor's neighbour values (q and w*C of the chunk edges) are published
//    with the speeds, and one barrier serves the maximum and the exchange.
//  * Every array is replaced in place (q -> q(n+1/2) -> fluxR, wC -> fluxL -> limited).
//  * FP64 divides by C and rho through one reciprocal each (LMath<double>::div): the
//    quotient is corrected by its exact remainder, which rounds it as the division does.
//  * Ghosts of transparent ends need one pchip interval only (their argument lies between
//    the third and the fourth node).  A ghost is written where the neighbour's value
//    would be read, so the cells next to an end need no selects.
//  * LDS: 20 rows of one value per thread, and what the PX pencils' ends need (PX known at
//    the launch: dynamic LDS).
//  * The argument block is read into scalar registers (uniform_load): FP64 4 cells per
//    thread 168 vector registers with spills -> 147, 2 cells 123; FP64 256^3 664 -> 621 us per
//    sweep, FP32 192^3 158 -> 147, a 1024-cell tube 18.0 -> 16.9.
//  * Three kernels (FORM): without ghost jobs where both ends are circular or constant (FP64
//    MHD, 2 cells per thread: 139 -> 120 vector registers; 100^3 47.5 -> 44.6 us per sweep, FP32
//    MHD 191^2 13.2 -> 12.4), with them, and with Neumann-Richtmyer viscosity (the sweep momentum
//    of the next chunk through two more LDS rows; FP64 96^3 with gravity and radiation 123 -> 43
//    against the general form).
// Measured against the general form (us per sweep, mean of the directions): FP64 125^3 175 ->
// 75, 256^3 1463 -> 594 (1.34 GB: 2.3 TB/s), 333x333 19 -> 15, FP32 192^3 372 -> 144,
// 1024x1024 37 -> 26, FP64 MHD 96^3 61 -> 43.  Spilling registers for one more wave per SIMD
// loses (FP64, 2 cells per thread at 4 waves: 782 -> 1130 at 256^3).
// Every expression keeps the .m evaluation order (FP64: bit for bit the general form; FP32
// the same contractions as the general form).
#pragma once

#include "fluid_math.h"
#include "fluid_tile.h"
#include "imh_common.h"
#include "imh_kernels.h"

#include <type_traits>

namespace imh {

// Arithmetic of the lean sweep.  FP32 is FMath<float>'s.
template <typename T>
struct LMath;

template <>
struct LMath<float> : FMath<float> {
    static __device__ __forceinline__ float divrho2(float x, float, float inv) { return x * inv; }
    // see LMath<double>::mm
    static __device__ __forceinline__ float mm(float a, float b) {
        const int ha = __float_as_int(a), hb = __float_as_int(b);
        const int f = (ha & int(0x80000000)) | 0x3E800000;      // +-0.25
        const float m = __int_as_float(f & ~((ha ^ hb) >> 31)) * fminf(fabsf(a), fabsf(b));
        return __builtin_isunordered(a, b) ? NAN : m;
    }
    static __device__ __forceinline__ float lim(int l, float dl, float dr) {
        if (l == IMH_LIM_VANLEER) return vanleer(dl, dr);
        if (l == IMH_LIM_SUPERBEE) {
            const bool c = fabsf(dl) < fabsf(dr);  // (1 + c) dl, (2 - c) dr
            return mm((c ? 2.0f : 1.0f) * dl, (c ? 1.0f : 2.0f) * dr);
        }
        return mm(dl, dr);
    }
};

template <>
struct LMath<double> {
    // 1 / y: hardware estimate and two Newton steps.
    static __device__ __forceinline__ double rcp(double y) {
        double r = __builtin_amdgcn_rcp(y);
        double e = fma(-y, r, 1.0);
        r = fma(r, e, r);
        e = fma(-y, r, 1.0);
        return fma(r, e, r);
    }
    // x / y with r = rcp(y): the quotient x*r, corrected by its remainder (Markstein's
    // scheme), is the correctly rounded x / y while no intermediate leaves the normal
    // range (|x| above 1e-290 or zero, y and the quotient within 1e+-290); below it the
    // remainder underflows and the last bit may be off.  Zeros, infinities and NaN go
    // through div_fixup, and so does a quotient past the largest value: its remainder makes
    // a NaN of it, which div_fixup takes, over finite operands, for an overflow and returns
    // as infinity of the right sign (gfx950; so does any x over a y below 5.6e-309, whose
    // reciprocal overflows: right where the quotient does).  Callers divide by densities
    // (above 1.5e-154, so that the square is normal), speeds, sums of two differences whose
    // product is x (subnormal only where x is 0) and, with x of 3 and more, the differences of
    // end_ghost.
    static __device__ __forceinline__ double div(double x, double y, double r) {
        const double q = x * r;
        const double e = fma(-y, q, x);
        return __builtin_amdgcn_div_fixup(fma(e, r, q), y, x);
    }
    static __device__ __forceinline__ double quot(double x, double y) { return div(x, y, rcp(y)); }
    static __device__ __forceinline__ double divrho2(double x, double rho, double r) {
        return div(x, rho, r);
    }
    // sqrt(x), x >= 0: hardware estimate of 1/sqrt, Goldschmidt's coupled iteration for the
    // root and half its reciprocal, and two steps on the root with its exact remainder
    // (correctly rounded as sqrt() is, without the scaling that only x below 1e-230 needs).
    static __device__ __forceinline__ double root(double x) {
        const double y = __builtin_amdgcn_rsq(x);
        double q = x * y, h = 0.5 * y;
        const double r = fma(-h, q, 0.5);
        q = fma(q, r, q);
        h = fma(h, r, h);
        double d = fma(-q, q, x);
        q = fma(d, h, q);
        d = fma(-q, q, x);
        q = fma(d, h, q);
        return (x == 0.0 || x == INFINITY) ? x : q;
    }
    // pressure.m 'totsnd' (pressure_totsnd): P and the fast speed c; inv = 1 / rho
    static __device__ __forceinline__ void press(double rho, double px, double py, double pz,
                                                 double E, double bx, double by, double bz,
                                                 MagUse u, double g, double& P, double& c,
                                                 double& inv) {
        inv = rcp(rho);
        const double v2 = quot(px * px + py * py + pz * pz, rho * rho);
        double b2 = 0.0;
        if (u.x) b2 = b2 + bx * bx;
        if (u.y) b2 = b2 + by * by;
        if (u.z) b2 = b2 + bz * bz;
        double r = (g - 1.0) * (E - 0.5 * rho * v2);
        c = root(fabs(div(g * (r - (g - 1.0) * 0.5 * b2) + 2.0 * b2, rho, inv)));
        r = r + 0.5 * (2.0 - g) * b2;
        P = r < 0.0 ? 0.0 : r;
    }
    // minmod as 0.125 * (sign a + sign b) * min(|a|, |b|): +-m / 4 where a and b have the
    // same sign bit (m is 0 where either is 0), else 0; NaN where either is NaN
    static __device__ __forceinline__ double mm(double a, double b) {
        const int ha = __double2hiint(a), hb = __double2hiint(b);
        const int f = (ha & int(0x80000000)) | 0x3FD00000;      // +-0.25
        const double s = __hiloint2double(f & ~((ha ^ hb) >> 31), 0);
        const double m = s * fmin(fabs(a), fabs(b));
        return __builtin_isunordered(a, b) ? NAN : m;
    }
    static __device__ __forceinline__ double lim(int l, double dl, double dr) {
        if (l == IMH_LIM_VANLEER) {
            const double t = quot(fmax(dl * dr, 0.0), dl + dr);
            return isnan(t) ? 0.0 : t;
        }
        if (l == IMH_LIM_SUPERBEE) {
            const bool c = fabs(dl) < fabs(dr);  // (1 + c) dl, (2 - c) dr
            return mm(__hiloint2double(c ? 0x40000000 : 0x3FF00000, 0) * dl,
                      __hiloint2double(c ? 0x3FF00000 : 0x40000000, 0) * dr);
        }
        return mm(dl, dr);
    }
};

namespace lean {

constexpr int PXMAX = LEAN_PXMAX;   // pencils per tile

// Dynamic LDS of a block: byte offsets of its parts and its size.  The 20 exchange rows
// hold one value per thread and, per pencil, the value past each end (lower, upper).
// With viscosity, two more rows: the sweep momentum of each chunk's first and last cell.
struct Lds {
    int trk, red, ends, visc, total;
};
__host__ __device__ constexpr int row_len(int bs) { return bs + 2 * PXMAX; }
__host__ __device__ constexpr Lds lds_layout(int bs, int px, int esz, bool visc = false) {
    Lds L{};
    L.trk = 20 * row_len(bs) * esz;
    L.red = L.trk + px * 30 * 8;                  // edge trackers [job][3], FP64
    L.ends = L.red + 2 * (bs / 64) * px * esz;    // pencil maxima per wave, 2 stages
    L.visc = L.ends + px * 40 * esz;              // (ends: [side][field][cell from the end][2])
    L.total = L.visc + (visc ? 2 * bs * esz : 0);
    return L;
}

// Maximum over the lanes of a wave that share a pencil (NaN ignored).  x pencils: blocks
// of min(TL, 64) adjacent lanes; y / z: lanes PX apart.  Row rotations (DPP) and row
// swaps: no LDS round trips.
template <typename T, int CTRL>
__device__ __forceinline__ T dpp_mov(T v) {
    if constexpr (sizeof(T) == 4) {
        const int x = __builtin_bit_cast(int, v);
        return __builtin_bit_cast(T, __builtin_amdgcn_update_dpp(x, x, CTRL, 0xF, 0xF, false));
    } else {
        typedef int I2 __attribute__((ext_vector_type(2)));
        I2 x = __builtin_bit_cast(I2, v);
        x.x = __builtin_amdgcn_update_dpp(x.x, x.x, CTRL, 0xF, 0xF, false);
        x.y = __builtin_amdgcn_update_dpp(x.y, x.y, CTRL, 0xF, 0xF, false);
        return __builtin_bit_cast(T, x);
    }
}
template <bool XM, typename T>
__device__ __forceinline__ T wave_pencil_max(T v, int TL, int PX) {
    if (XM && TL < 16) {
        for (int off = TL >> 1; off >= 1; off >>= 1) v = fmax(v, __shfl_xor(v, off, 64));
        return v;
    }
    // lane distances 1, 2, 4, 8 within a row of 16 (a rotation by each)
    const int lo = XM ? 1 : PX;
    if (lo <= 1) v = fmax(v, dpp_mov<T, 0x121>(v));
    if (lo <= 2) v = fmax(v, dpp_mov<T, 0x122>(v));
    if (lo <= 4) v = fmax(v, dpp_mov<T, 0x124>(v));
    if (lo <= 8) v = fmax(v, dpp_mov<T, 0x128>(v));
    if (XM ? TL >= 32 : lo <= 16) v = fmax(v, __shfl_xor(v, 16, 64));
    if (XM ? TL >= 64 : true) v = fmax(v, __shfl_xor(v, 32, 64));
    return v;
}

// Fixes where a value is computed: the compiler otherwise moves work of one field behind
// another's, and keeps all fields' inputs in registers at once.
template <typename T>
__device__ __forceinline__ void pin(T& x) {
    asm volatile("" : "+v"(x));
}
// The same for a value that is one for all lanes.
__device__ __forceinline__ void pin_s(int& x) { asm volatile("" : "+s"(x)); }

// Ghost of a one-cell shift past a pencil end (ghost_values() with m = 1) for every mode
// but circ and wormhole, whose ghost comes from elsewhere.  c0, c1: the end cell and the
// next.  neg: the shifted component is the shift's direction; zero: zero_shift's
// ghost of this flux object is 0.  At a transparent end the cubic's argument, 4, lies
// between its nodes 3 and bcInfinity, and the slope at the far node is 0 (the stored edge
// repeats there), so one interval's coefficients, from two cells and the edge, suffice;
// bcInfinity = 4 is that node.
// Ahead of a front the differences next to the third node fall below 2e-307 in whole rows of
// cells; the slope's quotients by them overflow to infinity (LMath<double>::div), and the slope
// is 0, as with divisions.
__device__ __forceinline__ double end_ghost(int mode, bool neg, bool zero, double c0, double c1,
                                            int active, int bc_inf, double& tracker) {
    if (mode == IMH_BC_TRANS) {
        double ev = 0.0;
        if (active) ev = edge_nudge(tracker, c0);
        double v = ev;
        if (bc_inf > 4) {
            pin_s(bc_inf);  // (its reciprocal is formed here each time, not kept)
            const double h = double(bc_inf) - 3.0;
            const double rh = LMath<double>::rcp(h);
            const double e1 = c0 - c1, e2 = LMath<double>::div(ev - c0, h, rh);
            double d = 0.0;
            if ((e1 > 0.0 && e2 > 0.0) || (e1 < 0.0 && e2 < 0.0)) {
                const double w1 = 2.0 * h + 1.0, w2 = h + 2.0;
                d = LMath<double>::quot(w1 + w2, LMath<double>::quot(w1, e1) + LMath<double>::quot(w2, e2));
            }
            const double dz = LMath<double>::div(e2 - d, h, rh);
            const double dd = LMath<double>::div(0.0 - e2, h, rh);
            v = LMath<double>::div(dd - dz, h, rh);
            v = v + (2.0 * dz - dd);
            v = v + d;
            v = v + c0;
        }
        return fabs(c0 - v) < 1e-4 ? c0 : v;
    }
    if (mode == IMH_BC_WALL) return tracker;
    if (mode == IMH_BC_ZERO) return zero ? 0.0 : c0;
    const double r = mode == IMH_BC_MIRROR ? c1 : c0;  // flip, const, upper wormhole: the end
    return (neg && (mode == IMH_BC_MIRROR || mode == IMH_BC_FLIP)) ? -r : r;
}

}  // namespace lean

// The sweep of one tile (PX pencils) of one simulation along D.  lds: lean::lds_layout; dt:
// the same for all lanes.
template <typename T, int BS, int K, bool MHD, int D, int FORM = LEAN_ENDS>
__device__ __forceinline__ void fluid_lean_body(const FluidArgs<T>& ap, long long tile, char* lds,
                                                double dt) {
    const FluidArgs<T> a = uniform_load(&ap);
    using M = LMath<T>;
    constexpr bool XM = D == 0;
    constexpr bool VISC = FORM == LEAN_VISC;
    constexpr int X = D + 1;
    constexpr int NW = BS / 64;
    constexpr int RL = lean::row_len(BS);
    // Fields whose U^n stays in registers (the others' is read again at the end, mostly past L2:
    // at FP64 256^3 1275 MB fetched per sweep for 671): all where that is cheap; with four FP64
    // cells per thread the three that still fit 168 registers (256^3 619 -> 594 us, 200^3 349 ->
    // 333, 125^3 78 -> 75), which MHD sweeps do not (200^3 358 -> 383).
    constexpr int KEEP = int(sizeof(T)) * K <= 16 ? 5
                         : (sizeof(T) == 8 && K == 4 && !MHD && FORM != LEAN_VISC ? 3 : 0);

    // not loop-invariant: in a loop over tiles the compiler would keep what follows from it
    // in registers over the whole body
    int tid = threadIdx.x;
    lean::pin(tid);
    const int wave = tid >> 6;
    const int PX = a.PX, TL = a.TL;              // powers of two
    const int lg = 31 - __builtin_clz(XM ? TL : PX);
    const int px = XM ? tid >> lg : tid & (PX - 1);
    const int ty = XM ? tid & (TL - 1) : tid >> lg;
    const int dstep = XM ? 1 : PX;
    const lean::Lds L = lean::lds_layout(BS, PX, int(sizeof(T)));
    double* const s_trk = reinterpret_cast<double*>(lds + L.trk);
    T* const s_red = reinterpret_cast<T*>(lds + L.red);
    T* const s_end = reinterpret_cast<T*>(lds + L.ends);
    auto row = [&](int r) __attribute__((always_inline)) -> T* {
        return reinterpret_cast<T*>(lds) + r * RL;
    };

    const long long pen0 = tile * PX;
    const int nn[3] = {a.n0, a.n1, a.n2};
    // face of slot p of the tile, -1 for padding (with a lower wormhole boundary the slots
    // hold pencil pairs, worm_face)
    auto slot_face = [&](int p) __attribute__((always_inline)) -> int {
        const long long sl = pen0 + p;
        if (sl >= a.npencil) return -1;
        return a.worm ? int(worm_face(nn, D, sl)) : int(sl);
    };
    const int pface = slot_face(px);
    const bool pen_ok = pface >= 0;
    const int N = sel3i(D, a.n0, a.n1, a.n2);
    int i0 = ty * K;
    long long base64 = 0, stride64 = 1;
    // padding pencils read a real one
    pencil_base(nn, D, pen_ok ? pface : (a.worm ? 0 : a.npencil - 1), base64, stride64);
    unsigned base = unsigned(base64);
    const unsigned stride = XM ? 1u : unsigned(stride64);
    const bool full = N % K == 0;
    const bool vec = XM && full;
    // start of the chunk, of x pencils that move whole chunks as vectors
    auto cb = [&]() __attribute__((always_inline)) -> unsigned { return base + unsigned(i0 < N ? i0 : N - K); };
    auto off = [&](int k) __attribute__((always_inline)) -> unsigned {
        const int i = i0 + k < N ? i0 + k : N - 1;
        return base + unsigned(i) * stride;
    };

    const double ff = dt / a.dx;          // fluxFactor = dTime ./ DGRID{X}
    const double hf = 0.5 * ff;
    const double g = a.gamma;
    const int mlo = mode_at(a.modes, 0, D), mhi = mode_at(a.modes, 1, D);
    // circular and constant ends take their ghosts from the exchange rows
    const bool simple = FORM == LEAN_PLAIN ||
                        (lean_plain_end(mlo) && lean_plain_end(mhi));
    const int ty_last = (N - 1) / K;
    const bool own_lo = ty == 0, own_hi = ty == ty_last;   // chunk with cell 0 / cell N-1
    // where the neighbouring chunks' values are read: past a pencil end, the other end's
    // chunk (circular) or the row's slot for the value past that end
    const int t_first = XM ? px << lg : px, t_last = XM ? t_first + ty_last : ty_last * PX + px;
    const int g_lo = BS + px, g_hi = BS + lean::PXMAX + px;
    const int tl_ = !own_lo ? tid - dstep : (simple && mlo == IMH_BC_CIRC ? t_last : g_lo);
    const int tr_ = ty < ty_last ? tid + dstep
                                 : (own_hi ? (simple && mhi == IMH_BC_CIRC ? t_first : g_hi) : tid);
    const bool clo = simple && mlo == IMH_BC_CONST && own_lo;
    const bool chi = simple && mhi == IMH_BC_CONST && own_hi;

    // ---- ghost jobs: thread j evaluates the ghosts of (pencil, side, field) j; their edge
    // trackers (store.fluxR lower / store.fluxL upper, fluxR, fluxL) are in LDS meanwhile ---
    // one register holds a job: pencil, side, field, the pencil whose end cells it reads
    // (past a lower wormhole the partner's, wormhole_shift.m:21-57), whether there is one
    int jobs = 0;
    if (!simple) {
        const int p = tid / 10, r = tid - p * 10, side = r >= 5, v = side ? r - 5 : r;
        const int pq = a.worm && !side && slot_face(p ^ 1) >= 0 ? (p ^ 1) : p;
        jobs = p | side << 8 | v << 12 | pq << 16;
        if (tid >= PX * 10 || slot_face(p) < 0) jobs = -1;
    }
    struct Job {
        int p, side, v, q, mode;
    };
    auto job = [&]() __attribute__((always_inline)) -> Job {
        Job j;
        j.p = jobs & 255;
        j.side = (jobs >> 8) & 1;
        j.v = (jobs >> 12) & 15;
        j.q = jobs >> 16;
        j.mode = j.side ? mhi : mlo;
        return j;
    };
    auto job_trk = [&](const Job& j) __attribute__((always_inline)) -> bool {
        return jobs >= 0 && (j.mode == IMH_BC_TRANS || j.mode == IMH_BC_WALL);
    };
    auto trk_at = [&](const Job& j, int r) __attribute__((always_inline)) {
        const int obj = r == 0 ? (j.side ? OBJ_SFL : OBJ_SFR) : (r == 1 ? OBJ_FR : OBJ_FL);
        return gmem(a.edges) + ((j.side ? a.eo[1] : a.eo[0]) + (long long)(obj + j.v) * a.eo_step + slot_face(j.p));
    };
    double trk[3] = {0.0, 0.0, 0.0};
    if (!simple) {
        const Job j = job();
        if (job_trk(j)) {
#pragma unroll
            for (int r = 0; r < 3; ++r) trk[r] = *trk_at(j, r);
        }
    }

    // ---- load the chunk (clamped at the pencil end: no branches) ----------------------
    T q[5][K], bm[3][K], un0[KEEP ? KEEP : 1][K];
    if (vec) {
#pragma unroll
        for (int v = 0; v < 5; ++v) chunk_load<T, K>(a.q[v] + cb(), q[v]);
        if constexpr (MHD) {
#pragma unroll
            for (int v = 0; v < 3; ++v) chunk_load<T, K>(a.bc[v] + cb(), bm[v]);
        }
    } else {
#pragma unroll
        for (int k = 0; k < K; ++k) {
            const unsigned o = off(k);
#pragma unroll
            for (int v = 0; v < 5; ++v) q[v][k] = gmem(a.q[v])[o];
            if constexpr (MHD) {
#pragma unroll
                for (int v = 0; v < 3; ++v) bm[v][k] = gmem(a.bc[v])[o];
            }
        }
    }
    if constexpr (KEEP) {
#pragma unroll
        for (int v = 0; v < KEEP; ++v)
#pragma unroll
            for (int k = 0; k < K; ++k) un0[v][k] = q[v][k];
    }

    // Numerators of wFluidFlux.m (w = numerator / C) of state Q into nu, and the largest
    // |u| + c of the chunk.
    T nu[5][K];
    auto numerators = [&](const T (&Q)[5][K], int obj) __attribute__((always_inline)) -> T {
        T lmax = T(NAN);
        // Neumann-Richtmyer viscosity (ArtificialViscosity.m:73-77): vm = min(p(i+1) - p(i), 0)
        // of the sweep momentum, whose objects are obj + X (the FluidArray in the predictor,
        // its StorageArray in the corrector); press gains vm .* (c1 .* c_f + c2 .* vm ./ rho)
        T vm[K];
        if constexpr (VISC) {
            T* const s_mv = reinterpret_cast<T*>(lds + L.visc);
            s_mv[tid] = Q[X][0];
            s_mv[BS + tid] = Q[X][K - 1];
            __syncthreads();
            T nb = Q[X][K - 1];
            if (ty < ty_last) nb = s_mv[tid + dstep];
            if (own_hi) {
                T c0 = Q[X][0], c1 = s_mv[BS + (ty > 0 ? tid - dstep : tid)];
#pragma unroll
                for (int k = 1; k < K; ++k)
                    if (i0 + k < N) {
                        c1 = c0;
                        c0 = Q[X][k];
                    }
                if (mhi == IMH_BC_CIRC) {
                    nb = s_mv[t_first];
                } else {
                    const bool trk = pen_ok && (mhi == IMH_BC_TRANS || mhi == IMH_BC_WALL);
                    double tv = 0.0;
                    IMH_GLOBAL_AS double* const tp =
                        gmem(a.edges) + (trk ? a.eoff[((obj + X) * 2 + 1) * 3 + D] + pface : 0);
                    if (trk) tv = *tp;
                    nb = T(lean::end_ghost(mhi, true, false, double(c0), double(c1), a.active_lin,
                                           a.bc_inf, tv));
                    if (trk && mhi == IMH_BC_TRANS) *tp = tv;
                }
            }
#pragma unroll
            for (int k = 0; k < K; ++k) {
                const T up = (k + 1 < K && i0 + k < N - 1) ? Q[X][k + 1 < K ? k + 1 : k] : nb;
                vm[k] = fmin(up - Q[X][k], T(0));  // MATLAB min(.., 0) skips NaN
            }
        }
#pragma unroll
        for (int k = 0; k < K; ++k) {
            const T bx = MHD ? bm[0][k] : T(0), by = MHD ? bm[1][k] : T(0),
                    bz = MHD ? bm[2][k] : T(0);
            T P, c, ir;
            M::press(Q[0][k], Q[1][k], Q[2][k], Q[3][k], Q[4][k], bx, by, bz, a.use, g, P, c, ir);
            const T U = M::divrho2(Q[X][k], Q[0][k], ir);
            const T sp = fabs(U) + c;
            lmax = fmax(lmax, sp);  // NaN-ignoring, like MATLAB max
            nu[0][k] = Q[X][k];
            if constexpr (VISC) {
                const T t = T(a.visc_quad) * vm[k];
                T tr;
                if constexpr (sizeof(T) == 8) tr = M::divrho2(t, Q[0][k], ir);
                else tr = t / Q[0][k];
                P = P + vm[k] * (T(a.visc_lin) * c + tr);
            }
            if constexpr (MHD) {
                const T bX = sel3(D, bx, by, bz);
                const T b[3] = {bx, by, bz};
#pragma unroll
                for (int v = 1; v < 4; ++v) {
                    if (v == X) {
                        nu[v][k] = U * Q[v][k] + P - bX * b[v - 1];
                    } else {
                        const T t = U * Q[v][k];
                        nu[v][k] = t - bX * b[v - 1];
                    }
                }
                T bdotp = bx * Q[1][k] + by * Q[2][k] + bz * Q[3][k];
                nu[4][k] = U * (Q[4][k] + P) - M::divrho2(bX * bdotp, Q[0][k], ir);
            } else {
#pragma unroll
                for (int v = 1; v < 4; ++v) {
                    if (v == X) nu[v][k] = U * Q[v][k] + P;
                    else nu[v][k] = U * Q[v][k];
                }
                nu[4][k] = U * (Q[4][k] + P);
            }
        }
        return lmax;
    };
    auto publish_max = [&](int stage, T v) __attribute__((always_inline)) {
        v = lean::wave_pencil_max<XM>(v, TL, PX);
        s_red[(stage * NW + wave) * PX + px] = v;
    };
    auto pencil_max = [&](int stage, int p) __attribute__((always_inline)) -> T {
        T m = T(NAN);
        if (XM) {
            const int w0 = (p << lg) >> 6, w1 = ((p << lg) + TL - 1) >> 6;
            for (int w = w0; w <= w1; ++w) m = fmax(m, s_red[(stage * NW + w) * PX + p]);
        } else {
#pragma unroll
            for (int w = 0; w < NW; ++w) m = fmax(m, s_red[(stage * NW + w) * PX + p]);
        }
        return m;
    };
    // two arrays' values at the two cells next to each pencil end, for the ghost jobs
    auto put_ends = [&](const T (&A)[5][K], const T (&B)[5][K]) __attribute__((always_inline)) {
        if (simple || !(i0 < 2 || i0 + K > N - 2) || i0 >= N) return;
        int p = px, i0_ = i0;
        lean::pin(p);
        lean::pin(i0_);
        T* const e0 = s_end + p * 40;
#pragma unroll
        for (int k = 0; k < K; ++k) {
            const int i = i0_ + k;
#pragma unroll
            for (int side = 0; side < 2; ++side) {
                const int c = side ? N - 1 - i : i;
                if (c >= 0 && c < 2) {
                    T* e = e0 + side * 20 + c * 2;
#pragma unroll
                    for (int v = 0; v < 5; ++v) {
                        e[v * 4] = A[v][k];
                        e[v * 4 + 1] = B[v][k];
                    }
                }
            }
        }
    };
    // Ghosts of one stage, into the rows' slots past the pencil ends: 0 predictor
    // (store.fluxR lower, store.fluxL upper; ends and rows hold q and w*C, so a ghost F goes
    // in as q = 2F, w*C = 0), 1 corrector (fluxR and fluxL, both sides), 2 final (limited
    // fluxR lower, limited fluxL upper).
    auto ghosts = [&](auto KIND) __attribute__((always_inline)) {
        constexpr int kind = decltype(KIND)::value;
        if (jobs < 0) return;
        const Job j = job();
        const bool worm = j.mode == IMH_BC_WORMHOLE && j.side == 0;
        // whose end cells: the other end's of a circular pencil
        const T* e = s_end + j.q * 40 + (j.mode == IMH_BC_CIRC ? 1 - j.side : j.side) * 20 + j.v * 4;
        const int slot = (j.side ? BS + lean::PXMAX : BS) + j.p;
        T Cp = T(0), rCp = T(0);
        if constexpr (kind == 0) {
            Cp = pencil_max(0, j.q);
            rCp = M::rcp(Cp);
        }
#pragma unroll 1
        for (int o = 0; o < (kind == 1 ? 2 : 1); ++o) {
            const int which = kind == 1 ? o : j.side;  // flux object: 0 fluxR, 1 fluxL
            double c[2];
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                if constexpr (kind == 0) {
                    const T w = M::div(e[2 * i + 1], Cp, rCp);
                    c[i] = double(which ? T(0.5) * (e[2 * i] - w) : T(0.5) * (e[2 * i] + w));
                } else {
                    c[i] = double(e[2 * i + which]);
                }
                lean::pin(c[i]);
            }
            double* const t = s_trk + tid * 3 + (kind == 0 ? 0 : 1 + which);
            double r;
            if (j.mode == IMH_BC_CIRC) {
                r = c[0];
            } else if (worm) {  // cell 0 of the partner, negated for mom(X) (isVecNorm)
                r = j.v == X ? -c[0] : c[0];
            } else {
                // zero_shift.m: fluxR keeps its upper side, fluxL its lower one
                double tv = *t;
                r = lean::end_ghost(j.mode, j.v == X, which != 1 - j.side, c[0], c[1],
                                    a.active_lin, a.bc_inf, tv);
                *t = tv;
            }
            if constexpr (kind == 0) {
                T* p = row(j.v * 4 + (j.side ? 0 : 2)) + slot;
                p[0] = T(2) * T(r);
                p[RL] = T(0);
            } else if constexpr (kind == 1) {
                row(j.v * 4 + o * 2 + (j.side ? 0 : 1))[slot] = T(r);
            } else {
                row(j.v * 2 + j.side)[slot] = T(r);
            }
        }
    };
    using Kind0 = std::integral_constant<int, 0>;
    using Kind1 = std::integral_constant<int, 1>;
    using Kind2 = std::integral_constant<int, 2>;

    // shift(X,-1) / shift(X,+1) of a row at chunk cell k; nb: the value next to the chunk.
    // In a chunk that the pencil end cuts short, end_fill() has put the value past the end
    // behind the last cell.
    auto lower_of = [&](const T (&A)[K], int k, T nb) __attribute__((always_inline)) -> T {
        return k > 0 ? A[k > 0 ? k - 1 : 0] : nb;
    };
    auto upper_of = [&](const T (&A)[K], int k, T nb) __attribute__((always_inline)) -> T {
        return k + 1 < K ? A[k + 1 < K ? k + 1 : k] : nb;
    };
    auto end_fill = [&](T (&A)[K], T nb) __attribute__((always_inline)) {
        if (full) return;
#pragma unroll
        for (int k = 1; k < K; ++k) A[k] = (i0 + k == N) ? nb : A[k];
    };
    // padding cells past the pencil end repeat the last cell
    auto pad_fill = [&](T (&A)[K]) __attribute__((always_inline)) {
        if (full) return;
#pragma unroll
        for (int k = 1; k < K; ++k) A[k] = (i0 + k < N) ? A[k] : A[k - 1];
    };

    // ================= predictor: W and C from U^n (wFluidFlux.m) ====================
    publish_max(0, numerators(q, OBJ_PRIM));
#pragma unroll
    for (int v = 0; v < 5; ++v) {
        row(v * 4 + 0)[tid] = q[v][0];
        row(v * 4 + 1)[tid] = nu[v][0];
        row(v * 4 + 2)[tid] = q[v][K - 1];
        row(v * 4 + 3)[tid] = nu[v][K - 1];
    }
    if (clo) {
#pragma unroll
        for (int v = 0; v < 5; ++v) {
            row(v * 4 + 2)[g_lo] = q[v][0];
            row(v * 4 + 3)[g_lo] = nu[v][0];
        }
    }
    if (chi) {
#pragma unroll
        for (int v = 0; v < 5; ++v) {
            row(v * 4 + 0)[g_hi] = q[v][K - 1];
            row(v * 4 + 1)[g_hi] = nu[v][K - 1];
        }
    }
    put_ends(q, nu);
    if (!simple && tid < PX * 10) {
#pragma unroll
        for (int r = 0; r < 3; ++r) s_trk[tid * 3 + r] = trk[r];
    }
    __syncthreads();
    const T C = pencil_max(0, px);
    const T rC = M::rcp(C);
    const T hfC = T(hf) * C;
    if (!simple) {
        ghosts(Kind0{});
        __syncthreads();
    }
#pragma unroll
    for (int v = 0; v < 5; ++v) {
        __builtin_amdgcn_sched_barrier(0);
        T FR[K], FL[K];
#pragma unroll
        for (int k = 0; k < K; ++k) {
            const T w = M::div(nu[v][k], C, rC);
            FR[k] = T(0.5) * (q[v][k] + w);
            FL[k] = T(0.5) * (q[v][k] - w);
        }
        const T nbR = T(0.5) * (row(v * 4 + 2)[tl_] + M::div(row(v * 4 + 3)[tl_], C, rC));
        const T nbL = T(0.5) * (row(v * 4 + 0)[tr_] - M::div(row(v * 4 + 1)[tr_], C, rC));
        end_fill(FL, nbL);
#pragma unroll
        for (int k = 0; k < K; ++k) {
            const T sR = lower_of(FR, k, nbR);
            const T sL = upper_of(FL, k, nbL);
            q[v][k] = q[v][k] - hfC * (FR[k] - sR + FL[k] - sL);
            lean::pin(q[v][k]);
        }
    }
    // mass.store.array = max(mass.store.array, MINMASS)
#pragma unroll
    for (int k = 0; k < K; ++k) q[0][k] = fmax(q[0][k], T(a.minmass));
#pragma unroll
    for (int v = 0; v < 5; ++v) pad_fill(q[v]);

    // ================= corrector: W' and C' from U^(n+1/2) ===========================
    {
        const T m = numerators(q, OBJ_FSTORE);
        publish_max(1, i0 < N ? m : T(NAN));
    }
    __syncthreads();  // also: every thread has read the predictor's rows
    const T C2 = pencil_max(1, px);
    const T rC2 = M::rcp(C2);
    const T ffC = T(ff) * C2;
    const int lim = a.limiter;
    // fluxR' in q, fluxL' in nu
#pragma unroll
    for (int v = 0; v < 5; ++v) {
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int k = 0; k < K; ++k) {
            const T w = M::div(nu[v][k], C2, rC2);
            const T h = q[v][k];
            q[v][k] = T(0.5) * (h + w);
            nu[v][k] = T(0.5) * (h - w);
            lean::pin(q[v][k]);
            lean::pin(nu[v][k]);
        }
        row(v * 4 + 0)[tid] = q[v][0];
        row(v * 4 + 1)[tid] = q[v][K - 1];
        row(v * 4 + 2)[tid] = nu[v][0];
        row(v * 4 + 3)[tid] = nu[v][K - 1];
    }
    if (clo) {
#pragma unroll
        for (int v = 0; v < 5; ++v) {
            row(v * 4 + 1)[g_lo] = q[v][0];
            row(v * 4 + 3)[g_lo] = nu[v][0];
        }
    }
    if (chi) {
#pragma unroll
        for (int v = 0; v < 5; ++v) {
            row(v * 4 + 0)[g_hi] = q[v][K - 1];
            row(v * 4 + 2)[g_hi] = nu[v][K - 1];
        }
    }
    put_ends(q, nu);
    __syncthreads();
    if (!simple) {
        ghosts(Kind1{});
        __syncthreads();
    }
    // limited fluxes, in place (each cell's update uses the values before it)
#pragma unroll
    for (int v = 0; v < 5; ++v) {
        __builtin_amdgcn_sched_barrier(0);
        const T nbRl = row(v * 4 + 1)[tl_], nbRr = row(v * 4 + 0)[tr_];
        const T nbLl = row(v * 4 + 3)[tl_], nbLr = row(v * 4 + 2)[tr_];
        end_fill(q[v], nbRr);
        end_fill(nu[v], nbLr);
        T R2[K], L2[K];
#pragma unroll
        for (int k = 0; k < K; ++k) {
            const T rm = lower_of(q[v], k, nbRl), rp = upper_of(q[v], k, nbRr);
            const T lm = lower_of(nu[v], k, nbLl), lp = upper_of(nu[v], k, nbLr);
            const T fr = q[v][k], fl = nu[v][k];
            R2[k] = fr + M::lim(lim, fr - rm, rp - fr);
            L2[k] = fl + M::lim(lim, lm - fl, fl - lp);
        }
        pad_fill(R2);
        pad_fill(L2);
#pragma unroll
        for (int k = 0; k < K; ++k) {
            q[v][k] = R2[k];
            nu[v][k] = L2[k];
            lean::pin(q[v][k]);
            lean::pin(nu[v][k]);
        }
    }
    __syncthreads();  // every thread has read this stage's rows and ends
#pragma unroll
    for (int v = 0; v < 5; ++v) {
        row(v * 2 + 0)[tid] = q[v][K - 1];
        row(v * 2 + 1)[tid] = nu[v][0];
        if (clo) row(v * 2 + 0)[g_lo] = q[v][0];
        if (chi) row(v * 2 + 1)[g_hi] = nu[v][K - 1];
    }
    put_ends(q, nu);
    __syncthreads();
    if (!simple) {
        ghosts(Kind2{});
        __syncthreads();
    }
    lean::pin(base);  // the cells' addresses are formed again, not kept since the loads
    lean::pin(i0);
#pragma unroll
    for (int v = 0; v < 5; ++v) {
        __builtin_amdgcn_sched_barrier(0);
        T un[K];
        if (v < KEEP) {
#pragma unroll
            for (int k = 0; k < K; ++k) un[k] = un0[v < KEEP ? v : 0][k];
        } else if (vec) {
            chunk_load<T, K>(a.q[v] + cb(), un);
        } else {
#pragma unroll
            for (int k = 0; k < K; ++k) un[k] = gmem(a.q[v])[off(k)];
        }
        const T nbR = row(v * 2 + 0)[tl_], nbL = row(v * 2 + 1)[tr_];
        end_fill(nu[v], nbL);
#pragma unroll
        for (int k = 0; k < K; ++k) {
            const T sR = lower_of(q[v], k, nbR);
            const T sL = upper_of(nu[v], k, nbL);
            const T dq = ffC * (q[v][k] - sR + nu[v][k] - sL);
            un[k] = un[k] - dq;
            if (v == 0) un[k] = fmax(un[k], T(a.minmass));  // mass.array = max(mass, MINMASS)
        }
        if (vec) {
            if (pen_ok && i0 < N) chunk_store<T, K>(a.q[v] + cb(), un);
        } else {
#pragma unroll
            for (int k = 0; k < K; ++k)
                if (pen_ok && i0 + k < N) gmem(a.q[v])[off(k)] = un[k];
        }
    }

    // ---- the edge trackers back -------------------------------------------------------
    if (!simple) {
        const Job j = job();
        if (job_trk(j)) {
#pragma unroll
            for (int r = 0; r < 3; ++r) *trk_at(j, r) = s_trk[tid * 3 + r];
        }
    }
}

#ifdef IMH_LEAN_OCCUPANCY
// Persistent batched form (tiles != nullptr) or one block per tile of args[0].
template <typename T, int BS, int K, bool MHD, int D, int FORM>
__global__ void __launch_bounds__(BS) IMH_LEAN_OCCUPANCY
fluid_lean_kernel(const FluidArgs<T>* args, const BatchTile* tiles, int ntiles) {
    extern __shared__ __attribute__((aligned(16))) char lean_lds[];
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
            tile = args[0].xcd_remap ? xcd_tile(blockIdx.x, ntiles) : (long long)blockIdx.x;
        }
        double dt;
        if (sweep_runs(args[arg], dt))
            fluid_lean_body<T, BS, K, MHD, D, FORM>(args[arg], tile, lean_lds, dt);
        __syncthreads();
    }
}
#endif

}  // namespace imh
