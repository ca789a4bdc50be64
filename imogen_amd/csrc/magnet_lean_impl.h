// magnet_lean_impl.h -- the magnetic sweep (magnet/magnetFlux.m, magnet/relaxingMagnet.m,
// MagnetArray.updateCellCentered) of the common case: no fade end, no first assignment of
// the flux objects, uniform spacing, pencils of 8 cells or more.  magnet_sweep_impl.h holds
// the general form.
//
// One magnetFlux(X, [I1 I2]) is two launches:
//   flow (mag_flow_body)  per component I: the grid-aligned velocity of every cell into
//                         LDS beside B_I, one barrier, then each thread advects four
//                         consecutive cells from a window of twelve: the smoothing, both
//                         upwind passes and the limiter are recomputed where windows
//                         overlap instead of being exchanged (the general form exchanges
//                         six times, two barriers each); the limited fluxes go to scratch.
//   CT (mag_ct_body)      both components' curl terms into B_X in one pass, the new B_X
//                         also into LDS; cell-centred B_I2 beside it; one barrier; the
//                         cell-centred B_X.
// The general form takes six launches, and its y / z pencils read one cell per row; here
// the lanes of y / z tiles run over adjacent pencils.  A tile is PX whole pencils, so that
// B_I and B_X can be updated in place.  What bounds it: HBM and L2 traffic on large grids (FP64
// 200^3: 150 us of advection and 107 of CT for 512 and 448 MB), the latency of a tile's chain
// (loads, LDS, windows, stores) on small ones; the arithmetic is some 100 instructions per
// cell and component.  Per magnetFlux call, general -> lean: FP64 100^3 85 -> 32 us, 512^2 52 ->
// 16 (x) and 22 (y); the 1-D lane's iteration (lane1d.hip) 181 -> 130.
//
// TRK: some boundary is transparent or a wall.  Without, the kernels hold no tracker code: FP64
// advection 147 -> 88 vector registers (3 -> 5 waves per SIMD), CT 89 -> 57.
//
// Past a pencil end the windows hold the wrapped cells (circular) or the ghosts of each
// shift call in the .m text's order, from the object's edge tracker (other modes), put in by
// the thread that owns the end cell: chunk 0 starts at cell 0 and the last chunk is moved
// back to end at cell N-1, so both ends sit at fixed places of a window.  The last chunk
// stores all its cells, the one before it those in front of N-4, whose windows then end
// within the pencil.
//
// Transverse ghosts of transparent faces nudge their tracker once per sweep: the flow
// evaluates every cell's velocity once (and stores the nudged trackers); the CT evaluates
// some fluxes twice, from the trackers as they were, and stores the nudged ones after its
// barrier.
#pragma once

#include "fluid_lean_impl.h"

namespace imh {

namespace mlean {

constexpr int CH = 4;  // cells of a chunk
// x rows: lanes read at a distance of one chunk
__device__ constexpr int pad(int p) { return p + (p >> 2); }

// One-cell transverse shift along I: where the neighbour is (an offset from the cell), and
// what the boundary makes of it.
struct Nb {
    int off;
    bool neg, zero, trk;
};
__device__ __forceinline__ Nb transverse(int mode, bool upper, bool flips, bool zeroes, int jI,
                                         int NI, int sI) {
    const int in = upper ? -sI : sI;   // towards the interior, from the face
    Nb n = {-in, false, false, false};
    if (upper ? jI < NI - 1 : jI > 0) return n;
    n.off = 0;                         // const, flip, zero: the cell itself
    if (mode == IMH_BC_CIRC) n.off = in * (NI - 1);
    else if (mode == IMH_BC_MIRROR) n.off = NI > 1 ? in : 0;
    else if (mode == IMH_BC_TRANS) n.off = NI > 2 ? in : 0;  // (shorter: the end cell repeats)
    n.trk = mode == IMH_BC_TRANS || mode == IMH_BC_WALL;
    n.neg = flips && (mode == IMH_BC_MIRROR || mode == IMH_BC_FLIP);
    n.zero = zeroes && mode == IMH_BC_ZERO;
    return n;
}

// Whether the ghosts of a boundary come from its edge tracker.
__host__ __device__ constexpr bool tracked(int mode) {
    return mode == IMH_BC_TRANS || mode == IMH_BC_WALL;
}
// The ghost of a one-cell shift past a pencil end (lean::end_ghost); without TRK no mode of the
// sweep is tracked, and the ghost is an element or 0.
template <bool TRK, typename T>
__device__ __forceinline__ T end_value(int mode, bool neg, bool zero, T c0, T c1, int active,
                                       int bc_inf, double& tracker) {
    if constexpr (TRK) {
        return T(lean::end_ghost(mode, neg, zero, double(c0), double(c1), active, bc_inf, tracker));
    } else {
        if (mode == IMH_BC_ZERO && zero) return T(0);
        const T r = mode == IMH_BC_MIRROR ? c1 : c0;
        return (neg && (mode == IMH_BC_MIRROR || mode == IMH_BC_FLIP)) ? -r : r;
    }
}

// The two ghosts of shift(X, 2) past the upper end; c0, c1, c2: the end cell and the two
// before it.
__device__ __forceinline__ void end_ghost2(int mode, double c0, double c1, double c2, int N,
                                           int active, int bc_inf, double& tracker, double& g0,
                                           double& g1) {
    if (mode == IMH_BC_TRANS) {
        const GhostSpec s = {mode, 1, 0, 0, active, bc_inf};
        const Ends e = {0.0, 0.0, 0.0, c2, c1, c0};
        ghost_values<2>(s, e, N, 2, &tracker, g0, g1);
        return;
    }
    g0 = g1 = c0;
    if (mode == IMH_BC_WALL) g0 = g1 = tracker;
    if (mode == IMH_BC_MIRROR) {
        g0 = c1;
        g1 = c2;
    }
}

// FP64: the lean sweep's quotient and limiter (the same bits as the division's).
__device__ __forceinline__ double quot(double x, double y) { return LMath<double>::quot(x, y); }
__device__ __forceinline__ float quot(float x, float y) { return x / y; }
__device__ __forceinline__ double limited(int l, double dl, double dr) {
    return LMath<double>::lim(l, dl, dr);
}
__device__ __forceinline__ float limited(int l, float dl, float dr) { return lim_delta(l, dl, dr); }

// Thread, pencil and geometry of a tile.
template <bool XM>
struct Tile {
    int px, ty, TL;
    long long pen;
    bool ok;
    unsigned base, stride;
    int pc[3];
    template <typename T>
    __device__ __forceinline__ Tile(const MagnetLeanArgs<T>& a, int d, int PX, int TL_,
                                    long long tile) {
        const int tid = threadIdx.x;
        TL = TL_;
        const int lg = 31 - __builtin_clz(XM ? TL : PX);
        px = XM ? tid >> lg : tid & (PX - 1);
        ty = XM ? tid & (TL - 1) : tid >> lg;
        pen = tile * PX + px;
        ok = pen < a.npencil;
        const int nn[3] = {a.n0, a.n1, a.n2};
        long long b, s;
        const long long p = ok ? pen : a.npencil - 1;  // padding pencils read a real one
        pencil_base(nn, d, p, b, s);
        pencil_coords(nn, d, p, pc);
        base = unsigned(b);
        stride = unsigned(s);
    }
};

}  // namespace mlean

// The advection of component I[comp] (relaxingMagnet.m:15-50) along D on one tile.
template <typename T, int D, bool TRK>
__device__ __forceinline__ void mag_flow_body(const MagnetLeanArgs<T>& ap, int comp,
                                              long long tile, T* lds, double dt) {
    const MagnetLeanArgs<T> a = uniform_load(&ap);
    constexpr bool XM = D == 0;
    constexpr int CH = mlean::CH;
    const int PX = a.PX;
    const mlean::Tile<XM> t(a, D, PX, a.TL, tile);
    const int N = sel3i(D, a.n0, a.n1, a.n2);
    const int nn[3] = {a.n0, a.n1, a.n2};
    const int dI = comp ? a.dI[1] : a.dI[0];
    const int linI = comp ? a.active_linI[1] : a.active_linI[0];
    T* const bI = comp ? a.bI[1] : a.bI[0];
    T* const flux = a.flux + (comp ? a.ncell : 0);
    const int mlo = mode_at(a.modes, 0, D), mhi = mode_at(a.modes, 1, D);
    const int f = a.bc_inf;
    // LDS slot of cell i (-4..N+3)
    const int rl = mag_lean_row(XM, N);
    T* const sr = lds + (XM ? t.px * rl : t.px);
    T* const sb = sr + PX * rl;
    auto slot = [&](int i) __attribute__((always_inline)) -> int {
        return XM ? mlean::pad(i + 4) : (i + 4) * PX;
    };

    // ---- (shift_I(p_X,-1) + p_X) ./ (shift_I(rho,-1) + rho), and B_I, into LDS ---------------
    {
        const int jI = sel3i(dI, t.pc[0], t.pc[1], t.pc[2]);  // constant along the pencil
        const int NI = sel3i(dI, a.n0, a.n1, a.n2);
        const int sI = dI == 0 ? 1 : (dI == 1 ? a.n0 : a.n0 * a.n1);
        const int mI = mode_at(a.modes, 0, dI);
        mlean::Nb nb = {0, false, false, false};
        if (dI < a.ndims) nb = mlean::transverse(mI, false, false, false, jI, NI, sI);
        constexpr int U = 4;
        for (int p0 = t.ty; p0 < N; p0 += U * t.TL) {
            T m0[U], r0[U], mn[U], rn[U], b[U];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int i = p0 + u * t.TL < N ? p0 + u * t.TL : N - 1;
                const unsigned cell = t.base + unsigned(i) * t.stride;
                m0[u] = gmem(a.mom)[cell];
                r0[u] = gmem(a.rho)[cell];
                mn[u] = gmem(a.mom)[cell + unsigned(nb.off)];
                rn[u] = gmem(a.rho)[cell + unsigned(nb.off)];
                b[u] = gmem(bI)[cell];
            }
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int i = p0 + u * t.TL;
                if (i >= N) break;
                if (TRK && nb.trk && t.ok) {
                    const long long fi = face_index(nn, dI, D == 0 ? i : t.pc[0],
                                                    D == 1 ? i : t.pc[1], D == 2 ? i : t.pc[2]);
                    const long long im = a.eoff[((OBJ_PRIM + D + 1) * 2 + 0) * 3 + dI] + fi;
                    const long long ir = a.eoff[((OBJ_PRIM + 0) * 2 + 0) * 3 + dI] + fi;
                    double em = a.edges[im], er = a.edges[ir];
                    mn[u] = T(lean::end_ghost(mI, false, false, double(m0[u]), double(mn[u]), linI,
                                              f, em));
                    rn[u] = T(lean::end_ghost(mI, false, false, double(r0[u]), double(rn[u]), linI,
                                              f, er));
                    if (mI == IMH_BC_TRANS) {
                        a.edges[im] = em;
                        a.edges[ir] = er;
                    }
                }
                const T v = mlean::quot(mn[u] + m0[u], rn[u] + r0[u]);
                sr[slot(i)] = v;
                sb[slot(i)] = b[u];
                if (i < 4 && mhi == IMH_BC_CIRC) {
                    sr[slot(N + i)] = v;
                    sb[slot(N + i)] = b[u];
                }
                if (i >= N - 4 && mlo == IMH_BC_CIRC) {
                    sr[slot(i - N)] = v;
                    sb[slot(i - N)] = b[u];
                }
            }
        }
    }
    __syncthreads();
    if (!t.ok) return;  // no barrier follows in this body

    const double ff = 0.5 * dt / a.dxX;       // relaxingMagnet.m:15
    const T hf = T(ff), hf2 = T(2.0 * ff);    // relaxingMagnet.m:32
    const int nch = (N + CH - 1) / CH;
    auto eidx = [&](int obj, int side) __attribute__((always_inline)) -> long long {
        return a.eoff[((obj + 3 * dI + D) * 2 + side) * 3 + D] + t.pen;
    };
    for (int c = t.ty; c < nch; c += t.TL) {
        const bool last = c == nch - 1;
        const int i0 = last ? N - CH : c * CH;
        const bool lo = c == 0 && mlo != IMH_BC_CIRC, hi = last && mhi != IMH_BC_CIRC;
        const bool tlo = TRK && lo && mlean::tracked(mlo), thi = TRK && hi && mlean::tracked(mhi);
        // edge trackers of this pencil along X
        double evg_lo = 0, esfr_lo = 0, ewm_lo = 0, efl_lo = 0, evg_hi = 0, esfr_hi = 0, ewm_hi = 0;
        if (tlo) {
            evg_lo = a.edges[eidx(OBJ_VG, 0)];
            esfr_lo = a.edges[eidx(OBJ_MSFR, 0)];
            ewm_lo = a.edges[eidx(OBJ_WMAG, 0)];
            efl_lo = a.edges[eidx(OBJ_MFLUX, 0)];
        }
        if (thi) {
            evg_hi = a.edges[eidx(OBJ_VG, 1)];
            esfr_hi = a.edges[eidx(OBJ_MSFR, 1)];
            ewm_hi = a.edges[eidx(OBJ_WMAG, 1)];
        }
        // ghosts of a one-cell shift along X (component I != X: no sign flips)
        auto glo = [&](bool zero, T c0, T c1, double& trk) __attribute__((always_inline)) -> T {
            return mlean::end_value<TRK>(mlo, false, zero, c0, c1, a.active_linX, f, trk);
        };
        auto ghi = [&](T c0, T c1, double& trk) __attribute__((always_inline)) -> T {
            return mlean::end_value<TRK>(mhi, false, false, c0, c1, a.active_linX, f, trk);
        };

        // arrays over cells -4..7 of the window (index 4 + j); each stage holds two less
        T vg[12], b[12];
#pragma unroll
        for (int j = 0; j < 12; ++j) vg[j] = sr[slot(i0 + j - 4)];
#pragma unroll
        for (int j = 1; j < 11; ++j) b[j] = sb[slot(i0 + j - 4)];
        if (lo) vg[3] = glo(false, vg[4], vg[5], evg_lo);
        if (hi) vg[8] = ghi(vg[7], vg[6], evg_hi);
        // smoothing: vg = 0.25*(vg.shift(X,-1) + vg.shift(X,1) + 2*vg)
        T s[12];
#pragma unroll
        for (int j = 1; j < 11; ++j) s[j] = T(0.25) * (vg[j - 1] + vg[j + 1] + T(2) * vg[j]);
        if (hi) s[8] = ghi(s[7], s[6], evg_hi);
        // velocityFlow = (vg + vg.shift(X,1)) < 0
        T vf[10];
#pragma unroll
        for (int j = 1; j < 10; ++j) vf[j] = (s[j] + s[j + 1] < T(0)) ? T(1) : T(0);
        // predictor: store.fluxR = B.*vg; upwind select; B_half
        T w[12], wu[10];
#pragma unroll
        for (int j = 1; j < 11; ++j) w[j] = b[j] * s[j];
        if (hi) w[8] = ghi(w[7], w[6], esfr_hi);
#pragma unroll
        for (int j = 1; j < 10; ++j) wu[j] = w[j] * (T(1) - vf[j]) + w[j + 1] * vf[j];
        if (lo) wu[3] = glo(true, wu[4], wu[5], esfr_lo);  // FLUXR: zero mode's lower ghost 0
        // corrector: wMag = store.*vg; flux; dFluxR, dFluxL; limiter
        T wm[10];
#pragma unroll
        for (int j = 2; j < 10; ++j) {
            const T st = b[j] - hf * (wu[j] - wu[j - 1]);
            wm[j] = st * s[j];
        }
        if (lo) wm[3] = glo(false, wm[4], wm[5], ewm_lo);
        // ghosts past the upper end, one set per shift call of the .m text
        T a7 = wm[8], b7 = wm[8], c7 = wm[8], d6 = wm[8], d7 = wm[9];
        if (hi) {
            a7 = ghi(wm[7], wm[6], ewm_hi);   // flux = ... shift(X,1)
            b7 = ghi(wm[7], wm[6], ewm_hi);   // dFluxR: shift(X,1)
            if constexpr (TRK) {              // dFluxR: shift(X,2)
                double g0, g1;
                mlean::end_ghost2(mhi, double(wm[7]), double(wm[6]), double(wm[5]), N, a.active_linX,
                                  f, ewm_hi, g0, g1);
                d6 = T(g0);
                d7 = T(g1);
            } else {
                d6 = mhi == IMH_BC_MIRROR ? wm[6] : wm[7];
                d7 = mhi == IMH_BC_MIRROR ? wm[5] : wm[7];
            }
            c7 = ghi(wm[7], wm[6], ewm_hi);   // dFluxL: shift(X,1)
        }
        const int lim = a.limiter;
        T F[8];
#pragma unroll
        for (int j = 3; j < 8; ++j) {
            const T a1 = j == 7 ? a7 : wm[j + 1];
            const T b1 = j == 7 ? b7 : wm[j + 1];
            const T c1 = j == 7 ? c7 : wm[j + 1];
            const T b2 = j == 7 ? d7 : (j == 6 ? d6 : wm[j + 2]);
            const T F0 = wm[j] * (T(1) - vf[j]) + a1 * vf[j];
            const T dR = b1 - (vf[j] * b2 + (T(1) - vf[j]) * wm[j]);
            const T dL = wm[j] - (vf[j] * c1 + (T(1) - vf[j]) * wm[j - 1]);
            F[j] = F0 + mlean::limited(lim, dL, dR);
        }
        if (lo) F[3] = glo(true, F[4], F[5], efl_lo);  // 'flux' type: zero mode's ghost 0
        // B_I = B_I - 2*fluxFactor .* (flux - flux.shift(X,-1))
#pragma unroll
        for (int k = 0; k < CH; ++k) {
            if (last || i0 + k < N - CH) {
                const unsigned cell = t.base + unsigned(i0 + k) * t.stride;
                gmem(bI)[cell] = b[4 + k] - hf2 * (F[4 + k] - F[3 + k]);
                gmem(flux)[cell] = F[4 + k];
            }
        }
        if (tlo && mlo == IMH_BC_TRANS) {
            a.edges[eidx(OBJ_VG, 0)] = evg_lo;
            a.edges[eidx(OBJ_MSFR, 0)] = esfr_lo;
            a.edges[eidx(OBJ_WMAG, 0)] = ewm_lo;
            a.edges[eidx(OBJ_MFLUX, 0)] = efl_lo;
        }
        if (thi && mhi == IMH_BC_TRANS) {
            a.edges[eidx(OBJ_VG, 1)] = evg_hi;
            a.edges[eidx(OBJ_MSFR, 1)] = esfr_hi;
            a.edges[eidx(OBJ_WMAG, 1)] = ewm_hi;
        }
    }
}

// Constrained transport of both components (relaxingMagnet.m:56-60: flux = flux -
// flux.shift(I,1); flux = flux.shift(X,-1); mag(X) = mag(X) - dt/DGRID{I} .* flux), then
// cellMag_k = 0.5*(B_k + B_k.shift(k,1)) (MagnetArray.m:36-38) of the last component and X.
template <typename T, int D, bool TRK>
__device__ __forceinline__ void mag_ct_body(const MagnetLeanArgs<T>& ap, long long tile, T* lds,
                                            double dt) {
    const MagnetLeanArgs<T> a = uniform_load(&ap);
    constexpr bool XM = D == 0;
    const int PX = a.PX;
    const mlean::Tile<XM> t(a, D, PX, a.TL, tile);
    const int N = sel3i(D, a.n0, a.n1, a.n2);
    const int nn[3] = {a.n0, a.n1, a.n2};
    const int f = a.bc_inf;
    const int mlo = mode_at(a.modes, 0, D), mhi = mode_at(a.modes, 1, D);
    T* const row = lds + (XM ? t.px * N : t.px);
    const int rs = XM ? 1 : PX;

    // G = F - shift_I(F,+1): flux object, component I == DIRECT (flips for mirror / flip),
    // type 'flux' (zero mode: ghost 0)
    mlean::Nb nb[2], nc;
    T ffI[2];
    bool onf[2];   // cells on a transparent upper I face: their trackers are nudged
#pragma unroll
    for (int q = 0; q < 2; ++q) {
        const int dI = a.dI[q];
        const int jI = sel3i(dI, t.pc[0], t.pc[1], t.pc[2]);
        const int NI = sel3i(dI, a.n0, a.n1, a.n2);
        const int sI = dI == 0 ? 1 : (dI == 1 ? a.n0 : a.n0 * a.n1);
        const int m = mode_at(a.modes, 1, dI);
        nb[q] = {0, false, false, false};
        if (dI < a.ndims) nb[q] = mlean::transverse(m, true, true, true, jI, NI, sI);
        if (q == 1) {
            nc = nb[1];
            nc.zero = false;  // not a flux: zero mode keeps constant ghosts
        }
        onf[q] = TRK && nb[q].trk && m == IMH_BC_TRANS;
        ffI[q] = T(dt / a.dxI[q]);
    }
    auto fidx = [&](int obj, int dI, int i) __attribute__((always_inline)) -> long long {
        return a.eoff[(obj * 2 + 1) * 3 + dI] +
               face_index(nn, dI, D == 0 ? i : t.pc[0], D == 1 ? i : t.pc[1], D == 2 ? i : t.pc[2]);
    };
    // the upper I neighbour's value v read at nb.off, as the boundary has it; trk: a copy
    auto shifted = [&](const mlean::Nb& n, int q, T self, T v, double& trk)
        __attribute__((always_inline)) -> T {
        if (TRK && n.trk)
            return T(lean::end_ghost(mode_at(a.modes, 1, a.dI[q]), true, n.zero, double(self),
                                     double(v), a.active_linI[q], f, trk));
        if (n.zero) return T(0);
        return n.neg ? -v : v;
    };
    auto curl = [&](int q, int i, T f0, T fn) __attribute__((always_inline)) -> T {
        double trk = 0;
        if (TRK && nb[q].trk) trk = a.edges[fidx(OBJ_MFLUX + 3 * a.dI[q] + D, a.dI[q], i)];
        return f0 - shifted(nb[q], q, f0, fn, trk);
    };
    // ghosts of flux.shift(X,-1) that are not an element of the array
    const bool glo = (TRK && mlean::tracked(mlo)) || mlo == IMH_BC_ZERO;
    const int ilo = mlo == IMH_BC_CIRC ? N - 1 : (mlo == IMH_BC_MIRROR ? 1 : 0);

    constexpr int U = 2;
    for (int p0 = t.ty; p0 < N; p0 += U * t.TL) {
        T f0[2][U], fn[2][U], bx[U], bi[U], bn[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int i = p0 + u * t.TL < N ? p0 + u * t.TL : N - 1;
            const unsigned cell = t.base + unsigned(i) * t.stride;
            const unsigned cm = t.base + unsigned(i > 0 ? i - 1 : ilo) * t.stride;
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                const T* F = a.flux + (q ? a.ncell : 0);
                f0[q][u] = gmem(F)[cm];
                fn[q][u] = gmem(F)[cm + unsigned(nb[q].off)];
            }
            bx[u] = gmem(a.bX)[cell];
            bi[u] = gmem(a.bI[1])[cell];
            bn[u] = gmem(a.bI[1])[cell + unsigned(nc.off)];
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int i = p0 + u * t.TL;
            if (i >= N || !t.ok) break;
            const unsigned cell = t.base + unsigned(i) * t.stride;
            T x = bx[u];
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                T h = curl(q, i > 0 ? i - 1 : ilo, f0[q][u], fn[q][u]);
                if (glo && i == 0) {
                    if (!TRK || mlo == IMH_BC_ZERO) {
                        h = T(0);
                    } else {
                        const long long ei =
                            a.eoff[((OBJ_MFLUX + 3 * a.dI[q] + D) * 2 + 0) * 3 + D] + t.pen;
                        double tr = a.edges[ei];
                        const T* F = a.flux + (q ? a.ncell : 0);
                        const unsigned c1 = t.base + t.stride;
                        const T h1 = curl(q, 1, gmem(F)[c1], gmem(F)[c1 + unsigned(nb[q].off)]);
                        h = mlean::end_value<TRK>(mlo, false, true, h, h1, a.active_linX, f, tr);
                        if (mlo == IMH_BC_TRANS) a.edges[ei] = tr;
                    }
                }
                x = x - ffI[q] * h;
            }
            gmem(a.bX)[cell] = x;
            row[i * rs] = x;
            double tc = 0;
            const bool trkc = TRK && nc.trk;
            const long long ic = trkc ? fidx(OBJ_MAG + a.dI[1], a.dI[1], i) : 0;
            if (trkc) tc = a.edges[ic];
            const T sh = shifted(nc, 1, bi[u], bn[u], tc);
            if (onf[1]) a.edges[ic] = tc;
            gmem(a.cI)[cell] = T(0.5) * (bi[u] + sh);
        }
    }
    __syncthreads();
    if (!t.ok) return;  // no barrier follows in this body
    for (int i = t.ty; i < N; i += t.TL) {
        const unsigned cell = t.base + unsigned(i) * t.stride;
        const T x = row[i * rs];
        T sh;
        if (i < N - 1) {
            sh = row[(i + 1) * rs];
        } else if (mhi == IMH_BC_CIRC) {
            sh = row[0];
        } else {
            const bool trk = TRK && mlean::tracked(mhi);
            const long long ei = trk ? a.eoff[((OBJ_MAG + D) * 2 + 1) * 3 + D] + t.pen : 0;
            double tr = 0;
            if (trk) tr = a.edges[ei];
            sh = mlean::end_value<TRK>(mhi, true, false, x, row[(N - 2) * rs], a.active_linX, f, tr);
            if (trk && mhi == IMH_BC_TRANS) a.edges[ei] = tr;
        }
        gmem(a.cX)[cell] = T(0.5) * (x + sh);
#pragma unroll
        for (int q = 0; q < 2; ++q)
            if (onf[q] && a.active_linI[q]) {
                const long long ei = fidx(OBJ_MFLUX + 3 * a.dI[q] + D, a.dI[q], i);
                double tr = a.edges[ei];
                edge_nudge(tr, double(gmem(a.flux + (q ? a.ncell : 0))[cell]));
                a.edges[ei] = tr;
            }
    }
}

}  // namespace imh
