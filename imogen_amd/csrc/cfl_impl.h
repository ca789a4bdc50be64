// cfl_impl.h -- device functions of the time update (TimeManager.m), shared by the CFL launches
// (cfl.hip) and the 1-D iteration kernel (line1d_variant.hip).
#pragma once

#include "fluid_lean_impl.h"
#include "imh_common.h"
#include "imh_kernels.h"

namespace imh {

namespace {

__device__ inline double wave_max(double v) {
    for (int off = 32; off >= 1; off >>= 1) v = fmax(v, __shfl_xor(v, off, 64));
    return v;
}

// Maxima of m over the block in every thread (NaN ignored: MATLAB max; 0 when all are NaN).
template <int BS>
__device__ __forceinline__ void block_max(double (&m)[3], double (*s_red)[BS / 64]) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        const double v = wave_max(m[k]);
        if (lane == 0) s_red[k][wave] = v;
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        double v = s_red[k][0];
#pragma unroll
        for (int w = 1; w < BS / 64; ++w) v = fmax(v, s_red[k][w]);
        m[k] = v >= 0.0 ? v : 0.0;
    }
}

// |p_i/rho| + c_s (pressure.m 'sound', the operations of pressure_sound) of one cell.
__device__ __forceinline__ void cell_speeds(double rho, double px, double py, double pz, double E,
                                            double bx, double by, double bz, const MagUse& u,
                                            double g, double (&m)[3]) {
#pragma clang fp contract(off)  // FP32 units contract; every unit rounds these alike
    using M = LMath<double>;
    const double inv = M::rcp(rho);
    const double v2 = M::quot(px * px + py * py + pz * pz, rho * rho);
    double b2 = 0.0;
    if (u.x) b2 = 0.0 + bx * bx;
    if (u.y) b2 = b2 + by * by;
    if (u.z) b2 = b2 + bz * bz;
    double r = (g - 1.0) * (E - 0.5 * rho * v2);
    r = r - (g - 1.0) * 0.5 * b2;
    const double cs = M::root(fabs(M::div(g * r + 2.0 * b2, rho, inv)));
    m[0] = fmax(m[0], fabs(M::div(px, rho, inv)) + cs);
    m[1] = fmax(m[1], fabs(M::div(py, rho, inv)) + cs);
    m[2] = fmax(m[2], fabs(M::div(pz, rho, inv)) + cs);
}

}  // namespace

// The speeds of cells [c0, c1), c0 a multiple of 4, into m.
template <int BS, typename T>
__device__ __forceinline__ void cfl_cells(const CflArgs<T>& a, long long c0, long long c1,
                                          double (&m)[3]) {
    typedef T V4 __attribute__((ext_vector_type(4)));
    for (long long c = c0 + 4 * threadIdx.x; c < c1; c += 4 * BS) {
        T q[5][4], b[3][4];
        if (c + 4 <= c1) {
#pragma unroll
            for (int v = 0; v < 5; ++v) {
                const V4 x = *(const IMH_GLOBAL_AS V4*)(gmem(a.q[v]) + c);
#pragma unroll
                for (int u = 0; u < 4; ++u) q[v][u] = x[u];
            }
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                V4 x = {T(0), T(0), T(0), T(0)};
                if (a.bc[k]) x = *(const IMH_GLOBAL_AS V4*)(gmem(a.bc[k]) + c);
#pragma unroll
                for (int u = 0; u < 4; ++u) b[k][u] = x[u];
            }
        } else {  // the last cells, the first of them again in place of those past c1
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const long long cu = c + u < c1 ? c + u : c;
#pragma unroll
                for (int v = 0; v < 5; ++v) q[v][u] = gmem(a.q[v])[cu];
#pragma unroll
                for (int k = 0; k < 3; ++k) b[k][u] = a.bc[k] ? gmem(a.bc[k])[cu] : T(0);
            }
        }
#pragma unroll
        for (int u = 0; u < 4; ++u)
            cell_speeds(double(q[0][u]), double(q[1][u]), double(q[2][u]), double(q[3][u]),
                        double(q[4][u]), double(b[0][u]), double(b[1][u]), double(b[2][u]), a.use,
                        a.gamma, m);
    }
}

// dt of one simulation from its reduced speeds (TimeManager.m:65-98).
__device__ inline void finalize_sim(SimDev& d, const SimParams& q, const double (&speed)[3]) {
#pragma clang fp contract(off)
    double cmax = 1e-2, dx = 0.0;
    int gi = 0;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        if (speed[k] > cmax) {
            cmax = speed[k];
            dx = q.dgrid[k];
            gi = k + 1;
        }
    }
    if (gi < 1) {
        d.error = IMH_ECFL;
        d.active = 0;
        return;
    }
    d.grid_index = gi;
    double upd = double(q.update_mode + 1);
    d.dt = q.cfl * dx / cmax;
    double newtime = d.time + upd * d.dt;
    if (newtime > q.time_max) {
        d.dt = (q.time_max - d.time) / upd;
        newtime = q.time_max;
    }
    d.time = newtime;
}

// TimeManager.running (TimeManager.m:36-39), evaluated at the top of the loop body.
__device__ inline int running(const SimDev& d, const SimParams& q) {
    return (d.iteration <= q.iter_max) && (d.time < q.time_max) && d.error == 0;
}

// Whether a simulation takes part in time update `step` (2: only with update_mode 0).
__device__ inline int cfl_runs(const SimDev& d, const SimParams& par, int gate, int step) {
    if (step > 1 && par.update_mode != 0) return -1;  // no second update
    return gate == CFL_ALWAYS ? 1 : (gate == CFL_ACTIVE ? d.active : running(d, par));
}

// The end of a time update, by one thread.  count: the loop body's iteration = iteration + 1
// (TimeManager.step) goes with its last time update; nothing reads it in between.
__device__ inline void cfl_finish(SimDev& d, const SimParams& par, int run, int gate, int step,
                                  int count, const double (&m)[3]) {
    if (gate != CFL_ACTIVE) d.active = run;
    if (!run) return;
    finalize_sim(d, par, m);
    if (count && d.active && step == (par.update_mode == 0 ? 2 : 1)) d.iteration += 1;
}

}  // namespace imh
