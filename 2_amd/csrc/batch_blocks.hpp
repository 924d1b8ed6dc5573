// batch_blocks.hpp -- device side of the batched stepping (batch.hip): the
// descriptors, one workgroup's share of each pass, and the step controller.
#pragma once

#include "comp_tiles.hpp"
#include "demag_tiles.hpp"

namespace mmx {

enum BatchPass { BP_XF = 0, BP_Y = 1, BP_Z = 2, BP_YI = 3, BP_XI = 4, BP_N = 5 };

// Per-simulation descriptor, read-only during a launch.
struct BatchSim {
    DemagGeom g;
    LineFFT<float> fx, fy, fz;
    FieldParams fp;
    float2 *xbuf, *ybuf;
    const float *kern;
    float *mbuf[2];
    float *mpred, *tau0;
    const float *msat_map;
    // composite-radix transforms with radices up to 16 (ns = 0: the generic
    // tiles), and whether z takes 64 columns per workgroup (z_column_tile)
    CompFFT cx, cy, cz;
    int zcol;
    int tile[BP_N];   // rows (XF, XI) or columns (Y, Z, YI) per workgroup
    int ntx[BP_N];    // column tiles per line set (Y, Z, YI)
    int first[BP_N];  // first block of this simulation in each pass
};

// Per-simulation RK12 state, owned by the device during a run.
struct BatchState {
    double t, dt, t0, t_stop, mindt, maxdt, maxerr, err, peakerr, gamma;
    long long step, step_stop, badsteps, evals;
    int cur, tries, need_stage0, active, error;
    float h;
    unsigned int err_bits;
    int pad_;
};

// ------------------------------------------------------------- kernels
//
// Which tiles a pass's kernel has to hold: the composite-radix ones, the
// 64-column z tile alone, or any, the generic ones included, whose registers
// (148 against 94 or fewer) leave three waves per SIMD instead of five; a batch
// with no simulation that needs them runs without.
enum BatchKind { KIND_COMP = 0, KIND_ZCOL = 1, KIND_ANY = 2 };

// Each pass is a device function of one virtual block `vb` (a tile of one
// simulation, from the pass's block table), called by the per-pass kernels
// with vb = blockIdx.x and by the persistent kernel for vb = blockIdx.x,
// blockIdx.x + gridDim.x, ...

template <int STAGE, int KIND>
__device__ __forceinline__ void bxf_block(const BatchSim *__restrict__ sims,
                                          const BatchState *__restrict__ st,
                                          const int *__restrict__ map, int vb, float2 *sm)
{
    const int s = map[vb];
    const BatchSim &S = sims[s];
    const BatchState &Z = st[s];
    if (!Z.active || (STAGE == 0 && !Z.need_stage0)) return;
    const long row0 = (long)(vb - S.first[BP_XF]) * S.tile[BP_XF];
    const float *m = S.mbuf[Z.cur];
    const bool comp = KIND != KIND_ANY || S.cx.ns;
    if (comp && STAGE == 0)
        xf_comp_tile<16, 0>(S.g, S.cx, S.tile[BP_XF], row0, m, S.msat_map, nullptr, 0.0f, nullptr,
                            nullptr, S.xbuf, sm);
    else if (comp)
        xf_comp_tile<16, 1>(S.g, S.cx, S.tile[BP_XF], row0, m, S.msat_map, S.tau0, Z.h, S.msat_map,
                            S.mpred, S.xbuf, sm);
    else if (STAGE == 0)
        xf_tile<0>(S.g, S.fx, S.tile[BP_XF], row0, m, S.msat_map, nullptr, 0.0f, nullptr, nullptr,
                   S.xbuf, sm);
    else
        xf_tile<1>(S.g, S.fx, S.tile[BP_XF], row0, m, S.msat_map, S.tau0, Z.h, S.msat_map,
                   S.mpred, S.xbuf, sm);
}

// log2 of the columns of a tile (a power of two on the composite passes)
__device__ __forceinline__ int log2_tile(int w) { return __builtin_ctz(w); }

__device__ __forceinline__ bool idle(const BatchState &Z, int stage)
{
    return !Z.active || (stage == 0 && !Z.need_stage0);
}

template <int KIND>
__device__ __forceinline__ void by_block(int stage, const BatchSim *__restrict__ sims,
                                         const BatchState *__restrict__ st,
                                         const int *__restrict__ map, int vb, float2 *sm)
{
    const int s = map[vb];
    const BatchSim &S = sims[s];
    if (idle(st[s], stage)) return;
    const DemagGeom &g = S.g;
    const int b = vb - S.first[BP_Y], W = S.tile[BP_Y], ntx = S.ntx[BP_Y];
    if (g.p0 == 1) {
        if (KIND != KIND_ANY || S.cy.ns) {
            CompLine c;
            c.kx0 = b * W;
            c.film = true;
            c.kfix = 0;
            c.n = g.n1;
            c.es = g.sx;
            c.cs = g.nrows * g.sx;
            c.base = S.xbuf + c.kx0;
            z_comp_tile<16>(g, S.cy, log2_tile(W), c, S.kern, sm);
        } else {
            y2d_tile(g, S.fy, W, b * W, S.kern, S.xbuf, sm);
        }
    } else {
        const int kt = b % ntx, line = b / ntx; // line = c n0 + i
        if (KIND != KIND_ANY || S.cy.ns)
            y_comp_tile<16, -1>(g, S.cy, log2_tile(W), kt * W, S.xbuf + (long)line * g.n1 * g.sx,
                                S.ybuf + (long)line * g.p1 * g.sx, sm);
        else
            yf_tile(g, S.fy, W, kt * W, line % g.n0, line / g.n0, S.xbuf, S.ybuf, sm);
    }
}

template <int KIND>
__device__ __forceinline__ void bz_block(int stage, const BatchSim *__restrict__ sims,
                                         const BatchState *__restrict__ st,
                                         const int *__restrict__ map, int vb, float2 *sm)
{
    const int s = map[vb];
    const BatchSim &S = sims[s];
    if (idle(st[s], stage)) return;
    const DemagGeom &g = S.g;
    const int b = vb - S.first[BP_Z], W = S.tile[BP_Z], ntx = S.ntx[BP_Z];
    if (KIND == KIND_ZCOL || S.zcol) {
        switch (g.n0) {
#define CASE(N) case N: z_column_tile<N>(g, S.kern, S.ybuf, b * kZCols, sm); break;
            CASE(2) CASE(3) CASE(4) CASE(5) CASE(6) CASE(7) CASE(8)
#undef CASE
        default: break;
        }
    } else if (KIND != KIND_ANY || S.cz.ns) {
        CompLine c;
        c.kx0 = (b % ntx) * W;
        c.film = false;
        c.kfix = b / ntx;
        c.n = g.n0;
        c.es = (long)g.p1 * g.sx;
        c.cs = g.n0 * c.es;
        c.base = S.ybuf + (long)c.kfix * g.sx + c.kx0;
        z_comp_tile<16>(g, S.cz, log2_tile(W), c, S.kern, sm);
    } else {
        z_tile(g, S.fz, W, (b % ntx) * W, b / ntx, S.kern, S.ybuf, sm);
    }
}

template <int KIND>
__device__ __forceinline__ void byi_block(int stage, const BatchSim *__restrict__ sims,
                                          const BatchState *__restrict__ st,
                                          const int *__restrict__ map, int vb, float2 *sm)
{
    const int s = map[vb];
    const BatchSim &S = sims[s];
    if (idle(st[s], stage)) return;
    const DemagGeom &g = S.g;
    const int b = vb - S.first[BP_YI], W = S.tile[BP_YI], ntx = S.ntx[BP_YI];
    const int kt = b % ntx, line = b / ntx;
    if (KIND != KIND_ANY || S.cy.ns)
        y_comp_tile<16, +1>(g, S.cy, log2_tile(W), kt * W, S.ybuf + (long)line * g.p1 * g.sx,
                            S.xbuf + (long)line * g.n1 * g.sx, sm);
    else
        yi_tile(g, S.fy, W, kt * W, line % g.n0, line / g.n0, S.ybuf, S.xbuf, sm);
}

// STAGE 0: tau0 = torque(m) (solve_rk12.go:97-115); STAGE 1: corrector,
// normalised m into the other buffer, max |tau1 - tau0| into err_bits.
template <int STAGE, int KIND>
__device__ __forceinline__ void bxi_block(const BatchSim *__restrict__ sims,
                                          BatchState *__restrict__ st,
                                          const int *__restrict__ map, int vb, float2 *sm)
{
    const int s = map[vb];
    const BatchSim &S = sims[s];
    BatchState &Z = st[s];
    if (!Z.active || (STAGE == 0 && !Z.need_stage0)) return;
    const long row0 = (long)(vb - S.first[BP_XI]) * S.tile[BP_XI];
    EpilogueIO io{};
    if (STAGE == 0) {
        io.m = S.mbuf[Z.cur];
        io.tout = S.tau0;
        if (KIND != KIND_ANY || S.cx.ns)
            xi_comp_tile<16, EPI_TAU0>(S.g, S.cx, S.tile[BP_XI], row0, S.xbuf, S.fp, io, sm);
        else
            xi_tile<EPI_TAU0>(S.g, S.fx, S.tile[BP_XI], row0, S.xbuf, S.fp, io, sm);
    } else {
        io.m = S.mpred;
        io.tau0 = S.tau0;
        io.mnew = S.mbuf[Z.cur ^ 1];
        io.h = Z.h;
        io.err = &Z.err_bits;
        io.err_mask = 0;
        if (KIND != KIND_ANY || S.cx.ns)
            xi_comp_tile<16, EPI_CORR>(S.g, S.cx, S.tile[BP_XI], row0, S.xbuf, S.fp, io, sm);
        else
            xi_tile<EPI_CORR>(S.g, S.fx, S.tile[BP_XI], row0, S.xbuf, S.fp, io, sm);
    }
}

// RK12Solver.Step's controller (solve_rk12.go:124-214) after one try, for one
// simulation; mirrors the host loop of mmx_sim_step.
__device__ __forceinline__ void control_one(BatchState &Z)
{
    if (!Z.active) return;
    const int maxTry = 10;
    const double headRoom = 0.8;
    const float maxdiff = __uint_as_float(Z.err_bits);
    Z.err_bits = 0u;
    Z.evals += Z.need_stage0 ? 2 : 1;
    if (!isfinite(maxdiff)) {
        Z.error = MMX_ERR_NAN;
        Z.active = 0;
        return;
    }
    const float stepDiff = maxdiff * Z.h;
    const double err = (double)stepDiff;
    const double dt = Z.dt;
    Z.t = Z.t0 + dt;
    Z.err = err;
    bool bad = false;
    if (err > Z.maxerr) {
        Z.badsteps++;
        bad = true;
    }
    if ((!bad || Z.tries == maxTry - 1) && err > Z.peakerr) Z.peakerr = err;
    double factor = bad ? pow(Z.maxerr / err, 1.0 / 3.0) : sqrt(Z.maxerr / err);
    factor *= headRoom;
    if (factor > 1.5) factor = 1.5;
    if (factor < 0.1) factor = 0.1;
    const double minFactor = factor < 2.0 ? factor : 2.0;
    double newDt = dt * minFactor;
    if (newDt < Z.mindt) newDt = Z.mindt;
    if (newDt > Z.maxdt) newDt = Z.maxdt;
    Z.dt = newDt;
    if (!bad || newDt == Z.mindt) {
        Z.cur ^= 1;
        Z.step++;
        Z.tries = 0;
        Z.need_stage0 = 1;
        Z.t0 = Z.t;
        if (Z.t >= Z.t_stop || Z.step >= Z.step_stop) Z.active = 0;
    } else {
        if (Z.tries > maxTry) {
            Z.error = MMX_ERR_CONVERGE;
            Z.active = 0;
            return;
        }
        Z.tries++;
        Z.need_stage0 = 0;
    }
    Z.h = (float)(Z.dt * Z.gamma);
}

// Arguments of the persistent launch (batch_persist.hip).
struct PersistArgs {
    const int *map[BP_N];
    int nblk[BP_N];
    int nsim;
    int tries;
    unsigned int *bar;   // [0]: arrivals, [1]: generation
    unsigned int *fail;  // nonzero: a barrier wait timed out
    int *nactive;        // active simulations after the last controller run
};

// The persistent kernel, for its attributes and launch.
const void *persist_kernel();

} // namespace mmx
