// comp_x.hip -- the x passes on composite-radix transforms (comp_tiles.hpp), one simulation, and the
// choice of radices.
#include <cstdint>
#include <initializer_list>

#include "comp_launch.hpp"

namespace mmx {

// ------------------------------------------------------------ the radices

static bool comp_radix(int r)
{
#define CASE(V) if (r == V) return true;
    MMX_COMP_RADICES_16(CASE)
    MMX_COMP_RADICES_32(CASE)
#undef CASE
    return false;
}

CompFFT comp_plan(int L, const LineFFT<float> &f, int top2)
{
    CompFFT c;
    c.L = L;
    c.tw = f.tw;
    c.rtw = f.rtw;
    int top = top2 + 1;
    // two stages, the larger radix first
    for (int r1 = 1; r1 <= top2; r1++) {
        const int r0 = L / r1;
        if (L % r1 || r0 < r1 || !comp_radix(r0) || !comp_radix(r1) || r0 >= top) continue;
        top = r0;
        c.ns = 2;
        c.R[0] = r0;
        c.R[1] = r1;
        c.R[2] = 1;
    }
    if (c.ns == 0) {
        top = 33;
        for (int r2 = 2; r2 <= 32; r2++)
            for (int r1 = r2; r1 <= 32 && L % r2 == 0; r1++) {
                const int r0 = L / r2 / r1;
                if (L % (r2 * r1) || r0 < r1 || r0 >= top || !comp_radix(r0) || !comp_radix(r1) ||
                    !comp_radix(r2))
                    continue;
                top = r0;
                c.ns = 3;
                c.R[0] = r0;
                c.R[1] = r1;
                c.R[2] = r2;
            }
    }
    c.Rl = c.ns == 3 ? c.R[2] : c.R[1];
    c.P = c.Rl | 1;
    c.Ml = L / c.Rl;
    for (int s = 0; s < 3; s++) c.byM[s].set(L / c.R[s]);
    c.byL.set(L);
    c.byRl.set(c.Rl);
    c.byR0.set(c.R[0]);
    c.byR1.set(c.R[1]);
    c.byMl.set(c.Ml);
    return c;
}

template <int RM, int PRED>
MMX_COMP_KERNEL xf_comp(DemagGeom g, CompFFT f, int RB, const float *__restrict__ m,
                        const float *__restrict__ msat_map, const float *__restrict__ tau0, float h,
                        const float *__restrict__ norm_map, float *__restrict__ mpred,
                        float2 *__restrict__ xb, unsigned int *ho_dev, unsigned int *ho_host, int pairs)
{
    extern __shared__ float2 sm[];
    // a hand-off takes a workgroup of its own, the last one
    const int nb = gridDim.x - (ho_dev != nullptr);
    if ((int)blockIdx.x == nb) return hand_off(ho_dev, ho_host);
    xf_comp_tile<RM, PRED>(g, f, RB, (long)xcd_tile(blockIdx.x, nb) * RB, m, msat_map, tau0, h, norm_map,
                           mpred, xb, sm, pairs != 0);
}

template <int RM, int MODE, int PAIR>
MMX_COMP_KERNEL xi_comp(DemagGeom g, CompFFT f, int RB, const float2 *__restrict__ xb, FieldParams fp,
                        EpilogueIO io)
{
    extern __shared__ float2 sm[];
    xi_comp_tile<RM, MODE, PAIR>(g, f, RB, (long)xcd_tile(blockIdx.x, gridDim.x) * RB, xb, fp, io, sm);
}

// Rows per workgroup: as few as leave all workgroups resident at once (a row's
// chain of loads, stages and epilogue is what a small grid waits for), up to
// 16 within 48 KB of LDS.
static int comp_rows(const DemagPlanImpl *P)
{
    int rb = 1;
    while (rb < 16 && div_up(P->g.nrows, rb) > kCompSlots && comp_x_lds(P->cx, rb + 1) <= 48 * 1024) rb++;
    return rb;
}

bool comp_x_applies(const DemagPlanImpl *P)
{
    return P->cx.ns > 0 && comp_x_lds(P->cx, 1) <= kLdsMax && comp_x_fits(P->g);
}

// 8-byte accesses of cell pairs (a component starts at an even cell when n2 is
// even; the caller's arrays may start anywhere)
static bool aligned8(std::initializer_list<const void *> ps)
{
    for (const void *p : ps)
        if (reinterpret_cast<uintptr_t>(p) % 8) return false;
    return true;
}

template <int RM, int PRED>
static int xf_go(const DemagPlanImpl *P, const float *m, const float *msat_map, const float *tau0, float h,
                 const float *norm_map, float *mpred, hipStream_t st)
{
    const int rb = comp_rows(P);
    const size_t b = comp_x_lds(P->cx, rb);
    comp_lds(xf_comp<RM, PRED>, b);
    unsigned int *ho = PRED ? nullptr : P->handoff_dev;
    const bool pairs = P->g.n2 % 2 == 0 && aligned8({m, msat_map, tau0, norm_map, mpred});
    xf_comp<RM, PRED><<<dim3(div_up(P->g.nrows, rb) + (ho ? 1 : 0)), dim3(kBlock), b, st>>>(
        P->g, P->cx, rb, m, msat_map, tau0, h, norm_map, mpred, P->xbuf, ho, P->handoff_host, pairs);
    MMX_CHECK_LAUNCH();
    return MMX_OK;
}

int comp_xf(const DemagPlanImpl *P, int pred, const float *m, const float *msat_map, const float *tau0,
            float h, const float *norm_map, float *mpred, hipStream_t st)
{
    const bool s = comp_top(P->cx) <= 16;
    if (pred)
        return s ? xf_go<16, 1>(P, m, msat_map, tau0, h, norm_map, mpred, st)
                 : xf_go<32, 1>(P, m, msat_map, tau0, h, norm_map, mpred, st);
    return s ? xf_go<16, 0>(P, m, msat_map, nullptr, 0.0f, nullptr, nullptr, st)
             : xf_go<32, 0>(P, m, msat_map, nullptr, 0.0f, nullptr, nullptr, st);
}

template <int RM, int MODE, int PAIR>
static int xi_go(const DemagPlanImpl *P, const FieldParams &fp, const EpilogueIO &io, hipStream_t st)
{
    const int rb = comp_rows(P);
    const size_t b = comp_x_lds(P->cx, rb);
    comp_lds(xi_comp<RM, MODE, PAIR>, b);
    xi_comp<RM, MODE, PAIR><<<dim3(div_up(P->g.nrows, rb)), dim3(kBlock), b, st>>>(P->g, P->cx, rb, P->xbuf,
                                                                                   fp, io);
    MMX_CHECK_LAUNCH();
    return MMX_OK;
}

template <int RM, int MODE>
static int xi_pair(const DemagPlanImpl *P, int pair, const FieldParams &fp, const EpilogueIO &io,
                   hipStream_t st)
{
    if constexpr (MODE == EPI_B)
        return pair ? xi_go<RM, MODE, 1>(P, fp, io, st) : xi_go<RM, MODE, 0>(P, fp, io, st);
    else
        return pair == 1   ? xi_go<RM, MODE, 1>(P, fp, io, st)
               : pair == 2 ? xi_go<RM, MODE, 2>(P, fp, io, st)
                           : xi_go<RM, MODE, 0>(P, fp, io, st);
}

template <int RM>
static int xi_mode(const DemagPlanImpl *P, int mode, const FieldParams &fp, const EpilogueIO &io,
                   hipStream_t st)
{
    // two cells at a time where the grid fills the chip: more rows than
    // workgroups wanted (below, half as many threads would each take longer)
    const bool even = P->g.n2 % 2 == 0 && P->g.nrows > kCompSlots &&
                      aligned8({io.m, io.hout, io.tout, io.tau0, io.mnew});
    const int pair = !even                                        ? 0
                     : (mode == EPI_B || fast_xi_applies(fp))     ? 1
                     : fast_xi_maps_applies(fp)                   ? 2
                                                                  : 0;
    switch (mode) {
    case EPI_B: return xi_pair<RM, EPI_B>(P, pair, fp, io, st);
    case EPI_HEFF: return xi_pair<RM, EPI_HEFF>(P, pair, fp, io, st);
    case EPI_TAU0: return xi_pair<RM, EPI_TAU0>(P, pair, fp, io, st);
    case EPI_CORR: return xi_pair<RM, EPI_CORR>(P, pair, fp, io, st);
    default: set_error("demag_inverse: bad mode %d", mode); return MMX_ERR_ARG;
    }
}

int comp_xi(const DemagPlanImpl *P, int mode, const FieldParams &fp, const EpilogueIO &io, hipStream_t st)
{
    return comp_top(P->cx) <= 16 ? xi_mode<16>(P, mode, fp, io, st) : xi_mode<32>(P, mode, fp, io, st);
}

} // namespace mmx
