// comp_y.hip -- the 3-D y passes on composite-radix transforms (comp_tiles.hpp), one simulation.
#include "comp_launch.hpp"

namespace mmx {

// tiles: column tile fastest, then plane, then component
template <int RM, int DIR>
MMX_COMP_KERNEL y_comp(DemagGeom g, CompFFT f, int lw, int ntx, const float2 *__restrict__ src,
                       float2 *__restrict__ dst)
{
    extern __shared__ float2 sm[];
    const int tile = xcd_tile(blockIdx.x, gridDim.x);
    const int tx = tile % ntx, line = tile / ntx; // line = c n0 + i
    const size_t x = (size_t)line * g.n1 * g.sx, y = (size_t)line * g.p1 * g.sx;
    y_comp_tile<RM, DIR>(g, f, lw, tx << lw, src + (DIR < 0 ? x : y), dst + (DIR < 0 ? y : x), sm);
}

bool comp_y_applies(const DemagPlanImpl *P)
{
    return P->cy.ns > 0 && comp_y_lds(P->cy, 0) <= kLdsMax;
}
template <int RM, int DIR> static int y_go(const DemagPlanImpl *P, hipStream_t st)
{
    const DemagGeom &g = P->g;
    const int lw = comp_cols(P->cy, 1, [&](int w) { return comp_y_lds(P->cy, w); }, 3L * g.n0, g.h2);
    const int ntx = div_up(g.h2, 1 << lw);
    const size_t b = comp_y_lds(P->cy, lw);
    comp_lds(y_comp<RM, DIR>, b);
    y_comp<RM, DIR><<<dim3(ntx * g.n0 * 3), dim3(kBlock), b, st>>>(
        g, P->cy, lw, ntx, DIR < 0 ? P->xbuf : P->ybuf, DIR < 0 ? P->ybuf : P->xbuf);
    MMX_CHECK_LAUNCH();
    return MMX_OK;
}

int comp_yf(const DemagPlanImpl *P, hipStream_t st)
{
    return comp_top(P->cy) <= 16 ? y_go<16, -1>(P, st) : y_go<32, -1>(P, st);
}
int comp_yi(const DemagPlanImpl *P, hipStream_t st)
{
    return comp_top(P->cy) <= 16 ? y_go<16, +1>(P, st) : y_go<32, +1>(P, st);
}

} // namespace mmx
