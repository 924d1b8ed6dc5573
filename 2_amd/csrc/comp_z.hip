// comp_z.hip -- the z pass, and a film's y pass, on composite-radix transforms
// (comp_tiles.hpp), one simulation.
#include "comp_launch.hpp"

namespace mmx {

// Threads: up to what the class's registers allow (128 per thread for radices up
// to 16, 256 up to 32)
constexpr int z_threads_max(int rm) { return rm <= 16 ? 1024 : 512; }

// 3-D z (film 0): tiles ordered so that ky and p1 - ky, which read the same
// octant rows, run back to back; film y (film 1)
template <int RM>
__global__ void __launch_bounds__(z_threads_max(RM)) z_comp(DemagGeom g, CompFFT f, int lw, int ntx, int film, const float *__restrict__ K,
                       float2 *__restrict__ buf)
{
    extern __shared__ float2 sm[];
    const int tile = xcd_tile(blockIdx.x, gridDim.x);
    const int tx = tile % ntx, o = tile / ntx;
    CompLine c;
    c.kx0 = tx << lw;
    c.film = film != 0;
    if (film) {
        c.kfix = 0;
        c.n = g.n1;
        c.es = g.sx;
        c.cs = g.nrows * g.sx;
        c.base = buf + c.kx0;
    } else {
        c.kfix = mirror_order(o, g.p1);
        c.n = g.n0;
        c.es = (long)g.p1 * g.sx;
        c.cs = g.n0 * c.es;
        c.base = buf + (long)c.kfix * g.sx + c.kx0;
    }
    z_comp_tile<RM>(g, f, lw, c, K, sm);
}

template <int N0>
MMX_COMP_KERNEL z_col(DemagGeom g, const float *__restrict__ K, float2 *__restrict__ yb)
{
    extern __shared__ float2 sm[];
    z_column_tile<N0>(g, K, yb, xcd_tile(blockIdx.x, gridDim.x) * kZCols, sm);
}

static bool zcol_applies(const DemagGeom &g) { return 2 * g.n0 == g.p0 && g.n0 >= 2 && g.n0 <= 16; }
bool comp_z_applies(const DemagPlanImpl *P)
{
    const DemagGeom &g = P->g;
    if (g.p0 == 1) return false;
    if (zcol_applies(g) && (double)g.p1 * g.h2 + kZCols < 2147483647.0) return true;
    const long es = (long)g.p1 * g.sx;
    return P->cz.ns > 0 && comp_z_lds(P->cz, 0) <= kLdsMax &&
           comp_line_fits(g.n0 * es, es, P->cz.L / P->cz.R[0]);
}
bool comp_y2d_applies(const DemagPlanImpl *P)
{
    const DemagGeom &g = P->g;
    return g.p0 == 1 && P->cy.ns > 0 && comp_z_lds(P->cy, 0) <= kLdsMax &&
           comp_line_fits(g.nrows * g.sx, g.sx, P->cy.L / P->cy.R[0]);
}

// Threads of a workgroup: the CU's waves (four per SIMD in class 16, three in
// class 32) shared by the workgroups that it holds at once, at most one DFT per
// thread and stage.  Long lines leave room for one workgroup, which then needs
// the waves (film of 1024 rows, 114 KB: 256 threads 95 us, 768 threads 76); with many
// small ones more threads each would leave fewer of them (z of 240x200x36, 36 KB:
// 576 threads 109 us, 256 threads 72).
static int z_threads(const CompFFT &f, int lw, size_t lds, long blocks, int rm)
{
    const long waves = rm <= 16 ? 16 : 12;
    const long held = std::max(1L, std::min((long)(kLdsMax / lds), (blocks + 255) / 256));
    const long nt = std::min(64L * std::max(4L, waves / held), 64L * div_up(comp_tasks(f, 3 << lw), 64));
    return (int)std::min((long)z_threads_max(rm), std::max(64L, nt));
}

template <int RM> static int z_go(const DemagPlanImpl *P, const CompFFT &f, int film, hipStream_t st)
{
    const DemagGeom &g = P->g;
    const int nline = film ? 1 : g.p1;
    const int lw = comp_cols(f, 3, [&](int w) { return comp_z_lds(f, w); }, nline, g.h2);
    const int ntx = div_up(g.h2, 1 << lw);
    const size_t b = comp_z_lds(f, lw);
    comp_lds(z_comp<RM>, b);
    z_comp<RM><<<dim3(ntx * nline), dim3(z_threads(f, lw, b, (long)ntx * nline, RM)), b, st>>>(
        g, f, lw, ntx, film, P->kern, film ? P->xbuf : P->ybuf);
    MMX_CHECK_LAUNCH();
    return MMX_OK;
}

int comp_z(const DemagPlanImpl *P, hipStream_t st)
{
    const DemagGeom &g = P->g;
    if (zcol_applies(g)) {
        const dim3 nb((unsigned)div_up((long)g.p1 * g.h2, kZCols));
        switch (g.n0) {
#define CASE(N) case N: z_col<N><<<nb, dim3(kBlock), zcol_lds(N), st>>>(g, P->kern, P->ybuf); break;
            CASE(2) CASE(3) CASE(4) CASE(5) CASE(6) CASE(7) CASE(8) CASE(9) CASE(10) CASE(11) CASE(12)
            CASE(13) CASE(14) CASE(15) CASE(16)
#undef CASE
        default: break;
        }
        MMX_CHECK_LAUNCH();
        return MMX_OK;
    }
    return comp_top(P->cz) <= 16 ? z_go<16>(P, P->cz, 0, st) : z_go<32>(P, P->cz, 0, st);
}

int comp_y2d(const DemagPlanImpl *P, hipStream_t st)
{
    return comp_top(P->cy) <= 16 ? z_go<16>(P, P->cy, 1, st) : z_go<32>(P, P->cy, 1, st);
}

} // namespace mmx
