// pair_epilogue.hpp -- the field, torque and RK stage of two neighbouring cells
// with 8-byte accesses, for the C2R passes (register-FFT and composite-radix).
#pragma once

#include "epilogue.hpp"

namespace mmx {

// Two neighbouring cells (k0 even, k0 + 1 < n2) of one row at once, for
// uniform material parameters (MAPS false) or the Msat, Aex, alpha and Ku
// maps, the B_ext and anisU masks, the thermal field and H_dex (MAPS true),
// and no spin-transfer term: the same per-cell arithmetic as cell_epilogue
// (exchange6 order dim 0, dim 2, dim 1; SumUpdater order), with 8-byte loads
// and stores of the cell pair.

__device__ __forceinline__ int nb_lo(int pos, int len, int wrap)
{
    int lo = pos - 1;
    lo = (lo < 0 && wrap) ? len + lo : lo;
    return max(lo, 0);
}
__device__ __forceinline__ int nb_hi(int pos, int len, int wrap)
{
    int hi = pos + 1;
    hi = (hi == len && wrap) ? hi - len : hi;
    return min(hi, len - 1);
}

// Aex/Msat of the cell pair at byte offset b (div_zero(mask_unity(aex),
// mask_unity(msat)) of exchange6_cell), and of one cell
__device__ __forceinline__ float2 lex_pair(const FieldParams &fp, unsigned b)
{
    const float2 a = fp.aex_map ? ld_off<float2>(fp.aex_map, b) : float2{1.0f, 1.0f};
    const float2 s = fp.msat_map ? ld_off<float2>(fp.msat_map, b) : float2{1.0f, 1.0f};
    return float2{div_zero(a.x, s.x), div_zero(a.y, s.y)};
}
__device__ __forceinline__ float lex_one(const FieldParams &fp, unsigned b)
{
    const float a = fp.aex_map ? ld_off<float>(fp.aex_map, b) : 1.0f;
    const float s = fp.msat_map ? ld_off<float>(fp.msat_map, b) : 1.0f;
    return div_zero(a, s);
}

template <int MODE, bool MAPS = false>
__device__ __forceinline__ void pair_epilogue(const DemagGeom &g, const FieldParams &fp,
                                              const EpilogueIO &io, unsigned I0, int i, int j,
                                              int k0, const float hd0[3], const float hd1[3],
                                              float &errmax)
{
    const size_t N = g.N;
    const unsigned b0 = I0 * 4u; // byte offset of cell I0 in a component array
    if (MODE == EPI_B) {
#pragma unroll
        for (int c = 0; c < 3; c++) st_off<float2>(io.hout + c * N, b0, float2{hd0[c], hd1[c]});
        return;
    }
    const float *__restrict__ m = io.m;
    float m0[3], m1[3], H0[3], H1[3];
#pragma unroll
    for (int c = 0; c < 3; c++) {
        const float2 a = ld_off<float2>(m + c * N, b0);
        m0[c] = a.x;
        m1[c] = a.y;
    }
    // neighbour byte offsets: dim 0 (planes), dim 2 (along the row), dim 1
    // (rows); negative steps wrap in the unsigned sum and land on valid cells
    const int s0 = g.n1 * g.n2, s1 = g.n2;
    const unsigned o0l = b0 + 4u * (unsigned)((nb_lo(i, g.n0, fp.pbc[0]) - i) * s0);
    const unsigned o0h = b0 + 4u * (unsigned)((nb_hi(i, g.n0, fp.pbc[0]) - i) * s0);
    const unsigned o1l = b0 + 4u * (unsigned)((nb_lo(j, g.n1, fp.pbc[1]) - j) * s1);
    const unsigned o1h = b0 + 4u * (unsigned)((nb_hi(j, g.n1, fp.pbc[1]) - j) * s1);
    const unsigned o2l = b0 + 4u * (unsigned)(nb_lo(k0, g.n2, fp.pbc[2]) - k0); // left of cell 0
    const unsigned o2h = b0 + 4u * (unsigned)(nb_hi(k0 + 1, g.n2, fp.pbc[2]) - k0); // right of 1
    const float p0 = fp.ex_pre * fp.ex_c[0], p1 = fp.ex_pre * fp.ex_c[1],
                p2 = fp.ex_pre * fp.ex_c[2];
    if constexpr (MAPS) {
        // exchange weights: harmonic mean of the pair's and each neighbour's
        // Aex/Msat (w<dim><lo|hi><cell>)
        const float2 lc = lex_pair(fp, b0);
        const float2 lzl = lex_pair(fp, o0l), lzh = lex_pair(fp, o0h);
        const float2 lyl = lex_pair(fp, o1l), lyh = lex_pair(fp, o1h);
        const float lxl = lex_one(fp, o2l), lxh = lex_one(fp, o2h);
        const float w0l0 = avg_geom_zero(lc.x, lzl.x), w0h0 = avg_geom_zero(lc.x, lzh.x);
        const float w0l1 = avg_geom_zero(lc.y, lzl.y), w0h1 = avg_geom_zero(lc.y, lzh.y);
        const float w2l0 = avg_geom_zero(lc.x, lxl), w2h0 = avg_geom_zero(lc.x, lc.y);
        const float w2l1 = avg_geom_zero(lc.y, lc.x), w2h1 = avg_geom_zero(lc.y, lxh);
        const float w1l0 = avg_geom_zero(lc.x, lyl.x), w1h0 = avg_geom_zero(lc.x, lyh.x);
        const float w1l1 = avg_geom_zero(lc.y, lyl.y), w1h1 = avg_geom_zero(lc.y, lyh.y);
#pragma unroll
        for (int c = 0; c < 3; c++) {
            const float *mc = m + c * N;
            const float2 zl = ld_off<float2>(mc, o0l), zh = ld_off<float2>(mc, o0h);
            const float2 yl = ld_off<float2>(mc, o1l), yh = ld_off<float2>(mc, o1h);
            const float xl = ld_off<float>(mc, o2l), xh = ld_off<float>(mc, o2h);
            float e0 = p0 * (w0l0 * (zl.x - m0[c]) + w0h0 * (zh.x - m0[c]));
            float e1 = p0 * (w0l1 * (zl.y - m1[c]) + w0h1 * (zh.y - m1[c]));
            e0 += p2 * (w2l0 * (xl - m0[c]) + w2h0 * (m1[c] - m0[c]));
            e1 += p2 * (w2l1 * (m0[c] - m1[c]) + w2h1 * (xh - m1[c]));
            e0 += p1 * (w1l0 * (yl.x - m0[c]) + w1h0 * (yh.x - m0[c]));
            e1 += p1 * (w1l1 * (yl.y - m1[c]) + w1h1 * (yh.y - m1[c]));
            // B_ext mask: multiplier * map (the SumUpdater's vecMadd)
            float hx0 = fp.hext[c], hx1 = fp.hext[c];
            if (fp.bext_map) {
                const float2 bm = ld_off<float2>(fp.bext_map + c * N, b0);
                hx0 = fp.hext[c] * bm.x;
                hx1 = fp.hext[c] * bm.y;
            }
            H0[c] = hd0[c] + e0 + hx0;
            H1[c] = hd1[c] + e1 + hx1;
        }
    } else {
#pragma unroll
        for (int c = 0; c < 3; c++) {
            const float *mc = m + c * N;
            const float2 zl = ld_off<float2>(mc, o0l), zh = ld_off<float2>(mc, o0h);
            const float2 yl = ld_off<float2>(mc, o1l), yh = ld_off<float2>(mc, o1h);
            const float xl = ld_off<float>(mc, o2l), xh = ld_off<float>(mc, o2h);
            float e0 = p0 * ((zl.x - m0[c]) + (zh.x - m0[c]));
            float e1 = p0 * ((zl.y - m1[c]) + (zh.y - m1[c]));
            e0 += p2 * ((xl - m0[c]) + (m1[c] - m0[c]));
            e1 += p2 * ((m0[c] - m1[c]) + (xh - m1[c]));
            e0 += p1 * ((yl.x - m0[c]) + (yh.x - m0[c]));
            e1 += p1 * ((yl.y - m1[c]) + (yh.y - m1[c]));
            H0[c] = hd0[c] + e0 + fp.hext[c];
            H1[c] = hd1[c] + e1 + fp.hext[c];
        }
    }
    // Msat of the pair (a zero Msat reads as 1 in the anisotropy constant and
    // masks the renormalised cell)
    float2 ms = float2{1.0f, 1.0f};
    if constexpr (MAPS) {
        if (fp.msat_map) ms = ld_off<float2>(fp.msat_map, b0);
    }
    if (fp.anis) {
        float k = fp.ku2, k1 = fp.ku2;
        if constexpr (MAPS) {
            k = fp.ku2 / (ms.x == 0.0f ? 1.0f : ms.x);
            k1 = fp.ku2 / (ms.y == 0.0f ? 1.0f : ms.y);
            if (fp.ku_map) {
                const float2 q = ld_off<float2>(fp.ku_map, b0);
                k *= q.x;
                k1 *= q.y;
            }
        }
        // the anisU mask gives each cell's axis as multiplier * map
        float u0[3] = {fp.u[0], fp.u[1], fp.u[2]}, u1[3] = {fp.u[0], fp.u[1], fp.u[2]};
        if constexpr (MAPS) {
            if (fp.u_map) {
#pragma unroll
                for (int c = 0; c < 3; c++) {
                    const float2 um = ld_off<float2>(fp.u_map + c * N, b0);
                    u0[c] = fp.u[c] * um.x;
                    u1[c] = fp.u[c] * um.y;
                }
            }
        }
        const float mu0 = m0[0] * u0[0] + m0[1] * u0[1] + m0[2] * u0[2];
        const float mu1 = m1[0] * u1[0] + m1[1] * u1[1] + m1[2] * u1[2];
#pragma unroll
        for (int c = 0; c < 3; c++) {
            H0[c] += k * mu0 * u0[c];
            H1[c] += k1 * mu1 * u1[c];
        }
    }
    // H_therm, the SumUpdater's last term, then H_dex from its own
    // convolution (demagexch with an Msat mask)
    if constexpr (MAPS) {
        if (fp.htherm) {
#pragma unroll
            for (int c = 0; c < 3; c++) {
                const float2 t = ld_off<float2>(fp.htherm + c * N, b0);
                H0[c] += t.x;
                H1[c] += t.y;
            }
        }
        if (fp.hdex) {
#pragma unroll
            for (int c = 0; c < 3; c++) {
                const float2 t = ld_off<float2>(fp.hdex + c * N, b0);
                H0[c] += t.x;
                H1[c] += t.y;
            }
        }
    }
    if (io.hout) {
#pragma unroll
        for (int c = 0; c < 3; c++) st_off<float2>(io.hout + c * N, b0, float2{H0[c], H1[c]});
    }
    if (MODE == EPI_HEFF && io.tout == nullptr) return;
    float t0[3], t1[3];
    float2 alpha = float2{fp.alpha, fp.alpha};
    if constexpr (MAPS) {
        if (fp.alpha_map) {
            const float2 a = ld_off<float2>(fp.alpha_map, b0);
            alpha = float2{fp.alpha * a.x, fp.alpha * a.y};
        }
    }
    llg_torque(m0, H0, alpha.x, t0);
    llg_torque(m1, H1, alpha.y, t1);
    if (io.tout) {
#pragma unroll
        for (int c = 0; c < 3; c++) st_off<float2>(io.tout + c * N, b0, float2{t0[c], t1[c]});
    }
    if (MODE == EPI_CORR) {
        const float hh = 0.5f * io.h, mh = -0.5f * io.h;
        float a0[3], a1[3], d0[3], d1[3];
#pragma unroll
        for (int c = 0; c < 3; c++) {
            const float2 p = ld_off<float2>(io.tau0 + c * N, b0);
            a0[c] = m0[c] + (hh * t0[c] + mh * p.x);
            a1[c] = m1[c] + (hh * t1[c] + mh * p.y);
            d0[c] = t0[c] - p.x;
            d1[c] = t1[c] - p.y;
        }
        errmax = err_fold(err_fold(errmax, d0[0], d0[1], d0[2]), d1[0], d1[1], d1[2]);
        const float l0 = sqrtf(a0[0] * a0[0] + a0[1] * a0[1] + a0[2] * a0[2]);
        const float l1 = sqrtf(a1[0] * a1[0] + a1[1] * a1[1] + a1[2] * a1[2]);
        const float s0 = (ms.x == 0.0f) ? 0.0f : 1.0f, s1 = (ms.y == 0.0f) ? 0.0f : 1.0f;
        const float q0 = (l0 != 0.0f) ? s0 / l0 : 0.0f;
        const float q1 = (l1 != 0.0f) ? s1 / l1 : 0.0f;
#pragma unroll
        for (int c = 0; c < 3; c++)
            st_off<float2>(io.mnew + c * N, b0, float2{a0[c] * q0, a1[c] * q1});
    }
}

} // namespace mmx
