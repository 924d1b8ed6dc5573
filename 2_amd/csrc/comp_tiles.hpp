// comp_tiles.hpp -- one workgroup's share of each demag pass on the composite
// radix transforms (comp_fft.hpp), given its tile coordinates and its LDS.
// Called by the single-simulation kernels (comp_x.hip, comp_y.hip, comp_z.hip) and by the
// batched kernels (batch.hip).  Same passes, buffers and epilogue as the
// generic tiles (demag_tiles.hpp).
#pragma once

#include "comp_fft.hpp"
#include "pair_epilogue.hpp"

namespace mmx {

// Twiddles of the pass's length into LDS (a barrier follows before their use).
__device__ __forceinline__ void load_tw(const CompFFT &f, float2 *stw)
{
    for (int t = threadIdx.x; t < f.L; t += (int)blockDim.x) stw[t] = f.tw[t];
}

// ------------------------------------------------------------------ x passes

// The x passes address cells and spectrum rows with 32-bit byte offsets.
__host__ __device__ inline bool comp_x_fits(const DemagGeom &g)
{
    return g.N < kMaxCells32 && ((double)g.nrows + 16) * g.sx * sizeof(float2) < 4294967295.0 &&
           (g.n2 == g.Lx || g.n2 == 2 * g.Lx);
}

// LDS (bytes): 3 RB lines, twiddles
__host__ __device__ inline size_t comp_x_lds(const CompFFT &f, int RB)
{
    return (3ull * RB * comp_slots(f) + f.L) * sizeof(float2);
}

// transform of the 3 RB lines in A, in place; ends with a barrier
template <int RM, int DIR>
__device__ __forceinline__ void row_lines_fft(const CompFFT &f, const RowLines &ln, float2 *A,
                                              const float2 *stw)
{
    stage_first_lds<RM, DIR>(f, ln, A);
    __syncthreads();
    if (f.ns == 3) {
        stage_mid<RM, DIR, false>(f, ln, A, stw);
        __syncthreads();
    }
    stage_last<RM, DIR>(f, ln, A, stw, [&](int l, int, int, int p, float2 v) { A[ln.at(l, p)] = v; });
    __syncthreads();
}

template <int RM, int PRED>
__device__ __forceinline__ void
xf_comp_tile(const DemagGeom &g, const CompFFT &f, int RB, long row0, const float *__restrict__ m,
             const float *__restrict__ msat_map, const float *__restrict__ tau0, float h,
             const float *__restrict__ norm_map, float *__restrict__ mpred,
             float2 *__restrict__ xb, float2 *sm, bool pairs = false)
{
    const int L = f.L;
    const RowLines ln{3 * RB, comp_slots(f)};
    float2 *A = sm, *stw = sm + ln.nl * ln.ls;
    const long N = g.N;
    load_tw(f, stw);
    for (int t = threadIdx.x; t < RB * L; t += kBlock) {
        const int r = f.byL.quot(t), e = t - r * L;
        const long row = row0 + r;
        float v[2][3] = {{0.0f, 0.0f, 0.0f}, {0.0f, 0.0f, 0.0f}};
        if (row < g.nrows && 2 * e < g.n2) {
            const unsigned I = 4u * (unsigned)((int)row * g.n2 + 2 * e); // byte offset
            const bool two = 2 * e + 1 < g.n2;
            // the cell pair of a component array; one cell at the end of an odd
            // row, and two loads where the array is not 8-byte aligned
            auto ld2 = [&](const float *p) {
                return pairs ? ld_off<float2>(p, I)
                             : float2{ld_off<float>(p, I), two ? ld_off<float>(p, I + 4u) : 0.0f};
            };
            float2 x[3] = {ld2(m), ld2(m + N), ld2(m + 2 * N)};
            if (PRED) {
                // predictor m = y0 + dt*gamma*tau0 (maddKern), then the
                // normUpdater (normalize.cu:14-43)
                const float2 t0[3] = {ld2(tau0), ld2(tau0 + N), ld2(tau0 + 2 * N)};
                const float2 nm = norm_map ? ld2(norm_map) : float2{1.0f, 1.0f};
#pragma unroll
                for (int c = 0; c < 3; c++) x[c] = float2{x[c].x + h * t0[c].x, x[c].y + h * t0[c].y};
                auto unit = [](float a, float b, float c, float norm) {
                    const float len = sqrtf(a * a + b * b + c * c);
                    const float scale = (norm == 0.0f) ? 0.0f : 1.0f;
                    return (len != 0.0f) ? scale / len : 0.0f;
                };
                const float s0 = unit(x[0].x, x[1].x, x[2].x, nm.x);
                const float s1 = unit(x[0].y, x[1].y, x[2].y, nm.y);
#pragma unroll
                for (int c = 0; c < 3; c++) {
                    x[c] = float2{x[c].x * s0, x[c].y * s1};
                    if (pairs) {
                        st_off<float2>(mpred + c * N, I, x[c]);
                    } else {
                        st_off<float>(mpred + c * N, I, x[c].x);
                        if (two) st_off<float>(mpred + c * N, I + 4u, x[c].y);
                    }
                }
            }
            const float2 ms = msat_map ? ld2(msat_map) : float2{1.0f, 1.0f};
#pragma unroll
            for (int c = 0; c < 3; c++) {
                v[0][c] = msat_map ? x[c].x * ms.x : x[c].x;
                v[1][c] = two ? (msat_map ? x[c].y * ms.y : x[c].y) : 0.0f;
            }
        }
#pragma unroll
        for (int c = 0; c < 3; c++) A[ln.at(c * RB + r, slot_in(f, e))] = float2{v[0][c], v[1][c]};
    }
    __syncthreads();
    row_lines_fft<RM, -1>(f, ln, A, stw);

    // split the half-length spectrum into the R2C output X[0..L]
    for (int t = threadIdx.x; t < RB * L; t += kBlock) {
        const int r = f.byL.quot(t), k = t - r * L;
        const long row = row0 + r;
        if (row >= g.nrows) continue;
        const float2 w = f.rtw[k];
        const int pa = slot_out(f, k), pb = slot_out(f, k == 0 ? 0 : L - k);
        const unsigned o = 8u * ((unsigned)row * (unsigned)g.sx + (unsigned)k);
#pragma unroll
        for (int c = 0; c < 3; c++) {
            const float2 a = A[ln.at(c * RB + r, pa)];
            const float2 b = cconj(A[ln.at(c * RB + r, pb)]);
            const float2 E = float2{0.5f * (a.x + b.x), 0.5f * (a.y + b.y)};
            const float2 O = float2{0.5f * (a.y - b.y), -0.5f * (a.x - b.x)};
            float2 *dst = xb + (long)c * g.nrows * g.sx;
            st_off<float2>(dst, o, cadd(E, cmul(O, w)));
            // the last bin, E(0) - O(0)
            if (k == 0) st_off<float2>(dst, o + 8u * (unsigned)L, float2{a.x - a.y, 0.0f});
        }
    }
}

// PAIR 0: one cell at a time, every term; 1, 2: two cells at a time with 8-byte
// accesses, uniform parameters or maps, no spin-transfer term, n2 even
// (pair_epilogue) -- for grids with enough rows that the epilogue's
// instructions, not its latency, take the time
template <int RM, int MODE, int PAIR = 0>
__device__ __forceinline__ void
xi_comp_tile(const DemagGeom &g, const CompFFT &f, int RB, long row0,
             const float2 *__restrict__ xb, const FieldParams &fp, const EpilogueIO &io, float2 *sm)
{
    const int L = f.L;
    const RowLines ln{3 * RB, comp_slots(f)};
    float2 *A = sm, *stw = sm + ln.nl * ln.ls;
    load_tw(f, stw);
    // n2 is L (zero-padded) or 2 L (periodic)
    const bool full = g.n2 != L;
    auto place = [&](int t, int &r, int &k, int &i, int &j) {
        r = full ? f.byL.quot(t >> 1) : f.byL.quot(t);
        k = t - r * g.n2;
        const int row = (int)row0 + r;
        i = row / g.n1;
        j = row - i * g.n1;
        return row < g.nrows;
    };
    // the terms of this thread's first cell that need no demag field, loaded
    // together with the spectrum (their latency would follow the transform's)
    CellLocal loc;
    int r, k, i, j;
    const bool have = PAIR == 0 && (int)threadIdx.x < RB * g.n2 && place(threadIdx.x, r, k, i, j);
    if (have)
        cell_local<MODE, unsigned>(g, fp, io, (unsigned)(((int)row0 + r) * g.n2 + k), i, j, k, loc);
    // C2R pre-processing (imaginary parts of DC and Nyquist ignored)
    for (int t = threadIdx.x; t < RB * L; t += kBlock) {
        const int r = f.byL.quot(t), k = t - r * L;
        const long row = row0 + r;
        const float2 w = f.rtw[k];
        const int p = slot_in(f, k);
        const unsigned o = 8u * (unsigned)row * (unsigned)g.sx;
#pragma unroll
        for (int c = 0; c < 3; c++) {
            float2 z = float2{0.0f, 0.0f};
            if (row < g.nrows) {
                const float2 *src = xb + (long)c * g.nrows * g.sx;
                float2 a = ld_off<float2>(src, o + 8u * (unsigned)k),
                       bb = ld_off<float2>(src, o + 8u * (unsigned)(L - k));
                if (k == 0) {
                    a.y = 0.0f;
                    bb.y = 0.0f;
                }
                const float2 b = cconj(bb);
                const float2 E = cadd(a, b);
                const float2 O = cmulc(csub(a, b), w);
                z = float2{E.x - O.y, E.y + O.x};
            }
            A[ln.at(c * RB + r, p)] = z;
        }
    }
    __syncthreads();
    row_lines_fft<RM, +1>(f, ln, A, stw);

    float errmax = 0.0f;
    if constexpr (PAIR > 0) {
        for (int t = threadIdx.x; t < RB * g.n2 / 2; t += kBlock) {
            if (!place(2 * t, r, k, i, j)) continue;
            float hd0[3], hd1[3];
            const int p = slot_out(f, k >> 1);
#pragma unroll
            for (int c = 0; c < 3; c++) {
                const float2 z = A[ln.at(c * RB + r, p)];
                hd0[c] = fp.demag_scale * z.x;
                hd1[c] = fp.demag_scale * z.y;
            }
            pair_epilogue<MODE, PAIR == 2>(g, fp, io, (unsigned)(((int)row0 + r) * g.n2 + k), i, j, k, hd0,
                                           hd1, errmax);
        }
        if (MODE == EPI_CORR) block_max_slot(errmax, io.err, io.err_mask);
        return;
    }
    for (int t = threadIdx.x; t < RB * g.n2; t += kBlock) {
        const bool ok = place(t, r, k, i, j);
        if (!ok) continue;
        const long I = (row0 + r) * g.n2 + k;
        if (t >= kBlock) cell_local<MODE, unsigned>(g, fp, io, (unsigned)I, i, j, k, loc);
        float hd[3];
        const int p = slot_out(f, k >> 1);
#pragma unroll
        for (int c = 0; c < 3; c++) {
            const float2 z = A[ln.at(c * RB + r, p)];
            hd[c] = fp.demag_scale * ((k & 1) ? z.y : z.x);
        }
        cell_finish<MODE>(g, fp, io, I, loc, hd, errmax);
    }
    if (MODE == EPI_CORR) block_max_slot(errmax, io.err, io.err_mask);
}

// ------------------------------------------------------------------ y passes

// LDS (bytes) of a y tile: W lines, twiddles
__host__ __device__ inline size_t comp_y_lds(const CompFFT &f, int lw)
{
    return (((size_t)comp_slots(f) << lw) + f.L) * sizeof(float2);
}

// forward (DIR -1): rows j < n1 of src in, p1 rows of dst out; inverse: p1
// rows in, j < n1 out.  Columns past h2 read column h2 - 1 and store nothing.
template <int RM, int DIR>
__device__ __forceinline__ void
y_comp_tile(const DemagGeom &g, const CompFFT &f, int lw, int kx0, const float2 *__restrict__ src,
            float2 *__restrict__ dst, float2 *sm)
{
    const int L = f.L, nin = DIR < 0 ? g.n1 : L, nout = DIR < 0 ? L : g.n1;
    const ColLines ln{lw};
    float2 *A = sm, *stw = A + (comp_slots(f) << lw);
    load_tw(f, stw);
    const int last = g.h2 - 1 - kx0;
    stage_first<RM, DIR>(f, ln, A, [&](int w, int j, int o) {
        const unsigned at = 8u * (unsigned)(j * g.sx + kx0 + min(w, last));
        return j + o < nin ? ld_off<float2>(src + (long)o * g.sx, at) : float2{0.0f, 0.0f};
    });
    __syncthreads();
    if (f.ns == 3) {
        stage_mid<RM, DIR, false>(f, ln, A, stw);
        __syncthreads();
    }
    stage_last<RM, DIR>(f, ln, A, stw, [&](int w, int q, int o, int, float2 v) {
        if (w <= last && q + o < nout)
            st_off<float2>(dst + (long)o * g.sx, 8u * (unsigned)(q * g.sx + kx0 + w), v);
    });
}

// ------------------------------------- z pass, and the y pass of a film
//
// Forward transform, 3x3 kernel multiply and inverse transform of W columns of
// all three components, the components in the LDS next to each other.  The
// multiply walks the slots.  (A thread that held the last stage's points of all
// three components and multiplied them in registers saved two barriers, but at
// 256 registers, two waves per SIMD, z of 240x200x36 took 112 us against 66.)

// The three components of a line's first R1 (R2) elements lie within 4 GiB of
// each other: 32-bit byte offsets from a scalar base.
__host__ __device__ inline bool comp_line_fits(long cs, long es, int m0)
{
    return (2.0 * cs + (double)m0 * es + 4096.0) * sizeof(float2) < 4294967295.0;
}

struct CompLine {            // the transformed axis in memory
    float2 *base;            // element 0, component 0, column kx0
    long cs, es;             // component and element strides
    int n, kx0, kfix;        // elements that hold data; the other kernel index
    bool film;               // y of a film: kernel at (0, e), else at (e, kfix)
};

__host__ __device__ inline size_t comp_z_lds(const CompFFT &f, int lw)
{
    return (3 * ((size_t)comp_slots(f) << lw) + f.L) * sizeof(float2);
}

// three components of W columns as lines: line l = c W + w
struct Col3Lines {
    int lw, span;            // span: LDS elements of one component
    __device__ __forceinline__ int at(int l, int pos) const
    {
        return (l >> lw) * span + (pos << lw) + (l & ((1 << lw) - 1));
    }
    __device__ __forceinline__ int count(int m) const { return 3 * (m << lw); }
    // tasks run over columns, then slots, then components
    __device__ __forceinline__ void split(int task, const FastDiv &d, int &l, int &j) const
    {
        const int n = (int)d.d << lw;
        const int c = (task >= n) + (task >= 2 * n), t = task - c * n;
        l = (c << lw) + (t & ((1 << lw) - 1));
        j = t >> lw;
    }
};

template <int RM>
__device__ __forceinline__ void z_comp_tile(const DemagGeom &g, const CompFFT &f, int lw,
                                            const CompLine &c, const float *__restrict__ K, float2 *sm)
{
    const int W = 1 << lw;
    const Col3Lines ln{lw, comp_slots(f) << lw};
    float2 *A = sm, *stw = sm + 3 * ln.span;
    load_tw(f, stw);
    const int last = g.h2 - 1 - c.kx0, NT = blockDim.x;
    // byte offset of element j of line l = (component, column) from c.base
    const unsigned cs8 = 8u * (unsigned)c.cs, es8 = 8u * (unsigned)c.es;
    auto lane_off = [&](int l, int j, int w) {
        return (unsigned)(l >> lw) * cs8 + (unsigned)j * es8 + 8u * (unsigned)w;
    };
    // slot t of the W columns: its LDS element and kernel values
    auto place = [&](int t, int &o) {
        const int w = t & (W - 1), e = t >> lw;
        const int j = f.byRl.quot(e), r = e - j * f.Rl;
        const int k = group_out(f, j) + r * f.Ml, kx = c.kx0 + min(w, last);
        o = ((j * f.P + r) << lw) + w;
        return c.film ? kern_at(g, K, 0, k, kx) : kern_at(g, K, k, c.kfix, kx);
    };
    stage_first<RM, -1>(f, ln, A, [&](int l, int j, int o) {
        const unsigned at = lane_off(l, j, min(l & (W - 1), last));
        return j + o < c.n ? ld_off<float2>(c.base + o * c.es, at) : float2{0.0f, 0.0f};
    });
    // the kernel values of a thread's first slots, their loads under the
    // remaining forward stages (four slots each cost registers: z of 240x200x36
    // 80 us against 72)
    constexpr int NPF = 2;
    Kern6 kp[NPF];
    int op[NPF];
#pragma unroll
    for (int u = 0; u < NPF; u++) kp[u] = place(min((int)threadIdx.x + u * NT, (f.L << lw) - 1), op[u]);
    __syncthreads();
    if (f.ns == 3) {
        stage_mid<RM, -1, false>(f, ln, A, stw);
        __syncthreads();
    }
    stage_last<RM, -1>(f, ln, A, stw, [&](int l, int, int, int p, float2 v) { A[ln.at(l, p)] = v; });
    __syncthreads();
#pragma unroll
    for (int u = 0; u < NPF; u++)
        if ((int)threadIdx.x + u * NT < (f.L << lw))
            kern_apply(kp[u], A[op[u]], A[ln.span + op[u]], A[2 * ln.span + op[u]]);
    for (int t = threadIdx.x + NPF * NT; t < (f.L << lw); t += NT) {
        int o;
        const Kern6 kk = place(t, o);
        kern_apply(kk, A[o], A[ln.span + o], A[2 * ln.span + o]);
    }
    __syncthreads();
    stage_last_back<RM>(f, ln, A, stw);
    __syncthreads();
    if (f.ns == 3) {
        stage_mid<RM, +1, true>(f, ln, A, stw);
        __syncthreads();
    }
    stage_first_back<RM>(f, ln, A, [&](int l, int j, int o, float2 v) {
        const int w = l & (W - 1);
        if (w <= last && j + o < c.n) st_off<float2>(c.base + o * c.es, lane_off(l, j, w), v);
    });
}

// Short zero-padded z (2 <= n0 <= 16, p0 = 2 n0): 64 spectrum columns per
// workgroup, one per lane, the three components on a wave each.  With the upper
// half of the line zero, the even and the odd outputs are the n0-point
// transforms of a[i] and of a[i] W_p^i, in registers; the components meet in the
// LDS for the kernel multiply, which all four waves share (kz and p0 - kz
// together, their octant points loaded at the start), and
// out[i] = even[i] + W_p^-i odd[i] on the way back.  One thread for a column's
// three components (no LDS) took 12.1 us at 100x100x10, its serial chain of
// some 3000 instructions.
constexpr int kZCols = 64;

__host__ __device__ inline size_t zcol_lds(int n0) { return 3ull * 2 * n0 * kZCols * sizeof(float2); }

template <int N0>
__device__ __forceinline__ void z_column_tile(const DemagGeom &g, const float *__restrict__ K,
                                              float2 *__restrict__ yb, int col0, float2 *sm)
{
    constexpr int P0 = 2 * N0, NI = (N0 + 4) / 4; // octant rows kz = wave + 4 t <= N0
    static_assert(kBlock == 4 * kZCols, "three transforming waves and a fourth");
    const int lane = threadIdx.x & 63;
    const int q = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int ncol = g.p1 * g.h2;
    const int col = min(col0 + lane, ncol - 1); // past the end: loads only
    const int o = col / g.h2, kx = col - o * g.h2, ky = mirror_order(o, g.p1);
    const long istride = (long)g.p1 * g.sx;
    float2 *base = yb + (long)q * N0 * istride + (long)ky * g.sx + kx;
    const bool my = ky > g.p1 / 2;
    const int kyp = my ? g.p1 - ky : ky;
    const float sy = my ? -1.0f : 1.0f;
    // line element (half, e) of component c at sm[((c * 2 + half) * N0 + e) * 64 + lane]
    auto at = [&](int c, int half, int e) -> float2 & { return sm[((c * 2 + half) * N0 + e) * kZCols + lane]; };
    Kern6 kp[NI];
    float2 a[N0], x[N0];
    if (q < 3) {
#pragma unroll
        for (int i = 0; i < N0; i++) a[i] = base[i * istride];
    }
#pragma unroll
    for (int t = 0; t < NI; t++) kp[t] = kern_octant(g, K, min(q + 4 * t, N0), kyp, kx, 1.0f, sy);
    if (q < 3) {
        static_for<N0>([&](auto I) {
            constexpr int i = decltype(I)::value;
            x[i] = twmul<P0, i, -1>(a[i]);
        });
        cdft<N0, -1>(a);
        cdft<N0, -1>(x);
#pragma unroll
        for (int e = 0; e < N0; e++) {
            at(q, 0, e) = a[e];
            at(q, 1, e) = x[e];
        }
    }
    __syncthreads();
#pragma unroll
    for (int t = 0; t < NI; t++) {
        const int kz = q + 4 * t;
        if (kz > N0) break;
        const int h = kz & 1, e = kz >> 1;
        kern_apply(kp[t], at(0, h, e), at(1, h, e), at(2, h, e));
        if (kz > 0 && kz < N0) {
            Kern6 km = kp[t];
            km.xz = -km.xz;
            km.xy = -km.xy;
            const int em = (P0 - kz) >> 1; // P0 - kz has kz's parity
            kern_apply(km, at(0, h, em), at(1, h, em), at(2, h, em));
        }
    }
    __syncthreads();
    if (q < 3) {
#pragma unroll
        for (int e = 0; e < N0; e++) {
            a[e] = at(q, 0, e);
            x[e] = at(q, 1, e);
        }
        cdft<N0, +1>(a);
        cdft<N0, +1>(x);
        if (col0 + lane < ncol) {
            static_for<N0>([&](auto I) {
                constexpr int i = decltype(I)::value;
                const float2 w = twmul<P0, i, +1>(x[i]);
                base[i * istride] = float2{a[i].x + w.x, a[i].y + w.y};
            });
        }
    }
}

} // namespace mmx
