// comp_fft.hpp -- line transforms of any length whose prime factors are at
// most 13, in two or three stages of composite radices held in registers.
//
// A length L = R0 R1 (or R0 R1 R2) is transformed in few, large stages: an
// R-point DFT (R up to 32) is evaluated in one thread's registers
// (cdft: radix 4, 2, then the odd primes, constants folded at compile time), so
// a line crosses the LDS once per stage instead of once per prime-power
// factor.  The radices are arguments of the kernel, chosen per length on the
// host (comp_plan), and a switch outside the task loop picks the DFT: one
// kernel serves every length.  Kernels come in two register classes RM (every
// radix at most 16, or at most 32).
//
// What bounds these passes at the sizes they run at (grids whose lengths have
// no register-FFT kernel, and the x passes of small grids) is latency: the
// earlier form, one stage per factor from {8, 4, 2, 3, 5, 7} with integer
// divisions per butterfly and twiddles read from global memory, spent
// 36 us in the z pass of 200x200x5 and 18 us in each y pass against 7 and 9
// here (kernel times), and 272 and 84 us in those of 240x200x36 against 72 and
// 41.
#pragma once

#include "demag_plan.hpp"
#include "reg_fft.hpp"

namespace mmx {

// ------------------------------------------------------- DFT in registers

// R-point DFT, R odd: the cosine sums of v[n] + v[R-n] and the sine sums of
// v[n] - v[R-n] give X[k] and X[R-k] together.
template <int R, int DIR> __device__ __forceinline__ void odd_dft(float2 *v)
{
    constexpr int H = (R - 1) / 2;
    float2 s[H], d[H];
    float2 sum = v[0];
    static_for<H>([&](auto I) {
        constexpr int n = decltype(I)::value;
        s[n] = float2{v[n + 1].x + v[R - 1 - n].x, v[n + 1].y + v[R - 1 - n].y};
        d[n] = float2{v[n + 1].x - v[R - 1 - n].x, v[n + 1].y - v[R - 1 - n].y};
        sum.x += s[n].x;
        sum.y += s[n].y;
    });
    const float2 v0 = v[0];
    v[0] = sum;
    static_for<H>([&](auto K) {
        constexpr int k = decltype(K)::value + 1;
        float2 a = v0, b = float2{0.0f, 0.0f};
        static_for<H>([&](auto I) {
            constexpr int n = decltype(I)::value;
            constexpr float c = (float)cx_cs((long)(n + 1) * k, R, false);
            constexpr float q = (float)((double)DIR * cx_cs((long)(n + 1) * k, R, true));
            a.x += s[n].x * c;
            a.y += s[n].y * c;
            b.x += d[n].x * q;
            b.y += d[n].y * q;
        });
        // X[k] = a + i b, X[R-k] = a - i b
        v[k] = float2{a.x - b.y, a.y + b.x};
        v[R - k] = float2{a.x + b.y, a.y - b.x};
    });
}

template <int R, int DIR> __device__ __forceinline__ void prime_dft(float2 *v)
{
    if constexpr (R == 2 || R == 4)
        SmallDFT<float2, R, DIR>::run(v);
    else
        odd_dft<R, DIR>(v);
}

constexpr int cdft_radix(int rem)
{
    return rem % 4 == 0 ? 4 : rem % 2 == 0 ? 2 : rem % 3 == 0 ? 3 : rem % 5 == 0 ? 5
         : rem % 7 == 0 ? 7 : rem % 11 == 0 ? 11 : 13;
}

template <int N, int DIR, int Ns>
__device__ __forceinline__ void cdft_stages(float2 *a, float2 *b, bool &in_b)
{
    if constexpr (Ns < N) {
        constexpr int R = cdft_radix(N / Ns);
        static_assert((N / Ns) % R == 0, "prime factors up to 13");
        static_for<N / R>([&](auto I) {
            constexpr int J = decltype(I)::value, k = J % Ns, base = (J / Ns) * Ns * R + k;
            float2 v[R];
            static_for<R>([&](auto Q) {
                constexpr int q = decltype(Q)::value;
                v[q] = twmul<Ns * R, k * q, DIR>(a[J + q * (N / R)]);
            });
            prime_dft<R, DIR>(v);
            static_for<R>([&](auto Q) {
                constexpr int q = decltype(Q)::value;
                b[base + q * Ns] = v[q];
            });
        });
        in_b = !in_b;
        cdft_stages<N, DIR, Ns * R>(b, a, in_b);
    }
}

// In-register DFT of N points, natural order in and out (exp(DIR 2 pi i nk/N)).
template <int N, int DIR> __device__ __forceinline__ void cdft(float2 (&v)[N])
{
    if constexpr (N > 1) {
        float2 tmp[N];
        bool in_b = false;
        cdft_stages<N, DIR, 1>(v, tmp, in_b);
        if (in_b) {
#pragma unroll
            for (int i = 0; i < N; i++) v[i] = tmp[i];
        }
    }
}

// -------------------------------------------------------------- the radices

#define MMX_COMP_RADICES_16(X)                                                               \
    X(1) X(2) X(3) X(4) X(5) X(6) X(7) X(8) X(9) X(10) X(11) X(12) X(13) X(14) X(15) X(16)
#define MMX_COMP_RADICES_32(X)                                                               \
    X(18) X(20) X(21) X(22) X(24) X(25) X(26) X(27) X(28) X(30) X(32)

// calls f(std::integral_constant<int, R>) for the run-time radix r of class RM
#define MMX_COMP_CASE(V) case V: f(std::integral_constant<int, V>{}); break;
template <int RM, typename F> __device__ __forceinline__ void with_radix(int r, F &&f)
{
    if constexpr (RM <= 16) {
        switch (r) {
            MMX_COMP_RADICES_16(MMX_COMP_CASE)
        default: break;
        }
    } else {
        switch (r) {
            MMX_COMP_RADICES_16(MMX_COMP_CASE)
            MMX_COMP_RADICES_32(MMX_COMP_CASE)
        default: break;
        }
    }
}

// ------------------------------------------------------- stages over LDS
//
// In place: n = (a R1 + b) R2 + c and k = k0 + R0 k1 + R0 R1 k2 (two stages:
// n = a R1 + c, k = k0 + R0 k2) give
//   W_L^(nk) = W_R0^(a k0) . W_L^(R2 b k0) W_R1^(b k1) . W_L^(c (k0 + R0 k1)) W_R2^(c k2),
// so stage s is a DFT over one digit, whose slots it reads and writes, and the
// transform ends in the order of the slots (k0, k1, k2).  One buffer, one
// barrier between stages; the inverse of a product runs the stages backwards.
// The last digit has the odd pitch P, which spreads the lanes of every stage
// over the banks.
//
// A tile holds several lines.  Columns (the strided y and z passes, W = 2^lw
// neighbouring spectrum columns) keep the lanes along the columns, rows (the x
// passes) along the slots.

struct ColLines {
    int lw;
    __device__ __forceinline__ int at(int l, int pos) const { return (pos << lw) + l; }
    __device__ __forceinline__ int count(int m) const { return m << lw; }
    __device__ __forceinline__ void split(int task, const FastDiv &, int &l, int &j) const
    {
        l = task & ((1 << lw) - 1);
        j = task >> lw;
    }
};

struct RowLines {
    int nl, ls;
    __device__ __forceinline__ int at(int l, int pos) const { return l * ls + pos; }
    __device__ __forceinline__ int count(int m) const { return nl * m; }
    __device__ __forceinline__ void split(int task, const FastDiv &d, int &l, int &j) const
    {
        l = d.quot(task);
        j = task - l * (int)d.d;
    }
};

// slots of one line
__host__ __device__ inline int comp_slots(const CompFFT &f) { return f.Ml * f.P; }

// slot of input n, and of output k
__device__ __forceinline__ int slot_in(const CompFFT &f, int n)
{
    return n + f.byRl.quot(n) * (f.P - f.Rl);
}
__device__ __forceinline__ int slot_out(const CompFFT &f, int k)
{
    const int kl = f.byMl.quot(k), q = k - kl * f.Ml; // q = k0 + R0 k1
    if (f.ns == 2) return q * f.P + kl;
    const int k1 = f.byR0.quot(q), k0 = q - k1 * f.R[0];
    return (k0 * f.R[1] + k1) * f.P + kl;
}
// k0 + R0 k1 of the j-th slot group (k0 R1 + k1) of the last stage
__device__ __forceinline__ int group_out(const CompFFT &f, int j)
{
    if (f.ns == 2) return j;
    const int k0 = f.byR1.quot(j), k1 = j - k0 * f.R[1];
    return k0 + f.R[0] * k1;
}

// Stage 0: ld(l, j, o) -> slots; the input is element j + o of the line, o the
// same for all lanes.
template <int RM, int DIR, typename Lines, typename LD>
__device__ __forceinline__ void stage_first(const CompFFT &f, const Lines &ln, float2 *A, LD &&ld)
{
    const int M = (int)f.byM[0].d, S = f.byRl.quot(M) * f.P;
    with_radix<RM>(f.R[0], [&](auto RR) {
        constexpr int R = decltype(RR)::value;
        for (int task = threadIdx.x; task < ln.count(M); task += (int)blockDim.x) {
            int l, j;
            ln.split(task, f.byM[0], l, j);
            float2 v[R];
#pragma unroll
            for (int r = 0; r < R; r++) v[r] = ld(l, j, r * M);
            cdft<R, DIR>(v);
            const int p = slot_in(f, j);
#pragma unroll
            for (int r = 0; r < R; r++) A[ln.at(l, p + r * S)] = v[r];
        }
    });
}

// The same, in place, for a line that lies in its slots.
template <int RM, int DIR, typename Lines>
__device__ __forceinline__ void stage_first_lds(const CompFFT &f, const Lines &ln, float2 *A)
{
    const int M = (int)f.byM[0].d, S = f.byRl.quot(M) * f.P;
    with_radix<RM>(f.R[0], [&](auto RR) {
        constexpr int R = decltype(RR)::value;
        for (int task = threadIdx.x; task < ln.count(M); task += (int)blockDim.x) {
            int l, j;
            ln.split(task, f.byM[0], l, j);
            const int p = slot_in(f, j);
            float2 v[R];
#pragma unroll
            for (int r = 0; r < R; r++) v[r] = A[ln.at(l, p + r * S)];
            cdft<R, DIR>(v);
#pragma unroll
            for (int r = 0; r < R; r++) A[ln.at(l, p + r * S)] = v[r];
        }
    });
}

// The inverse of stage 0: slots -> st(l, j, o, value), element j + o.
template <int RM, typename Lines, typename ST>
__device__ __forceinline__ void stage_first_back(const CompFFT &f, const Lines &ln, const float2 *A,
                                                 ST &&st)
{
    const int M = (int)f.byM[0].d, S = f.byRl.quot(M) * f.P;
    with_radix<RM>(f.R[0], [&](auto RR) {
        constexpr int R = decltype(RR)::value;
        for (int task = threadIdx.x; task < ln.count(M); task += (int)blockDim.x) {
            int l, j;
            ln.split(task, f.byM[0], l, j);
            const int p = slot_in(f, j);
            float2 v[R];
#pragma unroll
            for (int r = 0; r < R; r++) v[r] = A[ln.at(l, p + r * S)];
            cdft<R, +1>(v);
#pragma unroll
            for (int r = 0; r < R; r++) st(l, j, r * M, v[r]);
        }
    });
}

// Middle stage of three, in place.  BACK: the inverse stage (twiddles after
// the DFT).
template <int RM, int DIR, bool BACK, typename Lines>
__device__ __forceinline__ void stage_mid(const CompFFT &f, const Lines &ln, float2 *A,
                                          const float2 *stw)
{
    const int M = (int)f.byM[1].d, R1P = f.R[1] * f.P;
    with_radix<RM>(f.R[1], [&](auto RR) {
        constexpr int R = decltype(RR)::value;
        for (int task = threadIdx.x; task < ln.count(M); task += (int)blockDim.x) {
            int l, j;
            ln.split(task, f.byM[1], l, j);
            const int k0 = f.byRl.quot(j), c = j - k0 * f.Rl, p = k0 * R1P + c, q = k0 * f.R[2];
            float2 v[R];
#pragma unroll
            for (int r = 0; r < R; r++) v[r] = A[ln.at(l, p + r * f.P)];
            if (!BACK) {
#pragma unroll
                for (int r = 1; r < R; r++)
                    v[r] = (DIR < 0) ? cmul(v[r], stw[r * q]) : cmulc(v[r], stw[r * q]);
            }
            cdft<R, DIR>(v);
            if (BACK) {
#pragma unroll
                for (int r = 1; r < R; r++)
                    v[r] = (DIR < 0) ? cmul(v[r], stw[r * q]) : cmulc(v[r], stw[r * q]);
            }
#pragma unroll
            for (int r = 0; r < R; r++) A[ln.at(l, p + r * f.P)] = v[r];
        }
    });
}

// Last stage: slots -> st(l, q, o, slot, value), output k = q + o; a task reads
// and writes the same slots, so st may store to A itself.
template <int RM, int DIR, typename Lines, typename ST>
__device__ __forceinline__ void stage_last(const CompFFT &f, const Lines &ln, const float2 *A,
                                           const float2 *stw, ST &&st)
{
    const FastDiv &d = f.ns == 3 ? f.byM[2] : f.byM[1];
    with_radix<RM>(f.Rl, [&](auto RR) {
        constexpr int R = decltype(RR)::value;
        for (int task = threadIdx.x; task < ln.count(f.Ml); task += (int)blockDim.x) {
            int l, j;
            ln.split(task, d, l, j);
            const int q = group_out(f, j);
            float2 v[R];
#pragma unroll
            for (int r = 0; r < R; r++) v[r] = A[ln.at(l, j * f.P + r)];
#pragma unroll
            for (int r = 1; r < R; r++)
                v[r] = (DIR < 0) ? cmul(v[r], stw[r * q]) : cmulc(v[r], stw[r * q]);
            cdft<R, DIR>(v);
#pragma unroll
            for (int r = 0; r < R; r++) st(l, q, r * f.Ml, j * f.P + r, v[r]);
        }
    });
}

// ... and its inverse, in place.
template <int RM, typename Lines>
__device__ __forceinline__ void stage_last_back(const CompFFT &f, const Lines &ln, float2 *A,
                                                const float2 *stw)
{
    const FastDiv &d = f.ns == 3 ? f.byM[2] : f.byM[1];
    with_radix<RM>(f.Rl, [&](auto RR) {
        constexpr int R = decltype(RR)::value;
        for (int task = threadIdx.x; task < ln.count(f.Ml); task += (int)blockDim.x) {
            int l, j;
            ln.split(task, d, l, j);
            const int q = group_out(f, j);
            float2 v[R];
#pragma unroll
            for (int r = 0; r < R; r++) v[r] = A[ln.at(l, j * f.P + r)];
            cdft<R, +1>(v);
#pragma unroll
            for (int r = 0; r < R; r++)
                A[ln.at(l, j * f.P + r)] = r ? cmulc(v[r], stw[r * q]) : v[r];
        }
    });
}

} // namespace mmx
