// kernel_build.hip -- one-time demag kernel construction in FP64 on the GPU.
//
// Compiled with -ffp-contract=off: the Kernel_Arne integration below performs
// the same IEEE double operations in the same order as the reference's Go code
// (modules/kernel_magnetostatic.go:30-181), so the float32 kernel it stores is
// the reference's kernel bit for bit (checked against the FP64 CPU oracle).
// The kernel is then transformed with an FP64 FFT (the reference uses a float32
// cuFFT here, maxwell_convolution.go:386-396), the real part of the octant
// kz <= p0/2, ky <= p1/2, kx <= p2/2 is kept and scaled by 1/(p0 p1 p2).
#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>

#include "demag_plan.hpp"

namespace mmx {

// tensor component of (source s, destination d) in the stored order
// XX,YY,ZZ,YZ,XZ,XY; -1 for the lower triangle (common/index.go:44-47)
__device__ __constant__ int kStoredIdx[3][3] = {{0, 5, 4}, {-1, 1, 3}, {-1, -1, 2}};

struct ArneArgs {
    int p[3];
    double cell[3];
    int x1, x2, y1, y2, z1, z2;
    double L;
    double accuracy;
    int reach[3];   // displacements within it are in arne_near's table
};

__device__ inline double delta_cells(int d)
{
    if (d < 0) d = -d;
    if (d > 0) d -= 1;
    return (double)d;
}

// First displacement in [lo, hi] whose wrapped index is w (w in [0, p)), or
// hi + 1 when there is none; the others follow at +p.  kernel.go:19-28 wraps
// x into [0, p) by adding or subtracting p.
__device__ inline int first_image(int w, int p, int lo)
{
    int x = w;
    while (x - p >= lo) x -= p;
    return x;
}

// The quadrature of one displacement of a unit S-dipole: the point counts,
// first point and spacing per axis, and the charge of one point
// (kernel_magnetostatic.go:94-146).  The source axis is a template argument so
// that every index is a constant (registers, not scratch).
template <int S> struct ArneQuad {
    static constexpr int U = S, V = (S + 1) % 3, W = (S + 2) % 3;
    int nv, nw, n[3];
    double v0, dv, w0, dw;   // face points: v0 + i dv, w0 + j dw
    double r0[3], dr[3];     // destination points: r0 + dr k
    double charge, pu1, pu2;
};

template <int S>
__device__ inline ArneQuad<S> arne_quad(const ArneArgs &a, int x, int y, int z)
{
    using Q = ArneQuad<S>;
    const double *cell = a.cell;
    Q q;
    const double R[3] = {(double)x * cell[0], (double)y * cell[1], (double)z * cell[2]};
    const double dx = delta_cells(x) * cell[0];
    const double dy = delta_cells(y) * cell[1];
    const double dz = delta_cells(z) * cell[2];
    double d = sqrt(dx * dx + dy * dy + dz * dz);
    if (d == 0) d = a.L;
    const double maxSize = d / a.accuracy;
#pragma unroll
    for (int c = 0; c < 3; c++) q.n[c] = (int)(fmax(cell[c] / maxSize, 1.) + 0.5);
    q.nv = 2 * q.n[Q::V];
    q.nw = 2 * q.n[Q::W];
    const double scale = 1 / (double)(q.nv * q.nw * q.n[0] * q.n[1] * q.n[2]);
    const double surface = cell[Q::V] * cell[Q::W];
    q.charge = surface * scale;
    q.pu1 = cell[Q::U] / 2.;
    q.pu2 = -q.pu1;
    q.v0 = -(cell[Q::V] / 2.) + cell[Q::V] / (double)(2 * q.nv);
    q.dv = cell[Q::V] / (double)q.nv;
    q.w0 = -(cell[Q::W] / 2.) + cell[Q::W] / (double)(2 * q.nw);
    q.dw = cell[Q::W] / (double)q.nw;
#pragma unroll
    for (int c = 0; c < 3; c++) {
        q.r0[c] = R[c] - cell[c] / 2. + cell[c] / (double)(2 * q.n[c]);
        q.dr[c] = cell[c] / (double)q.n[c];
    }
    return q;
}

// Field of the two charged face points (i, j) at the point (k0, k1, k2) of the
// destination cell: the term that kernel_magnetostatic.go:128-165 adds to B,
// same operations in the same order.
template <int S>
__device__ inline void arne_term(const ArneQuad<S> &q, int i, int j, int k0, int k1, int k2,
                                 double t[3])
{
    using Q = ArneQuad<S>;
    double R2[3], pole[3], b[3];
    pole[Q::V] = q.v0 + (double)i * q.dv;
    pole[Q::W] = q.w0 + (double)j * q.dw;
    const double rc[3] = {q.r0[0] + q.dr[0] * (double)k0, q.r0[1] + q.dr[1] * (double)k1,
                          q.r0[2] + q.dr[2] * (double)k2};
    pole[Q::U] = q.pu1;
#pragma unroll
    for (int c = 0; c < 3; c++) R2[c] = rc[c] - pole[c];
    double r = sqrt(R2[0] * R2[0] + R2[1] * R2[1] + R2[2] * R2[2]);
    double qr = q.charge / (4. * kPi * r * r * r);
#pragma unroll
    for (int c = 0; c < 3; c++) b[c] = R2[c] * qr;
    pole[Q::U] = q.pu2;
    R2[Q::U] = rc[Q::U] - pole[Q::U];
    r = sqrt(R2[0] * R2[0] + R2[1] * R2[1] + R2[2] * R2[2]);
    qr = -q.charge / (4. * kPi * r * r * r);
#pragma unroll
    for (int c = 0; c < 3; c++) t[c] = b[c] + R2[c] * qr;
}

// B (FP64) at displacement (x, y, z) of a unit S-dipole: the surface-charge /
// volume integration of kernel_magnetostatic.go:94-165, its terms added in the
// reference's loop order.
template <int S>
__device__ inline void arne_point(const ArneArgs &a, int x, int y, int z, double Bf[3])
{
    const ArneQuad<S> q = arne_quad<S>(a, x, y, z);
    Bf[0] = Bf[1] = Bf[2] = 0.0;
    for (int i = 0; i < q.nv; i++)
        for (int j = 0; j < q.nw; j++)
            for (int al = 0; al < q.n[0]; al++)
                for (int be = 0; be < q.n[1]; be++)
                    for (int ga = 0; ga < q.n[2]; ga++) {
                        double t[3];
                        arne_term<S>(q, i, j, al, be, ga, t);
                        for (int c = 0; c < 3; c++) Bf[c] += t[c];
                    }
}

// The displacements |x_a| <= reach[a], whose quadratures have more than the
// four points of the far field (up to (2 accuracy)^2 accuracy^3 and more where
// the cells are not cubes), are integrated beforehand, one workgroup each:
// wave 0 adds the terms one after another in the loop order of arne_point (so
// the sum has the same bits) while the other eight waves work out the next 512.
// A single thread's serial chain of square roots and divisions took 15 ms per
// source axis for cubic cells (31104 points per displacement at accuracy 6), 27
// for 4x4x3 nm (98304) and 640 for 8x8x3 nm; here the chain is the additions,
// 6 ns each: all three axes of 4x4x3 nm in 0.60 ms (1.39 ms when the adding
// wave waited for the LDS at every second term).
constexpr int kNearWaves = 8;
constexpr int kNearChunk = 64 * kNearWaves;

template <int S>
__device__ __forceinline__ void arne_near_one(const ArneArgs &a, float *__restrict__ tab,
                                              double (&buf)[2][3][kNearChunk])
{
    const int e1 = 2 * a.reach[1] + 1, e2 = 2 * a.reach[2] + 1;
    const int x = (int)blockIdx.x / (e1 * e2) - a.reach[0];
    const int y = (int)blockIdx.x / e2 % e1 - a.reach[1];
    const int z = (int)blockIdx.x % e2 - a.reach[2];
    const ArneQuad<S> q = arne_quad<S>(a, x, y, z);
    // the point's indices as digits (i, j, al, be, ga), advanced by one chunk
    // at a time with carries (no division per point)
    const int base[4] = {q.n[2], q.n[1], q.n[0], q.nw};
    const long npts = (long)q.nv * q.nw * q.n[0] * q.n[1] * q.n[2];
    const long nchunk = (npts + kNearChunk - 1) / kNearChunk;
    const int lane = threadIdx.x;
    int dig[5], step[5];
    for (int part = 0; part < 2; part++) {
        int r = part ? kNearChunk : lane - 64;
        int *d = part ? step : dig;
        for (int c = 0; c < 4; c++) {
            d[c] = r % base[c];
            r /= base[c];
        }
        d[4] = r;
    }
    double B = 0.0;
    for (long k = 0; k <= nchunk; k++) {
        if (lane >= 64 && k < nchunk) {
            const int e = lane - 64;
            if (k * kNearChunk + e < npts) {
                double t[3];
                arne_term<S>(q, dig[4], dig[3], dig[2], dig[1], dig[0], t);
                for (int c = 0; c < 3; c++) buf[k & 1][c][e] = t[c];
            }
            int carry = 0;
            for (int c = 0; c < 4; c++) {
                dig[c] += step[c] + carry;
                carry = dig[c] >= base[c] ? 1 : 0;
                dig[c] -= carry ? base[c] : 0;
            }
            dig[4] += step[4] + carry;
        }
        if (lane < 3 && k > 0) {
            const double *t = buf[(k - 1) & 1][lane];
            const long left = npts - (k - 1) * kNearChunk;
            if (left >= kNearChunk) {
                // 16 terms ahead in registers: the additions wait for each
                // other, not for the LDS
                double now[16], next[16];
#pragma unroll
                for (int e = 0; e < 16; e++) now[e] = t[e];
                for (int at = 16; at <= kNearChunk; at += 16) {
                    const double *tn = t + (at < kNearChunk ? at : 0);
#pragma unroll
                    for (int e = 0; e < 16; e++) next[e] = tn[e];
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int e = 0; e < 16; e++) B += now[e];
#pragma unroll
                    for (int e = 0; e < 16; e++) now[e] = next[e];
                }
            } else {
                for (int e = 0; e < (int)left; e++) B += t[e];
            }
        }
        __syncthreads();
    }
    if (lane < 3) tab[3 * ((size_t)S * gridDim.x + blockIdx.x) + lane] = (float)B;
}

__global__ void __launch_bounds__(64 + kNearChunk) __attribute__((amdgpu_waves_per_eu(3, 3)))
arne_near(ArneArgs a, float *__restrict__ tab)
{
    __shared__ double buf[2][3][kNearChunk];
    switch (blockIdx.y) {
    case 0: arne_near_one<0>(a, tab, buf); break;
    case 1: arne_near_one<1>(a, tab, buf); break;
    default: arne_near_one<2>(a, tab, buf); break;
    }
}

// One thread per padded-grid element (xw, yw, zw) and source axis: the element
// is the float32 sum, starting from 0, of float32(B) over every displacement (x, y, z) in the
// loop ranges that wraps onto it, added in the reference's loop order (x, then
// y, then z ascending; kernel_magnetostatic.go:91-101,168-172).  Without
// periodic images an element has at most one displacement; with them the
// element is the same float32 sum the reference forms, with no atomics, so the
// kernel is deterministic and bit-identical to it.  Every element is written.
// Near displacements come from arne_near's table.
__global__ void __launch_bounds__(kBlock) arne_kernel(ArneArgs a, const float *__restrict__ tab,
                                                      float *__restrict__ K6)
{
    const int X = 0, Y = 1, Z = 2;
    const int s = blockIdx.y;
    const long P = (long)a.p[X] * a.p[Y] * a.p[Z];
    const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= P) return;
    const int zw = (int)(t % a.p[Z]);
    const int yw = (int)((t / a.p[Z]) % a.p[Y]);
    const int xw = (int)(t / ((long)a.p[Z] * a.p[Y]));
    const int xs = first_image(xw, a.p[X], a.x1);
    const int ys = first_image(yw, a.p[Y], a.y1);
    const int zs = first_image(zw, a.p[Z], a.z1);
    const int *r = a.reach;
    const int e0 = 2 * r[0] + 1, e1 = 2 * r[1] + 1, e2 = 2 * r[2] + 1;
    float acc[3] = {0.0f, 0.0f, 0.0f};
    for (int x = xs; x <= a.x2; x += a.p[X])
        for (int y = ys; y <= a.y2; y += a.p[Y])
            for (int z = zs; z <= a.z2; z += a.p[Z]) {
                if (abs(x) <= r[0] && abs(y) <= r[1] && abs(z) <= r[2]) {
                    const size_t d = ((size_t)(x + r[0]) * e1 + (y + r[1])) * e2 + (z + r[2]);
                    const float *b = tab + 3 * ((size_t)s * e0 * e1 * e2 + d);
                    for (int dd = 0; dd < 3; dd++) acc[dd] += b[dd];
                    continue;
                }
                double Bf[3];
                switch (s) {
                case 0: arne_point<0>(a, x, y, z, Bf); break;
                case 1: arne_point<1>(a, x, y, z, Bf); break;
                default: arne_point<2>(a, x, y, z, Bf); break;
                }
                for (int dd = 0; dd < 3; dd++) acc[dd] += (float)Bf[dd];
            }
    for (int dd = 0; dd < 3; dd++) {
        const int idx = kStoredIdx[s][dd];
        if (idx >= 0) K6[idx * P + t] = acc[dd];
    }
}

// Reach of the near table per axis: an axis is cut into more than one piece
// while cell / (d / accuracy) >= 1.5 for the largest cell, d measured from
// one cell on.  Limited to the grid's displacements, and to 2^20 of them in
// all (an accuracy in the hundreds): the rest is integrated element by element.
static void arne_reach(ArneArgs &a)
{
    const int most[3] = {a.x2 > -a.x1 ? a.x2 : -a.x1, a.y2 > -a.y1 ? a.y2 : -a.y1,
                         a.z2 > -a.z1 ? a.z2 : -a.z1};
    // (finite, so that the loop ends for any cell)
    const double far = fmin(a.accuracy * fmax(a.cell[0], fmax(a.cell[1], a.cell[2])) / 1.5, 1e300);
    for (double d = far;; d *= 0.8) {
        double count = 1.0;
        for (int c = 0; c < 3; c++) {
            const double cells = floor(d / a.cell[c]) + 1.0;
            a.reach[c] = cells < (double)most[c] ? (int)cells : most[c];
            count *= 2.0 * a.reach[c] + 1.0;
        }
        if (count <= (double)(1 << 20)) return;
    }
}

// ------------------------------------------------------------ Newell, FP64
//
// No reference counterpart (the reference's dipole kernel is Kernel_Arne).
// Newell, Williams & Dunlop, J. Geophys. Res. 98 (1993) 9551: the cell-pair
// averaged tensor is a 27-point sixth-order difference of f (diagonal) and g
// (off-diagonal).  That difference cancels ~log10(64 |R|^6 / V^2) digits, so
// from NEWELL_RSWITCH largest cell sizes on the tensor is the point-dipole
// tensor averaged over the offset of two points drawn uniformly from the two
// cells (triangular density 1 - |t| per axis), with a 5-point Gauss rule of
// that density per axis (error below 1e-10 relative there).  K = -N.

constexpr double kNewellRSwitch = 8.0;
constexpr int kNewellNQ = 5;

struct NewellArgs {
    double d[3];
    double rs2;        // (kNewellRSwitch * largest cell size)^2
    double t[kNewellNQ], w[kNewellNQ];
    int e[3];          // octant extent per axis
};

__device__ inline double nw_f(double x, double y, double z)
{
    x = fabs(x); y = fabs(y); z = fabs(z);
    const double x2 = x * x, y2 = y * y, z2 = z * z;
    const double R = sqrt(x2 + y2 + z2);
    double t = 0.0;
    if (y > 0 && x2 + z2 > 0) t += 0.5 * y * (z2 - x2) * asinh(y / sqrt(x2 + z2));
    if (z > 0 && x2 + y2 > 0) t += 0.5 * z * (y2 - x2) * asinh(z / sqrt(x2 + y2));
    if (x * y * z > 0) t -= x * y * z * atan(y * z / (x * R));
    t += (2.0 * x2 - y2 - z2) * R / 6.0;
    return t;
}

__device__ inline double nw_g(double x, double y, double z)
{
    const double sgn = ((x < 0) != (y < 0)) ? -1.0 : 1.0;
    x = fabs(x); y = fabs(y); z = fabs(z);
    const double x2 = x * x, y2 = y * y, z2 = z * z;
    const double R = sqrt(x2 + y2 + z2);
    double t = 0.0;
    if (z > 0 && x2 + y2 > 0) t += x * y * z * asinh(z / sqrt(x2 + y2));
    if (x > 0 && y2 + z2 > 0) t += y / 6.0 * (3.0 * z2 - y2) * asinh(x / sqrt(y2 + z2));
    if (y > 0 && x2 + z2 > 0) t += x / 6.0 * (3.0 * z2 - x2) * asinh(y / sqrt(x2 + z2));
    if (z > 0) t -= z2 * z / 6.0 * atan(x * y / (z * R));
    if (y > 0) t -= z * y2 / 2.0 * atan(x * z / (y * R));
    if (x > 0) t -= z * x2 / 2.0 * atan(y * z / (x * R));
    t -= x * y * R / 3.0;
    return sgn * t;
}

// stored component c = axis pair (a, b), XX,YY,ZZ,YZ,XZ,XY
__device__ __constant__ int kNwA[6] = {0, 1, 2, 1, 0, 0};
__device__ __constant__ int kNwB[6] = {0, 1, 2, 2, 2, 1};

// One thread per octant displacement R = (i,j,k) * d, i < e0, j < e1, k < e2;
// writes the 6 components of K(R) to oct[6*t + c].
__global__ void __launch_bounds__(kBlock) newell_octant(NewellArgs a, double *__restrict__ oct)
{
    const long ne = (long)a.e[0] * a.e[1] * a.e[2];
    const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= ne) return;
    const int k = (int)(t % a.e[2]);
    const int j = (int)((t / a.e[2]) % a.e[1]);
    const int i = (int)(t / ((long)a.e[2] * a.e[1]));
    const double R[3] = {i * a.d[0], j * a.d[1], k * a.d[2]};
    const double V = a.d[0] * a.d[1] * a.d[2];
    double out[6];
    if (R[0] * R[0] + R[1] * R[1] + R[2] * R[2] >= a.rs2) {
        double acc[6] = {0, 0, 0, 0, 0, 0};
        for (int qi = 0; qi < kNewellNQ; qi++)
            for (int qj = 0; qj < kNewellNQ; qj++)
                for (int qk = 0; qk < kNewellNQ; qk++) {
                    const double x[3] = {R[0] + a.t[qi] * a.d[0], R[1] + a.t[qj] * a.d[1],
                                         R[2] + a.t[qk] * a.d[2]};
                    const double r2 = x[0] * x[0] + x[1] * x[1] + x[2] * x[2];
                    const double W = a.w[qi] * a.w[qj] * a.w[qk] / (r2 * r2 * sqrt(r2));
                    acc[0] += W * (3.0 * x[0] * x[0] - r2);
                    acc[1] += W * (3.0 * x[1] * x[1] - r2);
                    acc[2] += W * (3.0 * x[2] * x[2] - r2);
                    acc[3] += W * (3.0 * x[1] * x[2]);
                    acc[4] += W * (3.0 * x[0] * x[2]);
                    acc[5] += W * (3.0 * x[0] * x[1]);
                }
        for (int c = 0; c < 6; c++) out[c] = V / (4.0 * kPi) * acc[c];
    } else {
        const double w3[3] = {-1.0, 2.0, -1.0};
        for (int c = 0; c < 6; c++) {
            const int ax = kNwA[c], bx = kNwB[c];
            int b2 = bx, c2 = 3 - ax - bx;
            if (ax == bx) { b2 = (ax + 1) % 3; c2 = (ax + 2) % 3; }
            double s = 0.0;
            for (int u = 0; u < 3; u++)
                for (int v = 0; v < 3; v++)
                    for (int w = 0; w < 3; w++) {
                        const double xa = R[ax] + (u - 1) * a.d[ax];
                        const double xb = R[b2] + (v - 1) * a.d[b2];
                        const double xc = R[c2] + (w - 1) * a.d[c2];
                        const double fv = (ax == bx) ? nw_f(xa, xb, xc) : nw_g(xa, xb, xc);
                        s += w3[u] * w3[v] * w3[w] * fv;
                    }
            out[c] = -s / (4.0 * kPi * V);
        }
    }
    // K_ab is odd in R_a and in R_b: exactly 0 on those planes
    if (i == 0 || k == 0) out[4] = 0.0;          // XZ: axes 0, 2
    if (j == 0 || k == 0) out[3] = 0.0;          // YZ: axes 1, 2
    if (i == 0 || j == 0) out[5] = 0.0;          // XY: axes 0, 1
    for (int c = 0; c < 6; c++) oct[6 * t + c] = out[c];
}

// Component c of the padded real-space kernel from the octant: displacement
// of padded index q is q (q < p/2) or q - p (q > p/2); the p/2 planes are 0
// (the displacement range Kernel_Arne fills).  Off-diagonal components are
// odd in both of their axes.  Optionally also the float32 copy (real_f32).
__global__ void __launch_bounds__(kBlock) newell_expand(const double *__restrict__ oct, int e0, int e1,
                                                        int e2, int p0, int p1, int p2, int c,
                                                        double *__restrict__ real,
                                                        float *__restrict__ real_f32)
{
    const long P = (long)p0 * p1 * p2;
    const int ax = kNwA[c], bx = kNwB[c];
    for (long t = (long)blockIdx.x * blockDim.x + threadIdx.x; t < P; t += (long)gridDim.x * blockDim.x) {
        const int q[3] = {(int)(t / ((long)p1 * p2)), (int)((t / p2) % p1), (int)(t % p2)};
        const int p[3] = {p0, p1, p2};
        int disp[3];
        bool zero = false;
        for (int x = 0; x < 3; x++) {
            if (p[x] == 1) { disp[x] = 0; continue; }
            if (2 * q[x] == p[x]) zero = true;
            disp[x] = (2 * q[x] < p[x]) ? q[x] : q[x] - p[x];
        }
        double v = 0.0;
        if (!zero) {
            const long o = ((long)abs(disp[0]) * e1 + abs(disp[1])) * e2 + abs(disp[2]);
            v = oct[6 * o + c];
            if (ax != bx) {
                if (disp[ax] < 0) v = -v;
                if (disp[bx] < 0) v = -v;
            }
        }
        real[t] = v;
        if (real_f32) real_f32[t] = (float)v;
    }
}

// The statistics of a build, one word each in a cache line of its own:
// workgroups merging into one line run one after another, about 10 ns each.
// That was all the time of the maximum kernels (75 us of maxabs_kernel, 26 us
// of each extract_octant at any size up to 200x200x5, with 1024 workgroups per
// component and every word in one line; 15 and 8 us so), hence also no more
// workgroups than 4 values per thread need (stat_blocks).
constexpr int kStats = 11, kStatStride = 16;
static int stat_blocks(long n, int most)
{
    return (int)std::max(1L, std::min((long)most, (n + 4 * kBlock - 1) / (4 * kBlock)));
}

// max |oct[6 t + c]| per component c into dst[c] (float bits)
__global__ void __launch_bounds__(kBlock) maxabs_oct6(const double *__restrict__ oct, long ne,
                                                      unsigned int *dst)
{
    float m[6] = {0, 0, 0, 0, 0, 0};
    for (long t = (long)blockIdx.x * blockDim.x + threadIdx.x; t < ne; t += (long)gridDim.x * blockDim.x)
        for (int c = 0; c < 6; c++) m[c] = fmaxf(m[c], (float)fabs(oct[6 * t + c]));
    for (int c = 0; c < 6; c++) {
        block_max_to(m[c], dst + c * kStatStride);
        __syncthreads();
    }
}

// 5-point Gauss rule on [-1,1] for the density 1 - |t|: nodes 0, +-sqrt(u1),
// +-sqrt(u2) with u1, u2 the roots of the quadratic orthogonal to 1 and u
// under u dmu(u), mu the distribution of u = t^2 (moments E[t^2j] =
// 2/((2j+1)(2j+2))); weights from the moment equations.
static void newell_rule5(double t[5], double w[5])
{
    long double mu[5];
    for (int j = 0; j < 5; j++) mu[j] = 2.0L / ((2.0L * j + 1.0L) * (2.0L * j + 2.0L));
    // u^2 + c1 u + c0:  mu3 + c1 mu2 + c0 mu1 = 0,  mu4 + c1 mu3 + c0 mu2 = 0
    const long double det = mu[2] * mu[2] - mu[1] * mu[3];
    const long double c1 = (-mu[3] * mu[2] + mu[1] * mu[4]) / det;
    const long double c0 = (-mu[2] * mu[4] + mu[3] * mu[3]) / det;
    const long double disc = sqrtl(c1 * c1 - 4.0L * c0);
    const long double u1 = (-c1 + disc) / 2.0L, u2 = (-c1 - disc) / 2.0L;
    // 2 (W1 u1 + W2 u2) = mu1,  2 (W1 u1^2 + W2 u2^2) = mu2
    const long double A = (mu[2] / 2.0L - u2 * mu[1] / 2.0L) / (u1 - u2);
    const long double B = mu[1] / 2.0L - A;
    const long double W1 = A / u1, W2 = B / u2;
    t[0] = (double)-sqrtl(u1); w[0] = (double)W1;
    t[1] = (double)-sqrtl(u2); w[1] = (double)W2;
    t[2] = 0.0;                w[2] = (double)(1.0L - 2.0L * (W1 + W2));
    t[3] = (double)sqrtl(u2);  w[3] = (double)W2;
    t[4] = (double)sqrtl(u1);  w[4] = (double)W1;
}

// max |x| of a float array into *dst (bits of a non-negative float)
// (component blockIdx.y of n floats)
__global__ void __launch_bounds__(kBlock) maxabs_kernel(const float *__restrict__ a, long n,
                                                        unsigned int *dst)
{
    a += blockIdx.y * n;
    dst += blockIdx.y * kStatStride;
    float m = 0.0f;
    for (long t = (long)blockIdx.x * blockDim.x + threadIdx.x; t < n; t += (long)gridDim.x * blockDim.x)
        m = fmaxf(m, fabsf(a[t]));
    block_max_to(m, dst);
}

// FP64 transform of the kernel, one component at a time.  The spectrum of a
// real kernel is kept as its half kx <= p2/2 (rows of h2 points), and the octant
// needs only ky <= p1/2 of the y transform's output, so the passes run over
// all rows along x, over kx < h2 along y and over ky < nky, kx < h2 along z.  A
// workgroup takes W neighbouring lines (consecutive in memory for y and z,
// 16 W bytes of each row); with one line per workgroup and every line of the
// full complex grid these passes took 3.0 ms at 200x200x5, here 0.41 ms.

// x: row r of the real input (float32 kernel, or FP64 for Newell's) -> h2 points
template <typename T>
__global__ void __launch_bounds__(kBlock) x_fft_f64(const T *__restrict__ a, long nrows, int W, int h2,
                                                    double2 *__restrict__ out, LineFFT<double> f)
{
    extern __shared__ double2 smd[];
    const int L = f.L, ls = L + 1;
    double2 *A = smd, *B = smd + W * ls;
    const long row0 = (long)blockIdx.x * W;
    for (int t = threadIdx.x; t < W * L; t += blockDim.x) {
        const int r = t / L, k = t - r * L;
        A[r * ls + k] = double2{row0 + r < nrows ? (double)a[row0 * L + t] : 0.0, 0.0};
    }
    __syncthreads();
    const double2 *R = lds_fft<double, -1>(A, B, W, ls, 1, f);
    for (int t = threadIdx.x; t < W * h2; t += blockDim.x) {
        const int r = t / h2, k = t - r * h2;
        if (row0 + r < nrows) out[row0 * h2 + t] = R[r * ls + k];
    }
}

// y or z, in place: line (o, q), o = blockIdx.y < outer planes, q < nline, has
// its element t at o * L * inner + t * inner + q
__global__ void __launch_bounds__(kBlock) axis_fft_f64(double2 *__restrict__ data, long inner,
                                                       long nline, int W, LineFFT<double> f)
{
    extern __shared__ double2 smd[];
    const int L = f.L, ls = L + 1;
    double2 *A = smd, *B = smd + W * ls;
    const long q0 = (long)blockIdx.x * W;
    double2 *base = data + (long)blockIdx.y * L * inner + q0;
    for (int e = threadIdx.x; e < W * L; e += blockDim.x) {
        const int t = e / W, w = e - t * W;
        A[w * ls + t] = q0 + w < nline ? base[t * inner + w] : double2{0.0, 0.0};
    }
    __syncthreads();
    const double2 *R = lds_fft<double, -1>(A, B, W, ls, 1, f);
    for (int e = threadIdx.x; e < W * L; e += blockDim.x) {
        const int t = e / W, w = e - t * W;
        if (q0 + w < nline) base[t * inner + w] = R[w * ls + t];
    }
}

// lines per workgroup: two buffers of W lines within 48 KB, at most 8 (128-byte
// pieces of a row); one line of up to 4096 points takes 131 KB
static int fft_f64_lines(int L)
{
    int w = 8;
    while (w > 1 && 2ull * w * (L + 1) * sizeof(double2) > 48 * 1024) w /= 2;
    return w;
}

static size_t fft_f64_lds(int L) { return 2ull * fft_f64_lines(L) * (L + 1) * sizeof(double2); }

template <typename K> static void allow_lds_f64(K kernel, size_t bytes)
{
    if (bytes > 65536)
        (void)hipFuncSetAttribute(reinterpret_cast<const void *>(kernel),
                                  hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
}

__global__ void __launch_bounds__(kBlock) zero_strided(float *__restrict__ out, long n)
{
    for (long t = (long)blockIdx.x * blockDim.x + threadIdx.x; t < n; t += (long)gridDim.x * blockDim.x)
        out[6 * t] = 0.0f;
}

// Octant extraction with the 1/Np scale; realness statistics over it.
__global__ void __launch_bounds__(kBlock) extract_octant(const double2 *__restrict__ full,
                                                         int p1, int ko0, int ko1,
                                                         int h2, double inv,
                                                         float *__restrict__ out,
                                                         unsigned int *maxbad,
                                                         unsigned int *maxgood)
{
    const long n = (long)ko0 * ko1 * h2;
    float bad = 0.0f, good = 0.0f;
    for (long t = (long)blockIdx.x * blockDim.x + threadIdx.x; t < n; t += (long)gridDim.x * blockDim.x) {
        int kx, ky, kz;
        if (n <= 0x7fffffffL) {
            const unsigned u = (unsigned)t, r = u / (unsigned)h2;
            kx = (int)(u - r * (unsigned)h2);
            kz = (int)(r / (unsigned)ko1);
            ky = (int)r - kz * ko1;
        } else {
            kx = (int)(t % h2);
            ky = (int)((t / h2) % ko1);
            kz = (int)(t / ((long)h2 * ko1));
        }
        const double2 v = full[((long)kz * p1 + ky) * h2 + kx];
        out[6 * t] = (float)(v.x * inv); // component slot of `out` set by the caller
        bad = fmaxf(bad, (float)fabs(v.y));
        good = fmaxf(good, (float)fabs(v.x));
    }
    block_max_to(bad, maxbad);
    __syncthreads();
    block_max_to(good, maxgood);
}

// The octant storage takes K at kz > p0/2 or ky > p1/2 from its mirror
// point, sign-flipped for the components odd in that axis (XZ and XY in axis
// 0, YZ and XY in axis 1).  For a kernel given by the caller this maximum
// deviation of the full FP64 spectrum from that rule is checked.
__global__ void __launch_bounds__(kBlock) octant_mirror_dev(const double2 *__restrict__ full,
                                                            int p0, int p1, int h2, int odd0,
                                                            int odd1,
                                                            unsigned int *maxdev)
{
    const long n = (long)p0 * p1 * h2;
    float dev = 0.0f;
    for (long t = (long)blockIdx.x * blockDim.x + threadIdx.x; t < n; t += (long)gridDim.x * blockDim.x) {
        const int kx = (int)(t % h2);
        const int ky = (int)((t / h2) % p1);
        const int kz = (int)(t / ((long)h2 * p1));
        const bool mz = kz > p0 / 2, my = ky > p1 / 2;
        if (!mz && !my) continue;
        const int kzp = mz ? p0 - kz : kz, kyp = my ? p1 - ky : ky;
        const double sign = ((mz && odd0) ? -1.0 : 1.0) * ((my && odd1) ? -1.0 : 1.0);
        const double a = full[((long)kz * p1 + ky) * h2 + kx].x;
        const double b = full[((long)kzp * p1 + kyp) * h2 + kx].x;
        dev = fmaxf(dev, (float)fabs(a - sign * b));
    }
    block_max_to(dev, maxdev);
}

// ------------------------------------------------------------ demagexch
//
// Exch6NgbrKernel (modules/kernel_exchange.go:102-124): the 6-neighbour
// Laplacian on the padded grid, the same for the three diagonal components,
// its seven float32 values assigned one after another at wrapped positions
// (kernel.go:19-27): a later value replaces an earlier one at the same
// position (on a length-1 axis the centre ends up 1/h_x^2).  dexKernUpdater
// (mod_demagexchange.go:134-149): dex = float32(Ms K_d + cex K_ex) with
// cex = 2 Aex / (mu0 Ms), from the float32 Arne kernel.

struct ExchPoints {
    long off[7];
    float val[7];
    int n;
};

static ExchPoints exch6_points(const int p[3], const double cell[3])
{
    const double h[3] = {cell[0] * cell[0], cell[1] * cell[1], cell[2] * cell[2]};
    const int d[7][3] = {{0, 0, 0}, {1, 0, 0}, {-1, 0, 0}, {0, 1, 0}, {0, -1, 0}, {0, 0, 1}, {0, 0, -1}};
    const float v[7] = {(float)(-2 / h[0] - 2 / h[1] - 2 / h[2]), (float)(1 / h[0]), (float)(1 / h[0]),
                        (float)(1 / h[1]), (float)(1 / h[1]), (float)(1 / h[2]), (float)(1 / h[2])};
    ExchPoints e{};
    for (int t = 0; t < 7; t++) {
        long off = 0;
        for (int a = 0; a < 3; a++) off = off * p[a] + ((d[t][a] % p[a]) + p[a]) % p[a];
        int k = 0;
        while (k < e.n && e.off[k] != off) k++;
        if (k == e.n) e.n++;
        e.off[k] = off;
        e.val[k] = v[t];
    }
    return e;
}

__global__ void __launch_bounds__(kBlock) dex_combine(float *__restrict__ K6, long Pn, double ms,
                                                      double cex, ExchPoints e)
{
    const long n = 6 * Pn;
    for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x) {
        const long c = i / Pn, o = i - c * Pn;
        double v = ms * (double)K6[i];
        if (c < 3)
            for (int k = 0; k < e.n; k++)
                if (e.off[k] == o) v += cex * (double)e.val[k];
        K6[i] = (float)v;
    }
}

__global__ void __launch_bounds__(kBlock) fold_kernel(const float *__restrict__ kd,
                                                      const float *__restrict__ kx, double inv_ms,
                                                      float *__restrict__ out, long n)
{
    for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x)
        out[i] = (float)((double)kd[i] + (double)kx[i] * inv_ms);
}

static int make_line_fft_f64(int L, LineFFT<double> &f, std::vector<double2> &host)
{
    f.L = L;
    if (!factor_radices(L, f.radix, &f.nstages)) {
        set_error("FFT length %d has more than %d prime factors", L, kMaxStages);
        return MMX_ERR_SIZE;
    }
    host.resize(L);
    for (int t = 0; t < L; t++) {
        const long double a = 2.0L * 3.14159265358979323846264338327950288L * (long double)t / (long double)L;
        host[t] = double2{(double)cosl(a), (double)(-sinl(a))};
    }
    return MMX_OK;
}

int build_demag_kernel(DemagPlanImpl *P, bool keep_real)
{
    const DemagGeom &g = P->g;
    const int p[3] = {g.p0, g.p1, g.p2};
    const long Pn = (long)p[0] * p[1] * p[2];
    const bool newell = P->cell_kernel_type == MMX_KERNEL_NEWELL;
    MMX_REQUIRE(P->cell_kernel_type == MMX_KERNEL_ARNE || newell, MMX_ERR_ARG,
                "kernel type %d not available", P->cell_kernel_type);
    MMX_REQUIRE(p[0] > 0 && p[1] > 1 && p[2] > 1, MMX_ERR_SIZE,
                "demag kernel needs padded sizes p1, p2 > 1 (got %d %d %d)", p[0], p[1], p[2]);
    MMX_REQUIRE(p[1] % 2 == 0 && p[2] % 2 == 0 && (p[0] == 1 || p[0] % 2 == 0), MMX_ERR_SIZE,
                "demag kernel needs even padded sizes (got %d %d %d)", p[0], p[1], p[2]);
    MMX_REQUIRE(p[0] <= 4096 && p[1] <= 4096 && p[2] <= 4096, MMX_ERR_SIZE,
                "kernel build: padded sizes above 4096 are not supported (%d %d %d)", p[0], p[1],
                p[2]);
    MMX_REQUIRE(!newell || (P->pbc[0] == 0 && P->pbc[1] == 0 && P->pbc[2] == 0), MMX_ERR_ARG,
                "the Newell kernel supports non-periodic grids only");

    float *K6 = nullptr;     // Arne: float32 real-space kernel (6 x Pn); Newell: kept copy
    float *tab = nullptr;    // Arne: near-field table
    double *oct = nullptr;   // Newell: FP64 octant table (6 per displacement)
    double *real64 = nullptr; // Newell: one component of the padded real-space kernel
    double2 *full = nullptr; // one component's half spectrum (p0 x p1 x h2)
    unsigned int *stats = nullptr;
    void *twd = nullptr;
    int rc = MMX_OK;
    auto fail = [&](int code) {
        rc = code;
        return code;
    };
    int e[3];
    for (int a = 0; a < 3; a++) e[a] = (p[a] == 1) ? 1 : p[a] / 2;
    const long ne = (long)e[0] * e[1] * e[2];
    hipError_t err = hipSuccess;
    if (!newell || keep_real) err = hipMalloc(&K6, sizeof(float) * 6 * Pn);
    if (err == hipSuccess && newell) err = hipMalloc(&oct, sizeof(double) * 6 * ne);
    if (err == hipSuccess && newell) err = hipMalloc(&real64, sizeof(double) * Pn);
    if (err == hipSuccess) err = hipMalloc(&full, sizeof(double2) * (size_t)p[0] * p[1] * g.h2);
    if (err == hipSuccess) err = hipMalloc(&stats, sizeof(unsigned int) * kStats * kStatStride);
    if (err != hipSuccess) {
        (void)hipFree(K6);
        (void)hipFree(oct);
        (void)hipFree(real64);
        (void)hipFree(full);
        (void)hipFree(stats);
        set_error("kernel build: cannot allocate the FP64 work arrays (%ld points)", Pn);
        return MMX_ERR_NOMEM;
    }
    do {
        if (K6 && hipMemset(K6, 0, sizeof(float) * 6 * Pn) != hipSuccess) { fail(MMX_ERR_HIP); break; }
        if (hipMemset(stats, 0, sizeof(unsigned int) * kStats * kStatStride) != hipSuccess) { fail(MMX_ERR_HIP); break; }

        if (newell) {
            NewellArgs a{};
            double dm = 0.0;
            for (int x = 0; x < 3; x++) {
                a.d[x] = P->cell[x];
                a.e[x] = e[x];
                dm = fmax(dm, P->cell[x]);
            }
            a.rs2 = kNewellRSwitch * kNewellRSwitch * dm * dm;
            newell_rule5(a.t, a.w);
            newell_octant<<<dim3(div_up(ne, kBlock)), dim3(kBlock)>>>(a, oct);
            maxabs_oct6<<<dim3(stat_blocks(6 * ne, 256)), dim3(kBlock)>>>(oct, ne, stats);
            if (hipGetLastError() != hipSuccess) { set_error("newell_octant launch failed"); fail(MMX_ERR_HIP); break; }
        } else if (P->host_kernel) {
            // ConvPlan.loadKernel (convplan.go:85-115): the caller's kernel
            for (int c = 0; c < 6; c++) {
                if (!P->host_kernel[c]) continue;
                if (hipMemcpy(K6 + c * Pn, P->host_kernel[c], sizeof(float) * Pn,
                              hipMemcpyHostToDevice) != hipSuccess) { fail(MMX_ERR_HIP); break; }
            }
            if (rc) break;
            maxabs_kernel<<<dim3(stat_blocks(Pn, 256), 6), dim3(kBlock)>>>(K6, Pn, stats);
            if (hipGetLastError() != hipSuccess) { set_error("maxabs launch failed"); fail(MMX_ERR_HIP); break; }
        } else {
            // ranges of Kernel_Arne (kernel_magnetostatic.go:50-65)
            ArneArgs a{};
            for (int i = 0; i < 3; i++) {
                a.p[i] = p[i];
                a.cell[i] = P->cell[i];
            }
            a.x1 = -(p[0] - 1) / 2; a.x2 = p[0] / 2 - 1;
            a.y1 = -(p[1] - 1) / 2; a.y2 = p[1] / 2 - 1;
            a.z1 = -(p[2] - 1) / 2; a.z2 = p[2] / 2 - 1;
            if (p[0] == 1 && P->pbc[0] == 0) a.x2 = 0;
            a.x1 *= (P->pbc[0] + 1); a.x2 *= (P->pbc[0] + 1);
            a.y1 *= (P->pbc[1] + 1); a.y2 *= (P->pbc[1] + 1);
            a.z1 *= (P->pbc[2] + 1); a.z2 *= (P->pbc[2] + 1);
            double L = P->cell[0];
            if (P->cell[1] < L) L = P->cell[1];
            if (P->cell[2] < L) L = P->cell[2];
            a.L = L;
            a.accuracy = (double)P->accuracy;
            arne_reach(a);
            const int near = (2 * a.reach[0] + 1) * (2 * a.reach[1] + 1) * (2 * a.reach[2] + 1);
            if (hipMalloc(&tab, sizeof(float) * 9 * (size_t)near) != hipSuccess) {
                set_error("kernel build: cannot allocate the near-field table (%d displacements)", near);
                fail(MMX_ERR_NOMEM);
                break;
            }
            arne_near<<<dim3(near, 3), dim3(64 + kNearChunk)>>>(a, tab);
            arne_kernel<<<dim3(div_up(Pn, kBlock), 3), dim3(kBlock)>>>(a, tab, K6);
            if (hipGetLastError() != hipSuccess) { set_error("arne_kernel launch failed"); fail(MMX_ERR_HIP); break; }
            if (P->dex) {
                dex_combine<<<dim3(4096), dim3(kBlock)>>>(K6, Pn, P->dex_ms, P->dex_cex,
                                                          exch6_points(p, P->cell));
                if (hipGetLastError() != hipSuccess) { set_error("dex_combine launch failed"); fail(MMX_ERR_HIP); break; }
            }
            // IsZero test per component (maxwell_convolution.go:412-418)
            maxabs_kernel<<<dim3(stat_blocks(Pn, 256), 6), dim3(kBlock)>>>(K6, Pn, stats);
            if (hipGetLastError() != hipSuccess) { set_error("maxabs launch failed"); fail(MMX_ERR_HIP); break; }
        }
        unsigned int hs[kStats * kStatStride];
        if (hipMemcpy(hs, stats, sizeof(hs), hipMemcpyDeviceToHost) != hipSuccess) { fail(MMX_ERR_HIP); break; }
        float cmax[6], kmax = 0.0f;
        for (int c = 0; c < 6; c++) {
            std::memcpy(&cmax[c], &hs[c * kStatStride], 4);
            kmax = fmaxf(kmax, cmax[c]);
        }

        // FP64 twiddles for the three lengths
        LineFFT<double> f[3];
        std::vector<double2> tw[3];
        size_t off[4] = {0, 0, 0, 0};
        for (int ax = 0; ax < 3; ax++) {
            if (make_line_fft_f64(p[ax], f[ax], tw[ax])) { fail(MMX_ERR_SIZE); break; }
            off[ax + 1] = off[ax] + tw[ax].size();
        }
        if (rc) break;
        if (hipMalloc(&twd, sizeof(double2) * off[3]) != hipSuccess) { fail(MMX_ERR_NOMEM); break; }
        for (int ax = 0; ax < 3; ax++) {
            if (hipMemcpy((double2 *)twd + off[ax], tw[ax].data(), sizeof(double2) * tw[ax].size(),
                          hipMemcpyHostToDevice) != hipSuccess) { fail(MMX_ERR_HIP); break; }
            f[ax].tw = (const double2 *)twd + off[ax];
        }
        if (rc) break;
        allow_lds_f64(x_fft_f64<float>, fft_f64_lds(p[2]));
        allow_lds_f64(x_fft_f64<double>, fft_f64_lds(p[2]));
        allow_lds_f64(axis_fft_f64, std::max(fft_f64_lds(p[1]), fft_f64_lds(p[0])));
        // the caller's kernel: every ky, for the symmetry check
        const int nky = P->host_kernel ? p[1] : g.ko1;

        const long octant = (long)g.ko0 * g.ko1 * g.h2;
        const double inv = 1.0 / (double)Pn;
        for (int c = 0; c < 6; c++) {
            // interleaved storage: component c of point o at P->kern[6*o + c]
            // (6*octant floats); extract_octant / zero_strided write out[6*t]
            float *dst = P->kern + c;
            // (ConvPlan.loadKernel, used by demagexch, transforms every
            // component: convplan.go:85-115)
            const bool unused = P->host_kernel ? P->host_kernel[c] == nullptr
                                               : (!P->dex && (kmax == 0.0f || cmax[c] / kmax < 1e-5f));
            if (unused) {
                zero_strided<<<dim3(1024), dim3(kBlock)>>>(dst, octant);
                if (hipGetLastError() != hipSuccess) { set_error("kernel zero launch failed"); fail(MMX_ERR_HIP); break; }
                continue;
            }
            const long nrows = (long)p[0] * p[1];
            const int wx = fft_f64_lines(p[2]), wy = fft_f64_lines(p[1]), wz = fft_f64_lines(p[0]);
            if (newell) {
                newell_expand<<<dim3(4096), dim3(kBlock)>>>(oct, e[0], e[1], e[2], p[0], p[1], p[2], c,
                                                            real64, K6 ? K6 + c * Pn : nullptr);
                x_fft_f64<double><<<dim3(div_up(nrows, wx)), dim3(kBlock), fft_f64_lds(p[2])>>>(
                    real64, nrows, wx, g.h2, full, f[2]);
            } else {
                x_fft_f64<float><<<dim3(div_up(nrows, wx)), dim3(kBlock), fft_f64_lds(p[2])>>>(
                    K6 + c * Pn, nrows, wx, g.h2, full, f[2]);
            }
            axis_fft_f64<<<dim3(div_up(g.h2, wy), p[0]), dim3(kBlock), fft_f64_lds(p[1])>>>(
                full, g.h2, g.h2, wy, f[1]);
            if (p[0] > 1)
                axis_fft_f64<<<dim3(div_up((long)nky * g.h2, wz), 1), dim3(kBlock), fft_f64_lds(p[0])>>>(
                    full, (long)p[1] * g.h2, (long)nky * g.h2, wz, f[0]);
            extract_octant<<<dim3(stat_blocks(octant, 1024)), dim3(kBlock)>>>(full, p[1], g.ko0, g.ko1, g.h2, inv, dst,
                                                         stats + 8 * kStatStride, stats + 9 * kStatStride);
            if (P->host_kernel) {
                // components XX,YY,ZZ,YZ,XZ,XY: odd in axis 0 for XZ, XY; in axis 1 for YZ, XY
                const int odd0 = (c == 4 || c == 5), odd1 = (c == 3 || c == 5);
                octant_mirror_dev<<<dim3(1024), dim3(kBlock)>>>(full, p[0], p[1], g.h2, odd0, odd1,
                                                                stats + 10 * kStatStride);
            }
            if (hipGetLastError() != hipSuccess) { set_error("kernel FFT launch failed"); fail(MMX_ERR_HIP); break; }
        }
        if (rc) break;
        if (hipMemcpy(hs, stats, sizeof(hs), hipMemcpyDeviceToHost) != hipSuccess) { fail(MMX_ERR_HIP); break; }
        float bad, good;
        std::memcpy(&bad, &hs[8 * kStatStride], 4);
        std::memcpy(&good, &hs[9 * kStatStride], 4);
        P->bad_over_good = good > 0 ? (double)bad / (double)good : 0.0;
        if (P->host_kernel) {
            // ConvPlan only warns about imaginary parts (convplan.go:143-152);
            // the octant storage needs the mirror symmetry, so that is enforced
            float mdev;
            std::memcpy(&mdev, &hs[10 * kStatStride], 4);
            if (good > 0 && (double)mdev / (double)good > 1e-5) {
                set_error("convolution kernel: transformed kernel deviates from the mirror "
                          "symmetry of a demag/exchange kernel by %g of its maximum",
                          (double)mdev / (double)good);
                fail(MMX_ERR_ARG);
                break;
            }
        } else if (P->bad_over_good > 1e-5) {
            set_error("FFT kernel max bad/good part = %g", P->bad_over_good);
            fail(MMX_ERR_STATE);
            break;
        }
    } while (0);
    if (rc == MMX_OK && keep_real) {
        P->real_kernel = K6;
        K6 = nullptr;
    }
    (void)hipFree(K6);
    (void)hipFree(tab);
    (void)hipFree(oct);
    (void)hipFree(real64);
    (void)hipFree(full);
    (void)hipFree(stats);
    (void)hipFree(twd);
    if (rc == MMX_OK && hipDeviceSynchronize() != hipSuccess) {
        set_error("kernel build: device error");
        return MMX_ERR_HIP;
    }
    return rc;
}

int build_dex_kernel(const DemagPlanImpl *P, int accuracy, double ms, double aex, float *out)
{
    MMX_REQUIRE(P && out && accuracy >= 0 && ms != 0.0, MMX_ERR_ARG, "build_dex_kernel: bad arguments");
    DemagPlanImpl Q = *P;   // geometry, cells, periodicity; nothing of P is written
    Q.kern = out;
    Q.real_kernel = nullptr;
    Q.accuracy = accuracy;
    Q.cell_kernel_type = MMX_KERNEL_ARNE;
    Q.dex = true;
    Q.dex_ms = ms;
    Q.dex_cex = (2.0 * aex) / (kMu0 * ms);
    return build_demag_kernel(&Q, false);
}

int fold_kernels(const float *kd, const float *kx, double ms, float *out, long n)
{
    MMX_REQUIRE(kd && kx && out && n > 0 && ms != 0.0, MMX_ERR_ARG, "fold_kernels: bad arguments");
    fold_kernel<<<dim3(1024), dim3(kBlock)>>>(kd, kx, 1.0 / ms, out, n);
    MMX_CHECK_LAUNCH();
    MMX_HIP(hipDeviceSynchronize());
    return MMX_OK;
}

} // namespace mmx
