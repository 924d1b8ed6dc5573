// surrogate.hip -- learned correction of a 2x-coarsened demag field.
//
// No reference counterpart (the reference has no learned component).  For a
// film of n0 <= 5 layers on an n1 x n2 in-plane grid (internal z,y,x order):
//
//   coarse m  = means of 2x2 in-plane blocks of m, layers kept (coarsening the
//               few layers of a film loses most of the field: 92 % error on a
//               random state against 23 % for in-plane coarsening);
//   coarse B  = exact demag of the coarse grid (its own demag plan);
//   net input = per in-plane pixel, channel c*n0+i = m_c of layer i,
//               3*n0 + c*n0+i = the upsampled coarse B_c / (mu0 Ms), and
//               6*n0, 6*n0+1 = the position in the coarse cell (+-1 for odd /
//               even y, x: the residual operator has period 2), in bf16;
//   net       = 4 conv 3x3 layers 32 -> 32 -> 32 -> 32 -> 16 (ReLU after the
//               first three), BF16 MFMA with FP32 accumulation (gfx950's
//               v_mfma_f32_16x16x32_bf16, 32 channels or pixels per
//               instruction; 16-channel inputs on v_mfma_f32_16x16x16_bf16),
//               as implicit GEMMs over 16 x 8 pixel tiles;
//   B_fine   ~= upsampled coarse B + mu0 Ms * out[c*n0+i].
//
// Training (on the GPU, by these kernels): relative squared error of the
// residual against the exact fine field (sum d^2 / sum target^2 per sample), backward-data as the same convolution kernel with flipped
// and transposed weights and a ReLU-mask epilogue, weight gradients as MFMA
// products over the pixel tiles with per-workgroup partial sums reduced in a fixed
// order (deterministic), Adam on FP32 master weights.  The CPU oracle
// (oracle/surrogate.py) rounds to bf16 at the same points.
//
// In the RK12 solver (sim.cpp) the corrector's field evaluation uses the
// surrogate; the first stage (at the accepted m) stays exact, and every
// `check_every` steps the exact field at the accepted m judges the surrogate's
// there: above the tolerance the solver falls back to the exact path.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <random>
#include <type_traits>
#include <vector>

#include "demag_tiles.hpp"
#include "sim_impl.hpp"

namespace mmx {


typedef unsigned short bf16_t;
typedef short sh4 __attribute__((ext_vector_type(4)));
typedef short sh8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf8 __attribute__((ext_vector_type(8)));
typedef float fl4 __attribute__((ext_vector_type(4)));

// D += A B over k = 32 on gfx950's double-K bf16 MFMA: lane (n = lane % 16,
// g = lane / 16) passes 8 values of row n of A and 8 of column n of B, and
// holds D[4 g + e][n], e < 4.  Both operands index their k by the same
// (g, element), so the sum covers each k once whatever order the unit uses.
__device__ __forceinline__ fl4 mfma_k32(sh8 a, sh8 b, fl4 c)
{
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf8, a),
                                                   __builtin_bit_cast(bf8, b), c, 0, 0, 0);
}

constexpr int kSurCh[5] = {32, 32, 32, 32, 16};

__device__ __forceinline__ bf16_t f2bf(float x)
{
    unsigned int u = __float_as_uint(x);
    if ((u & 0x7f800000u) == 0x7f800000u) return (bf16_t)((u >> 16) | ((u & 0xffffu) ? 0x40u : 0u));
    u += 0x7fffu + ((u >> 16) & 1u);
    return (bf16_t)(u >> 16);
}
__device__ __forceinline__ float bf2f(bf16_t h) { return __uint_as_float((unsigned int)h << 16); }

struct SurGeom {
    int n0, n1, n2;       // fine grid
    int c0, c1, c2;       // coarse grid
    int f0;               // z coarsening factor (1 or 2)
    long N, Nc;
    float inv_mu0ms;      // 1 / (mu0 Ms)
    float msat;
};

// --------------------------------------------------------- field kernels

// Block means of m (times the Msat map) on the coarse grid; with PRED the fine
// m is first the RK predictor normalize(m0 + h tau0) (maddKern + normUpdater,
// as in the exact predictor), written to mpred.
template <int PRED>
__global__ void __launch_bounds__(kBlock)
sur_coarsen(SurGeom s, const float *__restrict__ m0, const float *__restrict__ tau0, float h,
            const float *__restrict__ msat_map, float *__restrict__ mpred, float *__restrict__ mc)
{
    const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= s.Nc) return;
    const int ck = (int)(t % s.c2), cj = (int)((t / s.c2) % s.c1), ci = (int)(t / ((long)s.c2 * s.c1));
    float acc[3] = {0.0f, 0.0f, 0.0f};
    for (int a = 0; a < s.f0; a++)
        for (int b = 0; b < 2; b++)
            for (int c = 0; c < 2; c++) {
                const long I = ((long)(ci * s.f0 + a) * s.n1 + (cj * 2 + b)) * s.n2 + (ck * 2 + c);
                float v0 = m0[I], v1 = m0[s.N + I], v2 = m0[2 * s.N + I];
                if (PRED) {
                    v0 = v0 + h * tau0[I];
                    v1 = v1 + h * tau0[s.N + I];
                    v2 = v2 + h * tau0[2 * s.N + I];
                    const float norm = msat_map ? msat_map[I] : 1.0f;
                    const float len = sqrtf(v0 * v0 + v1 * v1 + v2 * v2);
                    float scale = (norm == 0.0f) ? 0.0f : 1.0f;
                    scale = (len != 0.0f) ? scale / len : 0.0f;
                    v0 *= scale;
                    v1 *= scale;
                    v2 *= scale;
                    mpred[I] = v0;
                    mpred[s.N + I] = v1;
                    mpred[2 * s.N + I] = v2;
                }
                const float ms = msat_map ? msat_map[I] : 1.0f;
                acc[0] += v0 * ms;
                acc[1] += v1 * ms;
                acc[2] += v2 * ms;
            }
    const float inv = 1.0f / (float)(s.f0 * 4);
    mc[t] = acc[0] * inv;
    mc[s.Nc + t] = acc[1] * inv;
    mc[2 * s.Nc + t] = acc[2] * inv;
}

__device__ __forceinline__ long coarse_of(const SurGeom &s, int i, int j, int k)
{
    return ((long)(i / s.f0) * s.c1 + j / 2) * s.c2 + k / 2;
}

// net input channel ch of pixel (y, x), from m and the coarse B (tesla)
__device__ __forceinline__ float input_channel(const SurGeom &s, const float *__restrict__ m,
                                               const float *__restrict__ bc, int y, int x, int ch)
{
    const int nm = 3 * s.n0;
    if (ch < nm) {
        const int c = ch / s.n0, i = ch - c * s.n0;
        return m[c * s.N + ((long)i * s.n1 + y) * s.n2 + x];
    }
    if (ch < 2 * nm) {
        const int q = ch - nm, c = q / s.n0, i = q - c * s.n0;
        return bc[c * s.Nc + coarse_of(s, i, y, x)] * s.inv_mu0ms;
    }
    if (ch == 2 * nm) return (y & 1) ? 1.0f : -1.0f;
    if (ch == 2 * nm + 1) return (x & 1) ? 1.0f : -1.0f;
    return 0.0f;
}

// Packed bf16 input [P][32].  Bound by the latency of its scattered plane
// reads: a wave takes 64 consecutive pixels and 8 channels, so every plane is
// read in whole lines and a pixel's 8 channels leave in one 16-byte store
// (256x256x4: 12.6 us with one channel per thread, which read 4 pixels of 16
// planes per wave, 8.0 us so).  A first convolution that forms its input itself
// reads them by pixel: 25.9 us (21.1 with 4 channels per thread) against 8.1 for
// this and 5.7 for the convolution of the packed input.
__global__ void __launch_bounds__(kBlock)
sur_pack(SurGeom s, const float *__restrict__ m, const float *__restrict__ bc,
         bf16_t *__restrict__ x0)
{
    const long P = (long)s.n1 * s.n2;
    const long p = (long)blockIdx.x * 64 + (threadIdx.x & 63);
    const int q = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6); // uniform plane arithmetic
    if (p >= P) return;
    const int y = (int)((unsigned)p / (unsigned)s.n2), x = (int)p - y * s.n2; // P < 2^31
    unsigned w[4];
#pragma unroll
    for (int e = 0; e < 4; e++)
        w[e] = (unsigned)f2bf(input_channel(s, m, bc, y, x, 8 * q + 2 * e)) |
               ((unsigned)f2bf(input_channel(s, m, bc, y, x, 8 * q + 2 * e + 1)) << 16);
    *reinterpret_cast<uint4 *>(x0 + p * 32 + 8 * q) = uint4{w[0], w[1], w[2], w[3]};
}

// ------------------------------------------------------------ convolution

enum { CE_RELU_BF16 = 0, CE_LINEAR_F32 = 1, CE_MASK_BF16 = 2 };

__device__ __forceinline__ fl4 mfma_any(sh8 a, sh8 b, fl4 c) { return mfma_k32(a, b, c); }
__device__ __forceinline__ fl4 mfma_any(sh4 a, sh4 b, fl4 c)
{
    return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, c, 0, 0, 0);
}

// out[p][co] = epilogue(sum_tap sum_ci in[p + off(tap)][ci] * wt[tap][co][ci])
// over a 16 x 8 pixel tile per workgroup of 4 waves.  The MFMA computes
// D = A B with A = weights (rows co, k = ci) and B = the input (k = ci,
// columns = 16 pixels of a row), so each lane ends up holding 4 consecutive
// output channels of one pixel.
//
// Bound by the latency of one load - LDS - MFMA chain per workgroup (512
// workgroups at 256x256, two per CU), not by the 36 MFMA of a wave.  A wave
// owns 16 output channels, so its nine weight fragments are loaded from global
// memory straight into registers while the tile is staged, and an input
// fragment read once from LDS serves the three output rows it belongs to.
// With the weights staged in LDS (18 KB per workgroup) and every fragment read
// per output row: 9.0 us a layer at 256x256, so 5.6 us.
template <int CIN, int COUT, int EPI>
__global__ void __launch_bounds__(kBlock)
sur_conv(const bf16_t *__restrict__ in, const bf16_t *__restrict__ wt,
         const float *__restrict__ bias, const bf16_t *__restrict__ mask, void *__restrict__ out,
         int H, int W)
{
    static_assert(CIN == 32 || CIN == 16, "one MFMA per tap");
    using Frag = std::conditional_t<CIN == 32, sh8, sh4>;
    constexpr int CP = CIN + 8; // LDS pitch per pixel (bf16 elements)
    constexpr int NQ = CIN / 8, TASKS = 10 * 18 * NQ, ITER = (TASKS + kBlock - 1) / kBlock;
    constexpr int MT = COUT / 16, ROWS = 2 * MT; // output rows of a wave
    __shared__ __align__(16) bf16_t tile[10 * 18 * CP];
    const int x0 = blockIdx.x * 16, y0 = blockIdx.y * 8;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int n = lane & 15, kq = (lane >> 4) * 4, kf = (lane >> 4) * (CIN / 4);
    const int mt = wave % MT, row0 = (wave / MT) * ROWS, co = mt * 16 + kq;

    uint4 u[ITER];
#pragma unroll
    for (int i = 0; i < ITER; i++) {
        const int t = threadIdx.x + i * kBlock;
        const int q = t % NQ, pc = t / NQ, cx = pc % 18, cy = pc / 18;
        const int gy = y0 + cy - 1, gx = x0 + cx - 1;
        u[i] = uint4{0u, 0u, 0u, 0u};
        if (t < TASKS && gy >= 0 && gy < H && gx >= 0 && gx < W)
            u[i] = *reinterpret_cast<const uint4 *>(in + ((long)gy * W + gx) * CIN + 8 * q);
    }
    Frag a[9];
#pragma unroll
    for (int tap = 0; tap < 9; tap++)
        a[tap] = *reinterpret_cast<const Frag *>(wt + (tap * COUT + mt * 16 + n) * CIN + kf);
#pragma unroll
    for (int i = 0; i < ITER; i++) {
        const int t = threadIdx.x + i * kBlock;
        if (t < TASKS) *reinterpret_cast<uint4 *>(tile + (t / NQ) * CP + 8 * (t % NQ)) = u[i];
    }
    __syncthreads();

    fl4 acc[ROWS];
#pragma unroll
    for (int r = 0; r < ROWS; r++) acc[r] = fl4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int ri = 0; ri < ROWS + 2; ri++) // input row row0 + ri - 1 of the tile
#pragma unroll
        for (int dx = 0; dx < 3; dx++) {
            const Frag b = *reinterpret_cast<const Frag *>(tile + ((row0 + ri) * 18 + n + dx) * CP + kf);
#pragma unroll
            for (int dy = 0; dy < 3; dy++)
                if (ri - dy >= 0 && ri - dy < ROWS)
                    acc[ri - dy] = mfma_any(a[dy * 3 + dx], b, acc[ri - dy]);
        }
#pragma unroll
    for (int r = 0; r < ROWS; r++) {
        const long pix = (long)(y0 + row0 + r) * W + x0 + n;
        float v[4] = {acc[r][0], acc[r][1], acc[r][2], acc[r][3]};
        if (EPI == CE_LINEAR_F32) {
#pragma unroll
            for (int e = 0; e < 4; e++) v[e] += bias[co + e];
            *reinterpret_cast<float4 *>(reinterpret_cast<float *>(out) + pix * COUT + co) =
                float4{v[0], v[1], v[2], v[3]};
        } else {
            if (EPI == CE_RELU_BF16) {
#pragma unroll
                for (int e = 0; e < 4; e++) v[e] = fmaxf(v[e] + bias[co + e], 0.0f);
            } else {
                const uint2 mk = *reinterpret_cast<const uint2 *>(mask + pix * COUT + co);
                const bf16_t mb[4] = {(bf16_t)(mk.x & 0xffffu), (bf16_t)(mk.x >> 16),
                                      (bf16_t)(mk.y & 0xffffu), (bf16_t)(mk.y >> 16)};
#pragma unroll
                for (int e = 0; e < 4; e++) v[e] = bf2f(mb[e]) > 0.0f ? v[e] : 0.0f;
            }
            const unsigned lo = (unsigned)f2bf(v[0]) | ((unsigned)f2bf(v[1]) << 16);
            const unsigned hi = (unsigned)f2bf(v[2]) | ((unsigned)f2bf(v[3]) << 16);
            *reinterpret_cast<uint2 *>(reinterpret_cast<bf16_t *>(out) + pix * COUT + co) =
                uint2{lo, hi};
        }
    }
}

// The four layers' operands of the weight gradients and of the update.
struct SurLayers {
    const bf16_t *x[4], *dz[4]; // layer input, gradient at its linear output
    bf16_t *wt[4], *wbt[4];     // bf16 weights, forward and backward-data order
    int off[5];                 // first parameter of each layer (weights, then bias), and the end
};
constexpr int kSurSlot = 9 * 32 * 32 + 32; // partial gradients of one workgroup and layer
// Workgroups of the weight gradients per layer: a tile each up to 128 tiles;
// beyond, a workgroup adds up several tiles (two workgroups per CU over the
// four layers), so the partial gradients stay below 19 MB.  256x256 with one
// tile each and 38 MB: 18.1 us and a longer reduction, against 16.4 us.
constexpr int kSurParts = 128;

// Weight and bias gradients of one layer over 16 x 16 pixel tiles:
// part[(tap*CIN + ci)*COUT + co] = sum_p dz[p][co] x[p + off(tap)][ci],
// part[9*CIN*COUT + co] = sum_p dz[p][co].  MFMA with A = dz^T (rows co,
// k = pixels) and B = the shifted input (k = pixels, columns ci).
//
// The contraction runs over pixels, so both operands are turned to
// channel-major order on their way into LDS: a fragment (8 pixels of one
// channel) is then one 16-byte read, where the pixel-major tile took eight
// 2-byte reads per operand and MFMA, which was what bound the kernel.  The
// three taps of an input row come out of one 16 + 4 byte read by register
// shifts, and the next tile's loads fly under the products.  A wave keeps one 16 x 16 block of (co, ci) for its taps and reads
// every dz fragment once.  Channel pitches are odd multiples of 16 bytes (no
// bank conflicts between the 16 channels of a read).  All four layers in one
// launch, 512 workgroups at 256x256: 77 us of four launches before, 16.4 us
// so.  What is left is the latency of the loads (33 MB at 2 TB/s).
constexpr int kWgRow = 24, kWgX = 18 * kWgRow + 8, kWgD = 256 + 8;
template <int COUT>
__device__ __forceinline__ void wgrad_tiles(const bf16_t *__restrict__ x, const bf16_t *__restrict__ dz,
                                            float *__restrict__ dst, int H, int W, int ntile,
                                            bf16_t *xt, bf16_t *dzt, float *bsum)
{
    constexpr int CIN = 32, NQX = CIN / 4, NQD = COUT / 4;
    constexpr int XT = 18 * 9 * NQX, XI = (XT + kBlock - 1) / kBlock; // pairs of pixels x 4 channels
    constexpr int DT = 128 * NQD, DI = DT / kBlock;
    // COUT 32: a wave per (mt, nt) with all three dy; 16: waves 0, 1 take dy
    // 0 and 1, waves 2, 3 take dy 2
    constexpr int MT = COUT / 16, NDY = MT == 2 ? 3 : 2;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int n = lane & 15, kq = (lane >> 4) * 4, kq8 = (lane >> 4) * 8;
    const int nt = wave & 1, mt = MT == 2 ? wave >> 1 : 0;
    const int dy0 = MT == 2 ? 0 : (wave >> 1) * 2;
    fl4 acc[3 * NDY];
#pragma unroll
    for (int i = 0; i < 3 * NDY; i++) acc[i] = fl4{0.0f, 0.0f, 0.0f, 0.0f};
    float sum = 0.0f;
    const int tw = W / 16;
    uint2 ua[XI][2], ud[DI][2];
    auto load = [&](int tile) {
        const int x0 = (tile % tw) * 16, y0 = (tile / tw) * 16;
#pragma unroll
        for (int i = 0; i < XI; i++) {
            const int t = threadIdx.x + i * kBlock;
            const int q = t % NQX, pp = t / NQX, cx = 2 * (pp % 9), cy = pp / 9;
            const int gy = y0 + cy - 1;
#pragma unroll
            for (int h = 0; h < 2; h++) {
                const int gx = x0 + cx + h - 1;
                ua[i][h] = uint2{0u, 0u};
                if (t < XT && gy >= 0 && gy < H && gx >= 0 && gx < W)
                    ua[i][h] = *reinterpret_cast<const uint2 *>(x + ((long)gy * W + gx) * CIN + 4 * q);
            }
        }
#pragma unroll
        for (int i = 0; i < DI; i++) {
            const int t = threadIdx.x + i * kBlock;
            const int q = t % NQD, p = 2 * (t / NQD);
            const long g = (long)(y0 + p / 16) * W + x0 + p % 16;
#pragma unroll
            for (int h = 0; h < 2; h++)
                ud[i][h] = *reinterpret_cast<const uint2 *>(dz + (g + h) * COUT + 4 * q);
        }
    };
    load(blockIdx.x);
    for (int tile = blockIdx.x; tile < ntile; tile += gridDim.x) {
        if (tile != (int)blockIdx.x) __syncthreads(); // the tile before is read
        auto put = [](bf16_t *d, int pitch, uint2 e0, uint2 e1) {
            *reinterpret_cast<unsigned *>(d) = (e0.x & 0xffffu) | (e1.x << 16);
            *reinterpret_cast<unsigned *>(d + pitch) = (e0.x >> 16) | (e1.x & 0xffff0000u);
            *reinterpret_cast<unsigned *>(d + 2 * pitch) = (e0.y & 0xffffu) | (e1.y << 16);
            *reinterpret_cast<unsigned *>(d + 3 * pitch) = (e0.y >> 16) | (e1.y & 0xffff0000u);
        };
#pragma unroll
        for (int i = 0; i < XI; i++) {
            const int t = threadIdx.x + i * kBlock;
            const int q = t % NQX, pp = t / NQX, cx = 2 * (pp % 9), cy = pp / 9;
            if (t < XT) put(xt + 4 * q * kWgX + cy * kWgRow + cx, kWgX, ua[i][0], ua[i][1]);
        }
#pragma unroll
        for (int i = 0; i < DI; i++) {
            const int t = threadIdx.x + i * kBlock;
            put(dzt + 4 * (t % NQD) * kWgD + 2 * (t / NQD), kWgD, ud[i][0], ud[i][1]);
        }
        __syncthreads();
        if (tile + (int)gridDim.x < ntile) load(tile + gridDim.x); // flies under the products
        // k = the tile's 256 pixels, 32 per MFMA
#pragma unroll 2
        for (int ks = 0; ks < 8; ks++) {
            const sh8 a = *reinterpret_cast<const sh8 *>(dzt + (mt * 16 + n) * kWgD + ks * 32 + kq8);
            const bf16_t *xr = xt + (nt * 16 + n) * kWgX + (2 * ks + (kq8 >> 4) + dy0) * kWgRow + (kq8 & 15);
#pragma unroll
            for (int d = 0; d < NDY; d++) {
                if (dy0 + d > 2) break; // wave-uniform
                const uint4 w = *reinterpret_cast<const uint4 *>(xr + d * kWgRow);
                const unsigned w4 = *reinterpret_cast<const unsigned *>(xr + d * kWgRow + 8);
                const uint4 b1 = uint4{(w.x >> 16) | (w.y << 16), (w.y >> 16) | (w.z << 16),
                                       (w.z >> 16) | (w.w << 16), (w.w >> 16) | (w4 << 16)};
                const uint4 b2 = uint4{w.y, w.z, w.w, w4};
                acc[3 * d] = mfma_k32(a, __builtin_bit_cast(sh8, w), acc[3 * d]);
                acc[3 * d + 1] = mfma_k32(a, __builtin_bit_cast(sh8, b1), acc[3 * d + 1]);
                acc[3 * d + 2] = mfma_k32(a, __builtin_bit_cast(sh8, b2), acc[3 * d + 2]);
            }
        }
        // bias gradient: wave w sums pixels 64 w .. 64 w + 63 of channel `lane`,
        // tile by tile (one chain over all tiles would round each pixel to the
        // running total)
        if (lane < COUT) {
            float part = 0.0f;
#pragma unroll
            for (int p = 0; p < 64; p += 8) {
                const uint4 w = *reinterpret_cast<const uint4 *>(dzt + lane * kWgD + 64 * wave + p);
                const unsigned e[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    part += bf2f((bf16_t)(e[i] & 0xffffu));
                    part += bf2f((bf16_t)(e[i] >> 16));
                }
            }
            sum += part;
        }
    }
    // D[m = co][n = ci]: lane holds co = mt*16 + kq + e, ci = nt*16 + n
#pragma unroll
    for (int i = 0; i < 3 * NDY; i++) {
        const int tap = 3 * dy0 + i;
        if (tap < 9)
            *reinterpret_cast<float4 *>(dst + (tap * CIN + nt * 16 + n) * COUT + mt * 16 + kq) =
                float4{acc[i][0], acc[i][1], acc[i][2], acc[i][3]};
    }
    // the four waves' bias sums in wave order
    if (lane < COUT) bsum[wave * 32 + lane] = sum;
    __syncthreads();
    if (threadIdx.x < COUT)
        dst[9 * CIN * COUT + threadIdx.x] =
            ((bsum[threadIdx.x] + bsum[32 + threadIdx.x]) + bsum[64 + threadIdx.x]) + bsum[96 + threadIdx.x];
}

// grid: (workgroups of a layer, 4 layers)
__global__ void __launch_bounds__(kBlock)
sur_conv_wgrad(SurLayers ly, float *__restrict__ part, int H, int W, int ntile)
{
    __shared__ __align__(16) bf16_t xt[32 * kWgX];
    __shared__ __align__(16) bf16_t dzt[32 * kWgD];
    __shared__ float bsum[4 * 32];
    const int l = blockIdx.y;
    float *dst = part + ((long)l * gridDim.x + blockIdx.x) * kSurSlot;
    if (l == 3) wgrad_tiles<16>(ly.x[3], ly.dz[3], dst, H, W, ntile, xt, dzt, bsum);
    else wgrad_tiles<32>(ly.x[l], ly.dz[l], dst, H, W, ntile, xt, dzt, bsum);
}

struct SurAdam {
    float lr, b1, b2, eps, c1, c2;
};

// bf16 copies of weight v at canonical place e (tap, ci, co) of layer l:
// forward [tap][co][ci], backward-data [tap][ci][co] with the tap flipped (the
// transposed convolution)
__device__ __forceinline__ void put_weight(const SurLayers &ly, int l, int e, float v)
{
    const int lc = l == 3 ? 4 : 5, cout = 1 << lc; // 32 input channels in every layer
    const int co = e & (cout - 1), ci = (e >> lc) & 31, tap = e >> (lc + 5);
    const bf16_t h = f2bf(v);
    ly.wt[l][(tap * cout + co) * 32 + ci] = h;
    ly.wbt[l][((8 - tap) * 32 + ci) * cout + co] = h;
}

__global__ void __launch_bounds__(kBlock)
sur_prep_weights(SurLayers ly, const float *__restrict__ params)
{
    const int l = blockIdx.y, e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e < 9 * 32 * (l == 3 ? 16 : 32)) put_weight(ly, l, e, params[ly.off[l] + e]);
}

// grad[e] = sum over the workgroups of part[.][e] in a fixed order, with the
// partial gradients split over the 16 waves of a workgroup: wave g sums
// [g per, (g + 1) per) for 64 consecutive elements, then wave 0 adds the 16
// partial sums in wave order (deterministic; one serial chain per element
// over all tiles was latency-bound: 98 us per layer at 256 tiles).  All
// layers in one launch (grid.y), and with UPDATE the Adam step (Kingma & Ba
// 2015) on the FP32 master parameters and the new bf16 weights follow in the
// same thread: nine launches of 30 us at 256x256 before, one of 4.8 us so.
constexpr int kRedGroups = 16;
template <int UPDATE>
__global__ void __launch_bounds__(64 * kRedGroups)
sur_reduce_update(SurLayers ly, const float *__restrict__ part, int nparts, float *__restrict__ grad,
                  float *__restrict__ w, float *__restrict__ m1, float *__restrict__ m2, SurAdam ad)
{
    __shared__ float ps[kRedGroups][64];
    const int lane = threadIdx.x & 63, grp = threadIdx.x >> 6;
    const int l = blockIdx.y, e = blockIdx.x * 64 + lane, len = ly.off[l + 1] - ly.off[l];
    if ((int)blockIdx.x * 64 >= len) return; // the whole workgroup
    const int per = (nparts + kRedGroups - 1) / kRedGroups;
    const int t0 = grp * per, t1 = min(nparts, t0 + per);
    const float *src = part + (long)l * nparts * kSurSlot;
    float s = 0.0f;
    if (e < len) {
#pragma unroll 8
        for (int t = t0; t < t1; t++) s += src[(long)t * kSurSlot + e];
    }
    ps[grp][lane] = s;
    __syncthreads();
    if (grp == 0 && e < len) {
        float r = 0.0f;
        for (int g = 0; g < kRedGroups; g++) r += ps[g][lane];
        const int o = ly.off[l] + e;
        grad[o] = r;
        if (UPDATE) {
            const float a = ad.b1 * m1[o] + (1.0f - ad.b1) * r;
            const float b = ad.b2 * m2[o] + (1.0f - ad.b2) * r * r;
            m1[o] = a;
            m2[o] = b;
            float v = w[o];
            v -= ad.lr * (a / ad.c1) / (sqrtf(b / ad.c2) + ad.eps);
            w[o] = v;
            if (e < 9 * 32 * (l == 3 ? 16 : 32)) put_weight(ly, l, e, v);
        }
    }
}

__device__ __forceinline__ float target_at(const SurGeom &s, const float *__restrict__ bfine,
                                           const float *__restrict__ bc,
                                           const float *__restrict__ tgt_direct, long p, int y, int x,
                                           int ch)
{
    const int nused = 3 * s.n0;
    if (tgt_direct) return tgt_direct[p * nused + ch];
    const int c = ch / s.n0, i = ch - c * s.n0;
    const long I = ((long)i * s.n1 + y) * s.n2 + x;
    return (bfine[c * s.N + I] - bc[c * s.Nc + coarse_of(s, i, y, x)]) * s.inv_mu0ms;
}

// per-block partial sums of target^2 (16 pixels of 16 channels each).  The scale
// of the gradients follows from their total, and a gradient rounds to bf16: one
// unit in the total's last place already moves the weight gradients by 1e-5,
// so the order of the sum is kept.  64 pixels of 4 channels per wave, turned
// through LDS to the same order, took 6.5 us at 256x256x4 against 5.6 us.
__global__ void __launch_bounds__(kBlock)
sur_target_sq(SurGeom s, const float *__restrict__ bfine, const float *__restrict__ bc,
              const float *__restrict__ tgt_direct, float *__restrict__ part)
{
    __shared__ float red[kBlock / 64];
    const long P = (long)s.n1 * s.n2;
    const long t = (long)blockIdx.x * blockDim.x + threadIdx.x; // pixel * 16 + channel
    float v2 = 0.0f;
    if (t < P * 16 && (int)(t & 15) < 3 * s.n0) {
        const long p = t >> 4;
        const int y = (int)((unsigned)p / (unsigned)s.n2), x = (int)p - y * s.n2; // P < 2^31
        const float v = target_at(s, bfine, bc, tgt_direct, p, y, x, (int)(t & 15));
        v2 = v * v;
    }
    v2 = wave_sum(v2);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v2;
    __syncthreads();
    if (threadIdx.x == 0) {
        float s2 = 0.0f;
        for (int w = 0; w < kBlock / 64; w++) s2 += red[w];
        part[blockIdx.x] = s2;
    }
}

// out[0] = sum of the n values of part in a fixed order: thread i of one
// workgroup sums i, i + 1024, ..., then a tree in LDS (deterministic).
__global__ void __launch_bounds__(1024)
sur_reduce_one(const float *__restrict__ part, int n, float *__restrict__ out)
{
    __shared__ float ps[1024];
    float s = 0.0f;
    for (int t = threadIdx.x; t < n; t += 1024) s += part[t];
    ps[threadIdx.x] = s;
    __syncthreads();
    for (int h = 512; h > 0; h >>= 1) {
        if (threadIdx.x < h) ps[threadIdx.x] += ps[threadIdx.x + h];
        __syncthreads();
    }
    if (threadIdx.x == 0) out[0] = ps[0];
}

// d loss / d out = 2 (out - target) / sum target^2 (bf16), *t2 = sum target^2;
// the per-block partial sums of the squared error, in 64 bits, go to host_part
// (pinned memory, at most kLossBlocks; a copy to pageable memory took 10 us), sum
// target^2 behind them.  A wave takes 64 consecutive pixels and 4 of the 16
// channels, so the target's planes are read in whole lines: 9.7 us with one
// channel per thread, 6.6 us so at 256x256x4.
constexpr int kLossBlocks = 1024;
__global__ void __launch_bounds__(kBlock)
sur_loss(SurGeom s, const float *__restrict__ out, const float *__restrict__ bfine,
         const float *__restrict__ bc, const float *__restrict__ tgt_direct,
         const float *__restrict__ t2, bf16_t *__restrict__ gout, double *__restrict__ host_part)
{
    __shared__ double red[kBlock / 64];
    const long P = (long)s.n1 * s.n2;
    const int ch0 = 4 * __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), nused = 3 * s.n0;
    const float gscale = 2.0f / fmaxf(*t2, 1e-30f);
    double e2 = 0.0;
    for (long p = (long)blockIdx.x * 64 + (threadIdx.x & 63); p < P; p += (long)gridDim.x * 64) {
        const int y = (int)((unsigned)p / (unsigned)s.n2), x = (int)p - y * s.n2;
        const float4 o = *reinterpret_cast<const float4 *>(out + p * 16 + ch0);
        const float ov[4] = {o.x, o.y, o.z, o.w};
        bf16_t g[4] = {0, 0, 0, 0};
#pragma unroll
        for (int e = 0; e < 4; e++)
            if (ch0 + e < nused) {
                const float d = ov[e] - target_at(s, bfine, bc, tgt_direct, p, y, x, ch0 + e);
                e2 += (double)d * (double)d;
                g[e] = f2bf(gscale * d);
            }
        *reinterpret_cast<uint2 *>(gout + p * 16 + ch0) =
            uint2{(unsigned)g[0] | ((unsigned)g[1] << 16), (unsigned)g[2] | ((unsigned)g[3] << 16)};
    }
    e2 = wave_sum(e2);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = e2;
    __syncthreads();
    if (threadIdx.x == 0) {
        double s2 = 0.0;
        for (int w = 0; w < kBlock / 64; w++) s2 += red[w];
        host_part[blockIdx.x] = s2;
        if (blockIdx.x == 0) host_part[gridDim.x] = *t2;
    }
}

// H_demag (A/m) = upsampled coarse B / mu0 + Ms * out, into the field epilogue;
// optionally also out_scale * H_demag into hd_out (1: A/m, mu0: tesla)
template <int MODE>
__global__ void __launch_bounds__(kBlock)
sur_epilogue(DemagGeom g, SurGeom s, FieldParams fp, EpilogueIO io, const float *__restrict__ out,
             const float *__restrict__ bc, float *__restrict__ hd_out, float out_scale)
{
    const long I = (long)blockIdx.x * blockDim.x + threadIdx.x;
    float errmax = 0.0f;
    if (I < s.N) {
        const int k = (int)(I % s.n2), j = (int)((I / s.n2) % s.n1), i = (int)(I / ((long)s.n2 * s.n1));
        const long p = (long)j * s.n2 + k;
        const long ic = coarse_of(s, i, j, k);
        float hd[3];
#pragma unroll
        for (int c = 0; c < 3; c++)
            hd[c] = bc[c * s.Nc + ic] * (1.0f / (float)kMu0) + s.msat * out[p * 16 + c * s.n0 + i];
        if (hd_out) {
#pragma unroll
            for (int c = 0; c < 3; c++) hd_out[c * s.N + I] = out_scale * hd[c];
        }
        if (MODE != EPI_B) cell_epilogue<MODE>(g, fp, io, I, i, j, k, hd, errmax);
    }
    if (MODE == EPI_CORR) block_max_slot(errmax, io.err, io.err_mask);
}

// sum (a - b)^2 and sum c^2 per block (FP64 partials)
__global__ void __launch_bounds__(kBlock)
sur_diff_norm(const float *__restrict__ a, const float *__restrict__ b, const float *__restrict__ c,
              long n, double *__restrict__ part)
{
    __shared__ double red[2][kBlock / 64];
    double d2 = 0.0, b2 = 0.0;
    for (long t = (long)blockIdx.x * blockDim.x + threadIdx.x; t < n; t += (long)gridDim.x * blockDim.x) {
        const double d = (double)a[t] - (double)b[t];
        d2 += d * d;
        b2 += (double)c[t] * (double)c[t];
    }
    for (int o = 32; o > 0; o >>= 1) {
        d2 += __shfl_down(d2, o);
        b2 += __shfl_down(b2, o);
    }
    if ((threadIdx.x & 63) == 0) {
        red[0][threadIdx.x >> 6] = d2;
        red[1][threadIdx.x >> 6] = b2;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        double x = 0.0, y = 0.0;
        for (int w = 0; w < kBlock / 64; w++) {
            x += red[0][w];
            y += red[1][w];
        }
        part[2 * blockIdx.x] = x;
        part[2 * blockIdx.x + 1] = y;
    }
}

} // namespace mmx

// ------------------------------------------------------------ host object

struct mmx_surrogate {
    mmx_sim *sim = nullptr;
    mmx::SurGeom s{};
    int H = 0, W = 0;
    long P = 0;
    mmx_demag_plan *cplan = nullptr;
    float *mc = nullptr, *bc = nullptr, *bfine = nullptr, *hd = nullptr;
    mmx::bf16_t *x0 = nullptr, *act[3] = {}, *gout = nullptr, *dz[3] = {};
    float *out = nullptr, *tgt = nullptr, *part = nullptr, *loss_part = nullptr;
    double *loss_host = nullptr; // pinned: partial sums of the loss, then sum target^2
    double *norm_part = nullptr;
    float *params = nullptr, *grads = nullptr, *adam_m = nullptr, *adam_v = nullptr;
    mmx::bf16_t *wt[4] = {}, *wbt[4] = {};
    int np = 0, off_w[4] = {}, off_b[4] = {};
    long adam_t = 0;
};

namespace mmx {
namespace {

template <typename T> int dalloc(T **p, size_t count)
{
    if (hipMalloc(p, sizeof(T) * count) != hipSuccess) {
        set_error("surrogate: cannot allocate %zu bytes", sizeof(T) * count);
        return MMX_ERR_NOMEM;
    }
    return MMX_OK;
}

void sur_free(mmx_surrogate *S)
{
    void *ptrs[] = {S->mc, S->bc, S->bfine, S->hd, S->x0, S->act[0], S->act[1], S->act[2],
                    S->gout, S->dz[0], S->dz[1], S->dz[2], S->out, S->tgt, S->part, S->loss_part,
                    S->norm_part, S->params, S->grads, S->adam_m, S->adam_v, S->wt[0], S->wt[1],
                    S->wt[2], S->wt[3], S->wbt[0], S->wbt[1], S->wbt[2], S->wbt[3]};
    for (void *p : ptrs) (void)hipFree(p);
    if (S->loss_host) (void)hipHostFree(S->loss_host);
    if (S->cplan) plan_destroy(S->cplan);
}

SurLayers sur_layers(const mmx_surrogate *S)
{
    SurLayers ly{};
    for (int l = 0; l < 4; l++) {
        ly.x[l] = l == 0 ? S->x0 : S->act[l - 1];
        ly.dz[l] = l == 3 ? S->gout : S->dz[l];
        ly.wt[l] = S->wt[l];
        ly.wbt[l] = S->wbt[l];
        ly.off[l] = S->off_w[l];
    }
    ly.off[4] = S->np;
    return ly;
}

int prep_weights(mmx_surrogate *S, hipStream_t st)
{
    sur_prep_weights<<<dim3(div_up(9 * 32 * 32, kBlock), 4), dim3(kBlock), 0, st>>>(sur_layers(S),
                                                                                    S->params);
    MMX_CHECK_LAUNCH();
    return MMX_OK;
}

// the net on the packed input S->x0, formed from (m, coarse B) first where m is given
int net_forward(mmx_surrogate *S, const float *m, hipStream_t st)
{
    const dim3 grid(S->W / 16, S->H / 8), blk(kBlock);
    const float *b[4] = {S->params + S->off_b[0], S->params + S->off_b[1], S->params + S->off_b[2],
                         S->params + S->off_b[3]};
    if (m)
        sur_pack<<<dim3((unsigned)div_up(S->P, 64)), dim3(kBlock), 0, st>>>(S->s, m, S->bc, S->x0);
    sur_conv<32, 32, CE_RELU_BF16><<<grid, blk, 0, st>>>(S->x0, S->wt[0], b[0], nullptr, S->act[0], S->H,
                                                         S->W);
    sur_conv<32, 32, CE_RELU_BF16><<<grid, blk, 0, st>>>(S->act[0], S->wt[1], b[1], nullptr, S->act[1],
                                                         S->H, S->W);
    sur_conv<32, 32, CE_RELU_BF16><<<grid, blk, 0, st>>>(S->act[1], S->wt[2], b[2], nullptr, S->act[2],
                                                         S->H, S->W);
    sur_conv<32, 16, CE_LINEAR_F32><<<grid, blk, 0, st>>>(S->act[2], S->wt[3], b[3], nullptr, S->out,
                                                          S->H, S->W);
    MMX_CHECK_LAUNCH();
    return MMX_OK;
}

// workgroups of the loss, partial gradients of a layer
int loss_blocks(long P) { return (int)std::min<long>(div_up(P, 64), kLossBlocks); }
int grad_parts(int H, int W) { return std::min((H / 16) * (W / 16), kSurParts); }

// loss (given the target: exact fine B + coarse B, or a direct target),
// backward, gradients into S->grads and, for lr > 0, the Adam step;
// *loss = mean squared error
int net_backward(mmx_surrogate *S, const float *tgt_direct, float lr, double *loss, hipStream_t st)
{
    const int nlb = loss_blocks(S->P);
    const int ntp = (int)(S->P / 16); // partial sums of target^2, their total behind them
    float *t2 = S->loss_part + ntp;
    sur_target_sq<<<dim3(ntp), dim3(kBlock), 0, st>>>(S->s, S->bfine, S->bc, tgt_direct, S->loss_part);
    sur_reduce_one<<<dim3(1), dim3(1024), 0, st>>>(S->loss_part, ntp, t2);
    sur_loss<<<dim3(nlb), dim3(kBlock), 0, st>>>(S->s, S->out, S->bfine, S->bc, tgt_direct, t2,
                                                 S->gout, S->loss_host);
    const dim3 grid(S->W / 16, S->H / 8), blk(kBlock);
    sur_conv<16, 32, CE_MASK_BF16><<<grid, blk, 0, st>>>(S->gout, S->wbt[3], nullptr, S->act[2], S->dz[2],
                                                         S->H, S->W);
    for (int l = 2; l > 0; l--)
        sur_conv<32, 32, CE_MASK_BF16><<<grid, blk, 0, st>>>(S->dz[l], S->wbt[l], nullptr, S->act[l - 1],
                                                             S->dz[l - 1], S->H, S->W);
    // weight gradients of all layers from the kept inputs and output gradients
    const SurLayers ly = sur_layers(S);
    const int ntile = (S->W / 16) * (S->H / 16), nparts = grad_parts(S->H, S->W);
    sur_conv_wgrad<<<dim3(nparts, 4), blk, 0, st>>>(ly, S->part, S->H, S->W, ntile);
    const dim3 rgrid(div_up(kSurSlot, 64), 4), rblk(64 * kRedGroups);
    if (lr > 0) {
        S->adam_t++;
        SurAdam ad{lr, 0.9f, 0.999f, 1e-8f, 0.0f, 0.0f};
        ad.c1 = 1.0f - (float)std::pow(0.9, (double)S->adam_t);
        ad.c2 = 1.0f - (float)std::pow(0.999, (double)S->adam_t);
        sur_reduce_update<1><<<rgrid, rblk, 0, st>>>(ly, S->part, nparts, S->grads, S->params, S->adam_m,
                                                     S->adam_v, ad);
    } else {
        sur_reduce_update<0><<<rgrid, rblk, 0, st>>>(ly, S->part, nparts, S->grads, S->params, S->adam_m,
                                                     S->adam_v, SurAdam{});
    }
    MMX_CHECK_LAUNCH();
    if (loss) {
        MMX_HIP(hipStreamSynchronize(st));
        double sum = 0.0;
        for (int b = 0; b < nlb; b++) sum += S->loss_host[b];
        const double t2 = S->loss_host[nlb];
        *loss = t2 > 0 ? sum / t2 : 0.0;
    }
    return MMX_OK;
}

// coarse m (optionally from the RK predictor) and coarse B
int coarse_field(mmx_surrogate *S, const float *m, const float *tau0, float h, float *mpred,
                 hipStream_t st)
{
    const int nb = (int)div_up(S->s.Nc, kBlock);
    const float *map = S->sim->msat_map;
    if (tau0)
        sur_coarsen<1><<<dim3(nb), dim3(kBlock), 0, st>>>(S->s, m, tau0, h, map, mpred, S->mc);
    else
        sur_coarsen<0><<<dim3(nb), dim3(kBlock), 0, st>>>(S->s, m, nullptr, 0.0f, map, nullptr, S->mc);
    MMX_CHECK_LAUNCH();
    const long Nc = S->s.Nc;
    return mmx_demag_update_b(S->cplan, S->bc, S->bc + Nc, S->bc + 2 * Nc, S->mc, S->mc + Nc,
                              S->mc + 2 * Nc, nullptr, (float)S->sim->msat, st);
}

} // namespace

// Surrogate field evaluation at m (or at the predictor of m0 when tau0 is
// given): H_demag estimate into the epilogue of MODE.  Used by sim.cpp.
int surrogate_eval(mmx_surrogate *S, int mode, const float *m0, const float *tau0, float h,
                   float *mpred, const FieldParams &fp, const EpilogueIO &io, float *hd_out,
                   hipStream_t st)
{
    const float *m = tau0 ? mpred : m0;
    MMX_TRY(coarse_field(S, m0, tau0, h, mpred, st));
    MMX_TRY(net_forward(S, m, st));
    const DemagGeom &g = S->sim->plan->impl.g;
    const int nb = (int)div_up(S->s.N, kBlock);
    switch (mode) {
    case EPI_B: sur_epilogue<EPI_B><<<dim3(nb), dim3(kBlock), 0, st>>>(g, S->s, fp, io, S->out, S->bc, hd_out, 1.0f); break;
    case EPI_HEFF: sur_epilogue<EPI_HEFF><<<dim3(nb), dim3(kBlock), 0, st>>>(g, S->s, fp, io, S->out, S->bc, hd_out, 1.0f); break;
    case EPI_TAU0: sur_epilogue<EPI_TAU0><<<dim3(nb), dim3(kBlock), 0, st>>>(g, S->s, fp, io, S->out, S->bc, hd_out, 1.0f); break;
    default: sur_epilogue<EPI_CORR><<<dim3(nb), dim3(kBlock), 0, st>>>(g, S->s, fp, io, S->out, S->bc, hd_out, 1.0f); break;
    }
    MMX_CHECK_LAUNCH();
    return MMX_OK;
}

// ||a - b|| / ||c|| over n floats (L2; synchronises)
int surrogate_rel_l2(mmx_surrogate *S, const float *a, const float *b, const float *c, long n,
                     hipStream_t st, double *rel)
{
    const int nb = 512;
    sur_diff_norm<<<dim3(nb), dim3(kBlock), 0, st>>>(a, b, c, n, S->norm_part);
    MMX_CHECK_LAUNCH();
    std::vector<double> h(2 * nb);
    MMX_HIP(hipMemcpyAsync(h.data(), S->norm_part, sizeof(double) * 2 * nb, hipMemcpyDeviceToHost, st));
    MMX_HIP(hipStreamSynchronize(st));
    double d2 = 0.0, b2 = 0.0;
    for (int i = 0; i < nb; i++) {
        d2 += h[2 * i];
        b2 += h[2 * i + 1];
    }
    *rel = b2 > 0 ? std::sqrt(d2 / b2) : 0.0;
    return MMX_OK;
}

float *surrogate_hd_buffer(mmx_surrogate *S) { return S->hd; }

} // namespace mmx

using namespace mmx;

extern "C" {

int mmx_surrogate_create(mmx_surrogate **sur, mmx_sim *sim, unsigned long long seed)
{
    MMX_REQUIRE(sur && sim, MMX_ERR_ARG, "mmx_surrogate_create: NULL argument");
    MMX_TRY(sim_prepare(sim));
    const int n0 = sim->n[0], n1 = sim->n[1], n2 = sim->n[2];
    MMX_REQUIRE(n0 >= 1 && n0 <= 5 && n1 % 16 == 0 && n2 % 16 == 0, MMX_ERR_SIZE,
                "surrogate: needs 1 <= n0 <= 5 and n1, n2 multiples of 16 (got %d %d %d)", n0, n1, n2);
    MMX_REQUIRE(!sim->pbc[0] && !sim->pbc[1] && !sim->pbc[2], MMX_ERR_ARG,
                "surrogate: periodic grids are not supported");
    mmx_surrogate *S = new mmx_surrogate();
    S->sim = sim;
    SurGeom &s = S->s;
    s.n0 = n0; s.n1 = n1; s.n2 = n2;
    s.f0 = 1; // the layers are kept
    s.c0 = n0 / s.f0; s.c1 = n1 / 2; s.c2 = n2 / 2;
    s.N = (long)n0 * n1 * n2;
    s.Nc = (long)s.c0 * s.c1 * s.c2;
    s.msat = (float)sim->msat;
    s.inv_mu0ms = (float)(1.0 / (kMu0 * sim->msat));
    S->H = n1;
    S->W = n2;
    S->P = (long)n1 * n2;
    int off = 0;
    for (int l = 0; l < 4; l++) {
        S->off_w[l] = off;
        off += 9 * kSurCh[l] * kSurCh[l + 1];
        S->off_b[l] = off;
        off += kSurCh[l + 1];
    }
    S->np = off;
    const double ccell[3] = {sim->cell[0] * s.f0, sim->cell[1] * 2, sim->cell[2] * 2};
    const int zero[3] = {0, 0, 0};
    int rc = plan_create(&S->cplan, s.c0, s.c1, s.c2, ccell, zero, sim->kernel_type, sim->accuracy);
    const long P = S->P;
    if (rc == MMX_OK) rc = dalloc(&S->mc, 3 * s.Nc);
    if (rc == MMX_OK) rc = dalloc(&S->bc, 3 * s.Nc);
    if (rc == MMX_OK) rc = dalloc(&S->bfine, 3 * s.N);
    if (rc == MMX_OK) rc = dalloc(&S->hd, 3 * s.N);
    if (rc == MMX_OK) rc = dalloc(&S->x0, P * 32);
    for (int l = 0; l < 3 && rc == MMX_OK; l++) rc = dalloc(&S->act[l], P * 32);
    for (int l = 0; l < 3 && rc == MMX_OK; l++) rc = dalloc(&S->dz[l], P * 32);
    if (rc == MMX_OK) rc = dalloc(&S->gout, P * 16);
    if (rc == MMX_OK) rc = dalloc(&S->out, P * 16);
    if (rc == MMX_OK) rc = dalloc(&S->tgt, P * 3 * n0);
    if (rc == MMX_OK) rc = dalloc(&S->part, (size_t)4 * grad_parts(n1, n2) * kSurSlot);
    if (rc == MMX_OK) rc = dalloc(&S->loss_part, P / 16 + 1);
    if (rc == MMX_OK && hipHostMalloc(&S->loss_host, sizeof(double) * (loss_blocks(P) + 1)) != hipSuccess) {
        set_error("surrogate: cannot allocate pinned memory");
        rc = MMX_ERR_NOMEM;
    }
    if (rc == MMX_OK) rc = dalloc(&S->norm_part, 2 * 512);
    if (rc == MMX_OK) rc = dalloc(&S->params, S->np);
    if (rc == MMX_OK) rc = dalloc(&S->grads, S->np);
    if (rc == MMX_OK) rc = dalloc(&S->adam_m, S->np);
    if (rc == MMX_OK) rc = dalloc(&S->adam_v, S->np);
    for (int l = 0; l < 4 && rc == MMX_OK; l++) rc = dalloc(&S->wt[l], 9 * kSurCh[l] * kSurCh[l + 1]);
    for (int l = 0; l < 4 && rc == MMX_OK; l++) rc = dalloc(&S->wbt[l], 9 * kSurCh[l] * kSurCh[l + 1]);
    if (rc == MMX_OK) {
        // He initialisation (first layer over its 6 n0 + 2 used inputs), a
        // small last layer, zero biases
        std::vector<float> w(S->np, 0.0f);
        std::mt19937_64 gen(seed);
        std::normal_distribution<double> nd(0.0, 1.0);
        for (int l = 0; l < 4; l++) {
            const int fan = 9 * (l == 0 ? 6 * n0 + 2 : kSurCh[l]);
            const double sd = std::sqrt(2.0 / fan) * (l == 3 ? 0.1 : 1.0);
            for (int e = 0; e < 9 * kSurCh[l] * kSurCh[l + 1]; e++) w[S->off_w[l] + e] = (float)(sd * nd(gen));
        }
        if (hipMemcpy(S->params, w.data(), sizeof(float) * S->np, hipMemcpyHostToDevice) != hipSuccess ||
            hipMemset(S->adam_m, 0, sizeof(float) * S->np) != hipSuccess ||
            hipMemset(S->adam_v, 0, sizeof(float) * S->np) != hipSuccess ||
            hipMemset(S->grads, 0, sizeof(float) * S->np) != hipSuccess) {
            set_error("surrogate: initialisation copy failed");
            rc = MMX_ERR_HIP;
        }
    }
    if (rc == MMX_OK) rc = prep_weights(S, sim->st);
    if (rc == MMX_OK && hipStreamSynchronize(sim->st) != hipSuccess) rc = MMX_ERR_HIP;
    if (rc != MMX_OK) {
        sur_free(S);
        delete S;
        return rc;
    }
    *sur = S;
    return MMX_OK;
}

int mmx_surrogate_destroy(mmx_surrogate *sur)
{
    if (!sur) return MMX_OK;
    if (sur->sim && sur->sim->st) (void)hipStreamSynchronize(sur->sim->st);
    sur_free(sur);
    delete sur;
    return MMX_OK;
}

int mmx_surrogate_num_params(const mmx_surrogate *sur, int *count)
{
    MMX_REQUIRE(sur && count, MMX_ERR_ARG, "mmx_surrogate_num_params: NULL argument");
    *count = sur->np;
    return MMX_OK;
}

int mmx_surrogate_get_params(mmx_surrogate *sur, float *host, int count)
{
    MMX_REQUIRE(sur && host && count == sur->np, MMX_ERR_ARG, "mmx_surrogate_get_params: bad arguments");
    MMX_HIP(hipStreamSynchronize(sur->sim->st));
    MMX_HIP(hipMemcpy(host, sur->params, sizeof(float) * count, hipMemcpyDeviceToHost));
    return MMX_OK;
}

int mmx_surrogate_set_params(mmx_surrogate *sur, const float *host, int count)
{
    MMX_REQUIRE(sur && host && count == sur->np, MMX_ERR_ARG, "mmx_surrogate_set_params: bad arguments");
    MMX_HIP(hipStreamSynchronize(sur->sim->st));
    MMX_HIP(hipMemcpy(sur->params, host, sizeof(float) * count, hipMemcpyHostToDevice));
    sur->adam_t = 0;
    MMX_HIP(hipMemset(sur->adam_m, 0, sizeof(float) * sur->np));
    MMX_HIP(hipMemset(sur->adam_v, 0, sizeof(float) * sur->np));
    MMX_TRY(prep_weights(sur, sur->sim->st));
    MMX_HIP(hipStreamSynchronize(sur->sim->st));
    return MMX_OK;
}

int mmx_surrogate_get_grads(mmx_surrogate *sur, float *host, int count)
{
    MMX_REQUIRE(sur && host && count == sur->np, MMX_ERR_ARG, "mmx_surrogate_get_grads: bad arguments");
    MMX_HIP(hipStreamSynchronize(sur->sim->st));
    MMX_HIP(hipMemcpy(host, sur->grads, sizeof(float) * count, hipMemcpyDeviceToHost));
    return MMX_OK;
}

int mmx_surrogate_net(mmx_surrogate *sur, const float *x_host, const float *tgt_host, float *out_host,
                      double *loss)
{
    MMX_REQUIRE(sur && x_host && out_host, MMX_ERR_ARG, "mmx_surrogate_net: NULL argument");
    mmx_surrogate *S = sur;
    hipStream_t st = S->sim->st;
    const long P = S->P;
    // the input rounded to bf16 on the host side of the copy (same rounding)
    std::vector<unsigned short> xb(P * 32);
    for (long e = 0; e < P * 32; e++) {
        unsigned int u;
        std::memcpy(&u, &x_host[e], 4);
        if ((u & 0x7f800000u) == 0x7f800000u) xb[e] = (unsigned short)(u >> 16);
        else xb[e] = (unsigned short)((u + 0x7fffu + ((u >> 16) & 1u)) >> 16);
    }
    MMX_HIP(hipMemcpyAsync(S->x0, xb.data(), sizeof(unsigned short) * P * 32, hipMemcpyHostToDevice, st));
    MMX_TRY(net_forward(S, nullptr, st));
    if (tgt_host) {
        MMX_HIP(hipMemcpyAsync(S->tgt, tgt_host, sizeof(float) * P * 3 * S->s.n0, hipMemcpyHostToDevice, st));
        MMX_TRY(net_backward(S, S->tgt, 0.0f, loss, st));
    }
    MMX_HIP(hipMemcpyAsync(out_host, S->out, sizeof(float) * P * 16, hipMemcpyDeviceToHost, st));
    MMX_HIP(hipStreamSynchronize(st));
    return MMX_OK;
}

int mmx_surrogate_train_step(mmx_surrogate *sur, const float *m_dev, float lr, double *loss)
{
    MMX_REQUIRE(sur && m_dev && lr >= 0, MMX_ERR_ARG, "mmx_surrogate_train_step: bad arguments");
    mmx_surrogate *S = sur;
    mmx_sim *x = S->sim;
    MMX_REQUIRE(!x->msat_map, MMX_ERR_ARG, "surrogate: an Msat map is not supported");
    hipStream_t st = x->st;
    const long N = S->s.N;
    // target: the exact fine field; input: the coarse field
    MMX_TRY(mmx_demag_update_b(x->plan, S->bfine, S->bfine + N, S->bfine + 2 * N, m_dev, m_dev + N,
                               m_dev + 2 * N, nullptr, (float)x->msat, st));
    MMX_TRY(coarse_field(S, m_dev, nullptr, 0.0f, nullptr, st));
    MMX_TRY(net_forward(S, m_dev, st));
    return net_backward(S, nullptr, lr, loss, st);
}

int mmx_surrogate_predict_b(mmx_surrogate *sur, const float *m_dev, float *b_dev, int coarse_only)
{
    MMX_REQUIRE(sur && m_dev && b_dev, MMX_ERR_ARG, "mmx_surrogate_predict_b: NULL argument");
    mmx_surrogate *S = sur;
    hipStream_t st = S->sim->st;
    MMX_TRY(coarse_field(S, m_dev, nullptr, 0.0f, nullptr, st));
    if (coarse_only) {
        MMX_HIP(hipMemsetAsync(S->out, 0, sizeof(float) * S->P * 16, st));
    } else {
        MMX_TRY(net_forward(S, m_dev, st));
    }
    const DemagGeom &g = S->sim->plan->impl.g;
    const FieldParams fp = sim_field_params(S->sim);
    EpilogueIO io{};
    sur_epilogue<EPI_B><<<dim3((unsigned)div_up(S->s.N, kBlock)), dim3(kBlock), 0, st>>>(
        g, S->s, fp, io, S->out, S->bc, b_dev, (float)kMu0);
    MMX_CHECK_LAUNCH();
    return MMX_OK;
}

} // extern "C"
