// pv_cnn.hip -- the learned pressure preconditioner: a 6-layer 3x3
// convolutional network (3 -> 32 -> 32 -> 32 -> 32 -> 32 -> 1 channels, ReLU
// between layers) with BF16 operands and FP32 accumulation on the CDNA4
// matrix cores, trained on the GPU by the kernels below.
//
// Tensors are NHWC: batch b, row y, column x, channel c fastest.  The image
// side lengths are multiples of 16.  Padding: zero outside rows [0, H);
// columns wrap when px != 0 (the x-periodic domain) and are zero-padded
// otherwise (training crops).
//
// Parameter vector (FP32 master copy, offsets in floats):
//   layer 1   W1[co 32][tap 9][ci 3]            0 ..   863, b1[32] 864 .. 895
//   layer k   Wk[tap 9][co 32][ci 32], bk[32]   896 + (k-2) 9248, k = 2..5
//   layer 6   W6[tap 9][ci 32] + b6             37888 .. 38176
// tap = 3 ky + kx reads input pixel (y + ky - 1, x + kx - 1).
//
// Layers 2..5 run on v_mfma_f32_16x16x16_bf16: a block computes a 16 x 16
// pixel tile for all 32 output channels; wave w owns tile rows 4w .. 4w+3.
// GEMM view per row and tap: D[pixel 16][co 16] += A[pixel][ci 16] B[ci][co].
// Operand lanes (16x16x16): lane l holds A[l % 16][4 (l / 16) + q],
// B[4 (l / 16) + q][l % 16], D[4 (l / 16) + q][l % 16], q = 0..3.
#include <hip/hip_runtime.h>
#include <math.h>
#include "pv_kernels.h"

typedef short v4s __attribute__((ext_vector_type(4)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef unsigned v4u __attribute__((ext_vector_type(4)));
typedef unsigned short bf16;

#define CNN_C 32
#define TILE 16
#define HALO 18
#define PSTR 40   // LDS shorts per pixel (32 channels + 8 pad: spreads lanes over banks)

__device__ __forceinline__ bf16 f2bf(float f)
{
    unsigned u = __float_as_uint(f);
    u += 0x7fffu + ((u >> 16) & 1u);     // round to nearest even (finite inputs)
    return (bf16)(u >> 16);
}
__device__ __forceinline__ float bf2f(bf16 h) { return __uint_as_float(((unsigned)h) << 16); }
__device__ __forceinline__ bool bfpos(bf16 h) { return h != 0 && !(h & 0x8000u); }

__device__ __forceinline__ int wrapx(int x, int W, int px, bool &ok)
{
    if (x >= 0 && x < W) return x;
    if (px) return (x < 0) ? x + W : x - W;
    ok = false;
    return 0;
}

// ---------------------------------------------------------------------------
// layer 1: 3 -> 32, FP32 FMA, ReLU, BF16 out
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(256) k_cnn_l1(const float *__restrict__ in3, const float *__restrict__ prm,
                                               bf16 *__restrict__ out, int H, int W, int px)
{
    __shared__ float w[896];
    for (int k = threadIdx.x; k < 896; k += 256) w[k] = prm[k];
    __syncthreads();
    const int b = blockIdx.y, p = blockIdx.x * 256 + threadIdx.x;
    if (p >= H * W) return;
    const int y = p / W, x = p - y * W;
    float v[27];
#pragma unroll
    for (int t = 0; t < 9; t++) {
        const int yy = y + t / 3 - 1;
        bool ok = (yy >= 0 && yy < H);
        const int xx = wrapx(x + t % 3 - 1, W, px, ok);
#pragma unroll
        for (int c = 0; c < 3; c++) v[3 * t + c] = ok ? in3[(((size_t)b * H + yy) * W + xx) * 3 + c] : 0.0f;
    }
    bf16 o[CNN_C];
#pragma unroll
    for (int co = 0; co < CNN_C; co++) {
        float a = w[864 + co];
#pragma unroll
        for (int k = 0; k < 27; k++) a += w[co * 27 + k] * v[k];
        o[co] = f2bf(fmaxf(a, 0.0f));
    }
    uint4 *dst = (uint4 *)(out + (((size_t)b * H + y) * W + x) * CNN_C);
#pragma unroll
    for (int q = 0; q < 4; q++) {
        uint4 u;
        u.x = o[8 * q + 0] | ((unsigned)o[8 * q + 1] << 16);
        u.y = o[8 * q + 2] | ((unsigned)o[8 * q + 3] << 16);
        u.z = o[8 * q + 4] | ((unsigned)o[8 * q + 5] << 16);
        u.w = o[8 * q + 6] | ((unsigned)o[8 * q + 7] << 16);
        dst[q] = u;
    }
}

// ---------------------------------------------------------------------------
// layers 2..5 (and the input gradient of the backward pass): 32 -> 32 on MFMA.
// wts: BF16 [tap 9][co 32][ci 32].  bias may be null.  With relu the output
// is max(., 0); with mask the output is zeroed where mask <= 0 (ReLU'(a)).
// ---------------------------------------------------------------------------
// A tile of pixels with its halo (18 x 18, 324 pixels of 4 x 16 bytes): every
// load first, from a clamped place, then the LDS stores.  In one loop, each
// load waited for before the next, k_cnn_mid took 11.6 us for 32 crops of 64 x 64
// (10.8 now).
#define HALO_K ((HALO * HALO * 4 + 255) / 256)
struct halo_regs { v4u u[HALO_K]; };
__device__ __forceinline__ void halo_load(const bf16 *__restrict__ in, halo_regs &h, int b, int ty0, int tx0, int H, int W,
                                          int px)
{
#pragma unroll
    for (int k = 0; k < HALO_K; k++) {
        const int idx = min((int)threadIdx.x + k * 256, HALO * HALO * 4 - 1), pix = idx >> 2, ch = idx & 3;
        const int ty = pix / HALO, tx = pix - ty * HALO, gy = ty0 + ty - 1;
        bool ok = (gy >= 0 && gy < H);
        const int gx = wrapx(tx0 + tx - 1, W, px, ok), yc = min(max(gy, 0), H - 1);
        h.u[k] = *(const v4u *)(in + (((size_t)b * H + yc) * W + gx) * CNN_C + ch * 8);
        if (!ok) h.u[k] = (v4u){0, 0, 0, 0};
    }
}
__device__ __forceinline__ void halo_store(const halo_regs &h, bf16 *lds)
{
#pragma unroll
    for (int k = 0; k < HALO_K; k++) {
        const int idx = threadIdx.x + k * 256;
        if (idx < HALO * HALO * 4) *(v4u *)(lds + (idx >> 2) * PSTR + (idx & 3) * 8) = h.u[k];
    }
}
// the tile itself (256 pixels)
struct tile_regs { v4u u[4]; };
__device__ __forceinline__ void tile_load(const bf16 *__restrict__ in, tile_regs &h, int b, int ty0, int tx0, int H, int W)
{
#pragma unroll
    for (int k = 0; k < 4; k++) {
        const int idx = threadIdx.x + k * 256, pix = idx >> 2;
        h.u[k] = *(const v4u *)(in + (((size_t)b * H + ty0 + pix / TILE) * W + tx0 + pix % TILE) * CNN_C + (idx & 3) * 8);
    }
}
__device__ __forceinline__ void tile_store(const tile_regs &h, bf16 *lds)
{
#pragma unroll
    for (int k = 0; k < 4; k++) {
        const int idx = threadIdx.x + k * 256;
        *(v4u *)(lds + (idx >> 2) * PSTR + (idx & 3) * 8) = h.u[k];
    }
}

template <bool RELU, bool MASK>
__global__ void __launch_bounds__(256) k_cnn_mid(const bf16 *__restrict__ in, const bf16 *__restrict__ wts,
                                                const float *__restrict__ bias, bf16 *__restrict__ out,
                                                const bf16 *__restrict__ mask, int H, int W, int px)
{
    __shared__ __attribute__((aligned(16))) bf16 sin[HALO * HALO * PSTR];
    __shared__ __attribute__((aligned(16))) bf16 sw[9 * CNN_C * PSTR];
    const int ntx = W / TILE, b = blockIdx.y;
    const int ty0 = (blockIdx.x / ntx) * TILE, tx0 = (blockIdx.x % ntx) * TILE;
    constexpr int WK = (9 * CNN_C * 4 + 255) / 256;
    halo_regs h;
    v4u wr[WK];
#pragma unroll
    for (int k = 0; k < WK; k++) wr[k] = *(const v4u *)(wts + min((int)threadIdx.x + k * 256, 9 * CNN_C * 4 - 1) * 8);
    halo_load(in, h, b, ty0, tx0, H, W, px);
#pragma unroll
    for (int k = 0; k < WK; k++) {
        const int idx = threadIdx.x + k * 256;
        if (idx < 9 * CNN_C * 4) *(v4u *)(sw + (idx >> 2) * PSTR + (idx & 3) * 8) = wr[k];
    }
    halo_store(h, sin);
    __syncthreads();
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, col = lane & 15, grp = lane >> 4;
    v4f acc[4][2];
#pragma unroll
    for (int r = 0; r < 4; r++) { acc[r][0] = (v4f){0, 0, 0, 0}; acc[r][1] = (v4f){0, 0, 0, 0}; }
#pragma unroll
    for (int tap = 0; tap < 9; tap++) {
        const int ky = tap / 3, kx = tap % 3;
#pragma unroll
        for (int kc = 0; kc < 2; kc++) {
            const int ci = kc * 16 + 4 * grp;
            const v4s b0 = *(const v4s *)(sw + (tap * CNN_C + col) * PSTR + ci);
            const v4s b1 = *(const v4s *)(sw + (tap * CNN_C + 16 + col) * PSTR + ci);
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int row = wv * 4 + r;
                const v4s a = *(const v4s *)(sin + ((row + ky) * HALO + col + kx) * PSTR + ci);
                acc[r][0] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b0, acc[r][0], 0, 0, 0);
                acc[r][1] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b1, acc[r][1], 0, 0, 0);
            }
        }
    }
    __syncthreads();
    // stage the 16 x 16 x 32 output tile in LDS (reusing sin), then store coalesced
    bf16 *so = sin;
#pragma unroll
    for (int r = 0; r < 4; r++)
#pragma unroll
        for (int h = 0; h < 2; h++)
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const int pcol = 4 * grp + q, co = h * 16 + col;
                float v = acc[r][h][q] + (bias ? bias[co] : 0.0f);
                if (RELU) v = fmaxf(v, 0.0f);
                so[((wv * 4 + r) * TILE + pcol) * PSTR + co] = f2bf(v);
            }
    __syncthreads();
    for (int idx = threadIdx.x; idx < TILE * TILE * 4; idx += 256) {
        const int pix = idx >> 2, ch = idx & 3;
        const int gy = ty0 + pix / TILE, gx = tx0 + pix % TILE;
        const size_t g = (((size_t)b * H + gy) * W + gx) * CNN_C + ch * 8;
        uint4 u = *(const uint4 *)(so + pix * PSTR + ch * 8);
        if (MASK) {
            const uint4 m = *(const uint4 *)(mask + g);
            unsigned *pu = &u.x;
            const unsigned *pm = &m.x;
#pragma unroll
            for (int e = 0; e < 4; e++) {
                unsigned lo = bfpos((bf16)(pm[e] & 0xffffu)) ? (pu[e] & 0xffffu) : 0u;
                unsigned hi = bfpos((bf16)(pm[e] >> 16)) ? (pu[e] & 0xffff0000u) : 0u;
                pu[e] = lo | hi;
            }
        }
        *(uint4 *)(out + g) = u;
    }
}

// ---------------------------------------------------------------------------
// layer 6: 32 -> 1, FP32 FMA over BF16 activations; out = bias + sum
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(256) k_cnn_l6(const bf16 *__restrict__ a5, const float *__restrict__ prm,
                                               float *__restrict__ out, int H, int W, int px)
{
    __shared__ float w[289];
    for (int k = threadIdx.x; k < 289; k += 256) w[k] = prm[37888 + k];
    __syncthreads();
    const int b = blockIdx.y, p = blockIdx.x * 256 + threadIdx.x;
    if (p >= H * W) return;
    const int y = p / W, x = p - y * W;
    float a = w[288];
    for (int t = 0; t < 9; t++) {
        const int yy = y + t / 3 - 1;
        bool ok = (yy >= 0 && yy < H);
        const int xx = wrapx(x + t % 3 - 1, W, px, ok);
        if (!ok) continue;
        const uint4 *src = (const uint4 *)(a5 + (((size_t)b * H + yy) * W + xx) * CNN_C);
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const uint4 u = src[q];
            const unsigned e[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
            for (int k = 0; k < 4; k++) {
                a += w[t * 32 + 8 * q + 2 * k] * bf2f((bf16)(e[k] & 0xffffu));
                a += w[t * 32 + 8 * q + 2 * k + 1] * bf2f((bf16)(e[k] >> 16));
            }
        }
    }
    out[(size_t)b * H * W + p] = a;
}

// ---------------------------------------------------------------------------
// backward
// ---------------------------------------------------------------------------
// Loss = sum over valid pixels of (out - t)^2 / nvalid; valid = at least
// `border` pixels from every image edge.  gout = dLoss/dout; per-block loss.
__global__ void __launch_bounds__(256) k_cnn_loss(const float *__restrict__ out, const float *__restrict__ tgt,
                                                 float *__restrict__ gout, float *__restrict__ part, int H, int W,
                                                 int border, float inv_n)
{
    __shared__ float sh[256];
    const int b = blockIdx.y, p = blockIdx.x * 256 + threadIdx.x;
    float l = 0.0f;
    if (p < H * W) {
        const int y = p / W, x = p - y * W;
        const size_t k = (size_t)b * H * W + p;
        const bool ok = y >= border && y < H - border && x >= border && x < W - border;
        const float d = ok ? out[k] - tgt[k] : 0.0f;
        gout[k] = 2.0f * d * inv_n;
        l = d * d * inv_n;
    }
    sh[threadIdx.x] = l;
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
        if (threadIdx.x < s) sh[threadIdx.x] += sh[threadIdx.x + s];
        __syncthreads();
    }
    if (threadIdx.x == 0) part[blockIdx.y * gridDim.x + blockIdx.x] = sh[0];
}

// The backward kernels below walk tiles t = blockIdx.x, blockIdx.x + gridDim.x,
// ... of the batch (b, tile row, tile column), keep their weight gradients in
// accumulators over all of them and write one row of partials a workgroup, in
// the parameter vector's own layout (at most PVK_CNN_ROWS rows, whatever the batch).
struct tile_at {
    int b, ty0, tx0;
};
__device__ __forceinline__ tile_at tile_of(int t, int H, int W)
{
    const int ntx = W / TILE, n = ntx * (H / TILE), b = t / n, r = t - b * n;
    return {b, (r / ntx) * TILE, (r % ntx) * TILE};
}

// Layer 6 backward: gz5 = (sum_tap W6[tap] gout(p - off)) * (a5 > 0), and
// dW6[tap][ci] = sum_p gout(p) a5(p + off)[ci], db6.  The weight gradient is
// a product in FP32 on the matrix cores (16x16x4): M = tap (9 of 16), N = ci, K =
// the 324 pixels q = p + off of the halo tile, A[tap][q] = gout(q - off), 0
// outside the tile; a wavefront takes 16 channels and every other K step, the
// two halves are added through LDS.  One output a thread, 256 LDS reads after
// each other: 30 us for 32 crops of 64 x 64; 15.
__global__ void __launch_bounds__(256) k_cnn_l6_back(const float *__restrict__ gout, const bf16 *__restrict__ a5,
                                                    const float *__restrict__ prm, bf16 *__restrict__ gz5,
                                                    float *__restrict__ part, int H, int W, int px, int ntile)
{
    __shared__ float sg[HALO * HALO];                  // gout with halo
    __shared__ __attribute__((aligned(16))) bf16 sa[HALO * HALO * PSTR];
    __shared__ float sx[2][16][17], sb[4];
    __shared__ v4f w[72];                              // [tap][ci], four of a row a read
    for (int k = threadIdx.x; k < 288; k += 256) ((float *)w)[k] = prm[37888 + k];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, col = lane & 15, grp = lane >> 4;
    const int nb = wv & 1, kh = wv >> 1, ky = col / 3, kx = col % 3;
    v4f acc = (v4f){0, 0, 0, 0};
    float bias = 0.0f;
    for (int t = blockIdx.x; t < ntile; t += gridDim.x) {
        const tile_at at = tile_of(t, H, W);
        halo_regs h;
        float gr[2];
        halo_load(a5, h, at.b, at.ty0, at.tx0, H, W, px);
#pragma unroll
        for (int k = 0; k < 2; k++) {
            const int idx = min((int)threadIdx.x + k * 256, HALO * HALO - 1), ty = idx / HALO, tx = idx - ty * HALO;
            const int gy = at.ty0 + ty - 1;
            bool ok = (gy >= 0 && gy < H);
            const int gx = wrapx(at.tx0 + tx - 1, W, px, ok), yc = min(max(gy, 0), H - 1);
            gr[k] = gout[((size_t)at.b * H + yc) * W + gx];
            if (!ok) gr[k] = 0.0f;
        }
        __syncthreads();                               // the last tile's readers are done
        halo_store(h, sa);
        sg[threadIdx.x] = gr[0];
        if (threadIdx.x < HALO * HALO - 256) sg[256 + threadIdx.x] = gr[1];
        __syncthreads();
        {   // input gradient: thread = pixel
            const int ty = threadIdx.x / TILE, tx = threadIdx.x % TILE;
            float g[9];
#pragma unroll
            for (int k = 0; k < 9; k++) g[k] = sg[(ty + 2 - k / 3) * HALO + tx + 2 - k % 3];
            bias += sg[(ty + 1) * HALO + tx + 1];
            uint4 *dst = (uint4 *)(gz5 + (((size_t)at.b * H + at.ty0 + ty) * W + at.tx0 + tx) * CNN_C);
            const bf16 *am = sa + ((ty + 1) * HALO + tx + 1) * PSTR;
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const v4u m = *(const v4u *)(am + 8 * q);
                v4f s0 = (v4f){0, 0, 0, 0}, s1 = s0;
#pragma unroll
                for (int k = 0; k < 9; k++) {
                    const v4f w0 = w[k * 8 + 2 * q], w1 = w[k * 8 + 2 * q + 1];
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        s0[e] += w0[e] * g[k];
                        s1[e] += w1[e] * g[k];
                    }
                }
                unsigned o[4];
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    const float a = e < 2 ? s0[2 * e] : s1[2 * e - 4], c = e < 2 ? s0[2 * e + 1] : s1[2 * e - 3];
                    o[e] = (bfpos((bf16)(m[e] & 0xffffu)) ? (unsigned)f2bf(a) : 0u) |
                           (bfpos((bf16)(m[e] >> 16)) ? (unsigned)f2bf(c) << 16 : 0u);
                }
                dst[q] = make_uint4(o[0], o[1], o[2], o[3]);
            }
        }
#pragma unroll 8
        for (int u = 0; u < (HALO * HALO / 4 + 1) / 2; u++) {
            const int qq = 4 * (2 * u + kh) + grp, q = min(qq, HALO * HALO - 1);
            const int qy = q / HALO, qx = q - qy * HALO, py = qy - ky, pxx = qx - kx;
            const bool in = col < 9 && qq == q && (unsigned)py < TILE && (unsigned)pxx < TILE;
            const float av = in ? sg[(py + 1) * HALO + pxx + 1] : 0.0f;
            acc = __builtin_amdgcn_mfma_f32_16x16x4f32(av, bf2f(sa[q * PSTR + nb * 16 + col]), acc, 0, 0, 0);
        }
    }
    float *pp = part + (size_t)blockIdx.x * PVK_CNN_PSTRIDE + 37888;
    if (kh == 1)
#pragma unroll
        for (int q = 0; q < 4; q++) sx[nb][4 * grp + q][col] = acc[q];
#pragma unroll
    for (int d = 32; d > 0; d >>= 1) bias += __shfl_down(bias, d, 64);
    if (lane == 0) sb[wv] = bias;
    __syncthreads();
    if (kh == 0)
#pragma unroll
        for (int q = 0; q < 4; q++)
            if (4 * grp + q < 9) pp[(4 * grp + q) * 32 + nb * 16 + col] = acc[q] + sx[nb][4 * grp + q][col];
    if (threadIdx.x == 0) pp[288] = (sb[0] + sb[1]) + (sb[2] + sb[3]);
}

// Weight gradient of a 32 -> 32 layer on MFMA: per tap,
// dW[tap][co][ci] += sum_p gz(p)[co] a(p + off(tap))[ci]  (M = co, N = ci,
// K = a tile row's 16 pixels), plus db[co] (the same product with ones for a).
// LDS reads bound it: row r of a serves the taps ky of the gz rows r - ky, so
// the rows of a are walked once, six pixels of a row giving the operands of all
// three kx, and gz of the last three rows stays in registers: 172 two-byte
// reads a lane and tile instead of 1152 for the 144 products.  32 crops of 64 x
// 64: 20.0 us a layer with an operand pair read for each product; 11.2.
__global__ void __launch_bounds__(256) k_cnn_dw(const bf16 *__restrict__ gz, const bf16 *__restrict__ a,
                                               float *__restrict__ part, int poff, int H, int W, int px, int ntile)
{
    __shared__ __attribute__((aligned(16))) bf16 sa[HALO * HALO * PSTR];
    __shared__ __attribute__((aligned(16))) bf16 sg[TILE * TILE * PSTR];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, col = lane & 15, grp = lane >> 4;
    const int mb = wv >> 1, nb = wv & 1;              // co block, ci block of this wave
    const v4s ones = (v4s){0x3f80, 0x3f80, 0x3f80, 0x3f80};
    v4f acc[9], accb = (v4f){0, 0, 0, 0};
#pragma unroll
    for (int k = 0; k < 9; k++) acc[k] = (v4f){0, 0, 0, 0};
    for (int t = blockIdx.x; t < ntile; t += gridDim.x) {
        const tile_at at = tile_of(t, H, W);
        halo_regs h;
        tile_regs gr;
        halo_load(a, h, at.b, at.ty0, at.tx0, H, W, px);
        tile_load(gz, gr, at.b, at.ty0, at.tx0, H, W);
        __syncthreads();                               // the last tile's readers are done
        halo_store(h, sa);
        tile_store(gr, sg);
        __syncthreads();
        const bf16 *pa = sa + (4 * grp) * PSTR + nb * 16 + col, *pg = sg + (4 * grp) * PSTR + mb * 16 + col;
        v4s av[3];                                     // gz of rows r, r - 1, r - 2 (slot row % 3)
#pragma unroll
        for (int r = 0; r < HALO; r++) {
            short e[6];
#pragma unroll
            for (int k = 0; k < 6; k++) e[k] = (short)pa[(r * HALO + k) * PSTR];
            if (r < TILE) {
#pragma unroll
                for (int q = 0; q < 4; q++) av[r % 3][q] = (short)pg[(r * TILE + q) * PSTR];
                if (nb == 0) accb = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(av[r % 3], ones, accb, 0, 0, 0);
            }
#pragma unroll
            for (int kx = 0; kx < 3; kx++) {
                const v4s bv = (v4s){e[kx], e[kx + 1], e[kx + 2], e[kx + 3]};
#pragma unroll
                for (int ky = 0; ky < 3; ky++)
                    if (r - ky >= 0 && r - ky < TILE)
                        acc[3 * ky + kx] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(av[(r - ky + 3) % 3], bv, acc[3 * ky + kx], 0, 0, 0);
            }
        }
    }
    float *pp = part + (size_t)blockIdx.x * PVK_CNN_PSTRIDE + poff;
#pragma unroll
    for (int tap = 0; tap < 9; tap++)
#pragma unroll
        for (int q = 0; q < 4; q++)
            pp[(tap * CNN_C + mb * 16 + 4 * grp + q) * CNN_C + nb * 16 + col] = acc[tap][q];
    if (nb == 0 && col == 0)
#pragma unroll
        for (int q = 0; q < 4; q++) pp[9216 + mb * 16 + 4 * grp + q] = accb[q];
}

// Layer 1 weight gradient: dW1[co][tap][ci] = sum_p gz1(p)[co] in3(p + off)[ci], db1,
// in FP32 on the matrix cores (16x16x4; the input is FP32): M = co, N = (tap, ci)
// and a column of ones for db1 (28 of 32), K = the tile's 256 pixels, one
// 16 x 16 block a wavefront.  One output a thread: 40 us for 32 crops of 64 x
// 64; 7.
__global__ void __launch_bounds__(256) k_cnn_l1_back(const bf16 *__restrict__ gz, const float *__restrict__ in3,
                                                    float *__restrict__ part, int H, int W, int px, int ntile)
{
    constexpr int NI = HALO * HALO * 3, IK = (NI + 255) / 256;
    __shared__ float si[NI];
    __shared__ __attribute__((aligned(16))) bf16 sg[TILE * TILE * PSTR];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, col = lane & 15, grp = lane >> 4;
    const int mb = wv >> 1, n = (wv & 1) * 16 + col, tap = n / 3;     // n = 27: the ones; above: zeros
    const int off = (n < 27) ? ((tap / 3) * HALO + tap % 3) * 3 + n % 3 : 0;
    v4f acc = (v4f){0, 0, 0, 0};
    for (int t = blockIdx.x; t < ntile; t += gridDim.x) {
        const tile_at at = tile_of(t, H, W);
        tile_regs gr;
        float ir[IK];
        tile_load(gz, gr, at.b, at.ty0, at.tx0, H, W);
#pragma unroll
        for (int k = 0; k < IK; k++) {
            const int idx = min((int)threadIdx.x + k * 256, NI - 1), pix = idx / 3, c = idx % 3, ty = pix / HALO, tx = pix % HALO;
            const int gy = at.ty0 + ty - 1;
            bool ok = (gy >= 0 && gy < H);
            const int gx = wrapx(at.tx0 + tx - 1, W, px, ok), yc = min(max(gy, 0), H - 1);
            ir[k] = in3[(((size_t)at.b * H + yc) * W + gx) * 3 + c];
            if (!ok) ir[k] = 0.0f;
        }
        __syncthreads();                               // the last tile's readers are done
        tile_store(gr, sg);
#pragma unroll
        for (int k = 0; k < IK; k++)
            if ((int)threadIdx.x + k * 256 < NI) si[threadIdx.x + k * 256] = ir[k];
        __syncthreads();
#pragma unroll 8
        for (int ks = 0; ks < TILE * TILE / 4; ks++) {
            const int p = 4 * ks + grp;
            const float bv = si[((p / TILE) * HALO + p % TILE) * 3 + off];
            acc = __builtin_amdgcn_mfma_f32_16x16x4f32(bf2f(sg[p * PSTR + mb * 16 + col]), n < 27 ? bv : (n == 27 ? 1.0f : 0.0f),
                                                       acc, 0, 0, 0);
        }
    }
    float *pp = part + (size_t)blockIdx.x * PVK_CNN_PSTRIDE;
#pragma unroll
    for (int q = 0; q < 4; q++) {
        const int co = mb * 16 + 4 * grp + q;
        if (n < 27) pp[co * 27 + n] = acc[q];
        else if (n == 27) pp[864 + co] = acc[q];
    }
}

// g[k] = sum over rows q of part[q][k] in a fixed order: group y of 16 adds rows
// y, y + 16, ..., then the groups are added in order.  All layers in one launch
// after the backward pass (a pair of launches a layer took 66 us, this 15).
#define RGRP 16
__global__ void __launch_bounds__(64 * RGRP) k_cnn_reduce(const float *__restrict__ part, int nrow, float *__restrict__ g)
{
    __shared__ float sh[RGRP][64];
    const int x = threadIdx.x & 63, y = threadIdx.x >> 6, k = min((int)blockIdx.x * 64 + x, PVK_CNN_NPARAM - 1);
    const float *p = part + k;
    float s = 0.0f;
    int q = y;
    for (; q + 7 * RGRP < nrow; q += 8 * RGRP) {       // eight rows in flight
        float v[8];
#pragma unroll
        for (int u = 0; u < 8; u++) v[u] = p[(size_t)(q + u * RGRP) * PVK_CNN_PSTRIDE];
#pragma unroll
        for (int u = 0; u < 8; u++) s += v[u];
    }
    for (; q < nrow; q += RGRP) s += p[(size_t)q * PVK_CNN_PSTRIDE];
    sh[y][x] = s;
    __syncthreads();
    if (y == 0 && (int)blockIdx.x * 64 + x < PVK_CNN_NPARAM) {
        for (int u = 1; u < RGRP; u++) s += sh[u][x];
        g[k] = s;
    }
}

// Adam (FP32 master weights)
__global__ void k_cnn_adam(float *w, const float *g, float *m, float *v, int n, float lr, float b1, float b2,
                           float eps, float c1, float c2)
{
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= n) return;
    const float gk = g[k];
    const float mk = b1 * m[k] + (1.0f - b1) * gk, vk = b2 * v[k] + (1.0f - b2) * gk * gk;
    m[k] = mk;
    v[k] = vk;
    w[k] -= lr * (mk / c1) / (sqrtf(vk / c2) + eps);
}

// BF16 copies of the 32 -> 32 layers: forward [tap][co][ci] and, for the
// input gradient, the flipped transpose wt[tap'][ci][co] = W[8 - tap'][co][ci].
__global__ void k_cnn_pack(const float *__restrict__ prm, bf16 *__restrict__ wb, bf16 *__restrict__ wt)
{
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= 4 * 9216) return;
    const int l = k / 9216, r = k % 9216, tap = r / 1024, co = (r / 32) % 32, ci = r % 32;
    const float v = prm[896 + l * 9248 + r];
    wb[k] = f2bf(v);
    wt[l * 9216 + ((8 - tap) * CNN_C + ci) * CNN_C + co] = f2bf(v);
}

// ---------------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------------
extern "C" void pvk_cnn_pack(const pvk_cnn *c, hipStream_t s)
{
    hipLaunchKernelGGL(k_cnn_pack, dim3((4 * 9216 + 255) / 256), dim3(256), 0, s, c->w, c->wb, c->wt);
}

// forward of a batch: in3 [B][H][W][3] -> out [B][H][W]; activations kept in c->act
extern "C" void pvk_cnn_forward(const pvk_cnn *c, const float *in3, float *out, int B, int H, int W, int px,
                                hipStream_t s)
{
    const dim3 gp((H * W + 255) / 256, B), gt((H / TILE) * (W / TILE), B);
    hipLaunchKernelGGL(k_cnn_l1, gp, dim3(256), 0, s, in3, (const float *)c->w, c->act[0], H, W, px);
    for (int l = 0; l < 4; l++)
        hipLaunchKernelGGL((k_cnn_mid<true, false>), gt, dim3(256), 0, s, (const bf16 *)c->act[l],
                           (const bf16 *)(c->wb + l * 9216), (const float *)(c->w + 896 + l * 9248 + 9216),
                           c->act[l + 1], (const bf16 *)0, H, W, px);
    hipLaunchKernelGGL(k_cnn_l6, gp, dim3(256), 0, s, (const bf16 *)c->act[4], (const float *)c->w, out, H, W, px);
}

// loss and full gradient (into c->g) of the last forward; returns nothing on
// the host: the per-block loss partials are left in c->lpart
extern "C" void pvk_cnn_backward(const pvk_cnn *c, const float *in3, const float *out, const float *tgt, int B,
                                 int H, int W, int px, int border, hipStream_t s)
{
    const dim3 gp((H * W + 255) / 256, B), gt((H / TILE) * (W / TILE), B);
    const int nt = (H / TILE) * (W / TILE) * B;
    const dim3 gr(nt < PVK_CNN_ROWS ? nt : PVK_CNN_ROWS);
    const int interior = (H - 2 * border) * (W - 2 * border) * B;
    hipLaunchKernelGGL(k_cnn_loss, gp, dim3(256), 0, s, out, tgt, c->gout, c->lpart, H, W, border,
                       1.0f / (float)(interior > 0 ? interior : 1));
    hipLaunchKernelGGL(k_cnn_l6_back, gr, dim3(256), 0, s, (const float *)c->gout, (const bf16 *)c->act[4],
                       (const float *)c->w, c->gz[0], c->part, H, W, px, nt);
    int cur = 0;
    for (int l = 3; l >= 0; l--) {       // layer l + 2: input act[l], output-side gradient gz[cur]
        hipLaunchKernelGGL(k_cnn_dw, gr, dim3(256), 0, s, (const bf16 *)c->gz[cur], (const bf16 *)c->act[l], c->part,
                           896 + l * 9248, H, W, px, nt);
        hipLaunchKernelGGL((k_cnn_mid<false, true>), gt, dim3(256), 0, s, (const bf16 *)c->gz[cur],
                           (const bf16 *)(c->wt + l * 9216), (const float *)0, c->gz[cur ^ 1],
                           (const bf16 *)c->act[l], H, W, px);
        cur ^= 1;
    }
    hipLaunchKernelGGL(k_cnn_l1_back, gr, dim3(256), 0, s, (const bf16 *)c->gz[cur], in3, c->part, H, W, px, nt);
    hipLaunchKernelGGL(k_cnn_reduce, dim3((PVK_CNN_NPARAM + 63) / 64), dim3(64 * RGRP), 0, s, (const float *)c->part,
                       (int)gr.x, c->g);
}

extern "C" void pvk_cnn_adam(const pvk_cnn *c, float lr, int t, hipStream_t s)
{
    const float b1 = 0.9f, b2 = 0.999f;
    const float c1 = 1.0f - powf(b1, (float)t), c2 = 1.0f - powf(b2, (float)t);
    hipLaunchKernelGGL(k_cnn_adam, dim3((PVK_CNN_NPARAM + 255) / 256), dim3(256), 0, s, c->w, (const float *)c->g,
                       c->m, c->v, PVK_CNN_NPARAM, lr, b1, b2, 1e-8f, c1, c2);
    pvk_cnn_pack(c, s);
}
