// pv_fftk.h -- radix-8/4/2 Stockham FFT of length M (a power of two, 4..2048)
// held in LDS as separate real and imaginary arrays.
//
// Pass with radix R and sub-transform size Ns (Ns = 1, R, R*R', ...): the
// butterfly bb < M/R reads x[bb + r M/R], r < R, multiplies element r by
// W^(k r), k = bb mod Ns, W = exp(-+2 pi i / (Ns R)), takes an R-point DFT in
// registers and writes y[(bb / Ns) Ns R + k + r Ns].  Input and output are
// in natural order (no bit reversal).  Passes: radix 8 while at least three
// factors of two remain, then one radix-4 or radix-2 pass.  With T = M/8
// threads per transform every thread holds 8 complex values in every pass.
//
// The twiddle table tw holds exp(-2 pi i t / M) for t < M as (cos, sin)
// pairs; W^(k r) of a pass is entry k r M / (Ns R).  The inverse transform
// uses conjugate twiddles and is unscaled.
//
// The load and store halves are __host__ __device__ so the same code is
// checked on the CPU against a direct DFT.
#ifndef PV_FFTK_H
#define PV_FFTK_H
#include <hip/hip_runtime.h>

#define SK_SQRT_HALF 0.70710678118654752440

// Where element i of a transform lies in LDS.  Flat: at i.  Padded: one slot
// is left after every eight elements, so the stride-8 stores of the first
// radix-8 pass (and the 64-element jumps of the second) spread over all banks
// instead of one double in sixteen.
struct SkFlat {
    static __host__ __device__ __forceinline__ int at(int i) { return i; }
};
struct SkPad {
    static __host__ __device__ __forceinline__ int at(int i) { return i + (i >> 3); }
};

// (x + i y) times -i (forward) or +i (inverse)
template <bool INV>
__host__ __device__ __forceinline__ void sk_rot(double &x, double &y)
{
    double t = x;
    if (INV) { x = -y; y = t; }
    else     { x = y;  y = -t; }
}

template <bool INV>
__host__ __device__ __forceinline__ void sk_dft2(double *vr, double *vi, int a, int b)
{
    double tr = vr[a] - vr[b], ti = vi[a] - vi[b];
    vr[a] = vr[a] + vr[b]; vi[a] = vi[a] + vi[b];
    vr[b] = tr; vi[b] = ti;
}

// 4-point DFT of v[o], v[o+s], v[o+2s], v[o+3s], results in natural order in place
template <bool INV>
__host__ __device__ __forceinline__ void sk_dft4(double *vr, double *vi, int o, int s)
{
    const int i0 = o, i1 = o + s, i2 = o + 2 * s, i3 = o + 3 * s;
    double ar = vr[i0] + vr[i2], ai = vi[i0] + vi[i2];
    double br = vr[i0] - vr[i2], bi = vi[i0] - vi[i2];
    double cr = vr[i1] + vr[i3], ci = vi[i1] + vi[i3];
    double dr = vr[i1] - vr[i3], di = vi[i1] - vi[i3];
    sk_rot<INV>(dr, di);                       // omega (a1 - a3), omega = -+i
    vr[i0] = ar + cr; vi[i0] = ai + ci;
    vr[i2] = ar - cr; vi[i2] = ai - ci;
    vr[i1] = br + dr; vi[i1] = bi + di;
    vr[i3] = br - dr; vi[i3] = bi - di;
}

// 8-point DFT of v[0..7] in place, natural order: X_k = E_k + w^k O_k,
// X_{k+4} = E_k - w^k O_k with E, O the 4-point DFTs of even and odd entries.
template <bool INV>
__host__ __device__ __forceinline__ void sk_dft8(double *vr, double *vi)
{
    sk_dft4<INV>(vr, vi, 0, 2);                // E_k at 0, 2, 4, 6
    sk_dft4<INV>(vr, vi, 1, 2);                // O_k at 1, 3, 5, 7
    const double h = SK_SQRT_HALF;
    double o1r = vr[3], o1i = vi[3], o2r = vr[5], o2i = vi[5], o3r = vr[7], o3i = vi[7];
    // w = exp(-+ i pi / 4)
    double w1r = (o1r + (INV ? -o1i : o1i)) * h, w1i = (o1i + (INV ? o1r : -o1r)) * h;
    double w2r = o2r, w2i = o2i;
    sk_rot<INV>(w2r, w2i);
    double w3r = (-o3r + (INV ? -o3i : o3i)) * h, w3i = (-o3i + (INV ? o3r : -o3r)) * h;
    double e0r = vr[0], e0i = vi[0], e1r = vr[2], e1i = vi[2], e2r = vr[4], e2i = vi[4], e3r = vr[6], e3i = vi[6];
    double o0r = vr[1], o0i = vi[1];
    vr[0] = e0r + o0r; vi[0] = e0i + o0i;
    vr[4] = e0r - o0r; vi[4] = e0i - o0i;
    vr[1] = e1r + w1r; vi[1] = e1i + w1i;
    vr[5] = e1r - w1r; vi[5] = e1i - w1i;
    vr[2] = e2r + w2r; vi[2] = e2i + w2i;
    vr[6] = e2r - w2r; vi[6] = e2i - w2i;
    vr[3] = e3r + w3r; vi[3] = e3i + w3i;
    vr[7] = e3r - w3r; vi[7] = e3i - w3i;
}

// Read butterfly bb of a radix-R pass (R = 2^LR), twiddle, DFT: v[0..R).
// All sizes are powers of two and passed as base-2 logarithms, so index
// arithmetic is shifts and masks.
template <int LR, bool INV, class IX = SkFlat>
__host__ __device__ __forceinline__ void sk_load(const double *sr, const double *si, int bb, int logM, int logNs,
                                                 const double *tw, double *vr, double *vi)
{
    constexpr int R = 1 << LR;
    const int stride = 1 << (logM - LR), k = bb & ((1 << logNs) - 1), step = k << (logM - logNs - LR);
#pragma unroll
    for (int r = 0; r < R; r++) {
        vr[r] = sr[IX::at(bb + r * stride)];
        vi[r] = si[IX::at(bb + r * stride)];
    }
    if (logNs > 0) {
#pragma unroll
        for (int r = 1; r < R; r++) {
            const int t = r * step;
            const double c = tw[2 * t], s = INV ? -tw[2 * t + 1] : tw[2 * t + 1];
            const double xr = vr[r], xi = vi[r];
            vr[r] = xr * c - xi * s;
            vi[r] = xr * s + xi * c;
        }
    }
    if (R == 8) sk_dft8<INV>(vr, vi);
    else if (R == 4) sk_dft4<INV>(vr, vi, 0, 1);
    else sk_dft2<INV>(vr, vi, 0, 1);
}

template <int LR, class IX = SkFlat>
__host__ __device__ __forceinline__ void sk_store(double *sr, double *si, int bb, int logNs, const double *vr,
                                                  const double *vi)
{
    constexpr int R = 1 << LR;
    const int Ns = 1 << logNs;
    const int base = ((bb >> logNs) << (logNs + LR)) + (bb & (Ns - 1));
#pragma unroll
    for (int r = 0; r < R; r++) {
        sr[IX::at(base + r * Ns)] = vr[r];
        si[IX::at(base + r * Ns)] = vi[r];
    }
}

// One radix-R pass over a transform whose T threads have lane ids 0..T-1;
// every thread of the block calls it (barriers inside).  bb >= M / R idle.
template <int LR, bool INV, class IX = SkFlat>
__device__ __forceinline__ void sk_pass(double *sr, double *si, int logM, int logNs, const double *tw, int lane,
                                        int T)
{
    constexpr int U = 8 >> LR;
    const int nbf = 1 << (logM - LR);
    double vr[8], vi[8];
#pragma unroll
    for (int u = 0; u < U; u++) {
        const int bb = lane + u * T;
        if (bb < nbf) sk_load<LR, INV, IX>(sr, si, bb, logM, logNs, tw, vr + (u << LR), vi + (u << LR));
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < U; u++) {
        const int bb = lane + u * T;
        if (bb < nbf) sk_store<LR, IX>(sr, si, bb, logNs, vr + (u << LR), vi + (u << LR));
    }
    __syncthreads();
}

// Whole transform of length M = 2^logM; the caller has synchronised after
// filling sr / si and reads the result after this returns.
template <bool INV>
__device__ __forceinline__ void sk_fft(double *sr, double *si, int logM, const double *tw, int lane, int T)
{
    int logNs = 0, rem = logM;
    for (; rem >= 3; rem -= 3, logNs += 3) sk_pass<3, INV>(sr, si, logM, logNs, tw, lane, T);
    if (rem == 2) sk_pass<2, INV>(sr, si, logM, logNs, tw, lane, T);
    else if (rem == 1) sk_pass<1, INV>(sr, si, logM, logNs, tw, lane, T);
}

// The same from a thread's eight values in registers, v[r] = x[lane + r T]: the
// first radix-8 pass (no twiddles) needs no LDS read.  M >= 8.
template <bool INV, class IX>
__device__ __forceinline__ void sk_fft_regs(double *vr, double *vi, double *sr, double *si, int logM, const double *tw,
                                            int lane, int T)
{
    sk_dft8<INV>(vr, vi);
    sk_store<3, IX>(sr, si, lane, 0, vr, vi);
    __syncthreads();
    int logNs = 3, rem = logM - 3;
    for (; rem >= 3; rem -= 3, logNs += 3) sk_pass<3, INV, IX>(sr, si, logM, logNs, tw, lane, T);
    if (rem == 2) sk_pass<2, INV, IX>(sr, si, logM, logNs, tw, lane, T);
    else if (rem == 1) sk_pass<1, INV, IX>(sr, si, logM, logNs, tw, lane, T);
}

// ---------------------------------------------------------------------------
// Mixed radix: lengths M = 2^a 3^b with 8 | M.  The same Stockham passes with
// general (not power-of-two) sub-transform sizes Ns: radix 8 while three
// factors of two remain, then a radix-4 or radix-2 pass, then one radix-3
// pass per factor of three.  T = M / 8 threads per transform; a radix-R pass
// has M / R butterflies, so a thread takes up to 8 / R of them (3 for R = 3).
// Threads whose transform index is out of range (act = false) only take part
// in the barriers.
// ---------------------------------------------------------------------------

// 3-point DFT of v[0..2] in place: X_1,2 = a - (b + c) / 2 -+ i (sqrt 3 / 2)(b - c)
// (forward: exp(-2 pi i / 3); the inverse swaps X_1 and X_2)
template <bool INV>
__host__ __device__ __forceinline__ void sk_dft3(double *vr, double *vi)
{
    const double h = 0.86602540378443864676;          // sqrt(3) / 2
    const double sr_ = vr[1] + vr[2], si_ = vi[1] + vi[2];
    const double tr = vr[0] - 0.5 * sr_, ti = vi[0] - 0.5 * si_;
    const double dr = h * (vr[1] - vr[2]), di = h * (vi[1] - vi[2]);
    vr[0] += sr_; vi[0] += si_;
    if (INV) { vr[1] = tr - di; vi[1] = ti + dr; vr[2] = tr + di; vi[2] = ti - dr; }
    else     { vr[1] = tr + di; vi[1] = ti - dr; vr[2] = tr - di; vi[2] = ti + dr; }
}

// A sub-transform size n = 2^lg 3^c.  Every pass but the radix-3 ones after
// the first has c = 0, a constant where the passes are inlined, so its index
// arithmetic is shifts and masks, and the others divide by the constant 3:
// with divisions by n at run time the forward row kernel took 14.2 us and the
// inverse one 9.4 at 768 x 491 (10.6 and 7.1 at 96 x 200), 12.9 and 8.2 (9.8
// and 6.3) now.
struct SgSize {
    int n, lg, c;
    __host__ __device__ __forceinline__ SgSize(int n_, int lg_, int c_) : n(n_), lg(lg_), c(c_) {}
    __host__ __device__ __forceinline__ SgSize(int n_) : n(n_), lg(0), c(0)
    {
        for (; n_ % 2 == 0; n_ /= 2) lg++;
        for (; n_ % 3 == 0; n_ /= 3) c++;
    }
    __host__ __device__ __forceinline__ int quo(int x) const     // x / n, x >= 0
    {
        unsigned q = (unsigned)x >> lg;
        for (int u = 0; u < c; u++) q /= 3u;
        return (int)q;
    }
    __host__ __device__ __forceinline__ int rem(int x) const { return c ? x - quo(x) * n : x & (n - 1); }
};

template <int R, bool INV, class IX = SkFlat>
__host__ __device__ __forceinline__ void sg_load(const double *sr, const double *si, int bb, int M, SgSize Ns,
                                                 const double *tw, double *vr, double *vi)
{
    const int stride = M / R, k = Ns.rem(bb), step = Ns.quo(stride) * k;
#pragma unroll
    for (int r = 0; r < R; r++) {
        vr[r] = sr[IX::at(bb + r * stride)];
        vi[r] = si[IX::at(bb + r * stride)];
    }
    if (Ns.n > 1) {
#pragma unroll
        for (int r = 1; r < R; r++) {
            const int t = r * step;
            const double c = tw[2 * t], s = INV ? -tw[2 * t + 1] : tw[2 * t + 1];
            const double xr = vr[r], xi = vi[r];
            vr[r] = xr * c - xi * s;
            vi[r] = xr * s + xi * c;
        }
    }
    if (R == 8) sk_dft8<INV>(vr, vi);
    else if (R == 4) sk_dft4<INV>(vr, vi, 0, 1);
    else if (R == 3) sk_dft3<INV>(vr, vi);
    else sk_dft2<INV>(vr, vi, 0, 1);
}

template <int R, class IX = SkFlat>
__host__ __device__ __forceinline__ void sg_store(double *sr, double *si, int bb, SgSize Ns, const double *vr,
                                                  const double *vi)
{
    const int k = Ns.rem(bb), base = (bb - k) * R + k;
#pragma unroll
    for (int r = 0; r < R; r++) {
        sr[IX::at(base + r * Ns.n)] = vr[r];
        si[IX::at(base + r * Ns.n)] = vi[r];
    }
}

template <int R, bool INV, class IX = SkFlat>
__device__ __forceinline__ void sg_pass(double *sr, double *si, int M, SgSize Ns, const double *tw, int lane, int T,
                                        bool act)
{
    constexpr int U = (R == 3) ? 3 : 8 / R;
    const int nbf = M / R;
    double vr[U * R], vi[U * R];
#pragma unroll
    for (int u = 0; u < U; u++) {
        const int bb = lane + u * T;
        if (act && bb < nbf) sg_load<R, INV, IX>(sr, si, bb, M, Ns, tw, vr + u * R, vi + u * R);
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < U; u++) {
        const int bb = lane + u * T;
        if (act && bb < nbf) sg_store<R, IX>(sr, si, bb, Ns, vr + u * R, vi + u * R);
    }
    __syncthreads();
}

// Whole transform of length M = 2^a 3^b (8 | M), from registers as sk_fft_regs
template <bool INV, class IX>
__device__ __forceinline__ void sg_fft_regs(double *vr, double *vi, double *sr, double *si, int M, const double *tw, int lane,
                                            int T, bool act)
{
    int lg = 3, two = M / 8;
    while (two % 3 == 0) two /= 3;                   // the rest of the power-of-two part
    sk_dft8<INV>(vr, vi);
    if (act) sg_store<8, IX>(sr, si, lane, SgSize(1, 0, 0), vr, vi);
    __syncthreads();
    for (; two % 8 == 0; two /= 8, lg += 3) sg_pass<8, INV, IX>(sr, si, M, SgSize(1 << lg, lg, 0), tw, lane, T, act);
    if (two == 4) { sg_pass<4, INV, IX>(sr, si, M, SgSize(1 << lg, lg, 0), tw, lane, T, act); lg += 2; }
    else if (two == 2) { sg_pass<2, INV, IX>(sr, si, M, SgSize(1 << lg, lg, 0), tw, lane, T, act); lg += 1; }
    int n = 1 << lg;
    if (n < M) { sg_pass<3, INV, IX>(sr, si, M, SgSize(n, lg, 0), tw, lane, T, act); n *= 3; }
    for (int c = 1; n < M; n *= 3, c++) sg_pass<3, INV, IX>(sr, si, M, SgSize(n, lg, c), tw, lane, T, act);
}
#endif
