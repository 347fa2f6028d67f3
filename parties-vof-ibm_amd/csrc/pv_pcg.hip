// pv_pcg.hip -- fused FFT-preconditioned PCG for the variable-coefficient
// pressure equation div(beta grad phi) = rhs, beta = 2 / (rho_i + rho_nb)
// (operator of lsolver/psolve_cg.c:302-344), preconditioned by the
// constant-coefficient FFT-x / DCT-y solve.
//
// One iteration = four launches and no one-block kernels:
//   K1 k_pcg_apply      d_n = z + beta d_{n-1} on the fly (double-buffered d),
//                       Ad = A d_n, partials <d, Ad>           (row bands)
//   K2 k_pcg_update_fwd alpha; phi += alpha d; r -= alpha Ad; partials <r,r>;
//                       forward real FFT of the new r rows    (R rows per block)
//   K4 k_tri_cols       stop test from <r,r>; the y solves in place on the
//                       columns of the spectrum                (columns)
//   K6 k_ifft_rows_dot  z = inverse real FFT; partials <r, z>
// The Cahn-Hilliard solve's spectral start replaces K4 by K3 k_transpose,
// k_dct_rows (DCT-II, divide, DCT-III along y) and K5 k_transpose.
// Scalars are never stored by one block and read by others in the same
// kernel: every block re-adds the few hundred partials of the previous
// kernel in the same fixed order, so all blocks see bit-identical alpha,
// beta and stop decisions and the result does not depend on scheduling.
// <r, z> partials alternate between two buffers by iteration parity so beta
// can be formed from gamma_n and gamma_{n-1}.
#include <hip/hip_runtime.h>
#include <math.h>
#include <mutex>
#include "pv_kernels.h"
#include "pv_block.h"
#include "pv_fftk.h"
#include "pv_stencil.h"

#define AT(a, i, j) (a)[(ptrdiff_t)(j) * P + (i)]

struct cplx2 { double x, y; };

// log2 of the threads per transform of length 2^logM in the Stockham FFT
// (pv_fftk.h): M / 8 threads, at least one
__device__ __forceinline__ int sk_logT(int logM) { return logM >= 3 ? logM - 3 : 0; }

// X_k, k = 0..M, of a real length-2M sequence from Z = FFT_M(x_{2m} + i x_{2m+1}):
// Z_k (k = M: Z_0), Z_{M-k} (k = 0, M: Z_0) and c, s = cos, sin of pi k / M
__device__ __forceinline__ cplx2 rpost(double zr, double zi, double br, double bi, double c, double s)
{
    double cr = br, ci = -bi;
    double er = 0.5 * (zr + cr), ei = 0.5 * (zi + ci);
    double dr = zr - cr, di = zi - ci;
    double or_ = 0.5 * di, oi = -0.5 * dr;
    cplx2 X;
    X.x = er + (c * or_ + s * oi);
    X.y = ei + (c * oi - s * or_);
    return X;
}
__device__ __forceinline__ cplx2 rpost(const double *sr, const double *si, int base, int M, int k, const double *rt)
{
    const int ka = (k == M) ? 0 : k, kb = (k == 0 || k == M) ? 0 : M - k;
    return rpost(sr[base + ka], si[base + ka], sr[base + kb], si[base + kb], rt[2 * k], rt[2 * k + 1]);
}

// Y_k from X_k and X_{M-k} for the half-length inverse
__device__ __forceinline__ cplx2 rpre(cplx2 Xk, cplx2 Xmk, double c, double s)
{
    double ar = Xk.x + Xmk.x, ai = Xk.y - Xmk.y;
    double dr = Xk.x - Xmk.x, di = Xk.y + Xmk.y;
    double pr = dr * c - di * s, pi_ = dr * s + di * c;
    cplx2 Y;
    Y.x = ar - pi_;
    Y.y = ai + pr;
    return Y;
}

// The y transforms handle R = 2048 / M columns of M complex points per block
// (T = M / 8 threads per transform, 256 threads), so each thread owns
// IT = R * M / 256 = 8 items of the sweeps; the sweeps load all of a
// thread's items before storing any, so the loads are in flight together.
#define IT 8
#define CPT 4

// Stockham twiddles (M complex) staged in LDS behind the 2 R M row values.
__device__ __forceinline__ double *stage_twiddles(double *lds, int RM, int M, const double *tw)
{
    double *t = lds + 2 * RM;
    for (int k = threadIdx.x; k < 2 * M; k += NTH) t[k] = tw[k];
    return t;
}

// ---------------------------------------------------------------------------
// Face coefficients of the operator, formed once per solve (rho is fixed):
// bx(i,j) = 2 / (rho_i + rho_{i+1}) idx^2 for i in [-1, NXM), by(i,j) the
// same along y for j in [-1, NYM).  Addition commutes exactly, so
// bx(i-1, j) is bit for bit the west coefficient of cell (i, j).
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(NTH) k_pcg_faces(pvk_grid g, pvk_pcg w)
{
    const int P = g.P, NXM = g.NXM, NYM = g.NYM;
    const int j = (int)blockIdx.x - 1;
    const double idx2 = g.idx_c[1] * g.idx_c[1], idy2 = g.idy_c[1] * g.idy_c[1];
    const double *__restrict__ rho = w.rho;
    for (int i = (int)threadIdx.x - 1; i < NXM; i += NTH) {
        const double r0 = AT(rho, i, j);
        AT(w.bx, i, j) = (2.0 / (r0 + AT(rho, i + 1, j))) * idx2;
        AT(w.by, i, j) = (2.0 / (r0 + AT(rho, i, j + 1))) * idy2;
    }
}

// ---------------------------------------------------------------------------
// K1: d_n = z + beta d_{n-1}, Ad = A d_n, partial <d_n, Ad>.  One block per
// row j: the y neighbours and row clamps are block-uniform.  A thread's CPT
// columns of the three rows are loaded ahead of the sums that give beta (all
// blocks of a grid this size run at once, so nothing else covers them); its
// row's east and west values go through LDS.  Bound by memory, 48 bytes a
// cell: 11.2 us at 1024^2 (50 MB; 14.9 with every stencil
// value formed from its own loads after the sums), 50 at 2048^2 (73), 6.6 at
// 768 x 491 (10.6).
// ---------------------------------------------------------------------------
template <bool FIRST>
__global__ void __launch_bounds__(NTH, 4) k_pcg_apply(pvk_grid g, pvk_scal *sc, pvk_pcg w, int n)
{
    __shared__ double sh[2 * NTH];
    __shared__ double sd[2][NTH * CPT + 2];
    if (sc->p_done) return;
    const int P = g.P, NXM = g.NXM, NYM = g.NYM, t = threadIdx.x;
    const double *__restrict__ z = w.z;
    const double *__restrict__ dold = w.d[(n + 1) & 1];
    const double *__restrict__ bx = w.bx, *__restrict__ by = w.by;
    double *__restrict__ dnew = w.d[n & 1];
    double *__restrict__ Ad = w.Ad;
    const int j = xcd_band(blockIdx.x, gridDim.x);
    const int jr[3] = {j, (j + 1 == NYM) ? j : j + 1, (j == 0) ? 0 : j - 1};
    double zv[CPT][3], ov[CPT][3], cx[CPT][2], cy[CPT][2], ze, oe;
    auto load = [&](int base) {
#pragma unroll
        for (int u = 0; u < CPT; u++)
            if (base + u * NTH < NXM) {
                const int i = min(base + u * NTH + t, NXM - 1);
#pragma unroll
                for (int r = 0; r < 3; r++) {
                    zv[u][r] = AT(z, i, jr[r]);
                    if (!FIRST) ov[u][r] = AT(dold, i, jr[r]);
                }
                cx[u][0] = AT(bx, i, j);
                cx[u][1] = AT(bx, i - 1, j);
                cy[u][0] = AT(by, i, j);
                cy[u][1] = AT(by, i, j - 1);
            }
        if (t < 2) {                                 // the columns west and east of the chunk
            const int e = base + NTH * CPT, ie = t ? (e < NXM ? e : 0) : (base ? base - 1 : NXM - 1);
            ze = AT(z, ie, j);
            if (!FIRST) oe = AT(dold, ie, j);
        }
    };
    load(0);
    double beta = 0.0, sa, sb;
    if (!FIRST && w.flex) {   // flexible CG: A-orthogonal to the previous direction only
        block_sum2(w.zad, w.nrz, w.dad[(n + 1) & 1], w.ndad, sh, sa, sb);
        beta = -sa / sb;
    } else if (!FIRST) {      // Fletcher-Reeves: gamma_n / gamma_{n-1}
        block_sum2(w.rz[n & 1], w.nrz, w.rz[(n + 1) & 1], w.nrz, sh, sa, sb);
        beta = sa / sb;
    }
    auto dn = [&](double zz, double oo) { return FIRST ? zz : zz + beta * oo; };
    double acc = 0.0, sacc = 0.0;
    int par = 0;
    for (int base = 0; base < NXM; base += NTH * CPT, par ^= 1) {
        const int nc = min(NTH * CPT, NXM - base);
        double dc[CPT];
        if (base) load(base);
#pragma unroll
        for (int u = 0; u < CPT; u++)
            if (u * NTH < nc) {
                dc[u] = dn(zv[u][0], ov[u][0]);
                if (u * NTH + t < nc) sd[par][u * NTH + t + 1] = dc[u];
            }
        if (t < 2) sd[par][t ? nc + 1 : 0] = dn(ze, oe);
        __syncthreads();
#pragma unroll
        for (int u = 0; u < CPT; u++)
            if (u * NTH + t < nc) {
                const int b = u * NTH + t, i = base + b;
                const double d0 = dc[u], dE = sd[par][b + 2], dW = sd[par][b];
                const double dN = dn(zv[u][1], ov[u][1]), dS = dn(zv[u][2], ov[u][2]);
                const double ad = cx[u][0] * (dE - d0) - cx[u][1] * (d0 - dW) + cy[u][0] * (dN - d0) - cy[u][1] * (d0 - dS);
                AT(dnew, i, j) = d0;
                AT(Ad, i, j) = ad;
                acc += d0 * ad;
                sacc += ad;
            }
    }
    block_store_partial(acc, w.dad[n & 1], j, sh);
    if (w.sad) block_store_partial(sacc, w.sad, j, sh);
}

// ---------------------------------------------------------------------------
// K2: alpha; phi, r update; <r,r>; forward real FFT of the r rows -> spec
// (also the start kernel when n < 0: r = rhs - mean, phi = 0)
// ---------------------------------------------------------------------------
//
// The row kernels: T = M / 8 threads a row, each with the row's items lane +
// u T, u < 8 (two cells an item, one 16-byte load), which are also what the
// first radix-8 pass of its transform takes, so that pass runs on registers.
// A block is NT threads: one wavefront (NT / T rows of it) where T <= 64, else
// T.  Every load of the kernel (cells, twiddles, the split table) is
// unconditional, from clamped places, and goes out before the stop flag and
// the scalar sums are waited for; LDS is padded (SkPad).  With guarded loads,
// the twiddles staged one by one and the split table read where it is used, a
// chain of ~12 us of memory latency whatever the grid, the forward kernel
// took 19.6 us and the inverse one 13.7 at 1024^2 (13.4 and 10.9 at 128 x 256);
// now 14.2 and 8.3 (7.9 and 5.3).  One wavefront a block against 256 threads
// (NT / T rows): 15.0 and 8.7 against 15.8 and 9.4 at 1024^2, 14.1 and 9.5
// against 15.0 and 11.6 at 768 x 491 (12.9 and 8.2 since the index arithmetic
// there is shifts), 7.9 and 5.3 against 9.9 and 7.0 at 128 x 256.
#define RU 8
#define TWK 8                    // twiddle pairs a thread stages: M <= 8 NT
typedef double v2d __attribute__((ext_vector_type(2)));

template <int NT> struct RowGeo {
    int M, T, q, lane, j, LS;    // LS: LDS doubles of one row's real (or imaginary) part
    bool act;
};
template <bool P2, int NT> __device__ __forceinline__ RowGeo<NT> row_geo(const pvk_grid &g, const pvk_fft &F, int R)
{
    RowGeo<NT> o;
    o.M = F.mx;
    o.T = o.M >> 3;
    o.q = P2 ? (int)threadIdx.x >> (F.logmx - 3) : (int)threadIdx.x / o.T;
    o.lane = threadIdx.x - o.q * o.T;
    o.LS = o.M + (o.M >> 3);
    const int j = blockIdx.x * R + o.q;
    o.act = o.q < R && j < g.NYM;
    o.j = min(j, g.NYM - 1);
    o.q = min(o.q, R - 1);
    return o;
}
// this thread's share of the twiddle table, on its way to LDS
template <int NT> __device__ __forceinline__ void tw_load(int M, const double *tw, v2d *v)
{
#pragma unroll
    for (int k = 0; k < TWK; k++) v[k] = *(const v2d *)(tw + 2 * min((int)threadIdx.x + k * NT, M - 1));
}
template <int NT> __device__ __forceinline__ void tw_stage(int M, const v2d *v, double *lds)
{
#pragma unroll
    for (int k = 0; k < TWK; k++) {
        const int t = threadIdx.x + k * NT;
        if (t < M) *(v2d *)(lds + 2 * t) = v[k];
    }
}
// Sums of partials by a block of NT threads, the same order in every block:
// the loads (16 a thread and array in flight; more partials than that are
// added in a loop) and, later, the sums.
#define RPB 16
template <int NT> struct RowSums { double a[RPB], b[RPB]; };
template <int NT> __device__ __forceinline__ void row_sums_load(const double *pa, int na, const double *pb, int nb, RowSums<NT> &v)
{
#pragma unroll
    for (int k = 0; k < RPB; k++) {
        const int b = threadIdx.x + k * NT;
        v.a[k] = (b < na) ? pa[b] : 0.0;
        v.b[k] = (b < nb) ? pb[b] : 0.0;
    }
}
template <int NT> __device__ __forceinline__ void row_sums(const double *pa, int na, const double *pb, int nb,
                                                           const RowSums<NT> &v, double *sh, double &ra, double &rb)
{
    const int t = threadIdx.x;
    double sa = 0.0, sb = 0.0;
#pragma unroll
    for (int k = 0; k < RPB; k++) { sa += v.a[k]; sb += v.b[k]; }
    for (int b = t + RPB * NT; b < na; b += NT) sa += pa[b];
    for (int b = t + RPB * NT; b < nb; b += NT) sb += pb[b];
    sa = lane_first(wave_sum(sa));
    sb = lane_first(wave_sum(sb));
    if (NT > 64) {
        if ((t & 63) == 0) { sh[t >> 6] = sa; sh[8 + (t >> 6)] = sb; }
        __syncthreads();
        sa = sh[0];
        sb = sh[8];
        for (int w = 1; w < NT / 64; w++) { sa += sh[w]; sb += sh[8 + w]; }
        __syncthreads();
    }
    ra = sa;
    rb = sb;
}
template <int NT> __device__ __forceinline__ void row_partial(double v, double *part, double *sh)
{
    const int t = threadIdx.x;
    v = wave_sum(v);
    if (NT > 64) {
        if ((t & 63) == 0) sh[t >> 6] = v;
        __syncthreads();
        for (int w = 1; t == 0 && w < NT / 64; w++) v += sh[w];
    }
    if (t == 0) part[blockIdx.x] = v;
}
template <bool INV, bool P2>
__device__ __forceinline__ void rows_fft(double *vr, double *vi, double *sr, double *si, int M, int logM, const double *tw,
                                         int lane, int T, bool act)
{
    if (P2) sk_fft_regs<INV, SkPad>(vr, vi, sr, si, logM, tw, lane, T);
    else sg_fft_regs<INV, SkPad>(vr, vi, sr, si, M, tw, lane, T, act);
}

// MODE: the step of iteration n, the start (r = rhs - mean, phi = 0), a warm
// restart (r = rhs - mean - A phi0, in Ad) or the transform of r as it is
enum { ROW_STEP, ROW_START, ROW_WARM, ROW_PLAIN };
template <bool P2, int NT, int MODE>
__global__ void __launch_bounds__(NT) k_pcg_update_fwd(pvk_grid g, pvk_fft F, pvk_scal *sc, pvk_pcg w, int n)
{
    extern __shared__ double lds[];
    __shared__ double sh[16];
    const int P = g.P, N = g.NXM, R = w.rrow;
    const RowGeo<NT> o = row_geo<P2, NT>(g, F, R);
    const int M = o.M, T = o.T, lane = o.lane, j = o.j;
    double *tw = lds, *sr = lds + 2 * M + 2 * o.q * o.LS, *si = sr + o.LS;
    const double *pa = (MODE == ROW_STEP) ? w.rz[n & 1] : w.mean, *pb = w.dad[n & 1];
    const int na = (MODE == ROW_STEP) ? w.nrz : (MODE == ROW_PLAIN ? 0 : w.nmean), nb = (MODE == ROW_STEP) ? w.ndad : 0;
    const double *__restrict__ d = w.d[n & 1], *__restrict__ Ad = w.Ad;
    const double *__restrict__ src = (MODE == ROW_STEP || MODE == ROW_PLAIN) ? w.r : w.rhs;
    double *__restrict__ phi = w.phi, *__restrict__ r = w.r;
    RowSums<NT> ps;
    v2d x[RU], e[RU], rv[RU], a[RU], rt[RU], tv[TWK];
#define ROW2(f, u) (*(const v2d *)&AT(f, 2 * (lane + (u) * T), j))
    if (MODE != ROW_PLAIN) row_sums_load<NT>(pa, na, pb, nb, ps);
#pragma unroll
    for (int u = 0; u < RU; u++) {
        rv[u] = ROW2(src, u);
        if (MODE == ROW_STEP || MODE == ROW_WARM) a[u] = ROW2(Ad, u);
    }
    tw_load<NT>(M, F.wx, tv);
#pragma unroll
    for (int u = 0; u < RU; u++) {
        if (MODE == ROW_STEP) { x[u] = ROW2(phi, u); e[u] = ROW2(d, u); }
        rt[u] = *(const v2d *)(F.rtx + 2 * (lane + u * T));
    }
    const v2d rtM = *(const v2d *)(F.rtx + 2 * M);
    if (w.chb == 0.0 && sc->p_done) return;
    double alpha = 0.0, mean = 0.0, s0, s1;
    if (MODE != ROW_PLAIN) row_sums<NT>(pa, na, pb, nb, ps, sh, s0, s1);
    if (MODE == ROW_STEP) alpha = s0 / s1;
    else if (MODE != ROW_PLAIN) mean = s0 / ((double)g.NXM * (double)g.NYM);
    tw_stage<NT>(M, tv, tw);
    double vr[RU], vi[RU], acc = 0.0;
#pragma unroll
    for (int u = 0; u < RU; u++) {
        if (MODE == ROW_STEP) {
            rv[u].x = rv[u].x - alpha * a[u].x;
            rv[u].y = rv[u].y - alpha * a[u].y;
        } else if (MODE == ROW_WARM) {
            rv[u].x = rv[u].x - mean - a[u].x;
            rv[u].y = rv[u].y - mean - a[u].y;
        } else if (MODE == ROW_START) {
            rv[u].x = rv[u].x - mean;
            rv[u].y = rv[u].y - mean;
        }
        vr[u] = rv[u].x;
        vi[u] = rv[u].y;
        if (o.act) acc += rv[u].x * rv[u].x + rv[u].y * rv[u].y;
    }
    if (o.act && MODE != ROW_PLAIN) {
#pragma unroll
        for (int u = 0; u < RU; u++) {
            v2d *pp = (v2d *)&AT(phi, 2 * (lane + u * T), j);
            if (MODE == ROW_STEP) {
                v2d t;
                t.x = x[u].x + alpha * e[u].x;
                t.y = x[u].y + alpha * e[u].y;
                *pp = t;
            } else if (MODE == ROW_START) *pp = (v2d){0.0, 0.0};
            *(v2d *)&AT(r, 2 * (lane + u * T), j) = rv[u];
        }
    }
#undef ROW2
    __syncthreads();                            // twiddles staged
    rows_fft<false, P2>(vr, vi, sr, si, M, F.logmx, tw, lane, T, o.act);
    row_partial<NT>(acc, w.rr, sh);
    const double scale = 1.0 / (double)N;
    // X_k, k < M (and X_M): halfcomplex row of spec
    double *row = F.spec + (size_t)j * N;
    if (!o.act) return;
#pragma unroll
    for (int u = 0; u < RU; u++) {
        const int k = lane + u * T, kb = (k == 0) ? 0 : M - k;
        const cplx2 X = rpost(sr[SkPad::at(k)], si[SkPad::at(k)], sr[SkPad::at(kb)], si[SkPad::at(kb)], rt[u].x, rt[u].y);
        row[k] = X.x * scale;
        if (k > 0) row[N - k] = X.y * scale;
    }
    if (lane == 0) row[M] = rpost(sr[0], si[0], sr[0], si[0], rtM.x, rtM.y).x * scale;
}

// ---------------------------------------------------------------------------
// K3 / K5: 32 x 32 tiled transpose of an (rows x cols) row-major array;
// with check != 0 the stop test of iteration n runs first (all blocks).
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(NTH) k_transpose(pvk_scal *sc, pvk_pcg w, const double *__restrict__ in,
                                                  double *__restrict__ out, int rows, int cols, int check, int n,
                                                  double tol, int maxit)
{
    __shared__ double tile[32][33];
    __shared__ double sh[NTH];
    // a stop flag set by an earlier iteration leaves <r,r> stale: no recount
    if (w.chb == 0.0 && sc->p_done) return;
    if (check && n != -3) {                 // n = -3: a plain M_fft solve, no stop test
        double rr = block_sum(w.rr, w.nrr, sh);
        // n = -1: cold start, ||r0|| = ||b - mean|| is the reference norm;
        // n = -2: warm restart, the cold start's norm is kept
        double bn = (n == -1) ? ((sqrt(rr) == 0.0) ? 1.0 : sqrt(rr)) : sc->p_bnorm;
        double rel = sqrt(rr) / bn;
        bool done = (rel <= tol) || (n + 1 >= maxit && n >= 0);
        if (blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x == 0) {
            if (n == -1) sc->p_bnorm = bn;
            sc->p_res = rel;
            sc->p_iter = (n < 0) ? 0 : n + 1;
            if (done) sc->p_done = (rel <= tol) ? 1 : 3;
        }
        if (done) return;
    }
    const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;   // 32 x 8
    const int c0 = blockIdx.x * 32, r0 = blockIdx.y * 32;
    double v[4];
#pragma unroll
    for (int k = 0; k < 4; k++) {
        int r = r0 + ty + 8 * k, c = c0 + tx;
        v[k] = (r < rows && c < cols) ? in[(size_t)r * cols + c] : 0.0;
    }
#pragma unroll
    for (int k = 0; k < 4; k++) tile[ty + 8 * k][tx] = v[k];
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 4; k++) {
        int r = c0 + ty + 8 * k, c = r0 + tx;      // out is cols x rows
        if (r < cols && c < rows) out[(size_t)r * rows + c] = tile[tx][ty + 8 * k];
    }
}

// ---------------------------------------------------------------------------
// K4: per row of specT (one halfcomplex x-index i, length NYM along y):
// DCT-II, multiply by -1/(lamx_i + lamy_k) ((0,0) -> 0), DCT-III.
// DCT-II of x_n as a real FFT of v_nn = x_vmap(nn) (evens ascending, odds
// descending); the row is read and written contiguously and permuted in LDS.
// ---------------------------------------------------------------------------
// LDS slot (sr or si, index) of row element n under the even/odd reordering
__device__ __forceinline__ int dct_slot(int n, int N)
{
    const int nn = (n & 1) ? N - 1 - (n >> 1) : (n >> 1);
    return nn;                       // complex index nn >> 1, part nn & 1
}

__global__ void __launch_bounds__(NTH) k_dct_rows(pvk_grid g, pvk_fft F, pvk_scal *sc, pvk_pcg w, double *specT)
{
    extern __shared__ double lds[];
    if (w.chb == 0.0 && sc && sc->p_done) return;
    const double a_ch = (w.chb > 0.0) ? 1.0 / (sc->dt * c_BET[w.chstage]) : 0.0;
    const int logM = F.logmy, M = 1 << logM, logN = logM + 1, N = 2 * M, R = w.rdct, NX = g.NXM, RM = R * M;
    double *sr = lds, *si = lds + RM;
    double *tw = stage_twiddles(lds, RM, M, F.wy);
    const int i0 = blockIdx.x * R;
    // R rows of N reals = 2 RM values: 2 IT per thread, contiguous per row
    {
        double v[2 * IT];
#pragma unroll
        for (int u = 0; u < 2 * IT; u++) {
            const int t = threadIdx.x + u * NTH, q = t >> logN, nidx = t & (N - 1), i = i0 + q;
            v[u] = (t < 2 * RM && i < NX) ? specT[(size_t)i * N + nidx] : 0.0;
        }
#pragma unroll
        for (int u = 0; u < 2 * IT; u++) {
            const int t = threadIdx.x + u * NTH, q = t >> logN, nidx = t & (N - 1);
            if (t < 2 * RM) {
                const int nn = dct_slot(nidx, N);
                ((nn & 1) ? si : sr)[q * M + (nn >> 1)] = v[u];
            }
        }
    }
    __syncthreads();
    const int lT = sk_logT(logM), T = 1 << lT, qq = threadIdx.x >> lT, lane = threadIdx.x & (T - 1);
    sk_fft<false>(sr + qq * M, si + qq * M, logM, tw, lane, T);
    // spectral step on the pairs (k, M - k): k < M/2 as IT/2 items per
    // thread, k = M/2 by threads t < R
    const int logH = logM - 1, H = M >> 1;
    cplx2 Ya[IT / 2 + 1], Yb[IT / 2 + 1];
    auto pair = [&](int q, int k, cplx2 &ya, cplx2 &yb) {
        const int i = i0 + q;
        const int kk[2] = {k, M - k};
        cplx2 Xp[2];
        const double lx = (i < NX) ? F.lamx[i] : 1.0;
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const int kv = kk[h];
            cplx2 V = rpost(sr, si, q * M, M, kv, F.rty);
            double c = F.dcty[2 * kv], s = F.dcty[2 * kv + 1];
            double Ck = c * V.x + s * V.y;
            double Sk = c * V.y - s * V.x;
            double CNk = -Sk;
            double gk, gN;
            if (w.chb > 0.0) {          // (a_dt + bih lambda^2)^-1, no null mode
                const double lk = lx + F.lamy[kv];
                gk = 1.0 / (a_ch + w.chb * lk * lk);
                gN = 0.0;
                if (kv != 0) {
                    const double lN = lx + F.lamy[N - kv];
                    gN = 1.0 / (a_ch + w.chb * lN * lN);
                }
            } else {
                gk = (kv == 0 && i == 0) ? 0.0 : -1.0 / (lx + F.lamy[kv]);
                gN = (kv == 0) ? 0.0 : -1.0 / (lx + F.lamy[N - kv]);
            }
            double Cp = Ck * gk, CNp = (kv == 0) ? 0.0 : CNk * gN;
            Xp[h].x = c * Cp + s * CNp;
            Xp[h].y = s * Cp - c * CNp;
        }
        ya = rpre(Xp[0], Xp[1], F.rty[2 * k], F.rty[2 * k + 1]);
        yb = rpre(Xp[1], Xp[0], F.rty[2 * (M - k)], F.rty[2 * (M - k) + 1]);
    };
#pragma unroll
    for (int u = 0; u < IT / 2; u++) {
        const int t = threadIdx.x + u * NTH;
        if (t < R * H) pair(t >> logH, t & (H - 1), Ya[u], Yb[u]);
    }
    if ((int)threadIdx.x < R) pair(threadIdx.x, H, Ya[IT / 2], Yb[IT / 2]);
    __syncthreads();
#pragma unroll
    for (int u = 0; u < IT / 2; u++) {
        const int t = threadIdx.x + u * NTH;
        if (t < R * H) {
            const int q = t >> logH, k = t & (H - 1);
            sr[q * M + k] = Ya[u].x; si[q * M + k] = Ya[u].y;
            if (k > 0) { sr[q * M + M - k] = Yb[u].x; si[q * M + M - k] = Yb[u].y; }
        }
    }
    if ((int)threadIdx.x < R) {
        const int q = threadIdx.x;
        sr[q * M + H] = Ya[IT / 2].x; si[q * M + H] = Ya[IT / 2].y;
    }
    __syncthreads();
    sk_fft<true>(sr + qq * M, si + qq * M, logM, tw, lane, T);
    const double invN = 1.0 / (double)N;
#pragma unroll
    for (int u = 0; u < 2 * IT; u++) {
        const int t = threadIdx.x + u * NTH, q = t >> logN, nidx = t & (N - 1), i = i0 + q;
        if (t < 2 * RM && i < NX) {
            const int nn = dct_slot(nidx, N);
            specT[(size_t)i * N + nidx] = ((nn & 1) ? si : sr)[q * M + (nn >> 1)] * invN;
        }
    }
}

// ---------------------------------------------------------------------------
// K4': the y solve of the FFT preconditioner: one tridiagonal system per
// halfcomplex column of spec (psolve_fft.c:1536-1802, tridiag :141-163), in
// place on spec[j][i] -- no transposes.  On the uniform grid with zero
// gradient at the walls every row of column k but the end ones reads
//   c (x_{j-1} - (2 + m) x_j + x_{j+1}) = f_j,   c = 1 / dy^2, m = mw_k / c,
// and with q + 1/q = 2 + m, 0 < q < 1, the walls' reflections included,
//   x_j = -K (y+_j + y-_j - f_j),  y+_j = f_j + q y+_{j-1},  y-_j = f_j + q y-_{j+1},
//   K = q / (1 - q^2) / c,
//   y+_{-1} = (A + q^N B) / (1 - q^{2N}),  y-_N = (B + q^N A) / (1 - q^{2N}),
// A and B the values of y- at row 0 and of y+ at row N - 1 for zero starts.
// So a column is two independent first-order recurrences: segments of tri_l
// rows a thread (lane kk of a row group owns column i0 + kk, so consecutive
// lanes read consecutive doubles of a row), their carries combined by a scan
// with powers of q.  q, K, q^N and 1 / (1 - q^{2N}) are tables (per column), so
// the kernel has no division; the elimination it replaces (partitioned
// Thomas, a pivot division a row and a cyclic reduction of the separators
// with two divisions a step) took 16.6 us at 1024^2 against 10.2 now, and 13.2
// at 768 x 491 against 7.7.
// Column 0 (m = 0, row 0 replaced by the pin x_0 = 0) is two running sums:
// x_{j+1} - x_j = -sum_{i > j} f_i / c.  With mean removal (the PCG's
// pseudo-inverse) it is shifted to zero mean afterwards.  In the PCG this
// kernel also runs the stop test of iteration n (every block, from the <r, r>
// partials).
// ---------------------------------------------------------------------------
// b^e, 0 <= e < 2^BITS
template <int BITS> __device__ __forceinline__ double tri_pow(double b, int e)
{
    double p = 1.0;
#pragma unroll
    for (int k = 0; k < BITS; k++) {
        if ((e >> k) & 1) p *= b;
        b *= b;
    }
    return p;
}

// The carries of a scan over the segments of each column: with segment
// values ep (prefix) and em (suffix) and the ratio Q of a whole segment, V_s =
// ep_s + Q V_{s-1} and W_s = em_s + Q W_{s+1}: returns V_{s-1}, W_{s+1} and W_0.
// pl = Q^sl, pr = Q^(segments of the wavefront after this one), QG = Q^(segments
// a wavefront).  Lanes of segments past the last carry zeros.  tp, tm: a
// wavefront's totals.
struct TriScan { double v, w, w0; };
__device__ __forceinline__ TriScan tri_scan(double ep, double em, double Q, double pl, double pr, double QG, int KW, int kk,
                                            int nw, double (*tp)[64], double (*tm)[64])
{
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    double qk = Q;
    for (int off = KW; off < 64; off <<= 1) {
        const double up = __shfl_up(ep, off, 64), dn = __shfl_down(em, off, 64);
        if (lane >= off) ep = __builtin_fma(qk, up, ep);
        if (lane + off < 64) em = __builtin_fma(qk, dn, em);
        qk *= qk;
    }
    double cp = __shfl_up(ep, KW, 64), cm = __shfl_down(em, KW, 64);
    if (lane < KW) cp = 0.0;
    if (lane + KW >= 64) cm = 0.0;
    __syncthreads();                        // tp, tm free again
    if (lane + KW >= 64) tp[wv][kk] = ep;
    if (lane < KW) tm[wv][kk] = em;
    __syncthreads();
    double cw = 0.0, mw = 0.0, a = 0.0;
    for (int u = 0; u < wv; u++) cw = __builtin_fma(QG, cw, tp[u][kk]);
    for (int u = nw - 1; u >= 0; u--) {
        if (u == wv) mw = a;
        a = __builtin_fma(QG, a, tm[u][kk]);
    }
    TriScan r;
    r.v = __builtin_fma(pl, cw, cp);
    r.w = __builtin_fma(pr, mw, cm);
    r.w0 = a;
    return r;
}

template <int TRI_LMAX>
__global__ void __launch_bounds__(512) k_tri_cols(pvk_grid g, pvk_fft F, pvk_scal *sc, pvk_pcg w, int n,
                                                   double tol, int maxit)
{
    __shared__ double tp[8][64], tm[8][64], tb[64], ts[8];
    const int NX = g.NXM, NY = g.NYM, KW = F.tri_kw, S = F.tri_s, L = F.tri_l, t = threadIdx.x;
    const int nt = blockDim.x, nw = nt >> 6, lane = t & 63, wv = t >> 6, G = 64 >> F.tri_lkw;
    const int kk = t & (KW - 1), s = t >> F.tri_lkw, sl = lane >> F.tri_lkw;
    const int grp = xcd_band(blockIdx.x, gridDim.x);     // neighbouring column groups share an XCD's L2
    const int col = grp * KW + kk, cc = min(col, NX - 1), j0 = s * L;
    const int nrow = (col < NX && s < S) ? min(L, NY - j0) : 0, rem = NY - (S - 1) * L;
    double *spec = F.spec;
    // every load, unconditional from clamped places, before the stop flag and
    // the sums are waited for
    double f[TRI_LMAX];
#pragma unroll
    for (int l = 0; l < TRI_LMAX; l++) f[l] = spec[(size_t)min(j0 + min(l, L - 1), NY - 1) * NX + cc];
    const double q = F.tri_q[cc], K = F.tri_k[cc], qN = F.tri_qn[cc], den = F.tri_den[cc];
    double rr = 0.0, rp[8];
#pragma unroll
    for (int k = 0; k < 8; k++) rp[k] = (n != -3 && t + k * nt < w.nrr) ? w.rr[t + k * nt] : 0.0;
    if (sc->p_done) return;
#pragma unroll
    for (int k = 0; k < 8; k++) rr += rp[k];
    if (n != -3)
        for (int b = t + 8 * nt; b < w.nrr; b += nt) rr += w.rr[b];
    if (n != -3) {                          // stop test of iteration n (as the transpose stage does)
        rr = wave_sum(rr);
        if (lane == 0) ts[wv] = rr;
        __syncthreads();
        rr = ts[0];
        for (int u = 1; u < nw; u++) rr += ts[u];
        const double bn = (n == -1) ? ((sqrt(rr) == 0.0) ? 1.0 : sqrt(rr)) : sc->p_bnorm;
        const double rel = sqrt(rr) / bn;
        const bool done = (rel <= tol) || (n + 1 >= maxit && n >= 0);
        if (blockIdx.x == 0 && t == 0) {
            if (n == -1) sc->p_bnorm = bn;
            sc->p_res = rel;
            sc->p_iter = (n < 0) ? 0 : n + 1;
            if (done) sc->p_done = (rel <= tol) ? 1 : 3;
        }
        if (done) return;
    }
    // powers of q for the carries: Q = q^L, Q^sl, Q^(G - 1 - sl), Q^G, Q^s,
    // q^(rows after this segment)
    const double Q = tri_pow<5>(q, L), qr = tri_pow<5>(q, rem);
    const double pl = tri_pow<6>(Q, sl), pr = tri_pow<6>(Q, G - 1 - sl), QG = tri_pow<7>(Q, G);
    const double ps = pl * tri_pow<4>(QG, wv), pn = (s < S - 1) ? qr * tri_pow<9>(Q, max(S - 2 - s, 0)) : 1.0;
#pragma unroll
    for (int l = 0; l < TRI_LMAX; l++) f[l] = (l < nrow) ? f[l] : 0.0;
    // zero-start values at the segment's end (y+) and start (y-)
    double ep = 0.0, em = 0.0;
#pragma unroll
    for (int l = 0; l < TRI_LMAX; l++) {
        if (l < nrow) ep = __builtin_fma(q, ep, f[l]);
        em = __builtin_fma(q, em, f[TRI_LMAX - 1 - l]);      // rows past the segment: zeros
    }
    const TriScan c = tri_scan(ep, em, Q, pl, pr, QG, KW, kk, nw, tp, tm);
    if (s == S - 1) tb[kk] = __builtin_fma(qr, c.v, ep);
    __syncthreads();
    const double A = c.w0, B = tb[kk];
    double yp = __builtin_fma(ps, __builtin_fma(qN, B, A) * den, c.v);
    double ym = __builtin_fma(pn, __builtin_fma(qN, A, B) * den, c.w);
    double x[TRI_LMAX];
#pragma unroll
    for (int l = 0; l < TRI_LMAX; l++) {
        if (l < nrow) yp = __builtin_fma(q, yp, f[l]);
        x[l] = yp - f[l];
    }
#pragma unroll
    for (int l = TRI_LMAX - 1; l >= 0; l--) {
        if (l < nrow) ym = __builtin_fma(q, ym, f[l]);
        x[l] = -K * (x[l] + ym);
    }
    if (grp == 0) {                          // block-uniform: column 0 lives in group 0
        double e = 0.0;
#pragma unroll
        for (int l = 0; l < TRI_LMAX; l++) e += f[l];
        double run = tri_scan(0.0, e, 1.0, 1.0, 1.0, 1.0, KW, kk, nw, tp, tm).w, d[TRI_LMAX], ed = 0.0;
#pragma unroll
        for (int l = TRI_LMAX - 1; l >= 0; l--) {            // x_{j+1} - x_j
            d[l] = (l < nrow) ? -(run * F.tri_ic) : 0.0;
            run += f[l];
        }
#pragma unroll
        for (int l = 0; l < TRI_LMAX; l++) ed += d[l];
        double x0 = tri_scan(ed, 0.0, 1.0, 1.0, 1.0, 1.0, KW, kk, nw, tp, tm).v, sum = 0.0;
#pragma unroll
        for (int l = 0; l < TRI_LMAX; l++) {
            const double v = x0;
            x0 += d[l];
            d[l] = v;
            sum += (l < nrow) ? v : 0.0;
        }
        double shift = 0.0;
        if (!w.keep_pin) {
            sum = wave_sum(col == 0 ? sum : 0.0);
            __syncthreads();
            if (lane == 0) ts[wv] = sum;
            __syncthreads();
            for (int u = 0; u < nw; u++) shift += ts[u];
            shift /= (double)NY;
        }
        if (col == 0)
#pragma unroll
            for (int l = 0; l < TRI_LMAX; l++) x[l] = d[l] - shift;
    }
#pragma unroll
    for (int l = 0; l < TRI_LMAX; l++)
        if (l < nrow) spec[(size_t)(j0 + l) * NX + col] = x[l];
}

// ---------------------------------------------------------------------------
// K6: z = inverse real FFT of spec rows; partials <r, z> into rz[(n+1)&1]
// ---------------------------------------------------------------------------
template <bool P2, int NT>
__global__ void __launch_bounds__(NT) k_ifft_rows_dot(pvk_grid g, pvk_fft F, pvk_scal *sc, pvk_pcg w, int n)
{
    extern __shared__ double lds[];
    __shared__ double sh[16];
    const int P = g.P, N = g.NXM, R = w.rrow;
    const RowGeo<NT> o = row_geo<P2, NT>(g, F, R);
    const int M = o.M, T = o.T, lane = o.lane, j = o.j;
    double *tw = lds, *sr = lds + 2 * M + 2 * o.q * o.LS, *si = sr + o.LS;
    const double *__restrict__ r = w.r;
    double *__restrict__ z = w.z;
    const double *row = F.spec + (size_t)j * N;
    v2d rt[RU], rv[RU], tv[TWK];
    double xr[RU], xi[RU], mr[RU], mi[RU];
#pragma unroll
    for (int u = 0; u < RU; u++) {              // X_k and X_{M-k}
        const int k = lane + u * T;
        xr[u] = row[k];
        xi[u] = row[k > 0 ? N - k : 0];
        mr[u] = row[M - k];
        mi[u] = row[M + k];
    }
    tw_load<NT>(M, F.wx, tv);
#pragma unroll
    for (int u = 0; u < RU; u++) rt[u] = *(const v2d *)(F.rtx + 2 * (lane + u * T));
#pragma unroll
    for (int u = 0; u < RU; u++) rv[u] = *(const v2d *)&AT(r, 2 * (lane + u * T), j);
    if (w.chb == 0.0 && sc->p_done) return;
    tw_stage<NT>(M, tv, tw);
    double vr[RU], vi[RU], acc = 0.0;
#pragma unroll
    for (int u = 0; u < RU; u++) {
        const int k = lane + u * T;
        cplx2 a, b;
        a.x = xr[u];
        a.y = (k == 0) ? 0.0 : xi[u];
        b.x = mr[u];
        b.y = (k == 0) ? 0.0 : mi[u];
        const cplx2 Y = rpre(a, b, rt[u].x, rt[u].y);
        vr[u] = Y.x;
        vi[u] = Y.y;
    }
    __syncthreads();                            // twiddles staged
    rows_fft<true, P2>(vr, vi, sr, si, M, F.logmx, tw, lane, T, o.act);
    if (o.act)
#pragma unroll
        for (int u = 0; u < RU; u++) {
            const int m = lane + u * T;
            v2d t;
            t.x = sr[SkPad::at(m)];
            t.y = si[SkPad::at(m)];
            *(v2d *)&AT(z, 2 * m, j) = t;
            acc += rv[u].x * t.x + rv[u].y * t.y;
        }
    row_partial<NT>(acc, w.rz[(n < 0) ? 0 : ((n + 1) & 1)], sh);
}

__global__ void k_pcg_clear_done(pvk_scal *sc) { sc->p_done = 0; }
extern "C" void pvk_pcg_clear_done(pvk_scal *sc, hipStream_t s)
{
    hipLaunchKernelGGL(k_pcg_clear_done, dim3(1), dim3(1), 0, s, sc);
}

// sc->red[slot] = sum of the <r, z> partials of slot rzs (the energy-norm
// proxy <r, M r> that judges a warm start)
__global__ void __launch_bounds__(NTH) k_pcg_gamma(pvk_scal *sc, pvk_pcg w, int rzs, int slot)
{
    __shared__ double sh[NTH];
    const double v = block_sum(w.rz[rzs], w.nrz, sh);
    if (threadIdx.x == 0) sc->red[slot] = v;
}
extern "C" void pvk_pcg_gamma(pvk_scal *sc, const pvk_pcg *w, int rzs, int slot, hipStream_t s)
{
    hipLaunchKernelGGL(k_pcg_gamma, dim3(1), dim3(NTH), 0, s, sc, *w, rzs, slot);
}

// out = A x (the operator of k_pcg_apply on a given field; faces formed by
// the start of the solve)
__global__ void __launch_bounds__(NTH) k_pcg_opx(pvk_grid g, pvk_pcg w, const double *__restrict__ x,
                                                double *__restrict__ out)
{
    __shared__ double sh[NTH];
    const int P = g.P, NXM = g.NXM, NYM = g.NYM, j = xcd_band(blockIdx.x, gridDim.x);
    const int jn = (j + 1 == NYM) ? j : j + 1, js = (j == 0) ? 0 : j - 1;
    double sacc = 0.0;
    for (int i = threadIdx.x; i < NXM; i += NTH) {
        const int ie = (i + 1 == NXM) ? 0 : i + 1, iw = (i == 0) ? NXM - 1 : i - 1;
        const double d0 = AT(x, i, j);
        const double v = AT(w.bx, i, j) * (AT(x, ie, j) - d0) - AT(w.bx, i - 1, j) * (d0 - AT(x, iw, j)) +
                         AT(w.by, i, j) * (AT(x, i, jn) - d0) - AT(w.by, i, j - 1) * (d0 - AT(x, i, js));
        AT(out, i, j) = v;
        sacc += v;
    }
    if (w.sad) block_store_partial(sacc, w.sad, j, sh);
}
extern "C" void pvk_pcg_opx(const pvk_grid *g, const pvk_pcg *w, const double *x, double *out, hipStream_t s)
{
    hipLaunchKernelGGL(k_pcg_opx, dim3(g->NYM), dim3(NTH), 0, s, *g, *w, x, out);
}

// partial sums of rhs (mean removal before the solve)
__global__ void __launch_bounds__(NTH) k_pcg_mean(pvk_grid g, pvk_scal *sc, pvk_pcg w)
{
    __shared__ double sh[NTH];
    if (blockIdx.x == 0 && threadIdx.x == 0) { sc->p_done = 0; sc->p_iter = 0; }
    const int P = g.P, NXM = g.NXM;
    const int j0 = blockIdx.x * w.band, j1 = min(g.NYM, j0 + w.band);
    double acc = 0.0;
    for (int c = threadIdx.x; c < (j1 - j0) * NXM; c += NTH) {
        int j = j0 + c / NXM, i = c - (c / NXM) * NXM;
        acc += AT(w.rhs, i, j);
    }
    block_store_partial(acc, w.mean, blockIdx.x, sh);
}

// threads of a block of the row kernels, and its LDS: R padded rows of N/2
// complex values + the N/2 complex twiddles
extern "C" int pvk_fft_row_threads(int N) { return N / 16 <= 64 ? 64 : (N / 16 <= 128 ? 128 : 256); }
static size_t lds_row(int R, int N)
{
    const size_t M = N / 2;
    return (2 * M + 2 * (size_t)R * (M + M / 8)) * sizeof(double);
}
#define FWD_STEP(P2, NT) k_pcg_update_fwd<P2, NT, ROW_STEP>
#define FWD_START(P2, NT) k_pcg_update_fwd<P2, NT, ROW_START>
#define FWD_WARM(P2, NT) k_pcg_update_fwd<P2, NT, ROW_WARM>
#define FWD_PLAIN(P2, NT) k_pcg_update_fwd<P2, NT, ROW_PLAIN>
#define INV_DOT(P2, NT) k_ifft_rows_dot<P2, NT>

// Rows of 3888 and 4096 take more than 64 KiB of dynamic LDS (the padding; up
// to 68 KiB), which a kernel must be allowed (gfx950: up to 160 KiB a
// workgroup): their forms are, on the current device, when a handle of that
// length is made.  A refusal leaves the launch to report the error.
extern "C" void pvk_fft_row_allow(int N)
{
    static std::mutex mu;                // handles may be made by several host threads
    const void *const k[] = {(const void *)FWD_STEP(true, 256),   (const void *)FWD_STEP(false, 256),
                             (const void *)FWD_START(true, 256),  (const void *)FWD_START(false, 256),
                             (const void *)FWD_WARM(true, 256),   (const void *)FWD_WARM(false, 256),
                             (const void *)FWD_PLAIN(true, 256),  (const void *)FWD_PLAIN(false, 256),
                             (const void *)(INV_DOT(true, 256)),  (const void *)(INV_DOT(false, 256))};
    if (lds_row(pvk_fft_row_threads(N) / (N / 16), N) <= 65536) return;
    std::lock_guard<std::mutex> lk(mu);
    for (const void *f : k)
        if (hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024) != hipSuccess)
            (void)hipGetLastError();
}

#define ROWS(KERNEL, N)                                                                                                    \
    do {                                                                                                                   \
        const int nt = pvk_fft_row_threads(g->NXM), nrow = (g->NYM + w->rrow - 1) / w->rrow;                               \
        const size_t l = lds_row(w->rrow, g->NXM);                                                                         \
        const dim3 gr(nrow);                                                                                               \
        if (F->pow2x && nt == 64) hipLaunchKernelGGL((KERNEL(true, 64)), gr, dim3(64), l, s, *g, *F, sc, *w, N);           \
        else if (F->pow2x && nt == 128) hipLaunchKernelGGL((KERNEL(true, 128)), gr, dim3(128), l, s, *g, *F, sc, *w, N);   \
        else if (F->pow2x) hipLaunchKernelGGL((KERNEL(true, 256)), gr, dim3(256), l, s, *g, *F, sc, *w, N);                \
        else if (nt == 64) hipLaunchKernelGGL((KERNEL(false, 64)), gr, dim3(64), l, s, *g, *F, sc, *w, N);                 \
        else if (nt == 128) hipLaunchKernelGGL((KERNEL(false, 128)), gr, dim3(128), l, s, *g, *F, sc, *w, N);              \
        else hipLaunchKernelGGL((KERNEL(false, 256)), gr, dim3(256), l, s, *g, *F, sc, *w, N);                             \
    } while (0)
// R columns of N/2 complex values + the N/2 complex twiddles (y transforms)
static size_t lds_rows(int R, int N) { return ((size_t)R * (size_t)(N / 2) * 2 + (size_t)N) * sizeof(double); }

extern "C" void pvk_pcg_start(const pvk_grid *g, const pvk_fft *F, pvk_scal *sc, const pvk_pcg *w, double tol,
                              hipStream_t s)
{
    int nband = (g->NYM + w->band - 1) / w->band;
    hipLaunchKernelGGL(k_pcg_faces, dim3(g->NYM + 1), dim3(NTH), 0, s, *g, *w);
    hipLaunchKernelGGL(k_pcg_mean, dim3(nband), dim3(NTH), 0, s, *g, sc, *w);
    ROWS(FWD_START, -1);
    (void)tol;
}

// face coefficients + partial sums of rhs (resets the stop flag): the start
// of a solve for preconditioners other than the FFT one
extern "C" void pvk_pcg_prep(const pvk_grid *g, pvk_scal *sc, const pvk_pcg *w, hipStream_t s)
{
    hipLaunchKernelGGL(k_pcg_faces, dim3(g->NYM + 1), dim3(NTH), 0, s, *g, *w);
    hipLaunchKernelGGL(k_pcg_mean, dim3((g->NYM + w->band - 1) / w->band), dim3(NTH), 0, s, *g, sc, *w);
}

// K1 alone (d_n = z + beta d_{n-1}, Ad, <d_n, Ad>), for any preconditioner
extern "C" void pvk_pcg_apply(const pvk_grid *g, pvk_scal *sc, const pvk_pcg *w, int n, hipStream_t s)
{
    if (n == 0) hipLaunchKernelGGL(k_pcg_apply<true>, dim3(g->NYM), dim3(NTH), 0, s, *g, sc, *w, n);
    else hipLaunchKernelGGL(k_pcg_apply<false>, dim3(g->NYM), dim3(NTH), 0, s, *g, sc, *w, n);
}

// ---------------------------------------------------------------------------
// Jacobi-PCG (psolve_cg.c:130-293): the reference's recurrences, absolute
// stop sqrt(<r, z>) < tol, its early return without iterations (flag 4) and
// EPS = 1e-30 in both step lengths.  Two launches an iteration, one block a
// row: the apply kernel takes the stop test and beta from the previous
// partials and forms d_n = z + beta d_{n-1} at the stencil points, the
// update kernel forms the step, r and z = M r.  A form with one launch for
// each of the ghost fill, operator, update, direction and two scalar steps
// took 23.7 us an iteration at 128 x 256, where each launch is ~3 us of
// latency; this one takes 9.8 (two RK3 steps 109 -> 64 ms).
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(NTH) k_jac_start(pvk_grid g, pvk_scal *sc, pvk_pcg w, const double *__restrict__ M)
{
    __shared__ double sh[NTH];
    const int P = g.P, NXM = g.NXM, j = blockIdx.x;
    if (j == 0 && threadIdx.x == 0) { sc->p_done = 0; sc->p_iter = 0; }
    double acc = 0.0;
    for (int i = threadIdx.x; i < NXM; i += NTH) {
        const double r = AT(w.rhs, i, j), z = r * AT(M, i, j);
        AT(w.phi, i, j) = 0.0;
        AT(w.r, i, j) = r;
        AT(w.z, i, j) = z;
        acc += r * z;
    }
    block_store_partial(acc, w.rz[0], j, sh);
}

// ONE: rows of at most NTH cells, one a thread; its loads go out before the
// scalar sums are waited for (wider rows would hold too many at once)
template <bool ONE>
__global__ void __launch_bounds__(NTH) k_jac_apply(pvk_grid g, pvk_scal *sc, pvk_pcg w, int n, double tol, int maxit)
{
    __shared__ double sh[2 * NTH];
    const int P = g.P, NXM = g.NXM, NYM = g.NYM, j = xcd_band(blockIdx.x, gridDim.x);
    const int jn = (j + 1 == NYM) ? j : j + 1, js = (j == 0) ? 0 : j - 1;
    const double *__restrict__ z = w.z, *__restrict__ dold = w.d[(n + 1) & 1];
    const double *__restrict__ bx = w.bx, *__restrict__ by = w.by;
    double zv[5], dv[5], cv[4];
    auto load = [&](int i) {
        const int ie = (i + 1 == NXM) ? 0 : i + 1, iw = (i == 0) ? NXM - 1 : i - 1;
        zv[0] = AT(z, i, j);  zv[1] = AT(z, ie, j); zv[2] = AT(z, iw, j); zv[3] = AT(z, i, jn); zv[4] = AT(z, i, js);
        if (n > 0) {
            dv[0] = AT(dold, i, j);  dv[1] = AT(dold, ie, j); dv[2] = AT(dold, iw, j);
            dv[3] = AT(dold, i, jn); dv[4] = AT(dold, i, js);
        }
        cv[0] = AT(bx, i, j); cv[1] = AT(bx, i - 1, j); cv[2] = AT(by, i, j); cv[3] = AT(by, i, j - 1);
    };
    if (ONE) load(min((int)threadIdx.x, NXM - 1));
    if (sc->p_done) return;
    double rz, rzo = 0.0, beta = 0.0;
    if (n > 0) block_sum2(w.rz[n & 1], w.nrz, w.rz[(n + 1) & 1], w.nrz, sh, rz, rzo);
    else rz = block_sum(w.rz[0], w.nrz, sh);
    const double res = sqrt(rz);
    const int stop = (res < tol) ? (n == 0 ? 4 : 1) : (n >= maxit ? 3 : 0);
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        sc->p_res = res;
        sc->p_iter = n;
        if (stop) sc->p_done = stop;
    }
    if (stop) return;
    if (n > 0) beta = rz / (rzo + 1e-30);
    double acc = 0.0;
    for (int i = threadIdx.x; i < NXM; i += NTH) {
        if (!ONE) load(i);
        double d[5];
#pragma unroll
        for (int k = 0; k < 5; k++) d[k] = (n > 0) ? zv[k] + beta * dv[k] : zv[k];
        const double ad = cv[0] * (d[1] - d[0]) - cv[1] * (d[0] - d[2]) + cv[2] * (d[3] - d[0]) - cv[3] * (d[0] - d[4]);
        AT(w.d[n & 1], i, j) = d[0];
        AT(w.Ad, i, j) = ad;
        acc += d[0] * ad;
    }
    block_store_partial(acc, w.dad[0], j, sh);
}

template <bool ONE>
__global__ void __launch_bounds__(NTH) k_jac_update(pvk_grid g, const pvk_scal *sc, pvk_pcg w, const double *__restrict__ M,
                                                    int n)
{
    __shared__ double sh[2 * NTH];
    const int P = g.P, NXM = g.NXM, j = xcd_band(blockIdx.x, gridDim.x);
    const double *__restrict__ d = w.d[n & 1], *__restrict__ Ad = w.Ad;
    double ph, dd, rr, aa, mm;
    auto load = [&](int i) {
        ph = AT(w.phi, i, j); dd = AT(d, i, j); rr = AT(w.r, i, j); aa = AT(Ad, i, j); mm = AT(M, i, j);
    };
    if (ONE) load(min((int)threadIdx.x, NXM - 1));
    if (sc->p_done) return;
    double rz, dad;
    block_sum2(w.rz[n & 1], w.nrz, w.dad[0], w.ndad, sh, rz, dad);
    const double alpha = rz / (dad + 1e-30);
    double acc = 0.0;
    for (int i = threadIdx.x; i < NXM; i += NTH) {
        if (!ONE) load(i);
        const double r = rr - alpha * aa, z = r * mm;
        AT(w.phi, i, j) = ph + alpha * dd;
        AT(w.r, i, j) = r;
        AT(w.z, i, j) = z;
        acc += r * z;
    }
    block_store_partial(acc, w.rz[(n + 1) & 1], j, sh);
}

extern "C" void pvk_jac_start(const pvk_grid *g, pvk_scal *sc, const pvk_pcg *w, const double *M, hipStream_t s)
{
    hipLaunchKernelGGL(k_pcg_faces, dim3(g->NYM + 1), dim3(NTH), 0, s, *g, *w);
    hipLaunchKernelGGL(k_jac_start, dim3(g->NYM), dim3(NTH), 0, s, *g, sc, *w, M);
}

extern "C" void pvk_jac_iter(const pvk_grid *g, pvk_scal *sc, const pvk_pcg *w, const double *M, int half, int n, double tol,
                             int maxit, hipStream_t s)
{
    const dim3 gr(g->NYM);
    if (half == 0) {
        if (g->NXM <= NTH) hipLaunchKernelGGL(k_jac_apply<true>, gr, dim3(NTH), 0, s, *g, sc, *w, n, tol, maxit);
        else hipLaunchKernelGGL(k_jac_apply<false>, gr, dim3(NTH), 0, s, *g, sc, *w, n, tol, maxit);
    } else {
        if (g->NXM <= NTH) hipLaunchKernelGGL(k_jac_update<true>, gr, dim3(NTH), 0, s, *g, (const pvk_scal *)sc, *w, M, n);
        else hipLaunchKernelGGL(k_jac_update<false>, gr, dim3(NTH), 0, s, *g, (const pvk_scal *)sc, *w, M, n);
    }
}

// stage: 0 = K1 apply, 1 = K2 update + forward rows, 2 = K3 check + transpose,
// 3 = K4 column DCTs, 4 = K5 transpose back, 5 = K6 inverse rows + <r, z>,
// 6 = K4' check + tridiagonal y solves in place (replaces 2..4 for the
// pressure).  n = -1 runs stages 2..5 (or 6, 5) on the start residual.
extern "C" void pvk_pcg_stage(const pvk_grid *g, const pvk_fft *F, pvk_scal *sc, const pvk_pcg *w, int stage, int n,
                              double tol, int maxit, hipStream_t s)
{
    switch (stage) {
    case 0:
        pvk_pcg_apply(g, sc, w, n, s);
        break;
    case 1:
        if (n >= 0) ROWS(FWD_STEP, n);
        else if (n == -2) ROWS(FWD_WARM, n);
        else if (n == -3) ROWS(FWD_PLAIN, n);
        else ROWS(FWD_START, n);
        break;
    case 2:
        hipLaunchKernelGGL(k_transpose, dim3((g->NXM + 31) / 32, (g->NYM + 31) / 32), dim3(NTH), 0, s, sc, *w,
                           (const double *)F->spec, w->specT, g->NYM, g->NXM, 1, n, tol, maxit);
        break;
    case 3:
        hipLaunchKernelGGL(k_dct_rows, dim3((g->NXM + w->rdct - 1) / w->rdct), dim3(NTH), lds_rows(w->rdct, g->NYM),
                           s, *g, *F, sc, *w, w->specT);
        break;
    case 4:
        hipLaunchKernelGGL(k_transpose, dim3((g->NYM + 31) / 32, (g->NXM + 31) / 32), dim3(NTH), 0, s, sc, *w,
                           (const double *)w->specT, F->spec, g->NXM, g->NYM, 0, n, tol, maxit);
        break;
    case 6: {
        const dim3 gr((g->NXM + F->tri_kw - 1) / F->tri_kw), nt((F->tri_kw * F->tri_s + 63) / 64 * 64);
        if (F->tri_l <= 8)                   // registers for 8 or 16 rows a thread
            hipLaunchKernelGGL(k_tri_cols<8>, gr, nt, 0, s, *g, *F, sc, *w, n, tol, maxit);
        else
            hipLaunchKernelGGL(k_tri_cols<16>, gr, nt, 0, s, *g, *F, sc, *w, n, tol, maxit);
    } break;
    default:
        ROWS(INV_DOT, n);
        break;
    }
}
