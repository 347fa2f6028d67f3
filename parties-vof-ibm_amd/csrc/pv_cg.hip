// pv_cg.hip -- fused Krylov loops of the Cahn-Hilliard biharmonic solve
// (VOF_DIFFUSE.c:339-429) and of the momentum Jacobi-PCG (msolve_cg.c:525-722).
//
// Each iteration is two launches of 256-thread blocks, each block owning a
// band of rows (pv_block.h):
//   K1 apply : stop test and beta from the previous partials; the new search
//              direction p = z + beta p_old evaluated on the fly at every
//              stencil point through the ghost-fill index maps (so no ghost
//              fill kernel runs); A p; partial <p, A p>.
//   K2 update: alpha; x += alpha p; r -= alpha A p; partials of the next
//              residual products.  (Momentum: the next K1 makes the x step.)
// A scalar that an earlier kernel already formed (||b||, the previous <r,z>)
// is stored by block 0 in a parity-indexed slot that only later kernels read,
// so a kernel re-adds at most two partial sets.  The arithmetic of every
// update is the reference's, in its order; only reduction order differs.
#include <hip/hip_runtime.h>
#include <math.h>
#include "pv_kernels.h"
#include "pv_stencil.h"
#include "pv_block.h"

#define CPT 4   // cells per thread per pass: loads of CPT cells issue before any store

// ---------------------------------------------------------------------------
// Cahn-Hilliard
// ---------------------------------------------------------------------------
// CH ghost fill as an index map: x periodic cell image, y zero gradient
// (VOF_DIFFUSE.c:571-683; all ghost layers equal the first interior value).
__device__ __forceinline__ int chy(int j, int n) { return j < 0 ? 0 : (j >= n ? n - 1 : j); }

// column index of the x-periodic CH map for a tile of W columns, i from 3
// left of the level's first to W right of its last
template <int W> __device__ __forceinline__ int chx(int i, int n)
{
    i += (i < 0) ? n : 0;
    i -= (i >= n) ? n : 0;
    if (n < W)                             // a level narrower than the tile: more than once round
        while (i >= n) i -= n;
    return i;
}

// The CH kernels below run 1024 threads on a tile of 1024 cells: what bounds
// them is a chain of latencies (loads, three or four phases through LDS with a
// barrier between), and a tile's phases are as long as a thread's share of
// them.  Their partial sums keep the order of 256 threads with four cells each.
#define NTC 1024

// block_store_partial of N values a cell, one cell a thread (sh: N NTC doubles)
template <int N> __device__ __forceinline__ void cells_store_partial(const double (&v)[N], double *const (&part)[N], int slot, double *sh)
{
    const int t = threadIdx.x;
#pragma unroll
    for (int k = 0; k < N; k++) sh[k * NTC + t] = v[k];
    __syncthreads();
    if (t < NTH) {
#pragma unroll
        for (int k = 0; k < N; k++) {
            double *q = sh + k * NTC, a = 0.0;
#pragma unroll
            for (int u = 0; u < NTC / NTH; u++) a += q[t + u * NTH];
            a = wave_sum(a);
            if ((t & 63) == 0) q[t] = a;                  // this wavefront's own words
        }
    }
    __syncthreads();
    if (t < N) {
        const double *q = sh + t * NTC;
        double a = q[0];
#pragma unroll
        for (int wv = 1; wv < NTH / 64; wv++) a += q[wv * 64];
        part[t][slot] = a;
    }
}

// The CG start kernels work on tiles of CIT_X x CIT_Y cells: C on the tile
// with a three-cell halo through the CH ghost maps, then on the tile with a
// one-cell halo S(C) and the inner Laplacian of C (CH ghost rules: column
// NXM is column 0, rows -1 / NYM are rows 0 / NYM-1), and the WENO face
// fluxes of the tile's faces, each formed once in LDS instead of once per
// stencil use.  Every value is the arithmetic of the per-cell helpers
// (weno_rhs_at, diffusion_at, bilap_at) on the same operands, so the result
// is bitwise that of the untiled form.  One <b, b> and <r, r> partial per
// tile (w.nt0 of them).
#define CIT_X 64
#define CIT_Y 16
#define CIT_NX (CIT_X + 6)

struct CitTile {
    double c[CIT_Y + 6][CIT_NX];           // C, halo 3
    double l[CIT_Y + 2][CIT_X + 2];        // inner Laplacian of C, halo 1
};
template <class R> struct CitLds : CitTile {
    R s[CIT_Y + 2][CIT_X + 2];             // S(C), halo 1
    double fx[CIT_Y][CIT_X + 1];           // u C_face at x face c0 + b of row j0 + a
    double fy[CIT_Y + 1][CIT_X];           // v C_face at y face j0 + a of column c0 + b
};
static_assert(CIT_X * CIT_Y == NTC, "one cell a thread");

// tile of this block (XCD-aware order), its origin, C and the inner Laplacian
__device__ __forceinline__ int cit_tile(int &c0, int &j0)
{
    const int t = xcd_band(blockIdx.y * gridDim.x + blockIdx.x, gridDim.x * gridDim.y);
    const int ty = t / gridDim.x, tx = t - ty * gridDim.x;
    c0 = tx * CIT_X;
    j0 = ty * CIT_Y;
    return t;
}
// C of the tile (two cells a thread at most)
#define CIT_K (((CIT_Y + 6) * CIT_NX + NTC - 1) / NTC)
__device__ __forceinline__ void cit_load(const pvk_grid &g, const double *C, int c0, int j0, double (&cv)[CIT_K])
{
    const int P = g.P;
#pragma unroll
    for (int k = 0; k < CIT_K; k++) {
        const int q = min((int)threadIdx.x + k * NTC, (CIT_Y + 6) * CIT_NX - 1), a = q / CIT_NX, b = q - a * CIT_NX;
        cv[k] = AT(C, chx<CIT_X + 3>(c0 + b - 3, g.NXM), chy(j0 + a - 3, g.NYM));
    }
}
__device__ __forceinline__ void cit_stage(const double (&cv)[CIT_K], CitTile &T)
{
#pragma unroll
    for (int k = 0; k < CIT_K; k++) {
        const int q = threadIdx.x + k * NTC;
        if (q < (CIT_Y + 6) * CIT_NX) (&T.c[0][0])[q] = cv[k];
    }
}
// the inner Laplacian of the staged tile
__device__ __forceinline__ void cit_lap(const pvk_grid &g, int c0, int j0, CitTile &T)
{
    for (int q = threadIdx.x; q < (CIT_Y + 2) * (CIT_X + 2); q += NTC) {
        const int a = q / (CIT_X + 2), b = q - a * (CIT_X + 2), jb = j0 + a - 1;
        if (jb >= 0 && jb < g.NYM)
            T.l[a][b] = lap_vals(g, chx<CIT_X + 3>(c0 + b - 1, g.NXM), jb, T.c[a + 2][b + 2], T.c[a + 2][b + 3],
                                 T.c[a + 2][b + 1], T.c[a + 3][b + 2], T.c[a + 1][b + 2]);
    }
}
// L(L C) at tile cell (tr, tc) = global (i, j)
__device__ __forceinline__ double cit_bilap(const pvk_grid &g, const CitTile &T, int tr, int tc, int i, int j)
{
    const double L0 = T.l[tr + 1][tc + 1];
    const double LN = (j + 1 == g.NYM) ? L0 : T.l[tr + 2][tc + 1];
    const double LS = (j == 0) ? L0 : T.l[tr][tc + 1];
    return lap_vals(g, i, j, L0, T.l[tr + 1][tc + 2], T.l[tr + 1][tc], LN, LS);
}

// Explicit CH right-hand side and CG start: rc -> rn, r = p = b - A C;
// partials ||b||^2, ||r||^2.  Every load goes out before the first is used.
// With four cells a thread and each phase's loads where they are used: 54 us
// at 1024^2 in the FP32 form, 164 at 2048^2, 22 at 96^2 in FP64; now 37, 124 and
// 13 (the start from a given b: 26 and 88 -> 16 and 58 at 1024^2 and 2048^2).
template <class R>
__global__ void __launch_bounds__(NTC) k_ccg_init_rhs(pvk_grid g, pvk_phys ph, int stage, pvk_scal *sc,
                                                     const double *__restrict__ C, const double *__restrict__ u,
                                                     const double *__restrict__ v, double *__restrict__ rn,
                                                     double *__restrict__ r, double *__restrict__ p, pvk_ccg w,
                                                     double *__restrict__ bout)
{
    constexpr int KX = (CIT_Y * (CIT_X + 1) + NTC - 1) / NTC, KY = ((CIT_Y + 1) * CIT_X + NTC - 1) / NTC;
    __shared__ double sh[2 * NTC];
    __shared__ CitLds<R> T;
    const int P = g.P, NXM = g.NXM, NYM = g.NYM, wo = ph.weno_order;
    if (blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x == 0) { sc->ch_done = 0; sc->ch_iter = 0; }
    int c0, j0;
    const int t = cit_tile(c0, j0);
    const int tr = threadIdx.x / CIT_X, tc = threadIdx.x - tr * CIT_X, i = c0 + tc, j = j0 + tr;
    const bool in = i < NXM && j < NYM;
    double cv[CIT_K], uv[KX], vv[KY], old = 0.0;
    cit_load(g, C, c0, j0, cv);
#pragma unroll
    for (int k = 0; k < KX; k++) {
        const int q = min((int)threadIdx.x + k * NTC, CIT_Y * (CIT_X + 1) - 1), a = q / (CIT_X + 1), b = q - a * (CIT_X + 1);
        uv[k] = AT(u, min(c0 + b, NXM), min(j0 + a, NYM - 1));
    }
#pragma unroll
    for (int k = 0; k < KY; k++) {
        const int q = min((int)threadIdx.x + k * NTC, (CIT_Y + 1) * CIT_X - 1), a = q / CIT_X, b = q - a * CIT_X;
        vv[k] = AT(v, min(c0 + b, NXM - 1), min(j0 + a, NYM));
    }
    if (stage != 0) old = AT(rn, min(i, NXM - 1), min(j, NYM - 1));
    const double a_dt = 1.0 / (sc->dt * c_BET[stage]);
    cit_stage(cv, T);
    __syncthreads();
    for (int q = threadIdx.x; q < (CIT_Y + 2) * (CIT_X + 2); q += NTC) {
        const int a = q / (CIT_X + 2), b = q - a * (CIT_X + 2);
        T.s[a][b] = bulkS<R>(R(T.c[a + 2][b + 2]));
    }
    cit_lap(g, c0, j0, T);
#pragma unroll
    for (int k = 0; k < KX; k++) {
        const int q = threadIdx.x + k * NTC, a = q / (CIT_X + 1), b = q - a * (CIT_X + 1);
        if (q < CIT_Y * (CIT_X + 1) && c0 + b <= NXM && j0 + a < NYM) {
            const double vel = uv[k], *cr = &T.c[a + 3][b];       // cr[k] = C at column i - 3 + k
            T.fx[a][b] = vel * (double)face_vals<R>(cr[0], cr[1], cr[2], cr[3], cr[4], cr[5], vel, wo);
        }
    }
#pragma unroll
    for (int k = 0; k < KY; k++) {
        const int q = threadIdx.x + k * NTC, a = q / CIT_X, b = q - a * CIT_X;
        if (q < (CIT_Y + 1) * CIT_X && c0 + b < NXM && j0 + a <= NYM) {
            const double vel = vv[k];
            T.fy[a][b] = vel * (double)face_vals<R>(T.c[a][b + 3], T.c[a + 1][b + 3], T.c[a + 2][b + 3],
                                                    T.c[a + 3][b + 3], T.c[a + 4][b + 3], T.c[a + 5][b + 3], vel, wo);
        }
    }
    __syncthreads();
    double sums[2] = {0.0, 0.0};
    if (in) {
        double rc = weno_div(g, i, j, T.fx[tr][tc], T.fx[tr][tc + 1], T.fy[tr][tc], T.fy[tr + 1][tc]);
        rc += diffusion_vals<R>(g, ph, i, j, T.s[tr + 1][tc + 1], T.s[tr + 1][tc + 2], T.s[tr + 1][tc],
                                T.s[tr + 2][tc + 1], T.s[tr][tc + 1]);
        double cc = T.c[tr + 3][tc + 3];
        double rv = (stage == 0) ? a_dt * cc + c_GAMB[0] * rc : a_dt * cc + c_GAMB[stage] * rc + c_ZETB[stage] * old;
        double L2 = cit_bilap(g, T, tr, tc, i, j);
        double b = rv - ph.bih * L2;
        double Ap = a_dt * cc + ph.bih * L2;
        double rr = b - Ap;
        if (bout) AT(bout, i, j) = b;
        AT(rn, i, j) = rc;
        AT(r, i, j) = rr;
        AT(p, i, j) = rr;
        sums[0] = ch_w(g, i, j, b, b);
        sums[1] = ch_w(g, i, j, rr, rr);
    }
    double *const part[2] = {w.bb, w.rr[0]};
    cells_store_partial(sums, part, t, sh);
}

// CG start from a given b (b already holds rhs - (Cn^2/Pe) L^2 C).
__global__ void __launch_bounds__(NTC) k_ccg_init_b(pvk_grid g, pvk_phys ph, int stage, pvk_scal *sc,
                                                   const double *__restrict__ C, const double *__restrict__ bv,
                                                   double *__restrict__ r, double *__restrict__ p, pvk_ccg w)
{
    __shared__ double sh[2 * NTC];
    __shared__ CitTile T;
    const int P = g.P, NXM = g.NXM, NYM = g.NYM;
    if (blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x == 0) { sc->ch_done = 0; sc->ch_iter = 0; }
    int c0, j0;
    const int t = cit_tile(c0, j0);
    const int tr = threadIdx.x / CIT_X, tc = threadIdx.x - tr * CIT_X, i = c0 + tc, j = j0 + tr;
    double cv[CIT_K];
    cit_load(g, C, c0, j0, cv);
    const double bb = AT(bv, min(i, NXM - 1), min(j, NYM - 1));
    const double a_dt = 1.0 / (sc->dt * c_BET[stage]);
    cit_stage(cv, T);
    __syncthreads();
    cit_lap(g, c0, j0, T);
    __syncthreads();
    double sums[2] = {0.0, 0.0};
    if (i < NXM && j < NYM) {
        double cc = T.c[tr + 3][tc + 3];
        double Ap = a_dt * cc + ph.bih * cit_bilap(g, T, tr, tc, i, j);
        double rr = bb - Ap;
        AT(r, i, j) = rr;
        AT(p, i, j) = rr;
        sums[0] = ch_w(g, i, j, bb, bb);
        sums[1] = ch_w(g, i, j, rr, rr);
    }
    double *const part[2] = {w.bb, w.rr[0]};
    cells_store_partial(sums, part, t, sh);
}

// K1: stop test on ||r_n|| (VOF_DIFFUSE.c:403-414), beta, p_n = r + beta p_{n-1}
// (:416-422), Ap = a_dt p + (Cn^2/Pe) L^2 p (:318-337), partials of
// <p, Ap> (one per block).  A block owns a tile of
// CHT_X x CHT_Y cells: p on the tile with a two-cell halo (CH ghost maps) and
// the inner Laplacian with a one-cell halo are formed once in LDS, so each p
// value is formed once per tile instead of once per stencil use; every value is formed by the arithmetic of bilap_at
// (inner Laplacian with the CH ghost rules, then the outer one).
// The tile's loads go out before the sums that give beta: 9.2 -> 6.1 us an
// iteration at 96^2, 10.2 -> 8.6 at 352 x 704, 15.1 -> 15.6 at 1024^2 (within the
// noise of a run; there the two rounds of 1024 tiles hide each other's latency).
#define CHT_X 128
#define CHT_Y 8
#define CHT_K (((CHT_Y + 4) * (CHT_X + 4) + NTC - 1) / NTC)
static_assert(CHT_X * CHT_Y == NTC, "one cell a thread");
__global__ void __launch_bounds__(NTC) k_ccg_apply(pvk_grid g, pvk_phys ph, int stage, pvk_scal *sc, pvk_ccg w,
                                                  const double *__restrict__ r, const double *__restrict__ pold,
                                                  double *__restrict__ pnew, double *__restrict__ Ap, int n,
                                                  int maxit, double tol)
{
    __shared__ double sh[NTC];
    __shared__ double sp[CHT_Y + 4][CHT_X + 4];
    __shared__ double sl[CHT_Y + 2][CHT_X + 2];
    if (sc->ch_done) return;
    const int P = g.P, NXM = g.NXM, NYM = g.NYM;
    const bool lead = (blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x == 0);
    const int t = xcd_band(blockIdx.y * gridDim.x + blockIdx.x, gridDim.x * gridDim.y);
    const int ty = t / gridDim.x, tx = t - ty * gridDim.x;
    const int c0 = tx * CHT_X, j0 = ty * CHT_Y;
    // the tile's loads, ahead of the sums
    double rv[CHT_K], pv[CHT_K];
#pragma unroll
    for (int k = 0; k < CHT_K; k++) {
        const int q = min((int)threadIdx.x + k * NTC, (CHT_Y + 4) * (CHT_X + 4) - 1);
        const int a = q / (CHT_X + 4), b = q - a * (CHT_X + 4);
        const int ia = chx<CHT_X + 2>(c0 + b - 2, NXM), jb = chy(j0 + a - 2, NYM);
        rv[k] = AT(r, ia, jb);
        pv[k] = (n == 0) ? 0.0 : AT(pold, ia, jb);
    }
    const double rr = 2.0 * block_sum_wide(w.rr[n & 1], (n == 0) ? w.nt0 : w.nb, sh);   // start: one per tile
    double bnorm;
    if (n == 0) {
        bnorm = sqrt(2.0 * block_sum_wide(w.bb, w.nt0, sh));
        if (bnorm < 1e-30) bnorm = 1.0;
        if (lead) sc->ch_bnorm = bnorm;
    } else {
        bnorm = sc->ch_bnorm;
    }
    const double rel = sqrt(rr) / bnorm;
    double beta = 0.0;
    bool stop = (rel < tol) || (n == 0 && maxit <= 0);
    if (!stop && n > 0) {
        beta = rr / (sc->ch_rzb[(n + 1) & 1] + 1e-30);
        stop = (n >= maxit);
    }
    if (lead) {
        sc->ch_rzb[n & 1] = rr;
        if (stop) {
            sc->ch_rel = rel;
            sc->ch_iter = n;
            sc->ch_done = (rel < tol || maxit <= 0) ? 1 : 3;
        }
    }
    if (stop) return;

    const double a_dt = 1.0 / (sc->dt * c_BET[stage]);
#pragma unroll
    for (int k = 0; k < CHT_K; k++) {
        const int q = threadIdx.x + k * NTC;
        if (q < (CHT_Y + 4) * (CHT_X + 4)) (&sp[0][0])[q] = (n == 0) ? rv[k] : rv[k] + beta * pv[k];
    }
    __syncthreads();
    for (int q = threadIdx.x; q < (CHT_Y + 2) * (CHT_X + 2); q += NTC) {
        const int a = q / (CHT_X + 2), b = q - a * (CHT_X + 2), jb = j0 + a - 1;
        if (jb >= 0 && jb < NYM)
            sl[a][b] = lap_vals(g, chx<CHT_X + 2>(c0 + b - 1, NXM), jb, sp[a + 1][b + 1], sp[a + 1][b + 2], sp[a + 1][b],
                                sp[a + 2][b + 1], sp[a][b + 1]);
    }
    __syncthreads();
    const int tr = threadIdx.x / CHT_X, tc = threadIdx.x - tr * CHT_X, i = c0 + tc, j = j0 + tr;
    double acc[1] = {0.0};
    if (i < NXM && j < NYM) {
        const double L0 = sl[tr + 1][tc + 1];
        const double LN = (j + 1 == NYM) ? L0 : sl[tr + 2][tc + 1];
        const double LS = (j == 0) ? L0 : sl[tr][tc + 1];
        const double pc = sp[tr + 2][tc + 2];
        const double ap = a_dt * pc + ph.bih * lap_vals(g, i, j, L0, sl[tr + 1][tc + 2], sl[tr + 1][tc], LN, LS);
        AT(pnew, i, j) = pc;
        AT(Ap, i, j) = ap;
        acc[0] = ch_w(g, i, j, pc, ap);
    }
    double *const part[1] = {w.pap};
    cells_store_partial(acc, part, t, sh);
}

// K2: alpha = <r,r> / <p,Ap> (VOF_DIFFUSE.c:384-390); x += alpha p;
// r -= alpha Ap (:390-405); partial <r, r> of the next iteration.
__global__ void __launch_bounds__(NTH) k_ccg_update(pvk_grid g, pvk_scal *sc, pvk_ccg w, double *__restrict__ x,
                                                   const double *__restrict__ p, double *__restrict__ r,
                                                   const double *__restrict__ Ap, int n)
{
    __shared__ double sh[NTH];
    if (sc->ch_done) return;
    const int P = g.P, NXM = g.NXM;
    const int band = xcd_band(blockIdx.x, gridDim.x);
    const double pAp = 2.0 * block_sum(w.pap, w.npap, sh);
    if (fabs(pAp) < 1e-30) {
        if (blockIdx.x == 0 && threadIdx.x == 0) { sc->ch_done = 2; sc->ch_iter = n; }
        return;
    }
    const double alpha = sc->ch_rzb[n & 1] / pAp;
    const int j0 = band * w.band, j1 = min(g.NYM, j0 + w.band);
    double acc = 0.0;
    for (int j = j0; j < j1; j++)
    for (int i = threadIdx.x; i < NXM; i += NTH) {
        AT(x, i, j) += alpha * AT(p, i, j);
        double rr = AT(r, i, j) - alpha * AT(Ap, i, j);
        AT(r, i, j) = rr;
        acc += ch_w(g, i, j, rr, rr);
    }
    block_store_partial(acc, w.rr[(n + 1) & 1], band, sh);
}

extern "C" void pvk_ccg_init(const pvk_grid *g, const pvk_phys *ph, int stage, pvk_scal *sc, const pvk_ccg *w,
                             const double *C, const double *u, const double *v, double *rn, const double *b,
                             double *r, double *p, double *bout, hipStream_t s)
{
    const dim3 gr((g->NXM + CIT_X - 1) / CIT_X, (g->NYM + CIT_Y - 1) / CIT_Y);
    if (b)
        hipLaunchKernelGGL(k_ccg_init_b, gr, dim3(NTC), 0, s, *g, *ph, stage, sc, C, b, r, p, *w);
    else if (ph->precision)
        hipLaunchKernelGGL(k_ccg_init_rhs<float>, gr, dim3(NTC), 0, s, *g, *ph, stage, sc, C, u, v, rn, r, p, *w,
                           bout);
    else
        hipLaunchKernelGGL(k_ccg_init_rhs<double>, gr, dim3(NTC), 0, s, *g, *ph, stage, sc, C, u, v, rn, r, p, *w,
                           bout);
}

extern "C" void pvk_ccg_iter(const pvk_grid *g, const pvk_phys *ph, int stage, pvk_scal *sc, const pvk_ccg *w,
                             int half, int n, double *x, double *r, double *Ap, hipStream_t s)
{
    if (half == 0)
        hipLaunchKernelGGL(k_ccg_apply, dim3((g->NXM + CHT_X - 1) / CHT_X, (g->NYM + CHT_Y - 1) / CHT_Y), dim3(NTC),
                           0, s, *g, *ph, stage, sc, *w, (const double *)r,
                           (const double *)w->p[(n + 1) & 1], w->p[n & 1], Ap, n, ph->ch_iter_max, ph->ch_tol);
    else
        hipLaunchKernelGGL(k_ccg_update, dim3(w->nb), dim3(NTH), 0, s, *g, sc, *w, x, (const double *)w->p[n & 1], r,
                           (const double *)Ap, n);
}

// ---------------------------------------------------------------------------
// Momentum (u and v solved in the same launches; blocks [0, nb[0]) take u)
// ---------------------------------------------------------------------------
// Unknown ranges (msolve_cg.c:525-722): u at i = 1..NXM, j = 0..NYM-1; v at
// i = 0..NXM-1, j = 1..NYM-1.  Ghost maps of the CG-type boundary update
// (Velocity.c:2427-2805): u is x periodic with column 0 = column NXM and
// ghost rows -1 / NYM holding minus rows 0 / NYM-1; v is x periodic (cell
// image) and its wall rows 0 and NYM are never written by the solve.
struct mom_band {
    int comp, band, j0, j1, i0, jlo;
};
__device__ __forceinline__ mom_band mom_locate(const pvk_grid &g, const pvk_mcg &w)
{
    mom_band m;
    const int vb = xcd_band(blockIdx.x, gridDim.x);
    m.comp = (vb < w.nb[0]) ? 0 : 1;
    m.band = m.comp ? vb - w.nb[0] : vb;
    m.jlo = m.comp ? 1 : 0;                          // unknown rows [jlo, NYM)
    m.j0 = m.jlo + m.band * w.band;
    m.j1 = min(g.NYM, m.j0 + w.band);
    m.i0 = m.comp ? 0 : 1;
    return m;
}
// The FP32 form keeps what is an FP32 value as one: A d, the diagonal.
template <class R> __device__ __forceinline__ const R *mom_Ad(const pvk_mcg &w, int c)
{
    if constexpr (sizeof(R) == sizeof(float)) return w.Adf[c];
    else return w.Ad[c];
}
template <class R> __device__ __forceinline__ const R *mom_dg(const pvk_mcg &w, int c)
{
    if constexpr (sizeof(R) == sizeof(float)) return w.dgf[c];
    else return w.dg[c];
}
// the diagonal + EPS (the FP64 form stores the sum)
__device__ __forceinline__ double mom_D(float d) { return (double)d + 1e-14; }
__device__ __forceinline__ double mom_D(double d) { return d; }

// A thread's cells of its band, row by row, each row in chunks of NTH columns
// (the order of its sums): position and the next one.
struct mom_walk {
    int j, cb;
    __device__ __forceinline__ void next(int NXM)
    {
        cb += NTH;
        if (cb >= NXM) { cb = 0; j++; }
    }
};

// r = rhs - A x; dg = diag + EPS; d = r / dg; partial <r, d>
// (msolve_cg.c:627-645), and what the iterations read instead of rho and mu:
// the FP32 form the five coefficients, the FP64 form the time factor and
// the corner viscosity, so that an iteration divides nothing to form A d.
// Two cells a thread are in flight at once, each component's code knows its
// stencil (one harmonic mean for the operator, the diagonal and the
// coefficients), and what the preconditioned start overwrites is not formed.
// Bound by memory latency: 74 us at 1024^2 in the FP32 form with one cell in
// flight and the means formed three times over, 38 now.
template <class R, int COMP>
__device__ __forceinline__ void mcg_init_rows(const pvk_grid &g, const pvk_phys &ph, double alpha_k, double dt,
                                              const pvk_mcg &w, const mom_band &m, double *sh)
{
    constexpr bool F32 = sizeof(R) == sizeof(float);
    constexpr int U = 2;
    const int P = g.P, NXM = g.NXM, NYM = g.NYM, t = threadIdx.x;
    const double *x = w.x[COMP], *rhs = w.rhs[COMP], *rho = w.rho, *mu = w.mu;
    double *r = w.r[COMP], *d = w.d[COMP][0];
    double acc = 0.0;
    for (mom_walk p = {m.j0, 0}; p.j < m.j1;) {
        double ad[U], rr[U], dgv[U];
        float cc[U][5], df[U];
        double ft[U], mc[U], mp[U];
        int jj[U], ii[U];
        bool ok[U];
#pragma unroll
        for (int k = 0; k < U; k++) {
            const int j = min(p.j, m.j1 - 1), i = m.i0 + min(p.cb + t, NXM - 1);
            jj[k] = j;
            ii[k] = i;
            ok[k] = p.j < m.j1 && p.cb + t < NXM;
            p.next(NXM);
            ad[k] = (double)mom_op_vals<R>(g, ph, alpha_k, dt, rho, mu, COMP, i, j, R(AT(x, i, j)), R(AT(x, i + 1, j)),
                                           R(AT(x, i - 1, j)), R(AT(x, i, j + 1)), R(AT(x, i, j - 1)));
            rr[k] = AT(rhs, i, j) - ad[k];
            const R dr = mom_diag<R>(g, ph, alpha_k, dt, rho, mu, COMP, i, j);
            dgv[k] = (double)dr + 1e-14;
            if constexpr (F32) {
                df[k] = dr;
                mom_coeffs(g, ph, alpha_k, dt, rho, mu, COMP, i, j, cc[k]);
            } else {
                ft[k] = mom_time<R>(g, alpha_k, dt, rho, COMP, i, j);
                mc[k] = mom_corner<R>(g, mu, COMP, i, j);
                mp[k] = COMP ? mom_corner<R>(g, mu, 1, i + 1, j) : mom_corner<R>(g, mu, 0, i, j + 1);
            }
        }
#pragma unroll
        for (int k = 0; k < U; k++) {
            if (!ok[k]) continue;
            const int i = ii[k], j = jj[k];
            AT(r, i, j) = rr[k];
            if constexpr (F32) {
#pragma unroll
                for (int q = 0; q < 5; q++) AT(w.cf[COMP][q], i, j) = cc[k][q];
                AT(w.dgf[COMP], i, j) = df[k];
            } else {
                AT(w.dg[COMP], i, j) = dgv[k];
                AT(w.ft[COMP], i, j) = ft[k];
                AT(w.mc[COMP], i, j) = mc[k];
                if (COMP == 0 && j == NYM - 1) AT(w.mc[0], i, NYM) = mp[k];      // the last face's
                if (COMP == 1 && i == NXM - 1) AT(w.mc[1], NXM, j) = mp[k];
            }
            if (w.maxit <= 0) AT(w.Ad[COMP], i, j) = ad[k];                     // else every A d comes after it
            if (!F32 || !w.pc) {
                const double dd = rr[k] / dgv[k];
                AT(d, i, j) = dd;
                acc += rr[k] * dd;
            }
        }
    }
    if (!F32 || !w.pc) block_store_partial(acc, w.rz[COMP][0], m.band, sh);
}
template <class R>
__global__ void __launch_bounds__(NTH) k_mcg_init(pvk_grid g, pvk_phys ph, int stage, pvk_scal *sc, pvk_mcg w)
{
    __shared__ double sh[NTH];
    const mom_band m = mom_locate(g, w);
    if (m.band == 0 && threadIdx.x == 0) { sc->m_done[m.comp] = (w.maxit <= 0); sc->m_iter[m.comp] = 0; }
    const double alpha_k = c_BET[stage], dt = sc->dt;
    if (m.comp) mcg_init_rows<R, 1>(g, ph, alpha_k, dt, w, m, sh);
    else mcg_init_rows<R, 0>(g, ph, alpha_k, dt, w, m, sh);
}

// K1: stop test sqrt(r.r / N) < CG_ETOL (msolve_cg.c:691-704), beta =
// rz_new / (rz + EPS) (w.exact: rz_new / rz, 0 when rz is 0),
// d_n = z + beta d_{n-1} (:705-713), z the preconditioned residual, evaluated
// at the five operator points through the ghost maps; Ad = A d_n; partial
// <d, Ad>.  The x step of iteration n - 1 (x += alpha d) is made here, where
// d_{n-1} is read anyway, and by the blocks that find the solve stopped.
//
// A block walks its band in chunks of MCH columns, a thread one column: its
// own rows and the rows above and below stay in registers (the south and
// north values), east and west go through LDS.  The first chunk's loads are
// issued before the sums that give beta.  Bound by memory: 72 bytes a cell and
// component in the FP64 form (84 MB at 512 x 1024), 64 in the FP32 form (537
// MB at 2048^2: 123 us, 4.4 TB/s).  With the harmonic means and the time
// factor formed anew in each iteration, r / dg divided at every stencil point
// and the x step in the update kernel, the two kernels of an iteration took
// 20.7 + 11.5 us at 512 x 1024 in FP64 (16.7 + 9.7 now), 37 + 19 at 1024^2
// (28 + 14.6), and 120 + 196 at 2048^2 in the FP32 form with the polynomial
// preconditioner (123 + 118).
#define MCH 256                                                  // columns per chunk of k_mcg_apply
template <class R, int BAND, bool FIRST>
__global__ void __launch_bounds__(NTH) k_mcg_apply(pvk_grid g, pvk_phys ph, pvk_scal *sc, pvk_mcg w, int n)
{
    constexpr bool F32 = sizeof(R) == sizeof(float);
    __shared__ double sh[2 * NTH];
    __shared__ double sd[2][BAND][MCH + 2];
    const mom_band m = mom_locate(g, w);
    const int c = m.comp, t = threadIdx.x;
    const int was = sc->m_done[c], it = sc->m_iter[c];
    if (was && (FIRST || it != n)) return;               // stopped, x complete
    const int P = g.P, NXM = g.NXM, NYM = g.NYM, nrow = m.j1 - m.j0;
    const bool lead = (m.band == 0 && t == 0);
    const double *zc = FIRST ? w.d[c][0] : w.z[c], *dold = w.d[c][(n + 1) & 1], *dwall = w.d[c][0];
    double *dnew = w.d[c][n & 1], *x = w.x[c];
    R *Ad = const_cast<R *>(mom_Ad<R>(w, c));

    // a chunk's values: z and d_{n-1} of rows j0 - 1 .. j0 + BAND, those of the
    // ring column this thread sees to, x, and the operator's factors
    double z[BAND + 2], o[BAND + 2], rz_, ro_, xv[BAND];
    R cf[BAND][5];                                       // FP32: the coefficients; FP64: ft, xp, xm in 0..2
    double yf[BAND + 1];                                 // FP64: the y face viscosities
    auto ghost = [&](int b) { return b < m.jlo || b >= NYM; };
    auto ncol = [&](int cb) { return min(MCH, NXM - cb); };
    auto load = [&](int cb) {
        const int i = m.i0 + cb + min(t, ncol(cb) - 1);
#pragma unroll
        for (int a = 0; a < BAND + 2; a++) {
            const int b = m.j0 - 1 + a, bc = min(max(b, m.jlo), NYM - 1);
            z[a] = (c && ghost(b)) ? AT(dwall, i, b < 1 ? 0 : NYM) : AT(zc, i, bc);
            if (!FIRST) o[a] = AT(dold, i, bc);
        }
        if (t < 2 * BAND) {                              // thread 2 a + side: row j0 + a, west or east column
            const int e = m.i0 + cb + ((t & 1) ? ncol(cb) : -1), b = min(m.j0 + (t >> 1), NYM - 1);
            const int ie = c ? wrapc(e, NXM) : wrapu(e, NXM);
            rz_ = AT(zc, ie, b);
            if (!FIRST) ro_ = AT(dold, ie, b);
        }
#pragma unroll
        for (int a = 0; a < BAND; a++) {
            const int b = min(m.j0 + a, NYM - 1);
            if (!FIRST) xv[a] = AT(x, i, b);
            if constexpr (F32) {
#pragma unroll
                for (int k = 0; k < 5; k++) cf[a][k] = AT(w.cf[c][k], i, b);
            } else {
                cf[a][0] = AT(w.ft[c], i, b);
                cf[a][1] = c ? AT(w.mc[1], i + 1, b) : AT(w.mu, i, b);
                cf[a][2] = c ? AT(w.mc[1], i, b) : AT(w.mu, i - 1, b);
            }
        }
        if constexpr (!F32) {
#pragma unroll
            for (int a = 0; a <= BAND; a++)
                yf[a] = c ? AT(w.mu, i, min(m.j0 - 1 + a, NYM - 1)) : AT(w.mc[0], i, min(m.j0 + a, NYM));
        }
    };
    load(0);

    double beta = 0.0, alpha = 0.0;
    if (FIRST) {
        const double rz = block_sum(w.rz[c][0], w.nb[c], sh);
        if (lead) sc->m_rzb[c][0] = rz;
    } else {
        double rz, rr;
        block_sum2(w.rz[c][n & 1], w.nb[c], w.rr[c], w.nb[c], sh, rz, rr);
        const double rms = sqrt(w.in_tot[c] * rr), rzo = sc->m_rzb[c][(n + 1) & 1];
        alpha = sc->m_alpha[c];
        if (rms < w.tol || n >= w.maxit) {
            if (lead) {
                sc->m_rms[c] = rms;
                sc->m_iter[c] = n;
                sc->m_done[c] = (rms < w.tol) ? 1 : 3;
            }
            // the last x step; the public fields of the last A d and residual
            for (int j = m.j0; j < m.j1; j++)
                for (int i = m.i0 + t; i < m.i0 + NXM; i += NTH) {
                    AT(x, i, j) += alpha * AT(dold, i, j);
                    if constexpr (F32) {
                        AT(w.Ad[c], i, j) = (double)AT(Ad, i, j);
                        if (w.pc && (n & 1)) AT(w.r[c], i, j) = AT(w.r2[c], i, j);
                    }
                }
            return;
        }
        beta = w.exact ? (rzo != 0.0 ? rz / rzo : 0.0) : rz / (rzo + 1e-14);
        if (lead) sc->m_rzb[c][n & 1] = rz;
    }

    double acc = 0.0;
    int par = 0;
    for (int cb = 0; cb < NXM; cb += MCH, par ^= 1) {
        if (cb) load(cb);
        const int nc = ncol(cb);
        double dv[BAND + 2];
#pragma unroll
        for (int a = 0; a < BAND + 2; a++) {
            const double v = FIRST ? z[a] : z[a] + beta * o[a];
            dv[a] = ghost(m.j0 - 1 + a) ? (c ? z[a] : -v) : v;
        }
        if (t < nc) {
#pragma unroll
            for (int a = 0; a < BAND; a++) sd[par][a][t + 1] = dv[a + 1];
        }
        if (t < 2 * BAND) sd[par][t >> 1][(t & 1) ? nc + 1 : 0] = FIRST ? rz_ : rz_ + beta * ro_;
        __syncthreads();
        if (t < nc) {
            const int i = m.i0 + cb + t;
#pragma unroll
            for (int a = 0; a < BAND; a++) {
                if (a < nrow) {
                    const int j = m.j0 + a;
                    const double dc = dv[a + 1], dE = sd[par][a][t + 2], dW = sd[par][a][t];
                    R ad;
                    if constexpr (F32)
                        ad = mom_op_coeffs(cf[a], float(dc), float(dE), float(dW), float(dv[a + 2]), float(dv[a]));
                    else
                        ad = mom_op_flux<R>(g, ph.iRe, c, i, j, cf[a][0], cf[a][1], cf[a][2], yf[a + 1], yf[a], dc, dE,
                                            dW, dv[a + 2], dv[a]);
                    if (!FIRST) {
                        AT(x, i, j) = xv[a] + alpha * o[a + 1];
                        AT(dnew, i, j) = dc;
                    }
                    AT(Ad, i, j) = ad;
                    acc += dc * (double)ad;
                }
            }
        }
    }
    block_store_partial(acc, w.dad[c], m.band, sh);
}

// the step of iteration n: alpha = rz / (dAd + EPS) (msolve_cg.c:674; w.exact:
// rz / dAd, 0 when dAd is 0)
__device__ __forceinline__ double mom_alpha(pvk_scal *sc, const pvk_mcg &w, const mom_band &m, int n, double *sh)
{
    const int c = m.comp;
    const double dAd = block_sum(w.dad[c], w.nb[c], sh);
    const double rzn = sc->m_rzb[c][n & 1];
    const double alpha = w.exact ? (dAd != 0.0 ? rzn / dAd : 0.0) : rzn / (dAd + 1e-14);
    if (m.band == 0 && threadIdx.x == 0) { sc->m_iter[c] = n + 1; sc->m_alpha[c] = alpha; }
    return alpha;
}

// K2: alpha; r -= alpha Ad; z = r / dg; partials of r^2 / dg and r^2
// (msolve_cg.c:676-690).  Four cells a thread in flight, the first four's
// loads ahead of the sums.
template <class R>
__global__ void __launch_bounds__(NTH) k_mcg_update(pvk_grid g, pvk_scal *sc, pvk_mcg w, int n)
{
    __shared__ double sh[NTH];
    const mom_band m = mom_locate(g, w);
    const int c = m.comp, t = threadIdx.x;
    if (sc->m_done[c]) return;
    const int P = g.P, NXM = g.NXM;
    double *r = w.r[c], *z = w.z[c];
    const R *Ad = mom_Ad<R>(w, c), *dg = mom_dg<R>(w, c);
    double rv[CPT];
    R av[CPT], gv[CPT];
    auto load = [&](mom_walk p) {
#pragma unroll
        for (int k = 0; k < CPT; k++) {
            const int j = min(p.j, m.j1 - 1), i = m.i0 + min(p.cb + t, NXM - 1);
            rv[k] = AT(r, i, j);
            av[k] = AT(Ad, i, j);
            gv[k] = AT(dg, i, j);
            p.next(NXM);
        }
    };
    mom_walk p = {m.j0, 0};
    load(p);
    const double alpha = mom_alpha(sc, w, m, n, sh);
    double a0 = 0.0, a1 = 0.0;
    while (p.j < m.j1) {
        mom_walk q = p;
#pragma unroll
        for (int k = 0; k < CPT; k++) {
            if (q.j < m.j1 && q.cb + t < NXM) {
                const int j = q.j, i = m.i0 + q.cb + t;
                const double ri = rv[k] - alpha * (double)av[k], D = mom_D(gv[k]);
                AT(r, i, j) = ri;
                AT(z, i, j) = ri / D;
                a0 += ri * ri / D;
                a1 += ri * ri;
            }
            q.next(NXM);
        }
        p = q;
        if (p.j < m.j1) load(p);
    }
    block_store_partial(a0, w.rz[c][(n + 1) & 1], m.band, sh);
    block_store_partial(a1, w.rr[c], m.band, sh);
}

// Momentum preconditioner pc = 1 (FP32 form), the first-order Neumann polynomial of
// the Jacobi splitting A = D - N: z = D^-1 (r + N D^-1 r), i.e.
// z_p = (r_p + sum_q c_pq r_q / D_q) / D_p over the unknown neighbours q of
// p (periodic in x, no coupling across the walls), c_pq the FP32 operator
// coefficients (E, W, N, S) the start kernel formed and D = dg.  On a
// uniform grid c_pq = c_qp, so M = D^-1 + D^-1 N D^-1 is symmetric, and it
// is positive definite where A is diagonally dominant (the spectral radius
// of D^-1/2 N D^-1/2 below one).  It takes about half the Jacobi-PCG's
// iterations for one more stencil of r per iteration, which the update
// kernel forms from r_n and A d_n at the neighbours (r is double-buffered:
// r_{n+1} goes to the other buffer while neighbours read r_n).
//
// START: d_0 = z_0 = M r_0, partial <r_0, z_0>.  Otherwise alpha as k_mcg_update,
// r_{n+1} = r_n - alpha A d_n, z_{n+1} = M r_{n+1}, partials <r, z>, <r, r>.
//
// A thread's column: the quotients r / D of its own, the row above and the
// row below it forms itself, east and west come through LDS (three divisions
// a cell instead of five); the next chunk's loads are in flight over this one.
// Bound by memory, 48 bytes a cell and component (80 with the x step here and
// A d and the diagonal as doubles): 36 -> 23 us at 1024^2, 196 -> 118 at
// 2048^2; the start 26 -> 18 and 162 -> 98.
template <bool START>
__global__ void __launch_bounds__(NTH) k_mcg_update_pc(pvk_grid g, pvk_scal *sc, pvk_mcg w, int n)
{
    __shared__ double sh[NTH];
    __shared__ double sq[2][NTH + 2];
    const mom_band m = mom_locate(g, w);
    const int c = m.comp, t = threadIdx.x;
    if (!START && sc->m_done[c]) return;
    const int P = g.P, NXM = g.NXM, NYM = g.NYM;
    const double *rold = (n & 1) ? w.r2[c] : w.r[c];
    double *rnew = (n & 1) ? w.r[c] : w.r2[c], *z = START ? w.d[c][0] : w.z[c];
    const float *Ad = w.Adf[c], *dg = w.dgf[c];
    struct cell { double r; float a, d; };
    struct chunk { cell o, n, s, e; float c[4]; };
    auto get = [&](cell &q, int i, int j) {
        q.r = AT(rold, i, j);
        if (!START) q.a = AT(Ad, i, j);
        q.d = AT(dg, i, j);
    };
    auto load = [&](chunk &k, mom_walk p) {
        const int nc = min(NTH, NXM - p.cb), i = m.i0 + p.cb + min(t, nc - 1);
        get(k.o, i, p.j);
        get(k.n, i, min(p.j + 1, NYM - 1));
        get(k.s, i, max(p.j - 1, m.jlo));
        if (t < 2) {                                    // the column west, east of the chunk
            const int e = m.i0 + p.cb + (t ? nc : -1);
            get(k.e, c ? wrapc(e, NXM) : wrapu(e, NXM), p.j);
        }
#pragma unroll
        for (int q = 0; q < 4; q++) k.c[q] = AT(w.cf[c][1 + q], i, p.j);
    };
    chunk k;
    mom_walk p = {m.j0, 0};
    load(k, p);
    const double alpha = START ? 0.0 : mom_alpha(sc, w, m, n, sh);
    auto rv = [&](const cell &q) { return START ? q.r : q.r - alpha * (double)q.a; };
    auto quo = [&](const cell &q) { return rv(q) / mom_D(q.d); };
    double a0 = 0.0, a1 = 0.0;
    for (int par = 0; p.j < m.j1; par ^= 1) {
        const int nc = min(NTH, NXM - p.cb), i = m.i0 + p.cb + t, j = p.j;
        const double ri = rv(k.o), qn = quo(k.n), qs = quo(k.s), D = mom_D(k.o.d);
        const float cE = k.c[0], cW = k.c[1], cN = k.c[2], cS = k.c[3];
        if (t < nc) sq[par][t + 1] = quo(k.o);
        if (t < 2) sq[par][t ? nc + 1 : 0] = quo(k.e);
        p.next(NXM);
        if (p.j < m.j1) load(k, p);
        lds_barrier();
        if (t < nc) {
            double s = ri;
            s += (double)cE * sq[par][t + 2];
            s += (double)cW * sq[par][t];
            if (j + 1 < NYM) s += (double)cN * qn;
            if (j - 1 >= m.jlo) s += (double)cS * qs;
            const double zz = s / D;
            if (!START) AT(rnew, i, j) = ri;
            AT(z, i, j) = zz;
            a0 += ri * zz;
            a1 += ri * ri;
        }
    }
    block_store_partial(a0, w.rz[c][START ? 0 : (n + 1) & 1], m.band, sh);
    if (!START) block_store_partial(a1, w.rr[c], m.band, sh);
}

// The same on bands of two rows, both rows of a chunk of columns at once.  Row
// by row, a band comes back to the rows it shares (with its own other row and
// with the next bands) half a launch later, when half of what the launch
// moves, twice an L2 at 1024^2, has gone by: r, A d and the diagonal came
// from HBM twice.  The second row's terms of the sums wait in registers until
// the first row is through (KC chunks at most: rows up to KC NTH cells), so the
// sums keep their order.  23.3 -> 18.1 us at 1024^2 and 118 -> 103 at 2048^2 (402
// MB, 3.9 TB/s); the start 18.5 -> 15.1 and 98 -> 94.
template <bool START, int KC>
__global__ void __launch_bounds__(NTH) k_mcg_update_pc2(pvk_grid g, pvk_scal *sc, pvk_mcg w, int n)
{
    __shared__ double sh[NTH];
    __shared__ double sq[2][2][NTH + 2];
    const mom_band m = mom_locate(g, w);
    const int c = m.comp, t = threadIdx.x;
    if (!START && sc->m_done[c]) return;
    const int P = g.P, NXM = g.NXM, NYM = g.NYM;
    const double *rold = (n & 1) ? w.r2[c] : w.r[c];
    double *rnew = (n & 1) ? w.r[c] : w.r2[c], *z = START ? w.d[c][0] : w.z[c];
    const float *Ad = w.Adf[c], *dg = w.dgf[c];
    const bool two = m.j0 + 1 < m.j1;
    struct cell { double r; float a, d; };
    cell v[4], e;                                       // rows j0 - 1 .. j0 + 2; the column beside the chunk
    float cf[2][4];
    auto get = [&](cell &q, int i, int j) {
        q.r = AT(rold, i, j);
        if (!START) q.a = AT(Ad, i, j);
        q.d = AT(dg, i, j);
    };
    auto load = [&](int cb) {
        const int nc = min(NTH, NXM - cb), i = m.i0 + cb + min(t, nc - 1);
#pragma unroll
        for (int a = 0; a < 4; a++) get(v[a], i, min(max(m.j0 - 1 + a, m.jlo), NYM - 1));
        if (t < 4) {                                    // thread 2 a + side: row j0 + a, west or east
            const int ie = m.i0 + cb + ((t & 1) ? nc : -1);
            get(e, c ? wrapc(ie, NXM) : wrapu(ie, NXM), min(m.j0 + (t >> 1), NYM - 1));
        }
#pragma unroll
        for (int a = 0; a < 2; a++)
#pragma unroll
            for (int q = 0; q < 4; q++) cf[a][q] = AT(w.cf[c][1 + q], i, min(m.j0 + a, NYM - 1));
    };
    load(0);
    const double alpha = START ? 0.0 : mom_alpha(sc, w, m, n, sh);
    auto rv = [&](const cell &q) { return START ? q.r : q.r - alpha * (double)q.a; };
    auto quo = [&](const cell &q) { return rv(q) / mom_D(q.d); };
    double a0 = 0.0, a1 = 0.0, p0[KC], p1[KC];
#pragma unroll
    for (int k = 0; k < KC; k++) {
        const int cb = k * NTH, par = k & 1;
        p0[k] = p1[k] = 0.0;
        if (cb < NXM) {
            const int nc = min(NTH, NXM - cb), i = m.i0 + cb + t;
            double q[4], r[2], D[2];
            float cc[2][4];
#pragma unroll
            for (int a = 0; a < 4; a++) q[a] = quo(v[a]);
#pragma unroll
            for (int a = 0; a < 2; a++) {
                r[a] = rv(v[a + 1]);
                D[a] = mom_D(v[a + 1].d);
                if (t < nc) sq[par][a][t + 1] = q[a + 1];
#pragma unroll
                for (int u = 0; u < 4; u++) cc[a][u] = cf[a][u];
            }
            if (t < 4) sq[par][t >> 1][(t & 1) ? nc + 1 : 0] = quo(e);
            if (cb + NTH < NXM) load(cb + NTH);
            lds_barrier();
            if (t < nc) {
#pragma unroll
                for (int a = 0; a < 2; a++) {
                    const int j = m.j0 + a;
                    double s = r[a];
                    s += (double)cc[a][0] * sq[par][a][t + 2];
                    s += (double)cc[a][1] * sq[par][a][t];
                    if (j + 1 < NYM) s += (double)cc[a][2] * q[a + 2];
                    if (j - 1 >= m.jlo) s += (double)cc[a][3] * q[a];
                    const double zz = s / D[a];
                    if (a == 0 || two) {
                        if (!START) AT(rnew, i, j) = r[a];
                        AT(z, i, j) = zz;
                        if (a == 0) {
                            a0 += r[a] * zz;
                            a1 += r[a] * r[a];
                        } else {
                            p0[k] = r[a] * zz;
                            p1[k] = r[a] * r[a];
                        }
                    }
                }
            }
        }
    }
#pragma unroll
    for (int k = 0; k < KC; k++) {
        a0 += p0[k];
        a1 += p1[k];
    }
    block_store_partial(a0, w.rz[c][START ? 0 : (n + 1) & 1], m.band, sh);
    if (!START) block_store_partial(a1, w.rr[c], m.band, sh);
}

// Two rows a band (the default) and at most eight chunks of terms to hold in
// registers (90 in all for four, 104 for eight; 128 keep four blocks on a CU):
// chunk by chunk; other bands and wider grids row by row.
template <bool START>
static void mcg_update_pc(const pvk_grid *g, pvk_scal *sc, const pvk_mcg *w, int n, hipStream_t s)
{
    const dim3 gr(w->nb[0] + w->nb[1]);
    if (w->band == 2 && g->NXM <= 4 * NTH)
        hipLaunchKernelGGL((k_mcg_update_pc2<START, 4>), gr, dim3(NTH), 0, s, *g, sc, *w, n);
    else if (w->band == 2 && g->NXM <= 8 * NTH)
        hipLaunchKernelGGL((k_mcg_update_pc2<START, 8>), gr, dim3(NTH), 0, s, *g, sc, *w, n);
    else
        hipLaunchKernelGGL(k_mcg_update_pc<START>, gr, dim3(NTH), 0, s, *g, sc, *w, n);
}

extern "C" void pvk_mcg_init(const pvk_grid *g, const pvk_phys *ph, int stage, pvk_scal *sc, const pvk_mcg *w,
                             hipStream_t s)
{
    const dim3 gr(w->nb[0] + w->nb[1]);
    if (ph->precision) {
        hipLaunchKernelGGL(k_mcg_init<float>, gr, dim3(NTH), 0, s, *g, *ph, stage, sc, *w);
        if (w->pc) mcg_update_pc<true>(g, sc, w, 0, s);
    } else
        hipLaunchKernelGGL(k_mcg_init<double>, gr, dim3(NTH), 0, s, *g, *ph, stage, sc, *w);
}

template <class R, bool FIRST>
static void mcg_apply(const pvk_grid *g, const pvk_phys *ph, pvk_scal *sc, const pvk_mcg *w, int n, hipStream_t s)
{
    const dim3 gr(w->nb[0] + w->nb[1]);
    if (w->band == 1) hipLaunchKernelGGL((k_mcg_apply<R, 1, FIRST>), gr, dim3(NTH), 0, s, *g, *ph, sc, *w, n);
    else if (w->band == 2) hipLaunchKernelGGL((k_mcg_apply<R, 2, FIRST>), gr, dim3(NTH), 0, s, *g, *ph, sc, *w, n);
    else hipLaunchKernelGGL((k_mcg_apply<R, 4, FIRST>), gr, dim3(NTH), 0, s, *g, *ph, sc, *w, n);
}

extern "C" void pvk_mcg_iter(const pvk_grid *g, const pvk_phys *ph, pvk_scal *sc, const pvk_mcg *w, int half, int n,
                             hipStream_t s)
{
    const dim3 gr(w->nb[0] + w->nb[1]);
    if (half == 0 && ph->precision) {
        if (n == 0) mcg_apply<float, true>(g, ph, sc, w, n, s);
        else mcg_apply<float, false>(g, ph, sc, w, n, s);
    } else if (half == 0) {
        if (n == 0) mcg_apply<double, true>(g, ph, sc, w, n, s);
        else mcg_apply<double, false>(g, ph, sc, w, n, s);
    } else if (!ph->precision)
        hipLaunchKernelGGL(k_mcg_update<double>, gr, dim3(NTH), 0, s, *g, sc, *w, n);
    else if (w->pc)                                  // the polynomial preconditioner: FP32 form only
        mcg_update_pc<false>(g, sc, w, n, s);
    else
        hipLaunchKernelGGL(k_mcg_update<float>, gr, dim3(NTH), 0, s, *g, sc, *w, n);
}
