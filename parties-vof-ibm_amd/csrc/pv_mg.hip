// pv_mg.hip -- multigrid-preconditioned CG for the variable-density pressure
// equation: the same operator, start, gauge and stopping rule as the
// FFT-preconditioned CG (csrc/pv_pcg.hip, psolve_cg.c:255-279), with one
// multigrid V-cycle as the preconditioner in place of the constant-density
// FFT solve.  With a density ratio of 1e-3 the FFT preconditioner leaves a
// spectrum spread over three decades (M_fft A ~ 1 in the liquid, ~1e3 in the
// gas); the V-cycle, built on the variable face coefficients, does not.
//
// Operator, as k_pcg_apply: (A x)_ij = bx_i (x_E - x) - bx_{i-1} (x - x_W)
//   + by_j (x_N - x) - by_{j-1} (x - x_S), periodic in x, zero-gradient walls.
// V-cycle (cell-centred, 2 x 2 aggregation; symmetric, so CG stays CG):
//   smoother      red-black Gauss-Seidel, nu = 1 or 2 sweeps: (red, black)
//                 before the coarse correction, (black, red) after it;
//   restriction   sum of the four fine residuals;
//   prolongation  piecewise constant;
//   coarse faces  half the sum of the two fine faces across the coarse face;
//   the last level (<= PVK_MG_BOTTOM cells) is solved exactly with the
//   inverse of its operator grounded at cell 0, both sides projected to zero
//   mean (built per solve by a band Cholesky, one column per workgroup).
// Each level above PVK_MG_LDS_CELLS cells is two launches (pre-smoothing +
// restriction; correction + post-smoothing) on LDS tiles with a halo, so f,
// the faces and x cross HBM once per launch; the levels below run in one
// workgroup from LDS.  The V-cycle stores and computes in T = double, or in
// T = float inside the FP64 CG (the mixed form: level 0 then reads r and
// writes z in FP64, its own x and faces are FP32).
#include <hip/hip_runtime.h>
#include <math.h>
#include <mutex>
#include "pv_kernels.h"
#include "pv_block.h"

#define AT(a, i, j) (a)[(ptrdiff_t)(j) * P + (i)]
#define TXP 64      // cells per block row of the per-cell kernels
#define TYR 4       // rows per block; TXP * TYR = NTH

// a level with arrays of the V-cycle's type
template <typename T> struct Lev {
    int nx, ny, pitch;
    T *x, *f, *bx, *by, *xp;
};
template <typename T> __host__ __device__ static Lev<T> lev(const pvk_mglev &l)
{
    Lev<T> v;
    v.nx = l.nx;
    v.ny = l.ny;
    v.pitch = l.pitch;
    v.x = (T *)l.x;
    v.f = (T *)l.f;
    v.bx = (T *)l.bx;
    v.by = (T *)l.by;
    v.xp = (T *)l.xp;
    return v;
}

template <typename T> __device__ __forceinline__ T ld(const T *a, int pitch, int i, int j)
{
    return a[(ptrdiff_t)j * pitch + i];
}

// f of level L at (i, j); level 0 of the FP32 V-cycle reads the FP64 r0
template <typename T> __device__ __forceinline__ T fget(const Lev<T> &L, const double *r0, int p0, int i, int j)
{
    return r0 ? (T)r0[(ptrdiff_t)j * p0 + i] : ld(L.f, L.pitch, i, j);
}

// stop test of CG iteration n on the <r, r> partials (as k_tri_cols):
// n = -1 sets the reference norm, n = -2 keeps it (warm restart).  The
// partials of r_{n+1} come from the level-0 pre-smoothing (rrt, per tile)
// when it forms r_{n+1}, else from the start or update kernels (rr, per row).
// Returns whether the solve stops here.  (Any workgroup of at least NTH threads.)
__device__ bool mg_stop_test(pvk_scal *sc, const pvk_pcg &w, int n, double tol, int maxit, double *sh)
{
    const bool tiles = (n >= 0 && w.nrrt > 0);
    const double rr = block_sum_wide(tiles ? w.rrt : w.rr, tiles ? w.nrrt : w.nrr, sh);
    const double bn = (n == -1) ? ((sqrt(rr) == 0.0) ? 1.0 : sqrt(rr)) : sc->p_bnorm;
    const double rel = sqrt(rr) / bn;
    const bool done = (rel <= tol) || (n + 1 >= maxit && n >= 0);
    if (threadIdx.x == 0) {
        if (n == -1) sc->p_bnorm = bn;
        sc->p_res = rel;
        sc->p_iter = (n < 0) ? 0 : n + 1;
        if (done) sc->p_done = (rel <= tol) ? 1 : 3;
    }
    return done;
}

// ---------------------------------------------------------------------------
// 2 x 2 blocks of cells (one coarse cell each), what a thread of the smoothing
// kernels owns: cells a (2I, 2J) and d (2I+1, 2J+1) are red, b (2I+1, 2J)
// and c (2I, 2J+1) black; faces between them, to the left (la, lc), right
// (br, dr), south (sa, sb) and north (nc, nd), 0 at a wall.  The faces, f,
// 1 / diagonal and x stay in registers; LDS holds x, one array per colour
// (row j, pair I at j hx + I: cells 2 I and 2 I + 1 of a row are one red,
// (i + j) even, and one black), at offsets R and B of the array x.
// ---------------------------------------------------------------------------
template <typename T> struct Blk {
    T ab, cd, la, lc, br, dr, ac, bd, sa, sb, nc, nd;
    T ia, ib, ic, id, fa, fb, fc, fd, a, b, c, d;
    int s, l, r, up, dn;            // slots of row 2J: own, left, right block; of rows 2J+2 and 2J-1
    int I, J;
    bool on;
};

// Two values of a row from column 2 I on, in one load: a smoothing level's
// width and pitch are even and its arrays, like the CG's fields, start on two
// values (pv_create, pv_mg_create).
template <typename T> __device__ __forceinline__ void ld2(const T *a, int pitch, int i, int j, T &v0, T &v1)
{
    typedef T T2 __attribute__((ext_vector_type(2)));
    const T2 v = *(const T2 *)(a + (ptrdiff_t)j * pitch + i);
    v0 = v.x;
    v1 = v.y;
}

template <typename T> __device__ __forceinline__ void st2(T *a, int pitch, int i, int j, T v0, T v1)
{
    typedef T T2 __attribute__((ext_vector_type(2)));
    T2 v;
    v.x = v0;
    v.y = v1;
    *(T2 *)(a + (ptrdiff_t)j * pitch + i) = v;
}

// faces of the blocks: every load unconditional, from clamped positions; the
// wall faces are masked in blk_diag
template <typename T, int NB> __device__ __forceinline__ void blk_faces(const Lev<T> &L, Blk<T> (&k)[NB])
{
#pragma unroll
    for (int u = 0; u < NB; u++) {
        const int i = 2 * k[u].I, j = 2 * k[u].J, iw = (i == 0) ? L.nx - 1 : i - 1, p = L.pitch;
        ld2(L.bx, p, i, j, k[u].ab, k[u].br);
        ld2(L.bx, p, i, j + 1, k[u].cd, k[u].dr);
        ld2(L.by, p, i, max(j - 1, 0), k[u].sa, k[u].sb);
        ld2(L.by, p, i, j, k[u].ac, k[u].bd);
        ld2(L.by, p, i, j + 1, k[u].nc, k[u].nd);
        k[u].la = ld(L.bx, p, iw, j);
        k[u].lc = ld(L.bx, p, iw, j + 1);
    }
}
// 1 / b of the Gauss-Seidel update: FP64 divides; FP32 takes the hardware
// reciprocal (1 ulp), which keeps the V-cycle a fixed symmetric operator
// (both sweep directions use the same value)
template <typename T> __device__ __forceinline__ T gs_rcp(T b) { return T(1) / b; }
template <> __device__ __forceinline__ float gs_rcp<float>(float b) { return __builtin_amdgcn_rcpf(b); }

// wall faces and 1 / diagonal (RCP: gs_rcp; else a division)
template <bool RCP, typename T, int NB> __device__ __forceinline__ void blk_diag(int ny, Blk<T> (&k)[NB])
{
    auto inv = [](T b) { return RCP ? gs_rcp(b) : T(1) / b; };
#pragma unroll
    for (int u = 0; u < NB; u++) {
        if (k[u].J == 0) k[u].sa = k[u].sb = T(0);
        if (k[u].J + 1 == (ny >> 1)) k[u].nc = k[u].nd = T(0);
        k[u].ia = inv(k[u].ab + k[u].la + k[u].ac + k[u].sa);
        k[u].ib = inv(k[u].br + k[u].ab + k[u].bd + k[u].sb);
        k[u].ic = inv(k[u].cd + k[u].lc + k[u].nc + k[u].ac);
        k[u].id = inv(k[u].dr + k[u].cd + k[u].nd + k[u].bd);
    }
}

// half-sweeps; each ends with a barrier (a colour's cells read only the other
// colour, whose last writes a barrier has already ordered)
template <int R, int B, typename T, int NB> __device__ __forceinline__ void sweep_red0(int hx, T *x, Blk<T> (&k)[NB])
{
#pragma unroll
    for (int u = 0; u < NB; u++)
        if (k[u].on) {
            x[R + k[u].s] = k[u].a = -k[u].fa * k[u].ia;
            x[R + k[u].s + hx] = k[u].d = -k[u].fd * k[u].id;
        }
    lds_barrier();
}
template <int R, int B, typename T, int NB> __device__ __forceinline__ void sweep_red(int hx, T *x, Blk<T> (&k)[NB])
{
    const T *q = x + B;
    T w[NB], s[NB], e[NB], n[NB];
#pragma unroll
    for (int u = 0; u < NB; u++)
        if (k[u].on) {
            w[u] = q[k[u].l];
            s[u] = q[k[u].dn];
            e[u] = q[k[u].r + hx];
            n[u] = q[k[u].up];
        }
#pragma unroll
    for (int u = 0; u < NB; u++)
        if (k[u].on) {
            k[u].a = (k[u].ab * k[u].b + k[u].la * w[u] + k[u].ac * k[u].c + k[u].sa * s[u] - k[u].fa) * k[u].ia;
            k[u].d = (k[u].dr * e[u] + k[u].cd * k[u].c + k[u].nd * n[u] + k[u].bd * k[u].b - k[u].fd) * k[u].id;
            x[R + k[u].s] = k[u].a;
            x[R + k[u].s + hx] = k[u].d;
        }
    lds_barrier();
}
template <int R, int B, typename T, int NB> __device__ __forceinline__ void sweep_black(int hx, T *x, Blk<T> (&k)[NB])
{
    const T *q = x + R;
    T e[NB], s[NB], w[NB], n[NB];
#pragma unroll
    for (int u = 0; u < NB; u++)
        if (k[u].on) {
            e[u] = q[k[u].r];
            s[u] = q[k[u].dn];
            w[u] = q[k[u].l + hx];
            n[u] = q[k[u].up];
        }
#pragma unroll
    for (int u = 0; u < NB; u++)
        if (k[u].on) {
            k[u].b = (k[u].br * e[u] + k[u].ab * k[u].a + k[u].bd * k[u].d + k[u].sb * s[u] - k[u].fb) * k[u].ib;
            k[u].c = (k[u].cd * k[u].d + k[u].lc * w[u] + k[u].nc * n[u] + k[u].ac * k[u].a - k[u].fc) * k[u].ic;
            x[B + k[u].s] = k[u].b;
            x[B + k[u].s + hx] = k[u].c;
        }
    lds_barrier();
}
// the four residuals f - A x of a block
template <int R, int B, typename T>
__device__ __forceinline__ void blk_residual(int hx, const T *x, const Blk<T> &k, T &ra, T &rb, T &rc, T &rd)
{
    const T a = k.a, b = k.b, c = k.c, d = k.d, *r = x + R, *q = x + B;
    ra = k.fa - (k.ab * (b - a) - k.la * (a - q[k.l]) + k.ac * (c - a) - k.sa * (a - q[k.dn]));
    rd = k.fd - (k.dr * (q[k.r + hx] - d) - k.cd * (d - c) + k.nd * (q[k.up] - d) - k.bd * (d - b));
    rb = k.fb - (k.br * (r[k.r] - b) - k.ab * (b - a) + k.bd * (d - b) - k.sb * (b - r[k.dn]));
    rc = k.fc - (k.cd * (d - c) - k.lc * (c - r[k.l + hx]) + k.nc * (r[k.up] - c) - k.ac * (c - a));
}

// ---------------------------------------------------------------------------
// Fused smoothing of one level (levels with more than PVK_MG_LDS_CELLS cells).
// A workgroup owns a core tile of TX x TY cells (64 x 16 on levels wider than
// 512, 32 x 16 up to 512, 32 x 8 up to 256: smaller tiles, more workgroups, on
// the levels whose time is latency) and works on it extended by a halo of 2 nu
// cells (periodic in x, cut at the walls in y): half-sweep k is right on the
// cells at distance >= k from the extended edge (the others read an own value
// where a neighbour would be), so after 2 nu half-sweeps the core (and the ring
// the residual needs) holds exactly what sweeping the whole level would give.
//
// A thread owns one 2 x 2 block of the extended tile, two on the widest tile.
// What bounded these kernels on large levels was instruction issue.  With a
// thread a cell (half the lanes idle in each half-sweep, four LDS reads an
// update, five loads, a column modulo and a position a cell) a launch took,
// pre and post, FP32, 21.7 and 15.4 us at 1024^2, 75 and 33 at 2048^2; with
// blocks 14.0 and 10.5, 58 and 26: the rate of the memory they touch (62 and
// 27 MB at 1024^2) within a factor of two, at 2048^2 4.2 TB/s.
// ---------------------------------------------------------------------------
template <int NU, int SH> struct MgTile {
    static constexpr int TX = (SH == 0) ? 64 : 32;    // core tile
    static constexpr int TY = (SH == 2) ? 8 : 16;
    static constexpr int H = 2 * NU;                  // halo
    static constexpr int HX = (TX + 2 * H) / 2;       // blocks a row of the extended tile
    static constexpr int HY = (TY + 2 * H) / 2;       // rows of blocks
    static constexpr int NBLK = HX * HY;
    static constexpr int NB = (NBLK + NTH - 1) / NTH; // blocks per thread
    static constexpr int R = 0, B = 2 * NBLK;         // x by colour
    static constexpr int KC = (TX * TY + NTH - 1) / NTH; // core cells per thread, row by row
};

// Positions of this thread's blocks: slots in the tile (at its edge and at a
// wall the own slot: finite, and not used or times a face of 0), columns wrapped
// into the level and rows clamped into it (off outside: those slots are never read).
// The mask of blocks in the core: bit u.
template <int NU, int SH, typename T>
__device__ __forceinline__ int tile_place(int nx, int ny, int bx, int by, Blk<T> (&k)[MgTile<NU, SH>::NB])
{
    using TT = MgTile<NU, SH>;
    const int hx = nx >> 1, hy = ny >> 1;
    int core = 0;
#pragma unroll
    for (int u = 0; u < TT::NB; u++) {
        const int q = min((int)threadIdx.x + u * NTH, TT::NBLK - 1), j = q / TT::HX, i = q - j * TT::HX;
        const int gi = bx * (TT::TX / 2) + i - TT::H / 2, gj = by * (TT::TY / 2) + j - TT::H / 2;
        int I = gi < 0 ? gi + hx : (gi >= hx ? gi - hx : gi);
        if (hx < TT::HX) {                              // a level narrower than the tile: round it more than once
            I %= hx;
            if (I < 0) I += hx;
        }
        k[u].on = (int)threadIdx.x + u * NTH < TT::NBLK && gj >= 0 && gj < hy;
        k[u].I = I;
        k[u].J = min(max(gj, 0), hy - 1);
        k[u].s = 2 * j * TT::HX + i;
        k[u].l = k[u].s - (i > 0);
        k[u].r = k[u].s + (i + 1 < TT::HX);
        k[u].dn = (j == 0 || gj <= 0) ? k[u].s : k[u].s - TT::HX;
        k[u].up = (j + 1 == TT::HY || gj + 1 >= hy) ? k[u].s : k[u].s + 2 * TT::HX;
        if (k[u].on && i >= TT::H / 2 && i < (TT::H + TT::TX) / 2 && j >= TT::H / 2 && j < (TT::H + TT::TY) / 2 && gi < hx)
            core |= 1 << u;
    }
    return core;
}

// f of the blocks: the level's, or from the FP64 field r0
template <typename T, int NB>
__device__ __forceinline__ void blk_rhs(const Lev<T> &L, const double *r0, int p0, Blk<T> (&k)[NB])
{
#pragma unroll
    for (int u = 0; u < NB; u++) {
        const int i = 2 * k[u].I, j = 2 * k[u].J;
        if (r0) {
            double a, b, c, d;
            ld2(r0, p0, i, j, a, b);
            ld2(r0, p0, i, j + 1, c, d);
            k[u].fa = (T)a;
            k[u].fb = (T)b;
            k[u].fc = (T)c;
            k[u].fd = (T)d;
        } else {
            ld2(L.f, L.pitch, i, j, k[u].fa, k[u].fb);
            ld2(L.f, L.pitch, i, j + 1, k[u].fc, k[u].fd);
        }
    }
}

// tile of this workgroup, XCD-aware (consecutive tiles of a run share an L2)
__device__ __forceinline__ void tile_of(int &bx, int &by)
{
    const int t = xcd_band(blockIdx.y * gridDim.x + blockIdx.x, gridDim.x * gridDim.y);
    by = t / gridDim.x;
    bx = t - by * gridDim.x;
}

// core cell q = threadIdx.x + m NTH, row by row: its place in the core and in
// the level (clamped into it); is it a cell of the level?
template <int NU, int SH>
__device__ __forceinline__ bool core_cell(int m, int bx, int by, int nx, int ny, int &q, int &gi, int &gj)
{
    using TT = MgTile<NU, SH>;
    const int t = threadIdx.x + m * NTH;
    q = min(t, TT::TX * TT::TY - 1);
    const int ly = q / TT::TX, lx = q - ly * TT::TX, x = bx * TT::TX + lx, y = by * TT::TY + ly;
    gi = min(x, nx - 1);
    gj = min(y, ny - 1);
    return t < TT::TX * TT::TY && x < nx && y < ny;
}

// pre-smoothing from x = 0 and restriction of the residual; the stop test of
// iteration n in block (0, 0) (check: the kernel after the one that formed
// the residual).  On level 0 with step (CG iteration n >= 0) the kernel
// first does the CG step: f = r_{n+1} = r_n - alpha (A d_n - mean) is formed on
// the fly from r_n = r0 (tile and halo), and the core writes r_{n+1} to rnew,
// phi += alpha d and the partial <r_{n+1}, r_{n+1}> of the tile.  The red x of
// the core goes to xp (the post kernel reads it with halos while it writes x;
// its first half-sweep overwrites the black), row j of it holding the row's
// reds side by side.
template <int NU, int SH, typename T>
__global__ void __launch_bounds__(NTH, sizeof(T) == 4 ? 4 : 3) k_mg_pre(Lev<T> L, Lev<T> C, const double *r0, double *rnew, int p0,
                                               pvk_scal *sc, pvk_pcg w, int n, double tol, int maxit, int check,
                                               int step, int ncell)
{
    using TT = MgTile<NU, SH>;
    constexpr int R = TT::R, B = TT::B, NB = TT::NB, KC = TT::KC;
    __shared__ T x[4 * TT::NBLK];
    __shared__ __align__(16) double rl[TT::TX * TT::TY];      // r_{n+1} of the core
    __shared__ double sh[3 * NTH];
    if (sc->p_done) return;
    if (check && n != -3 && blockIdx.x == 0 && blockIdx.y == 0) mg_stop_test(sc, w, n, tol, maxit, sh);
    int bx, by;
    tile_of(bx, by);
    Blk<T> k[NB];
    const int core = tile_place<NU, SH>(L.nx, L.ny, bx, by, k);
    const bool on = step && n >= 0;
    double acc = 0.0;
    blk_faces(L, k);
    if (on) {
        // the tile's loads go out first and are in flight while the step's
        // scalars are summed (the three sums' loads together), the core's
        // d_n and phi while f is formed; every load is unconditional
        double r[NB][4], a[NB][4], dd[KC], pp[KC];
        const double *d = w.d[n & 1];
        double *phi = w.phi;
#pragma unroll
        for (int u = 0; u < NB; u++) {
            const int i = 2 * k[u].I, j = 2 * k[u].J;
            ld2(r0, p0, i, j, r[u][0], r[u][1]);
            ld2(r0, p0, i, j + 1, r[u][2], r[u][3]);
            ld2(w.Ad, p0, i, j, a[u][0], a[u][1]);
            ld2(w.Ad, p0, i, j + 1, a[u][2], a[u][3]);
        }
        double rz, dad, sad;
        block_sum3(w.rz[n & 1], w.nrz, w.dad[n & 1], w.ndad, w.sad, w.ndad, sh, rz, dad, sad);
        const double alpha = rz / dad, mad = sad / (double)ncell;
#pragma unroll
        for (int m = 0; m < KC; m++) {
            int q, gi, gj;
            core_cell<NU, SH>(m, bx, by, L.nx, L.ny, q, gi, gj);
            const size_t idx = (size_t)gj * p0 + gi;
            dd[m] = d[idx];
            pp[m] = phi[idx];
        }
#pragma unroll
        for (int u = 0; u < NB; u++) {
#pragma unroll
            for (int e = 0; e < 4; e++) r[u][e] -= alpha * (a[u][e] - mad);
            k[u].fa = (T)r[u][0];
            k[u].fb = (T)r[u][1];
            k[u].fc = (T)r[u][2];
            k[u].fd = (T)r[u][3];
            if (core >> u & 1) {
                const int j = k[u].s / TT::HX - TT::H, i = 2 * (k[u].s % TT::HX) - TT::H;
                st2(rl, TT::TX, i, j, r[u][0], r[u][1]);
                st2(rl, TT::TX, i, j + 1, r[u][2], r[u][3]);
            }
        }
        blk_diag<false>(L.ny, k);
        sweep_red0<R, B>(TT::HX, x, k);         // its barrier orders rl too
#pragma unroll
        for (int m = 0; m < KC; m++) {
            int q, gi, gj;
            if (core_cell<NU, SH>(m, bx, by, L.nx, L.ny, q, gi, gj)) {
                const size_t idx = (size_t)gj * p0 + gi;
                const double rn = rl[q];
                rnew[idx] = rn;
                phi[idx] = pp[m] + alpha * dd[m];
                acc += rn * rn;
            }
        }
    } else {
        blk_rhs(L, r0, p0, k);
        blk_diag<false>(L.ny, k);
        sweep_red0<R, B>(TT::HX, x, k);
    }
    sweep_black<R, B>(TT::HX, x, k);
    if constexpr (NU == 2) {
        sweep_red<R, B>(TT::HX, x, k);
        sweep_black<R, B>(TT::HX, x, k);
    }
#pragma unroll
    for (int u = 0; u < NB; u++)
        if (core >> u & 1) {                    // a core block's coarse cell is its own
            T ra, rb, rc, rd;
            blk_residual<R, B>(TT::HX, x, k[u], ra, rb, rc, rd);
            C.f[(ptrdiff_t)k[u].J * C.pitch + k[u].I] = ra + rb + rc + rd;
            T *xp = L.xp + (ptrdiff_t)(2 * k[u].J) * L.pitch + k[u].I;
            xp[0] = k[u].a;
            xp[L.pitch] = k[u].d;
        }
    if (on) block_store_partial(acc, w.rrt, by * gridDim.x + bx, sh);
}

// coarse correction xp + xc(parent) and post-smoothing (black first, so only
// the red xp is there); the result goes to x, or to the FP64 z0 on level 0 of the FP32 V-cycle.  The
// input (xp) and the output are separate arrays: a block reads its halo from
// the neighbouring tiles' cores, which their blocks overwrite, and when the
// level has more tiles than the GPU holds at once those blocks may already
// have finished.
// dot: partial <f, x> of the core (FP64, with r0 on that level) into w.rz[slot]
template <int NU, int SH, typename T>
__global__ void __launch_bounds__(NTH, sizeof(T) == 4 ? 4 : 3) k_mg_post(Lev<T> L, Lev<T> C, const double *r0, double *z0, int p0,
                                                const pvk_scal *sc, pvk_pcg w, int dot, int slot)
{
    using TT = MgTile<NU, SH>;
    constexpr int R = TT::R, B = TT::B, NB = TT::NB, KC = TT::KC;
    __shared__ T x[4 * TT::NBLK];
    __shared__ double sh[NTH];
    if (sc->p_done) return;
    int bx, by;
    tile_of(bx, by);
    Blk<T> k[NB];
    tile_place<NU, SH>(L.nx, L.ny, bx, by, k);
    // every global load of the kernel first, unconditional (clamped positions)
    T xc[NB];
    double fd[KC];
    blk_faces(L, k);
    blk_rhs(L, r0, p0, k);
#pragma unroll
    for (int u = 0; u < NB; u++) {
        const T *xp = L.xp + (ptrdiff_t)(2 * k[u].J) * L.pitch + k[u].I;
        k[u].a = xp[0];
        k[u].d = xp[L.pitch];
        xc[u] = ld(C.x, C.pitch, k[u].I, k[u].J);
    }
#pragma unroll
    for (int m = 0; m < KC; m++) {              // the core's f for the dot
        fd[m] = 0.0;
        if (dot) {
            int q, gi, gj;
            core_cell<NU, SH>(m, bx, by, L.nx, L.ny, q, gi, gj);
            fd[m] = r0 ? r0[(ptrdiff_t)gj * p0 + gi] : (double)ld(L.f, L.pitch, gi, gj);
        }
    }
    blk_diag<false>(L.ny, k);
#pragma unroll
    for (int u = 0; u < NB; u++)                // x = xp + the parent's correction
        if (k[u].on) {
            x[R + k[u].s] = k[u].a = k[u].a + xc[u];
            x[R + k[u].s + TT::HX] = k[u].d = k[u].d + xc[u];
        }
    lds_barrier();
    sweep_black<R, B>(TT::HX, x, k);
    sweep_red<R, B>(TT::HX, x, k);
    if constexpr (NU == 2) {
        sweep_black<R, B>(TT::HX, x, k);
        sweep_red<R, B>(TT::HX, x, k);
    }
    double acc = 0.0;
#pragma unroll
    for (int m = 0; m < KC; m++) {
        int q, gi, gj;
        if (core_cell<NU, SH>(m, bx, by, L.nx, L.ny, q, gi, gj)) {
            const int ly = q / TT::TX + TT::H, lx = q % TT::TX + TT::H;
            const T v = x[(((lx + ly) & 1) ? B : R) + ly * TT::HX + (lx >> 1)];
            if (z0) z0[(ptrdiff_t)gj * p0 + gi] = (double)v;
            else L.x[(ptrdiff_t)gj * L.pitch + gi] = v;
            if (dot) acc += fd[m] * (double)v;
        }
    }
    if (dot) block_store_partial(acc, w.rz[slot], by * gridDim.x + bx, sh);
}

// coarse face coefficients from the fine ones (the fine level may be the
// FP64 level 0 of the FP32 V-cycle)
template <typename TF, typename T> __global__ void __launch_bounds__(NTH) k_mg_faces(Lev<TF> L, Lev<T> C)
{
    const int I = blockIdx.x * TXP + (threadIdx.x & (TXP - 1)), J = blockIdx.y * TYR + (threadIdx.x >> 6);
    if (I >= C.nx || J >= C.ny) return;
    const int p = L.pitch;
    C.bx[(ptrdiff_t)J * C.pitch + I] = (T)(0.5 * ((double)ld(L.bx, p, 2 * I + 1, 2 * J) +
                                                  (double)ld(L.bx, p, 2 * I + 1, 2 * J + 1)));
    C.by[(ptrdiff_t)J * C.pitch + I] = (T)(0.5 * ((double)ld(L.by, p, 2 * I, 2 * J + 1) +
                                                  (double)ld(L.by, p, 2 * I + 1, 2 * J + 1)));
}

// FP32 copies of the level-0 faces
__global__ void __launch_bounds__(NTH) k_mg_faces0(Lev<double> L, Lev<float> C)
{
    const int I = blockIdx.x * TXP + (threadIdx.x & (TXP - 1)), J = blockIdx.y * TYR + (threadIdx.x >> 6);
    if (I >= C.nx || J >= C.ny) return;
    C.bx[(ptrdiff_t)J * C.pitch + I] = (float)ld(L.bx, L.pitch, I, J);
    C.by[(ptrdiff_t)J * C.pitch + I] = (float)ld(L.by, L.pitch, I, J);
}

// H = P G P, G the inverse of the bottom operator M = -A_B + s e0 e0^T (s its
// (0,0) entry: grounded at cell 0, symmetric positive definite) and P the
// projection to zero mean, in FP64: the bottom solve is then x = -H f.
// Numbered x fastest, M is banded: the x neighbours (the periodic one
// included) lie within nx - 1 of the diagonal, the y neighbours at nx.  Once
// per solve: k_mg_bottom_factor (one wavefront) factors M = L L^T in LDS in
// band storage and writes the band out; k_mg_bottom_cols solves L L^T g = e_c
// for one column c per lane (the lanes of a block share the band in LDS and
// keep their vectors there; no lane waits on another), writes g as row c of
// G (G is symmetric) and its mean; k_mg_bottom_proj forms
// (P G P)_rc = G_rc - m_r - m_c + mean of the m, m the column means (the row
// means of a symmetric G), in the cycle's type.
#define BW 64
// Bottoms at most 16 wide (all the common sizes; a window of 16 x 16 fits the
// registers of a wavefront, a wider one does not) go to k_mg_bottom_factor16 and
// k_mg_bottom_cols16, whose band is padded: row stride 17 and 16 zero rows
// after the last, so every loop runs its full, compile-time length with no
// bounds tests (entries past the band stay zero through the factorisation).
#define BK 16
#define BKT 256

// lane moves within a quad, compile-time pattern
template <int CTRL> __device__ __forceinline__ double quad_move(double v)
{
    const int lo = __builtin_amdgcn_mov_dpp(__double2loint(v), CTRL, 0xf, 0xf, true);
    const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(v), CTRL, 0xf, 0xf, true);
    return __hiloint2double(hi, lo);
}
#define QUAD_ALL(k) ((k) * 0x55)           // lane k of the quad to all four
#define QUAD_UP 0x90                       // lane g takes lane g - 1 (lane 0 its own)
#define QUAD_X1 0xB1                       // lane g takes lane g ^ 1
#define QUAD_X2 0x4E                       // lane g takes lane g ^ 2

__device__ __forceinline__ double read_lane(double v, int lane)
{
    return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), lane),
                            __builtin_amdgcn_readlane(__double2loint(v), lane));
}

// Right-looking band Cholesky of a bottom at most 16 wide, the trailing 16 x 16
// window in the registers of one wavefront: lane 4 (r % 16) + g holds row r's
// columns c with c % 4 = g, one register for each c % 16 / 4.  Row k + 16 takes
// row k's place in step k; its entry in column k is untouched until then and
// comes separately.  A step (unrolled 16 times, so registers and lanes are
// compile-time): the unscaled column k goes round through LDS while 1 / sqrt of
// the pivot is formed, then each lane updates its four entries; the next pivot
// needs no LDS (its row's own factor, squared).  Bound by these two chains, 0.16
// us a step.  One wavefront on the band in LDS, the pivot, the column and
// the updated entries read and written there in each step, took 87 us for 16 x
// 16 and 51 for 12 x 12; 41 and 24 here.
template <typename T> __global__ void __launch_bounds__(BKT) k_mg_bottom_factor16(Lev<T> B, double *Lg, double *dinv)
{
    constexpr int W = BK + 1;
    extern __shared__ double in[];         // in[r BK + c % 4 * 4 + c % 16 / 4] = M[r][c], r - 16 < c <= r
    const int nx = B.nx, ny = B.ny, nb = nx * ny, p = B.pitch, t = threadIdx.x;
    const int nbp = (nb + BK - 1) / BK * BK, RP = nbp + BK + 1;    // rows past nb: those of the identity
    double *in16 = in + (size_t)RP * BK, *col = in16 + RP;         // M[r][r - 16]; the column of a step
    for (int q = t; q < RP * W; q += BKT) in[q] = 0.0;
    __syncthreads();
    // row r's diagonal and its couplings to the columns before it: the west
    // neighbour, the periodic east neighbour (of i = nx - 1) and the south one
    for (int r = t; r < nb; r += BKT) {
        const int j = r / nx, i = r - j * nx;
        const int ie = (i + 1 == nx) ? 0 : i + 1, iw = (i == 0) ? nx - 1 : i - 1;
        const double ce = ld(B.bx, p, i, j), cw = ld(B.bx, p, iw, j);
        const double cn = (j + 1 < ny) ? (double)ld(B.by, p, i, j) : 0.0;
        const double cs = (j > 0) ? (double)ld(B.by, p, i, j - 1) : 0.0;
        double dg = ce + cw + cn + cs;
        if (ie == i) dg -= ce;             // nx = 1: the periodic image is the cell itself
        if (iw == i) dg -= cw;
        if (r == 0) dg += dg;              // grounding: the (0, 0) entry doubled
        auto entry = [&](int d) -> double & {
            const int c = (r - d) & (BK - 1);
            return (d == BK) ? in16[r] : in[r * BK + (c & 3) * 4 + (c >> 2)];
        };
        entry(0) = dg;
        if (iw < i) entry(i - iw) -= cw;
        if (ie < i) entry(i - ie) -= ce;
        if (j > 0) entry(nx) -= cs;
    }
    for (int r = nb + t; r < nbp; r += BKT) in[r * BK + (r & 3) * 4 + ((r & (BK - 1)) >> 2)] = 1.0;
    // the couplings in the padded band that no step writes
    for (int q = t; q < (nbp + BK) * W; q += BKT) {
        const int r = q / W, c = r - (q - r * W);
        if (c < 0 || c >= nbp) Lg[q] = 0.0;
    }
    __syncthreads();
    if (t >= 64) return;
    const int row = t >> 2, g = t & 3;
    double A[4], nA[4], n16;
#pragma unroll
    for (int u = 0; u < 4; u++) A[u] = in[row * BK + g * 4 + u];
#pragma unroll
    for (int u = 0; u < 4; u++) nA[u] = in[BK * BK + g * 4 + u];
    n16 = in16[BK];
    double piv = read_lane(A[0], 0);
    // lanes g = 0 store their row's factor, at row * W + (row - k), lane 1
    // stores 1 / L[k][k] (L[k][k] itself is not used)
    const bool keep = (g == 0);
    int off = keep ? row * W + row : (int)(dinv - Lg);
    const int wrap = keep ? BK * (W + 1) : 0, next = keep ? -1 : 1;
    for (int kb = 0; kb < nbp; kb += BK) {
#pragma unroll
        for (int s = 0; s < BK; s++) {
            const int k = kb + s;
            const double As = (row == s) ? n16 : A[s >> 2];      // column k, in lanes g = k % 4
            if (g == (s & 3)) col[(row & 3) * 4 + (row >> 2)] = As;
            __builtin_amdgcn_wave_barrier();
            double cj[4];
#pragma unroll
            for (int u = 0; u < 4; u++) cj[u] = col[g * 4 + u];
            const double c = ((s & 3) == 0) ? quad_move<QUAD_ALL(0)>(As) : ((s & 3) == 1) ? quad_move<QUAD_ALL(1)>(As)
                           : ((s & 3) == 2) ? quad_move<QUAD_ALL(2)>(As) : quad_move<QUAD_ALL(3)>(As);
            if (row == s) {
                off += wrap;
#pragma unroll
                for (int u = 0; u < 4; u++) A[u] = nA[u];
            }
#pragma unroll
            for (int u = 0; u < 4; u++) nA[u] = in[(k + BK + 1) * BK + g * 4 + u];
            n16 = in16[k + BK + 1];
            __builtin_amdgcn_wave_barrier();
            // 1 / sqrt(piv): the hardware estimate (about 23 bits) and two Newton
            // steps (quadratic: to FP64 rounding), far shorter a chain than an
            // IEEE sqrt and divide; L[k][k] = piv / sqrt(piv)
            double inv = __builtin_amdgcn_rsq(piv);
            inv = inv * (1.5 - 0.5 * piv * inv * inv);
            inv = inv * (1.5 - 0.5 * piv * inv * inv);
            const double li = c * inv;
            constexpr int N = BK - 1;
            piv = read_lane(A[((s + 1) & N) >> 2] - li * li, 4 * ((s + 1) & N) + ((s + 1) & 3));
#pragma unroll
            for (int u = 0; u < 4; u++) A[u] = A[u] - li * (cj[u] * inv);  // M[i][j] -= L[i][k] L[j][k]
            const double out = keep ? li : inv;
            if (keep || t == 1) *(double *)((char *)Lg + (unsigned)off * 8u) = out;
            off += next;
        }
    }
}

template <typename T, int NX> __global__ void __launch_bounds__(BW) k_mg_bottom_factor(Lev<T> B, double *Lg, double *dinv)
{
    constexpr int TRI_PER_LANE = (NX * (NX + 1) / 2 + BW - 1) / BW;
    extern __shared__ double lb[];         // lb[r W + d] = M[r][r - d] (L after the factorisation)
    const int nx = B.nx, ny = B.ny, nb = nx * ny, p = B.pitch, t = threadIdx.x;
    const int W = nx + 1;
    const int ntri = nx * (nx + 1) / 2;
    // this lane's pairs (i, j), 1 <= j <= i <= nx, of the trailing update:
    // q = t + BW u in the order (1,1), (2,1), (2,2), (3,1), ...
    int ti[TRI_PER_LANE], tj[TRI_PER_LANE];
#pragma unroll
    for (int u = 0; u < TRI_PER_LANE; u++) {
        const int q = t + BW * u;
        int i = 1, base = 0;
        while (base + i <= q) { base += i; i++; }
        ti[u] = (q < ntri) ? i : nx + 1;                 // nx + 1: never active
        tj[u] = q - base + 1;
    }
    for (int q = t; q < nb * W; q += BW) lb[q] = 0.0;
    __syncthreads();
    // row r's diagonal and its couplings to the columns before it: the west
    // neighbour, the periodic east neighbour (of i = nx - 1) and the south one
    for (int r = t; r < nb; r += BW) {
        const int j = r / nx, i = r - j * nx;
        const int ie = (i + 1 == nx) ? 0 : i + 1, iw = (i == 0) ? nx - 1 : i - 1;
        const double ce = ld(B.bx, p, i, j), cw = ld(B.bx, p, iw, j);
        const double cn = (j + 1 < ny) ? (double)ld(B.by, p, i, j) : 0.0;
        const double cs = (j > 0) ? (double)ld(B.by, p, i, j - 1) : 0.0;
        double dg = ce + cw + cn + cs;
        if (ie == i) dg -= ce;             // nx = 1: the periodic image is the cell itself
        if (iw == i) dg -= cw;
        if (r == 0) dg += dg;              // grounding: the (0, 0) entry doubled
        lb[r * W] = dg;
        if (iw < i) lb[r * W + (i - iw)] -= cw;
        if (ie < i) lb[r * W + (i - ie)] -= ce;
        if (j > 0) lb[r * W + nx] -= cs;
    }
    __syncthreads();
    // right-looking band Cholesky.  The block is
    // one wavefront, whose LDS accesses complete in program order, so a step
    // needs no workgroup barrier: it reads the pivot, column k (unscaled) and
    // its pairs' entries, then writes L[k][k], the scaled column and the
    // updated entries -- no two lanes write, or write and read, one entry in
    // a step (the updated entries have j >= 1, the column entries d = i), and
    // the next step's reads come after these writes.  The wave barriers keep
    // the compiler from moving LDS accesses across steps.
    for (int k = 0; k < nb; k++) {
        const int m = min(nx, nb - 1 - k);
        const double piv = lb[k * W];
        const double ck = (t >= 1 && t <= m) ? lb[(k + t) * W + t] : 0.0;
        double mi[TRI_PER_LANE], mj[TRI_PER_LANE], mij[TRI_PER_LANE];
#pragma unroll
        for (int u = 0; u < TRI_PER_LANE; u++) {
            const int i = ti[u], j = tj[u];
            mi[u] = mj[u] = mij[u] = 0.0;
            if (i <= m) {
                mi[u] = lb[(k + i) * W + i];
                mj[u] = lb[(k + j) * W + j];
                mij[u] = lb[(k + i) * W + (i - j)];
            }
        }
        // 1 / sqrt(piv): the hardware estimate (about 23 bits) and two Newton
        // steps (quadratic: to FP64 rounding), far shorter a chain than an
        // IEEE sqrt and divide; L[k][k] = piv / sqrt(piv)
        double inv = __builtin_amdgcn_rsq(piv);
        inv = inv * (1.5 - 0.5 * piv * inv * inv);
        inv = inv * (1.5 - 0.5 * piv * inv * inv);
        const double dkk = piv * inv;
        __builtin_amdgcn_wave_barrier();
        if (t == 0) {
            lb[k * W] = dkk;
            dinv[k] = inv;
        }
        if (t >= 1 && t <= m) lb[(k + t) * W + t] = ck * inv;
#pragma unroll
        for (int u = 0; u < TRI_PER_LANE; u++) {           // M[k+i][k+j] -= L[k+i][k] L[k+j][k]
            const int i = ti[u], j = tj[u];
            if (i <= m) lb[(k + i) * W + (i - j)] = mij[u] - (mi[u] * inv) * (mj[u] * inv);
        }
        __builtin_amdgcn_wave_barrier();
    }
    __syncthreads();
    for (int q = t; q < nb * W; q += BW) Lg[q] = lb[q];
}

// sum over d = 2 .. NX of a[d] w[d - 1] as a pairwise tree: these terms do
// not depend on the newest value w[0], so only one product and two adds of a
// step wait on the step before
template <int NX> __device__ __forceinline__ double band_sum(const double *a, const double *w)
{
    double p[NX];
#pragma unroll
    for (int d = 0; d < NX; d++) p[d] = (d >= 1) ? a[d + 1] * w[d] : 0.0;   // p[d] = a[d+1] w[d], d >= 1
#pragma unroll
    for (int h = 1; h < NX; h <<= 1)
#pragma unroll
        for (int d = 0; d + h < NX; d += 2 * h) p[d] += p[d + h];
    return p[0];
}

// columns c = blockIdx * cpb + lane of G from the band L and 1 / diag(L),
// both staged in LDS.  Each lane keeps the last NX values of its recurrence
// in registers and reads the next band row while the current one is used,
// so a step waits on one product, not on LDS.
template <int NX>
__global__ void __launch_bounds__(BW) k_mg_bottom_cols(int nx, int nb, int cpb, const double *Lg, const double *dinv,
                                                       double *G, double *cm)
{
    extern __shared__ double sm[];
    const int W = nx + 1, t = threadIdx.x;
    double *lb = sm, *di = sm + (size_t)nb * W, *y = di + nb;    // y[r cpb + lane]
    for (int q = t; q < nb * W; q += BW) lb[q] = Lg[q];
    for (int q = t; q < nb; q += BW) di[q] = dinv[q];
    __syncthreads();
    const int c = blockIdx.x * cpb + t;
    if (t >= cpb || c >= nb) return;
    // a band entry, 0 past the band or past the last row
    auto band = [&](int row, int d) -> double {
        return (d <= nx && row < nb) ? lb[row * W + d] : 0.0;
    };
    double w[NX], a[NX + 1], an[NX + 1];
    // L y = e_c: every lane runs all rows (y_r = 0 before row c comes out of
    // the same recurrence), so the loops stay uniform; w[d - 1] = y_{r - d},
    // a[d] = L[r][r - d], a[0] = 1 / L[r][r]
#pragma unroll
    for (int d = 0; d < NX; d++) w[d] = 0.0;
#pragma unroll
    for (int d = 0; d <= NX; d++) a[d] = (d == 0) ? di[0] : band(0, d);
    for (int r = 0; r < nb; r++) {
        const int rn = (r + 1 < nb) ? r + 1 : r;
#pragma unroll
        for (int d = 0; d <= NX; d++) an[d] = (d == 0) ? di[rn] : band(rn, d);
        const double v = ((r == c ? 1.0 : 0.0) - (band_sum<NX>(a, w) + a[1] * w[0])) * a[0];
#pragma unroll
        for (int d = NX - 1; d >= 1; d--) w[d] = w[d - 1];
        w[0] = v;
        y[r * cpb + t] = v;
#pragma unroll
        for (int d = 0; d <= NX; d++) a[d] = an[d];
    }
    // L^T g = y, in place; w[d - 1] = g_{r + d}, a[d] = L[r + d][r],
    // a[0] = 1 / L[r][r]
#pragma unroll
    for (int d = 0; d < NX; d++) w[d] = 0.0;
#pragma unroll
    for (int d = 0; d <= NX; d++) a[d] = (d == 0) ? di[nb - 1] : band(nb - 1 + d, d);
    for (int r = nb - 1; r >= 0; r--) {
        const int rp = (r > 0) ? r - 1 : 0;
#pragma unroll
        for (int d = 0; d <= NX; d++) an[d] = (d == 0) ? di[rp] : band(rp + d, d);
        const double yr = y[r * cpb + t];
        const double v = (yr - (band_sum<NX>(a, w) + a[1] * w[0])) * a[0];
#pragma unroll
        for (int d = NX - 1; d >= 1; d--) w[d] = w[d - 1];
        w[0] = v;
        y[r * cpb + t] = v;
#pragma unroll
        for (int d = 0; d <= NX; d++) a[d] = an[d];
    }
    double s = 0.0;
    for (int r = 0; r < nb; r++) {
        const double g = y[r * cpb + t];
        G[(size_t)c * nb + r] = g;
        s += g;
    }
    cm[c] = s / nb;
}

// The columns of bottoms at most 16 wide, 16 a block.  A quad of lanes shares a
// column: lane g forms the products with the values 4 g + 1 .. 4 g + 4 rows
// back (its window x, a ring of four at compile-time places, the row loop
// unrolled by 16; a value goes from lane to lane as it ages), the pairwise
// tree of band_sum ends in two moves within the quad, and all four lanes form
// the new value, so only one product and two adds of a step wait on the step
// before.  Rows are taken up to a multiple of 16, past nb the band and 1 / diag
// are zero, so those rows yield zero.  Three wavefronts only help to stage the
// band and to store the columns.  With a lane a column, all 16 products in
// it and 17 LDS reads a row, 94 us for 16 x 16 and 45 for 12 x 12; 53 and 31 here.
#define BYP (BK + 1)                       // pitch of y: no bank conflicts down a column
__global__ void __launch_bounds__(BKT) k_mg_bottom_cols16(int nb, const double *Lg, const double *dinv, double *G,
                                                          double *cm)
{
    constexpr int W = BK + 1;
    extern __shared__ double sm[];
    const int t = threadIdx.x, nbp = (nb + BK - 1) / BK * BK, RP = nbp + BK, c0 = blockIdx.x * BK;
    double *lb = sm, *di = sm + (size_t)RP * W, *y = di + RP;    // y[r BYP + column]
#pragma unroll 6
    for (int q = t; q < RP * W; q += BKT) lb[q] = (q < (nb + BK) * W) ? Lg[q] : 0.0;
    for (int q = t; q < RP; q += BKT) di[q] = (q < nb) ? dinv[q] : 0.0;
    __syncthreads();
    if (t < 64) {
        const int cc = t >> 2, g = t & 3, c = c0 + cc;
        double x[4] = {0.0, 0.0, 0.0, 0.0}, a[2][4], d[2], v = 0.0;
        // one row: sum, new value; xs the slot of the value before, m-th back in slot ord(m)
        auto step = [&](const double (&A)[4], double D, double e, double &x0, double x1, double x2, double x3) {
            const double o = quad_move<QUAD_UP>(x0);             // the value 4 g + 1 rows back, g > 0
            double p0 = A[0] * o, p2 = A[2] * x2;
            if (g == 0) p0 = 0.0;
            p0 += A[1] * x1;
            p2 += A[3] * x3;
            p0 += p2;
            p0 += quad_move<QUAD_X1>(p0);
            p0 += quad_move<QUAD_X2>(p0);
            const double a1 = quad_move<QUAD_ALL(0)>(A[0]), w0 = v;
            x0 = (g == 0) ? w0 : o;
            v = (e - (p0 + a1 * w0)) * D;
        };
        // L y = e_c, from the first row of this block's columns (y is zero
        // before its column): A[m] = L[r][r - 4 g - 1 - m]
        auto row_f = [&](double (&A)[4], double &D, int r) {
#pragma unroll
            for (int m = 0; m < 4; m++) A[m] = lb[r * W + 4 * g + 1 + m];
            D = di[r];
        };
        row_f(a[0], d[0], c0);
        for (int rb = c0; rb < nbp; rb += BK) {
#pragma unroll
            for (int s = 0; s < BK; s++) {
                const int r = rb + s;
                row_f(a[(s + 1) & 1], d[(s + 1) & 1], r + 1);
                step(a[s & 1], d[s & 1], (r == c) ? 1.0 : 0.0, x[(s + 3) & 3], x[(s + 2) & 3], x[(s + 1) & 3], x[s & 3]);
                if (g == 0) y[r * BYP + cc] = v;
            }
        }
        // L^T g = y in place, from the last row: A[m] = L[r + 4 g + 1 + m][r]
        auto row_b = [&](double (&A)[4], double &D, int r) {
#pragma unroll
            for (int m = 0; m < 4; m++) A[m] = lb[r * W + (4 * g + 1 + m) * (W + 1)];
            D = di[r];
        };
        v = 0.0;
#pragma unroll
        for (int q = 0; q < 4; q++) x[q] = 0.0;
        row_b(a[0], d[0], nbp - 1);
        for (int rb = nbp - BK; rb >= 0; rb -= BK) {
#pragma unroll
            for (int q = 0; q < BK; q++) {
                const int s = BK - 1 - q, r = rb + s;
                row_b(a[(q + 1) & 1], d[(q + 1) & 1], max(r - 1, 0));
                const double yr = (rb >= c0) ? y[r * BYP + cc] : 0.0;
                step(a[q & 1], d[q & 1], yr, x[(s + 1) & 3], x[(s + 2) & 3], x[(s + 3) & 3], x[s & 3]);
                if (g == 0) y[r * BYP + cc] = v;
            }
        }
    }
    __syncthreads();
    for (int u = t >> 6; u < BK; u += BKT / 64)
        if (c0 + u < nb)
            for (int r = t & 63; r < nb; r += 64) G[(size_t)(c0 + u) * nb + r] = y[r * BYP + u];
    if (t < BK && c0 + t < nb) {
        double sum = 0.0;
        for (int r = 0; r < nb; r++) sum += y[r * BYP + t];
        cm[c0 + t] = sum / nb;
    }
}

template <typename T> __global__ void __launch_bounds__(NTH) k_mg_bottom_proj(int nb, const double *G, const double *cm, T *H)
{
    __shared__ double sh[NTH];
    const int r = blockIdx.x, t = threadIdx.x;
    double s = 0.0;
    for (int q = t; q < nb; q += NTH) s += cm[q];
    sh[t] = s;
    __syncthreads();
    for (int w = NTH / 2; w > 0; w >>= 1) {
        if (t < w) sh[t] += sh[t + w];
        __syncthreads();
    }
    const double tm = sh[0] / nb, mr = cm[r];
    for (int c = t; c < nb; c += NTH) H[(size_t)r * nb + c] = (T)(((G[(size_t)r * nb + c] - mr) - cm[c]) + tm);
}

// ---------------------------------------------------------------------------
// Levels c0 .. nlev-1 in one workgroup.  The kernel runs on one CU, so its
// time is a chain of barrier-separated half-sweeps and bottom visits, and it
// is bound by their latency: at 1024^2 (64^2, 32^2 and the 16^2 bottom, W on
// both, FP32) a wavefront spends 53 % of its time waiting for the L2, LDS or a
// barrier, 16 % for an issue slot and 31 % on an instruction, a SIMD's vector
// unit is busy for 30 % (FP64, V at 96^2: 64, 14, 22 and 26 %).
//
// A thread owns 2 x 2 blocks of cells (one coarse cell each): two blocks of
// level c0, one of each level below.  It keeps their faces, 1 / diagonal, f
// and x in registers for the whole kernel; LDS holds only x, one array per
// colour (so neighbouring lanes read neighbouring words), and the coarse
// right-hand sides.  A half-sweep of a block is then four LDS reads (the
// neighbours outside the block), two updates and two writes, the restricted
// residual of a block is its owner's own sum, and every LDS address is an
// offset from the one dynamic array, so the accesses are LDS instructions.
// Reading the level descriptors (with their pointers) from LDS instead, as
// an earlier form did, made every access a flat one, and each pass reloaded
// the coefficients: at 1024^2 as above 53.4 us a launch, FP64, V at 96^2, 26;
// now 33.3 and 13.8 (kernel traces of whole runs).
// ---------------------------------------------------------------------------
#define CT 512
static_assert(PVK_MG_LDS_CELLS <= 8 * CT, "level c0 has at most two 2 x 2 blocks a thread");
static_assert(PVK_MG_LOW <= 3, "k_mg_coarse is instantiated for up to three smoothing levels");

__device__ __forceinline__ int ilog2_or_neg(int n) { return (n > 0 && (n & (n - 1)) == 0) ? __ffs(n) - 1 : -1; }

// In-LDS layout, in units of T and at fixed places (the most a level can
// need), so an access is an index register and an immediate offset: smoothing
// level K's red and black x (row j, pair I at j hx + I: cells 2 I and 2 I + 1
// of a row are one red, (i + j) even, and one black) and, below c0, its f;
// the bottom's x; then in doubles the bottom's f and partial sums.
template <int K> struct CLds {
    static constexpr int N = PVK_MG_LDS_CELLS >> (2 * K);                 // cells at most
    static constexpr int R = K ? CLds<(K ? K - 1 : 0)>::END : 0, B = R + N / 2, F = R + N, END = F + (K ? N : 0);
};
#define MG_BX CLds<2>::END                          // the bottom's x
#define MG_BD (MG_BX + PVK_MG_BOTTOM)               // end of the T part
#define MG_BF (PVK_MG_BOTTOM + 8)                   // the bottom's f
static_assert(MG_BD % 2 == 0, "the doubles start on 8 bytes");
template <typename T> static constexpr size_t coarse_lds_bytes()
{
    return MG_BD * sizeof(T) + sizeof(double) * (MG_BF + 3 * PVK_MG_BOTTOM);
}
static_assert(coarse_lds_bytes<double>() <= 65536, "a launch gets 64 KiB without asking for more");

struct CGeo {
    int nx, ny, hx, nblk;           // cells, blocks a row, blocks
};

// The blocks' positions.  A neighbour beyond a wall has face 0; its slot is
// the block's own (finite once the level has been swept, and 0 times it is 0).
template <typename T, int NB> __device__ __forceinline__ void blk_place(const CGeo &g, Blk<T> (&k)[NB])
{
    const int lhx = ilog2_or_neg(g.hx);
#pragma unroll
    for (int u = 0; u < NB; u++) {
        const int q = threadIdx.x + u * CT, hx = g.hx, hy = g.ny >> 1;
        k[u].on = q < g.nblk;
        const int qq = k[u].on ? q : 0;
        const int j = (lhx >= 0) ? (qq >> lhx) : qq / hx, i = qq - j * hx;
        k[u].I = i;
        k[u].J = j;
        k[u].s = 2 * j * hx + i;
        k[u].l = k[u].s + ((i == 0) ? hx - 1 : -1);
        k[u].r = k[u].s + ((i + 1 == hx) ? 1 - hx : 1);
        k[u].dn = (j == 0) ? k[u].s : k[u].s - hx;
        k[u].up = (j + 1 == hy) ? k[u].s : k[u].s + 2 * hx;
    }
}

// the first black half-sweep after the coarse correction: the red neighbours
// are read as x + x_coarse(their parent); the red cells themselves need not be
// corrected, the red half-sweep that follows overwrites them
template <int K, bool BOT, typename T, int NB>
__device__ __forceinline__ void sweep_black_corr(const CGeo &g, T *x, Blk<T> (&k)[NB])
{
    // x of the coarse cell (i, j)
    auto px = [&](int i, int j) {
        if constexpr (BOT) return x[MG_BX + j * g.hx + i];
        else return x[CLds<K + 1>::R + (((i + j) & 1) ? CLds<K + 1>::N / 2 : 0) + j * (g.hx >> 1) + (i >> 1)];
    };
    const T *R = x + CLds<K>::R;
    T e[NB], s[NB], w[NB], n[NB], pc[NB];
#pragma unroll
    for (int u = 0; u < NB; u++)
        if (k[u].on) {
            const int i = k[u].I, j = k[u].J, d = k[u].dn != k[u].s, h = k[u].up != k[u].s;
            e[u] = R[k[u].r] + px(i + k[u].r - k[u].s, j);
            s[u] = R[k[u].dn] + px(i, j - d);
            w[u] = R[k[u].l + g.hx] + px(i + k[u].l - k[u].s, j);
            n[u] = R[k[u].up] + px(i, j + h);
            pc[u] = px(i, j);
        }
#pragma unroll
    for (int u = 0; u < NB; u++)
        if (k[u].on) {
            const T a = k[u].a + pc[u], d = k[u].d + pc[u];
            k[u].b = (k[u].br * e[u] + k[u].ab * a + k[u].bd * d + k[u].sb * s[u] - k[u].fb) * k[u].ib;
            k[u].c = (k[u].cd * d + k[u].lc * w[u] + k[u].nc * n[u] + k[u].ac * a - k[u].fc) * k[u].ic;
            x[CLds<K>::B + k[u].s] = k[u].b;
            x[CLds<K>::B + k[u].s + g.hx] = k[u].c;
        }
    lds_barrier();
}

// Residual of the blocks, summed over each block: the coarse cell's f (with
// row sums first, as (red + black) of row 2J plus (red + black) of row 2J+1),
// to the next smoothing level's f, or to the bottom's in FP64
template <int K, bool BOT, typename T, int NB>
__device__ __forceinline__ void restrict_res(const CGeo &g, T *x, const Blk<T> (&k)[NB], double *bf)
{
#pragma unroll
    for (int u = 0; u < NB; u++)
        if (k[u].on) {
            T ra, rb, rc, rd;
            blk_residual<CLds<K>::R, CLds<K>::B>(g.hx, x, k[u], ra, rb, rc, rd);
            const T v = (ra + rb) + (rd + rc);
            const int q = threadIdx.x + u * CT;
            if constexpr (BOT) bf[q] = (double)v;
            else x[CLds<K + 1>::F + q] = v;
        }
    lds_barrier();
}

// Bottom level, x = -H f (H = P G P, symmetric, in the cycle's type), in
// FP64.  Wavefronts 2 q and 2 q + 1 sum quarter q of the columns, a thread for
// two rows r and r + 1 (each f from LDS serves two products), reading
// H[c][r], H[c][r+1] = H[r][c], H[r+1][c]; the four quarters are added in order
// through LDS.  H comes from the L2 through one CU (256 KiB or
// 512 KiB a visit), so the loads are what it costs: they go out in chunks of
// PF columns, one chunk ahead of the sums and the first one before the residual
// that the solve waits for.  Two buffers are read in turn (copying one to the
// other would wait for it), and a quarter's bounds and addresses are scalars:
// launched alone, back to back (faster than in a run, where other kernels come
// between), with the copy, and tests a lane, a launch took 44 us in FP64 (64^2,
// W on both levels), 29 (44 x 88, W on one) and 14.3 (48^2, V), 32.6 in FP32
// (64^2), and 38, 25, 12.4 and 30.8 without.  Wider FP32 loads (four rows a
// lane, halves of the wavefront swapped) gave nothing.
template <typename T> struct HChunk {
    static constexpr int PF = sizeof(T) == 4 ? 8 : 4;
    T h[PF][2];
};
struct BotGeo {
    int n, c0, nq, row;             // this quarter's columns [c0, c0 + nq), this thread's first row
};
__device__ __forceinline__ BotGeo bottom_geo(int n)
{
    const int q = __builtin_amdgcn_readfirstlane(threadIdx.x >> 7), m = (n + 3) / 4, c0 = q * m;
    return {n, c0, min(m, n - c0), 2 * ((int)threadIdx.x & 127)};
}
template <typename T> __device__ __forceinline__ void bottom_load(const BotGeo &g, const T *H, int c, HChunk<T> &k)
{
    constexpr int PF = HChunk<T>::PF;
    typedef T T2 __attribute__((ext_vector_type(2)));
    c += g.c0;
    if ((g.n & 1) == 0) {                                          // rows r, r + 1 in one aligned load
        const int r = min(g.row, g.n - 2);
#pragma unroll
        for (int u = 0; u < PF; u++) {
            const T2 v = *(const T2 *)(H + (size_t)min(c + u, g.n - 1) * g.n + r);       // past the end: not used
            k.h[u][0] = v.x;
            k.h[u][1] = v.y;
        }
    } else {
        const int r0 = min(g.row, g.n - 1), r1 = min(g.row + 1, g.n - 1);
#pragma unroll
        for (int u = 0; u < PF; u++) {
            const T *p = H + (size_t)min(c + u, g.n - 1) * g.n;
            k.h[u][0] = p[r0];
            k.h[u][1] = p[r1];
        }
    }
}
// v - h f: fused where the product is exact in FP64 (FP32 entries), which rounds alike
__device__ __forceinline__ double bottom_acc(float h, double f, double v) { return __builtin_fma(-(double)h, f, v); }
__device__ __forceinline__ double bottom_acc(double h, double f, double v) { return v - h * f; }
// columns c .. c + PF - 1 of the quarter
template <typename T>
__device__ __forceinline__ void bottom_add(const BotGeo &g, const HChunk<T> &k, const double *f, int c, double &v0, double &v1)
{
    constexpr int PF = HChunk<T>::PF;
    f += c;
    if (c + PF <= g.nq) {
#pragma unroll
        for (int u = 0; u < PF; u++) {
            v0 = bottom_acc(k.h[u][0], f[u], v0);
            v1 = bottom_acc(k.h[u][1], f[u], v1);
        }
    } else {
#pragma unroll
        for (int u = 0; u < PF; u++)
            if (c + u < g.nq) {
                v0 = bottom_acc(k.h[u][0], f[u], v0);
                v1 = bottom_acc(k.h[u][1], f[u], v1);
            }
    }
}

template <typename T>
__device__ __forceinline__ void bottom_solve(int n, const T *H, HChunk<T> &k, const double *bf, double *part, T *X)
{
    static_assert(CT == 2 * PVK_MG_BOTTOM, "four quarters of the bottom's columns, two rows a thread");
    constexpr int PF = HChunk<T>::PF;
    const BotGeo g = bottom_geo(n);
    const int r = g.row, q = threadIdx.x >> 7;
    const double *f = bf + g.c0;
    double v0 = 0.0, v1 = 0.0;
    for (int c = 0; c < g.nq; c += 2 * PF) {
        HChunk<T> k2;
        bottom_load(g, H, c + PF, k2);
        bottom_add(g, k, f, c, v0, v1);
        if (c + 2 * PF < g.nq) bottom_load(g, H, c + 2 * PF, k);
        if (c + PF < g.nq) bottom_add(g, k2, f, c + PF, v0, v1);
    }
    if (q > 0) {
        part[(q - 1) * PVK_MG_BOTTOM + r] = v0;
        part[(q - 1) * PVK_MG_BOTTOM + r + 1] = v1;
    }
    lds_barrier();
    if (q == 0) {
        if (r < n) X[r] = (T)(((v0 + part[r]) + part[PVK_MG_BOTTOM + r]) + part[2 * PVK_MG_BOTTOM + r]);
        if (r + 1 < n)
            X[r + 1] = (T)(((v1 + part[r + 1]) + part[PVK_MG_BOTTOM + r + 1]) + part[2 * PVK_MG_BOTTOM + r + 1]);
    }
    lds_barrier();
}

// everything a thread keeps: its blocks of each smoothing level
template <typename T, int NL> struct CState {
    CGeo g[NL + 1];                 // smoothing levels and the bottom
    Blk<T> k0[2], k1[1], k2[1];
    HChunk<T> h;                    // the bottom solve's first columns
    T *x;
    double *bf, *part;
};

// One visit of smoothing level K: a V, or with the level's bit in wmask two
// coarse corrections with smoothing between them (pre-smooth, correct,
// post-smooth, pre-smooth, correct, post-smooth: the error propagation
// S^T C S S^T C S stays symmetric in the energy inner product).  From x = 0
// the first red update is -f / diag; the second pre-smoothing leaves its red
// half-sweep out: the post-smoothing just ended with one and no black cell
// has changed since, so it would reproduce the same values.
template <int K, typename T, int NL> __device__ __forceinline__ void cycle(const pvk_mg &m, CState<T, NL> &S);
template <int K, int NB, typename T, int NL>
__device__ __forceinline__ void cycle_level(const pvk_mg &m, CState<T, NL> &S, Blk<T> (&k)[NB])
{
    constexpr bool BOT = (K + 1 == NL);
    const CGeo g = S.g[K];
    T *x = S.x;
    if constexpr (K > 0) {
#pragma unroll
        for (int u = 0; u < NB; u++)
            if (k[u].on) {
                const T *f = x + CLds<K>::F + 2 * k[u].J * g.nx + 2 * k[u].I;
                k[u].fa = f[0];
                k[u].fb = f[1];
                k[u].fc = f[g.nx];
                k[u].fd = f[g.nx + 1];
            }
    }
    const int visits = 1 + ((m.wmask >> (m.c0 + K)) & 1);
    for (int v = 0; v < visits; v++) {
        if (v == 0) sweep_red0<CLds<K>::R, CLds<K>::B>(g.hx, x, k);
        sweep_black<CLds<K>::R, CLds<K>::B>(g.hx, x, k);
        for (int sw = 1; sw < m.nu; sw++) {
            sweep_red<CLds<K>::R, CLds<K>::B>(g.hx, x, k);
            sweep_black<CLds<K>::R, CLds<K>::B>(g.hx, x, k);
        }
        if constexpr (BOT) {
            const int n = S.g[NL].nx * S.g[NL].ny;
            bottom_load(bottom_geo(n), (const T *)m.H, 0, S.h);
        }
        restrict_res<K, BOT>(g, x, k, S.bf);
        cycle<K + 1>(m, S);
        sweep_black_corr<K, BOT>(g, x, k);
        sweep_red<CLds<K>::R, CLds<K>::B>(g.hx, x, k);
        for (int sw = 1; sw < m.nu; sw++) {
            sweep_black<CLds<K>::R, CLds<K>::B>(g.hx, x, k);
            sweep_red<CLds<K>::R, CLds<K>::B>(g.hx, x, k);
        }
    }
}
template <int K, typename T, int NL> __device__ __forceinline__ void cycle(const pvk_mg &m, CState<T, NL> &S)
{
    if constexpr (K == NL) bottom_solve(S.g[NL].nx * S.g[NL].ny, (const T *)m.H, S.h, S.bf, S.part, S.x + MG_BX);
    else if constexpr (K == 0) cycle_level<0>(m, S, S.k0);
    else if constexpr (K == 1) cycle_level<1>(m, S, S.k1);
    else cycle_level<2>(m, S, S.k2);
}

// check: the stop test of iteration n first (grids with at most one tiled level;
// as a launch of its own 2 us and a gap an iteration)
template <typename T, int NL>
__global__ void __launch_bounds__(CT) k_mg_coarse(pvk_mg m, pvk_scal *sc, pvk_pcg w, int n, double tol, int maxit, int check)
{
    extern __shared__ double lds_raw[];
    T *x = (T *)lds_raw;
    CState<T, NL> S;
    S.x = x;
#pragma unroll
    for (int K = 0; K <= NL; K++) {
        const pvk_mglev &L = m.L[m.c0 + K];
        S.g[K].nx = L.nx;
        S.g[K].ny = L.ny;
        S.g[K].hx = L.nx >> 1;
        S.g[K].nblk = (L.nx >> 1) * (L.ny >> 1);
    }
    S.bf = (double *)(x + MG_BD);
    S.part = S.bf + MG_BF;
    const int nbot = S.g[NL].nx * S.g[NL].ny;
    // level 0 of the FP32 cycle: r in, z out in FP64
    const Lev<T> G0 = lev<T>(m.L[m.c0]);
    const bool ext = sizeof(T) == 4 && m.c0 == 0;
    // The loads below are valid whatever the stop flag says, so they are
    // issued before it is read, every one before the first use: one memory
    // round trip.
    if constexpr (NL > 0) {
        blk_place(S.g[0], S.k0);
        blk_faces(G0, S.k0);
#pragma unroll
        for (int u = 0; u < 2; u++) {
            const int i = 2 * S.k0[u].I, j = 2 * S.k0[u].J;
            if (ext) {
                double a, b, c, d;
                ld2(m.r0, m.p0, i, j, a, b);
                ld2(m.r0, m.p0, i, j + 1, c, d);
                S.k0[u].fa = (T)a;
                S.k0[u].fb = (T)b;
                S.k0[u].fc = (T)c;
                S.k0[u].fd = (T)d;
            } else {
                ld2(G0.f, G0.pitch, i, j, S.k0[u].fa, S.k0[u].fb);
                ld2(G0.f, G0.pitch, i, j + 1, S.k0[u].fc, S.k0[u].fd);
            }
        }
    } else {
        for (int q = threadIdx.x; q < nbot; q += CT) {
            const int j = q / G0.nx, i = q - j * G0.nx;
            S.bf[q] = ext ? (double)(T)m.r0[(ptrdiff_t)j * m.p0 + i] : (double)ld(G0.f, G0.pitch, i, j);
        }
    }
    if constexpr (NL > 1) {
        blk_place(S.g[1], S.k1);
        blk_faces(lev<T>(m.L[m.c0 + 1]), S.k1);
    }
    if constexpr (NL > 2) {
        blk_place(S.g[2], S.k2);
        blk_faces(lev<T>(m.L[m.c0 + 2]), S.k2);
    }
    if constexpr (NL == 0) bottom_load(bottom_geo(nbot), (const T *)m.H, 0, S.h);
    if (sc->p_done) return;
    if (check && mg_stop_test(sc, w, n, tol, maxit, S.bf + (NL > 0 ? 0 : MG_BF))) return;
    if constexpr (NL > 0) blk_diag<true>(S.g[0].ny, S.k0);
    if constexpr (NL > 1) blk_diag<true>(S.g[1].ny, S.k1);
    if constexpr (NL > 2) blk_diag<true>(S.g[2].ny, S.k2);
    __syncthreads();
    cycle<0>(m, S);
    if constexpr (NL == 0) {
        for (int q = threadIdx.x; q < nbot; q += CT) {
            const int j = q / G0.nx, i = q - j * G0.nx;
            if (ext) m.z0[(ptrdiff_t)j * m.p0 + i] = (double)x[MG_BX + q];
            else G0.x[(ptrdiff_t)j * G0.pitch + i] = x[MG_BX + q];
        }
    } else {
#pragma unroll
        for (int u = 0; u < 2; u++)
            if (S.k0[u].on) {
                const int i = 2 * S.k0[u].I, j = 2 * S.k0[u].J;
                if (ext) {
                    st2(m.z0, m.p0, i, j, (double)S.k0[u].a, (double)S.k0[u].b);
                    st2(m.z0, m.p0, i, j + 1, (double)S.k0[u].c, (double)S.k0[u].d);
                } else {
                    st2(G0.x, G0.pitch, i, j, S.k0[u].a, S.k0[u].b);
                    st2(G0.x, G0.pitch, i, j + 1, S.k0[u].c, S.k0[u].d);
                }
            }
    }
}

// stop test alone, and <r, z> alone (grids small enough for one workgroup)
__global__ void __launch_bounds__(NTH) k_mg_check(pvk_scal *sc, pvk_pcg w, int n, double tol, int maxit)
{
    __shared__ double sh[NTH];
    if (sc->p_done || n == -3) return;
    mg_stop_test(sc, w, n, tol, maxit, sh);
}
__global__ void __launch_bounds__(NTH) k_mg_dot(const pvk_scal *sc, pvk_pcg w, pvk_grid g, int slot)
{
    __shared__ double sh[NTH];
    if (sc->p_done) return;
    const int P = g.P;
    double acc = 0.0;
    for (int q = threadIdx.x; q < g.NXM * g.NYM; q += NTH) {
        const int j = q / g.NXM, i = q - j * g.NXM;
        acc += AT(w.r, i, j) * AT(w.z, i, j);
    }
    block_store_partial(acc, w.rz[slot], 0, sh);
}

// ---------------------------------------------------------------------------
// CG vector kernels, one block per row
// ---------------------------------------------------------------------------
// The pressure operator is singular (constants are its null space) and the
// V-cycle, unlike the FFT solve, does not drop the mean of its input: a mean
// left in r by rounding in A d is a part of the system no iteration can
// reduce, and once ||r|| comes down to it the CG stalls.  So the residual is
// kept at zero mean: every A d is used less its mean (sum(A d) is zero in
// exact arithmetic; the partials come from the kernel that forms A d).
//
// start: r = rhs - mean (phi = 0), or with warm != 0 r = rhs - mean - (Ad - mean(Ad))
// (Ad = A phi0, phi kept); partial <r, r>
__global__ void __launch_bounds__(NTH) k_mg_start(pvk_grid g, const pvk_scal *sc, pvk_pcg w, int warm)
{
    __shared__ double sh[NTH];
    const int P = g.P, j = xcd_band(blockIdx.x, gridDim.x);
    const double ncell = (double)g.NXM * (double)g.NYM;
    const double mean = block_sum(w.mean, w.nmean, sh) / ncell;
    const double mad = (warm && w.sad) ? block_sum(w.sad, w.ndad, sh) / ncell : 0.0;
    double acc = 0.0;
    for (int i = threadIdx.x; i < g.NXM; i += NTH) {
        double r = AT(w.rhs, i, j) - mean;
        if (warm) r -= AT(w.Ad, i, j) - mad;
        else AT(w.phi, i, j) = 0.0;
        AT(w.r, i, j) = r;
        acc += r * r;
    }
    block_store_partial(acc, w.rr, j, sh);
    (void)sc;
}

// alpha = <r, z> / <d, A d>; phi += alpha d; r -= alpha (A d - mean(A d));
// partial <r, r>
__global__ void __launch_bounds__(NTH) k_mg_update(pvk_grid g, const pvk_scal *sc, pvk_pcg w, int n)
{
    __shared__ double sh[3 * NTH];
    if (sc->p_done) return;
    const int P = g.P, j = xcd_band(blockIdx.x, gridDim.x);
    double rz, dad, sad = 0.0;
    if (w.sad) block_sum3(w.rz[n & 1], w.nrz, w.dad[n & 1], w.ndad, w.sad, w.ndad, sh, rz, dad, sad);
    else block_sum2(w.rz[n & 1], w.nrz, w.dad[n & 1], w.ndad, sh, rz, dad);
    const double alpha = rz / dad;
    const double mad = sad / ((double)g.NXM * (double)g.NYM);
    const double *d = w.d[n & 1];
    double acc = 0.0;
    for (int i = threadIdx.x; i < g.NXM; i += NTH) {
        AT(w.phi, i, j) += alpha * AT(d, i, j);
        const double r = AT(w.r, i, j) - alpha * (AT(w.Ad, i, j) - mad);
        AT(w.r, i, j) = r;
        acc += r * r;
    }
    block_store_partial(acc, w.rr, j, sh);
}

// ---------------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------------
// tile shape by level width: 0 = 64 x 16, 1 = 32 x 16, 2 = 32 x 8
// (level 0: m->sh0 when it is set)
static int tile_shape(const pvk_mg *m, int l)
{
    const pvk_mglev &L = m->L[l];
    if (l == 0 && m->sh0 >= 0) return m->sh0;
    return (L.nx > 512) ? 0 : (L.nx > 256 ? 1 : 2);
}
static dim3 tile_grid(const pvk_mg *m, int l)
{
    const pvk_mglev &L = m->L[l];
    const int sh = tile_shape(m, l), tx = sh ? 32 : 64, ty = (sh == 2) ? 8 : 16;
    return dim3((L.nx + tx - 1) / tx, (L.ny + ty - 1) / ty);
}
static dim3 cell_grid(const pvk_mglev &L) { return dim3((L.nx + TXP - 1) / TXP, (L.ny + TYR - 1) / TYR); }

extern "C" int pvk_mg_nrz(const pvk_mg *m)
{
    if (m->c0 == 0) return 1;
    const dim3 gr = tile_grid(m, 0);
    return (int)(gr.x * gr.y);
}

// above 64 KiB of dynamic LDS a kernel must be allowed it (gfx950: up to 160
// KiB per workgroup); raised once per device and kernel, under a lock
static void allow_lds(const void *k, int slot)
{
    static std::mutex mu;
    static unsigned char raised[64][4];
    int dev = 0;
    (void)hipGetDevice(&dev);
    std::lock_guard<std::mutex> lk(mu);
    if (dev >= 0 && dev < 64 && !raised[dev][slot]) {
        if (hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024) == hipSuccess)
            raised[dev][slot] = 1;
        else
            (void)hipGetLastError();
    }
}

// the bottom matrix of a solve: factor, columns of G, then P G P
template <typename T> static void bottom_setup(const pvk_mg *m, hipStream_t s)
{
    const pvk_mglev &Lb = m->L[m->nlev - 1];
    const int nx = Lb.nx, nb = nx * Lb.ny;
    double *dinv = m->Lb + (size_t)PVK_MG_BOTTOM * (PVK_MG_BOTTOM_NX + 1);
    if (nx <= BK) {
        const size_t nbp = ((size_t)nb + BK - 1) / BK * BK;
        const size_t fac = sizeof(double) * ((nbp + BK + 1) * (BK + 1) + BK);
        const size_t cols = sizeof(double) * ((nbp + BK) * (BK + 2) + nbp * BYP);
        hipLaunchKernelGGL(k_mg_bottom_factor16<T>, dim3(1), dim3(BKT), fac, s, lev<T>(Lb), m->Lb, dinv);
        if (cols > 65536) allow_lds((const void *)k_mg_bottom_cols16, 2);
        hipLaunchKernelGGL(k_mg_bottom_cols16, dim3((unsigned)(nbp / BK)), dim3(BKT), cols, s, nb,
                           (const double *)m->Lb, (const double *)dinv, m->G, m->cm);
    } else {
        const size_t band = sizeof(double) * (size_t)nb * (nx + 1), budget = 160 * 1024;
        int cpb = BW;                               // columns per block: as many as LDS holds
        while (cpb > 1 && band + sizeof(double) * (size_t)nb * (cpb + 1) > budget) cpb >>= 1;
        const size_t need_cols = band + sizeof(double) * (size_t)nb * (cpb + 1);
        if (band > 65536) allow_lds((const void *)k_mg_bottom_factor<T, PVK_MG_BOTTOM_NX>, sizeof(T) == 4 ? 0 : 1);
        hipLaunchKernelGGL((k_mg_bottom_factor<T, PVK_MG_BOTTOM_NX>), dim3(1), dim3(BW), band, s, lev<T>(Lb), m->Lb,
                           dinv);
        if (need_cols > 65536) allow_lds((const void *)k_mg_bottom_cols<PVK_MG_BOTTOM_NX>, 3);
        hipLaunchKernelGGL(k_mg_bottom_cols<PVK_MG_BOTTOM_NX>, dim3((nb + cpb - 1) / cpb), dim3(BW), need_cols, s,
                           nx, nb, cpb, (const double *)m->Lb, (const double *)dinv, m->G, m->cm);
    }
    hipLaunchKernelGGL(k_mg_bottom_proj<T>, dim3(nb), dim3(NTH), 0, s, nb, (const double *)m->G,
                       (const double *)m->cm, (T *)m->H);
}

// per solve: coarse faces of every level (FP32: and the level-0 copies) and,
// when asked, the bottom inverse, from the FP64 level-0 faces bx0, by0 (pitch pf)
extern "C" void pvk_mg_setup(const pvk_mg *m, const double *bx0, const double *by0, int pf, int bottom,
                             hipStream_t s)
{
    Lev<double> F0;
    F0.nx = m->L[0].nx;
    F0.ny = m->L[0].ny;
    F0.pitch = pf;
    F0.x = F0.f = nullptr;
    F0.bx = (double *)bx0;
    F0.by = (double *)by0;
    if (m->fp32) {
        hipLaunchKernelGGL(k_mg_faces0, cell_grid(m->L[0]), dim3(NTH), 0, s, F0, lev<float>(m->L[0]));
        if (m->nlev > 1)
            hipLaunchKernelGGL((k_mg_faces<double, float>), cell_grid(m->L[1]), dim3(NTH), 0, s, F0,
                               lev<float>(m->L[1]));
        for (int l = 1; l + 1 < m->nlev; l++)
            hipLaunchKernelGGL((k_mg_faces<float, float>), cell_grid(m->L[l + 1]), dim3(NTH), 0, s,
                               lev<float>(m->L[l]), lev<float>(m->L[l + 1]));
        if (bottom) bottom_setup<float>(m, s);
    } else {
        for (int l = 0; l + 1 < m->nlev; l++)
            hipLaunchKernelGGL((k_mg_faces<double, double>), cell_grid(m->L[l + 1]), dim3(NTH), 0, s,
                               lev<double>(m->L[l]), lev<double>(m->L[l + 1]));
        if (bottom) bottom_setup<double>(m, s);
    }
}

// One V-cycle z = V(r) for CG iteration n is, in order: pvk_mg_pre for
// levels 0 .. c0-1, pvk_mg_coarse, pvk_mg_post for levels c0-1 .. 0.  The
// stop test of n runs in the kernel after the one that formed r_{n+1}
// (n = -3: none); <r, z> partials go to w->rz[(n < 0) ? 0 : (n + 1) & 1].
// With tiled levels (c0 > 0) the level-0 pre kernel of iteration n >= 0 does
// the CG step, r_n -> r_{n+1}, between w->r and w->r2 by parity; without
// them (c0 = 0) pvk_mg_update does it in place in w->r.
static int rz_slot(int n) { return (n < 0) ? 0 : ((n + 1) & 1); }
static double *r_of(const pvk_mg *m, const pvk_pcg *w, int k)     // r_k, k >= 0
{
    return (m->c0 > 0 && (k & 1)) ? w->r2 : w->r;
}
// the residual a V-cycle of iteration n reads: r_{n+1} (r_0 for n < 0)
static const double *r_in(const pvk_mg *m, const pvk_pcg *w, int n) { return r_of(m, w, n < 0 ? 0 : n + 1); }

#define MG_SHAPES(KERNEL, NU, ...)                                                                         \
    do {                                                                                                   \
        if (sh == 0) hipLaunchKernelGGL((KERNEL<NU, 0, T>), gr, dim3(NTH), 0, s, __VA_ARGS__);             \
        else if (sh == 1) hipLaunchKernelGGL((KERNEL<NU, 1, T>), gr, dim3(NTH), 0, s, __VA_ARGS__);        \
        else hipLaunchKernelGGL((KERNEL<NU, 2, T>), gr, dim3(NTH), 0, s, __VA_ARGS__);                     \
    } while (0)

template <typename T>
static void pre_t(const pvk_mg *m, int l, pvk_scal *sc, const pvk_pcg *w, int n, double tol, int maxit,
                  hipStream_t s)
{
    const dim3 gr = tile_grid(m, l);
    const Lev<T> L = lev<T>(m->L[l]), C = lev<T>(m->L[l + 1]);
    const int step = (l == 0 && n >= 0);
    const double *r0 = (l == 0) ? (step ? r_of(m, w, n) : r_in(m, w, n)) : nullptr;
    double *rnew = step ? r_of(m, w, n + 1) : nullptr;
    const int sh = tile_shape(m, l), chk = (l == 1), nc = m->L[0].nx * m->L[0].ny;
    if (m->nu == 1) MG_SHAPES(k_mg_pre, 1, L, C, r0, rnew, m->p0, sc, *w, n, tol, maxit, chk, step, nc);
    else MG_SHAPES(k_mg_pre, 2, L, C, r0, rnew, m->p0, sc, *w, n, tol, maxit, chk, step, nc);
}

template <typename T> static void post_t(const pvk_mg *m, int l, pvk_scal *sc, const pvk_pcg *w, int n, hipStream_t s)
{
    const dim3 gr = tile_grid(m, l);
    const Lev<T> L = lev<T>(m->L[l]), C = lev<T>(m->L[l + 1]);
    const double *r0 = (l == 0) ? r_in(m, w, n) : nullptr;
    double *z0 = (l == 0) ? m->z0 : nullptr;
    const pvk_scal *cs = sc;
    const int sh = tile_shape(m, l), slot = rz_slot(n), dot = (l == 0);
    if (m->nu == 1) MG_SHAPES(k_mg_post, 1, L, C, r0, z0, m->p0, cs, *w, dot, slot);
    else MG_SHAPES(k_mg_post, 2, L, C, r0, z0, m->p0, cs, *w, dot, slot);
}

extern "C" void pvk_mg_pre(const pvk_mg *m, int l, pvk_scal *sc, const pvk_pcg *w, int n, double tol, int maxit,
                           hipStream_t s)
{
    if (m->fp32) pre_t<float>(m, l, sc, w, n, tol, maxit, s);
    else pre_t<double>(m, l, sc, w, n, tol, maxit, s);
}

template <typename T>
static void coarse_t(const pvk_mg *m, pvk_scal *sc, const pvk_pcg *w, int n, double tol, int maxit, hipStream_t s)
{
    constexpr size_t need = coarse_lds_bytes<T>();
    const int chk = m->c0 <= 1 && n != -3;
#define MG_COARSE(NL) hipLaunchKernelGGL((k_mg_coarse<T, NL>), dim3(1), dim3(CT), need, s, *m, sc, *w, n, tol, maxit, chk)
    switch (m->nlev - 1 - m->c0) {
    case 0: MG_COARSE(0); break;
    case 1: MG_COARSE(1); break;
    case 2: MG_COARSE(2); break;
    default: MG_COARSE(3); break;
    }
#undef MG_COARSE
}

extern "C" void pvk_mg_coarse(const pvk_mg *m, const pvk_grid *g, pvk_scal *sc, const pvk_pcg *w, int n,
                              double tol, int maxit, hipStream_t s)
{
    if (m->fp32) coarse_t<float>(m, sc, w, n, tol, maxit, s);
    else coarse_t<double>(m, sc, w, n, tol, maxit, s);
    if (m->c0 == 0)
        hipLaunchKernelGGL(k_mg_dot, dim3(1), dim3(NTH), 0, s, (const pvk_scal *)sc, *w, *g, rz_slot(n));
}

extern "C" void pvk_mg_post(const pvk_mg *m, int l, pvk_scal *sc, const pvk_pcg *w, int n, hipStream_t s)
{
    if (m->fp32) post_t<float>(m, l, sc, w, n, s);
    else post_t<double>(m, l, sc, w, n, s);
}

// phi = src unless the solve has already stopped (a zero right-hand side:
// phi stays 0)
__global__ void __launch_bounds__(NTH) k_mg_take(pvk_grid g, const pvk_scal *sc, const double *src, double *phi)
{
    if (sc->p_done) return;
    const int P = g.P, j = blockIdx.x;
    for (int i = threadIdx.x; i < g.NXM; i += NTH) AT(phi, i, j) = AT(src, i, j);
}

extern "C" void pvk_mg_check(pvk_scal *sc, const pvk_pcg *w, int n, double tol, int maxit, hipStream_t s)
{
    hipLaunchKernelGGL(k_mg_check, dim3(1), dim3(NTH), 0, s, sc, *w, n, tol, maxit);
}

extern "C" void pvk_mg_take(const pvk_grid *g, const pvk_scal *sc, const double *src, double *phi, hipStream_t s)
{
    hipLaunchKernelGGL(k_mg_take, dim3(g->NYM), dim3(NTH), 0, s, *g, sc, src, phi);
}

extern "C" void pvk_mg_start(const pvk_grid *g, pvk_scal *sc, const pvk_pcg *w, int warm, hipStream_t s)
{
    hipLaunchKernelGGL(k_mg_start, dim3(g->NYM), dim3(NTH), 0, s, *g, (const pvk_scal *)sc, *w, warm);
}

extern "C" void pvk_mg_update(const pvk_grid *g, pvk_scal *sc, const pvk_pcg *w, int n, hipStream_t s)
{
    hipLaunchKernelGGL(k_mg_update, dim3(g->NYM), dim3(NTH), 0, s, *g, (const pvk_scal *)sc, *w, n);
}
