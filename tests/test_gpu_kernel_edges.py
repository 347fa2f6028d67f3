"""Kernels at the sizes where their shape can go wrong: the edges of what a
block or thread owns, remainders, and the smallest and largest of a range.
Each against the restatement the repository has for it."""
import ctypes as C

import numpy as np
import pytest

import cnn_ref
import mg_ref
import oracle_lib
import pvof
from helpers import regions, relerr

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def lib(gpu):
    return pvof.load_lib()


def params(nx, ny, **kw):
    base = dict(NXM=nx, NYM=ny, xmax=1.0, ymax=ny / nx, Re=100.0, We=200.0, rho1=1.0, rho2=1e-3, mu1=1.0, mu2=1e-2,
                Cn=2.0 / nx, Pe_CH=nx / 2.0, cfl=0.2, default_dt=1e-4, max_dt=1e-3, ch_tol=1e-12, CG_ETOL=1e-9,
                pressure_solver=pvof.PV_PSOLVE_MG_PCG, p_rel_tol=1e-10, p_max_iter=3000)
    base.update(kw)
    return pvof.default_params(**base)


def canonical(p, a):
    """Cell array [ny][nx] -> canonical layout, x-ghosts periodic, y-ghosts copied."""
    return np.pad(np.pad(a, ((3, 4), (0, 0)), mode="edge"), ((0, 0), (3, 4)), mode="wrap")


# in-workgroup levels: none but the bottom (16 x 16, 8 x 12); one with an odd
# bottom (18 x 26 -> 9 x 13); two, blocks not filling the threads (44 x 36);
# the most blocks (64 x 64) and rows that are no power of two (60 x 68); a
# bottom 64 wide (128 x 32 -> 64 x 16 -> 32 x 8); three smoothing levels
# down to rows of two (512 x 8 -> ... -> 64 x 1); a tiled level above them
# with an odd number of coarse columns (88 x 56 -> 44 x 28 -> 22 x 14 -> 11 x 7)
@pytest.mark.parametrize("nx,ny", [(16, 16), (8, 12), (18, 26), (44, 36), (64, 64), (60, 68), (128, 32), (512, 8),
                                   (88, 56)])
@pytest.mark.parametrize("nu,w", [(2, 0), (1, 1), (2, 3)])
@pytest.mark.parametrize("fp32", [0, 1])
def test_in_workgroup_levels(lib, nx, ny, nu, w, fp32):
    p = params(nx, ny)
    s = pvof.Solver(p, lib)
    s.check(lib.pv_set_mg_sweeps(s.h, nu))
    s.check(lib.pv_set_mg_precision(s.h, fp32))
    s.check(lib.pv_set_mg_cycle(s.h, w))
    rho = mg_ref.bubbles(nx, ny, seed=nx + ny, nb=6)
    f = np.random.default_rng(nx * ny).standard_normal((ny, nx))
    f -= f.mean()
    s.set("RHO", canonical(p, rho))
    s.set("P_RES", canonical(p, f))
    s.call("mg_vcycle_apply")
    z = s.get("SCRATCH0")[regions(p)["cell"]]
    bx, by = mg_ref.faces(rho, float(nx * nx), float(nx * nx))
    lv, G = mg_ref.build(bx, by)
    sizes = mg_ref.level_sizes(nx, ny)
    c0 = next(i for i, sz in enumerate(sizes) if sz[0] * sz[1] <= mg_ref.LDS_CELLS)
    zr = mg_ref.vcycle(lv, G, f, nu, wl=tuple(range(c0, min(c0 + w, len(lv) - 1))))
    assert relerr(z, zr) < (1e-5 if fp32 else 1e-11)


# the grid is the bottom itself: full 16 x 16, rows no multiple of 16 (odd
# widths, 255 and 247 of 256 cells), the fewest cells and columns, and two
# wider than 16 (the other factorisation); a second density on the same handle
@pytest.mark.parametrize("nx,ny", [(16, 16), (15, 17), (13, 19), (9, 28), (8, 8), (10, 25), (17, 15), (32, 8)])
@pytest.mark.parametrize("fp32", [0, 1])
def test_bottom_inverse(lib, nx, ny, fp32):
    p = params(nx, ny)
    s = pvof.Solver(p, lib)
    s.check(lib.pv_set_mg_precision(s.h, fp32))
    for seed in (1, 2):
        rho = mg_ref.bubbles(nx, ny, seed=seed, nb=4)
        f = np.random.default_rng(seed).standard_normal((ny, nx))
        f -= f.mean()
        s.set("RHO", canonical(p, rho))
        s.set("P_RES", canonical(p, f))
        s.call("mg_vcycle_apply")
        z = s.get("SCRATCH0")[regions(p)["cell"]]
        lv, G = mg_ref.build(*mg_ref.faces(rho, float(nx * nx), float(nx * nx)))
        assert len(lv) == 1
        assert relerr(z, mg_ref.vcycle(lv, G, f, 2)) < (1e-5 if fp32 else 1e-11)


# one row of a buffer's worth left over, exactly one buffer (2048-value rows,
# 128 of them), one row more, and many buffers
@pytest.mark.parametrize("nx,ny", [(8, 8), (1000, 300), (2041, 121), (2041, 122), (3001, 700)])
def test_field_transfers(lib, nx, ny):
    """Fields set and read back through the staged transfers, ghosts
    included, bit for bit; two sets in a row do not overtake each other, and
    a missing array is an error."""
    p = params(nx, ny, pressure_solver=pvof.PV_PSOLVE_JACOBI_PCG)
    s = pvof.Solver(p, lib)
    rng = np.random.default_rng(nx + ny)
    a, b = rng.standard_normal(s.shape), rng.standard_normal(s.shape)
    for _ in range(2):
        s.set("U", a)
        s.set("V", b)
        assert np.array_equal(s.get("U"), a) and np.array_equal(s.get("V"), b)
        a, b = b, a
    null = C.POINTER(C.c_double)()
    assert lib.pv_get_field(s.h, pvof.F["U"], null) != 0 and lib.pv_set_field(s.h, pvof.F["U"], null) != 0


# rows of one thread (16), of three (48: threads left over in a wavefront), of
# a whole wavefront (1024) and of blocks of 128 and 256 threads (2048; 3072
# and 4096), with rows left over in the last block, and column counts of one
# segment, a short last segment and several wavefronts of segments
@pytest.mark.parametrize("nx,ny", [(16, 130), (48, 43), (1024, 9), (1152, 21), (2048, 13), (3072, 10), (4096, 17),
                                   (64, 1031)])
def test_fft_rows_and_columns(lib, nx, ny):
    p = pvof.default_params(NXM=nx, NYM=ny, ymax=ny / nx)
    o, s = oracle_lib.Oracle(p), pvof.Solver(p, lib)
    R = regions(p)["cell"]
    rhs = np.zeros(o.shape)
    rhs[R] = np.random.default_rng(nx + ny).standard_normal((ny, nx))
    rhs[R] -= rhs[R].mean()
    for x in (o, s):
        x.set("SCRATCH0", rhs)
        x.call("Pressure_solve_fft", pvof.F["SCRATCH0"], pvof.F["SCRATCH1"])
    got, ref = s.get("SCRATCH1")[R], o.get("SCRATCH1")[R]
    assert np.isfinite(got).all()
    assert relerr(got, ref) < 1e-10


# rows of 2^a 3^b whose passes differ: one, two, three and four radix-3 passes, the
# power-of-two part ending with radix 8 alone (48, 144, 432, 1296), 4 (192, 576) or 2
# (96, 288, 864), and with a second radix-8 pass before them (3072, 768)
@pytest.mark.parametrize("nx", [48, 144, 432, 1296, 192, 576, 96, 288, 864, 768, 3072])
def test_fft_mixed_radix_rows(lib, nx):
    test_fft_rows_and_columns(lib, nx, 24)


# columns: less than a chunk of 256, one short of one, exactly one, one over,
# two and a remainder; rows: every remainder of the bands of 1, 2 and 4 rows
# of u (NYM rows) and v (NYM - 1)
@pytest.mark.parametrize("nx,ny", [(16, 8), (96, 11), (255, 9), (256, 8), (257, 13), (520, 10)])
@pytest.mark.parametrize("rows", [1, 2, 4])
@pytest.mark.parametrize("form", ["fp64", "mixed", "mixed_pc"])
def test_momentum_cg(lib, nx, ny, rows, form):
    """Five iterations from a random start over random densities and
    viscosities: x against the oracle's, and in FP64, where the path is the
    same to rounding, r and A d.  The polynomial preconditioner takes another
    path, so it is solved out on both sides and the velocity compared.  The diagonal dominates (dt / dx^2 below 1), so
    rounding is not amplified: FP64 order of sums 1e-11, FP32 operator 1e-5."""
    pc = form == "mixed_pc"
    kw = dict(CG_ETOL=1e-11, CG_MAXIT=200) if pc else dict(CG_ETOL=1e-30, CG_MAXIT=5)
    p = params(nx, ny, pressure_solver=pvof.PV_PSOLVE_JACOBI_PCG, **kw)
    pm = params(nx, ny, pressure_solver=pvof.PV_PSOLVE_JACOBI_PCG,
                precision=pvof.PV_PREC_FP64 if form == "fp64" else pvof.PV_PREC_MIXED, **kw)
    o, s = oracle_lib.Oracle(p), pvof.Solver(pm, lib)
    rng = np.random.default_rng(nx * ny + rows)
    fields = dict(RHO=canonical(p, rng.uniform(0.5, 1.0, (ny, nx))), MU=canonical(p, rng.uniform(0.1, 1.0, (ny, nx))))
    for f in ("U", "V", "U_RHS", "V_RHS"):
        fields[f] = rng.standard_normal(o.shape) * (1e4 if "RHS" in f else 1.0)
    for x in (o, s):
        for f, a in fields.items():
            x.set(f, a)
        x.call("set_time_state", 0.0, 2e-4, 2e-4, 2)
    s.check(lib.pv_set_momentum_rows(s.h, rows))
    if pc:
        s.check(lib.pv_set_momentum_preconditioner(s.h, 1))
        s.check(lib.pv_set_momentum_cg_steps(s.h, 1))
        o.call("set_momentum_cg_steps", 1)
    R = regions(p)
    tol = 1e-11 if form == "fp64" else 1e-5
    for c in ("u", "v"):
        n, it = o.call("Velocity_solve_cg", ord(c)), C.c_int()
        s.call("Velocity_solve_cg", ord(c), C.byref(it))
        names = [c.upper()]
        if not pc:
            assert n == it.value == 5
        if form == "fp64":
            names += [c.upper() + q for q in ("_R", "_AD")]
        for f in names:
            assert np.isfinite(s.get(f)).all()
            assert relerr(s.get(f)[R[c]], o.get(f)[R[c]]) < tol, (f, relerr(s.get(f)[R[c]], o.get(f)[R[c]]))


# two rows a band chunk by chunk: four chunks short of full, full, one column
# over (the form that holds eight), eight full, one over (row by row); bands of
# one row left over in u or v
@pytest.mark.parametrize("nx,ny", [(1023, 9), (1024, 8), (1025, 9), (2048, 8), (2049, 9)])
def test_momentum_preconditioner_chunks(lib, nx, ny):
    test_momentum_cg(lib, nx, ny, 2, "mixed_pc")


# tiled levels: narrower than a tile, the halo going round more than once
# (16 x 1024), tiles of 32 x 8 with a part left over (200 x 56), of 32 x 16 with
# one in both directions (400 x 40), and of 64 x 16 down to 32 x 16 (1056 x 64:
# 1056, 528 and 264 wide)
@pytest.mark.parametrize("nx,ny", [(16, 1024), (200, 56), (400, 40), (1056, 64)])
@pytest.mark.parametrize("nu", [1, 2])
@pytest.mark.parametrize("fp32", [0, 1])
def test_tiled_levels(lib, nx, ny, nu, fp32):
    """The V-cycle against the restatement, and a solve (whose level-0 kernel
    makes the CG step) against the system it solves, with the tolerances the
    other sizes have."""
    p = params(nx, ny)
    s = pvof.Solver(p, lib)
    s.check(lib.pv_set_mg_sweeps(s.h, nu))
    s.check(lib.pv_set_mg_precision(s.h, fp32))
    rho = mg_ref.bubbles(nx, ny, seed=nx + ny, nb=6)
    f = np.random.default_rng(nx * ny).standard_normal((ny, nx))
    f -= f.mean()
    s.set("RHO", canonical(p, rho))
    s.set("P_RES", canonical(p, f))
    s.call("mg_vcycle_apply")
    R = regions(p)["cell"]
    z = s.get("SCRATCH0")[R]
    bx, by = mg_ref.faces(rho, float(nx * nx), float(nx * nx))
    lv, G = mg_ref.build(bx, by)
    assert relerr(z, mg_ref.vcycle(lv, G, f, nu)) < (1e-5 if fp32 else 1e-11)
    s.set("P_RHS", canonical(p, f))
    it = C.c_int()
    s.call("Pressure_solve_cg", C.byref(it))
    phi = s.get("PHI")[R]
    assert 0 < it.value < p.p_max_iter
    assert np.linalg.norm(mg_ref.apply_a(bx, by, phi) - f) <= 1.05e-10 * np.linalg.norm(f)


# rows of less than a block (48), exactly one thread a column (256), a chunk of
# 1024 columns and a part (1152) and two chunks (2048)
@pytest.mark.parametrize("nx,ny", [(48, 43), (256, 9), (1152, 21), (2048, 13)])
def test_pressure_apply_rows(lib, nx, ny):
    """A d of the FFT-PCG's last iteration (the first, the third: the second
    direction buffer in between) against the operator on that d.  Both sides
    round four products and their sum: at most eight ulp of |A| |d| a cell."""
    R = regions(params(nx, ny))["cell"]
    rho = mg_ref.bubbles(nx, ny, seed=nx, nb=6)
    bx, by = mg_ref.faces(rho, float(nx * nx), float(nx * nx))
    f = np.random.default_rng(ny).standard_normal((ny, nx))
    f -= f.mean()
    for its in (1, 3):
        p = params(nx, ny, pressure_solver=pvof.PV_PSOLVE_FFT_PCG, p_max_iter=its, p_rel_tol=1e-14)
        s = pvof.Solver(p, lib)
        s.set("RHO", canonical(p, rho))
        s.set("P_RHS", canonical(p, f))
        it = C.c_int()
        s.call("Pressure_solve_cg", C.byref(it))
        assert it.value == its
        d, ad = s.get("P_D")[R], s.get("P_AD")[R]
        assert np.abs(d).max() > 0
        big = 4 * max(bx.max(), by.max()) * np.abs(d).max()
        assert np.abs(ad - mg_ref.apply_a(bx, by, d)).max() <= 8 * np.finfo(float).eps * big
        s.close()


# the Cahn-Hilliard tiles (64 x 16 and 128 x 8): a level narrower than the halo
# goes round several times (8 x 8), one tile with a part empty (48 x 17), a tile
# and one column or row (129 x 9, 65 x 33), several with remainders (200 x 35)
@pytest.mark.parametrize("nx,ny", [(8, 8), (48, 17), (129, 9), (65, 33), (200, 35)])
@pytest.mark.parametrize("stage", [0, 1])
def test_cahn_hilliard_tiles(lib, nx, ny, stage):
    """One implicit Cahn-Hilliard step against the oracle's: the explicit
    right-hand side, the CG's start and its operator.  Both solve to 1e-13 of
    the right-hand side and the system's condition number is below 10."""
    p = params(nx, ny, pressure_solver=pvof.PV_PSOLVE_JACOBI_PCG, ch_tol=1e-13)
    o, s = oracle_lib.Oracle(p), pvof.Solver(p, lib)
    F = pvof.ic(lib, "bubbles", p, seed=nx + ny, nmin=2, nmax=4, rmin=0.05, rmax=0.2, gas_inside=1)
    rng = np.random.default_rng(nx * ny)
    old, u, v = (canonical(p, rng.standard_normal((ny, nx))) for _ in range(3))
    for x in (o, s):
        x.init_from_F(F)
        x.set("U", u)
        x.set("V", v)
        x.set("CH_RHS_N", old)
        x.call("set_time_state", 0.1, 1e-4, 1e-4, stage)
        x.call("VOF_DIFFUSE_step")
    R = regions(p)["cell"]
    assert relerr(s.get("CH_RHS_N")[R], o.get("CH_RHS_N")[R]) < 1e-12
    assert relerr(s.get("C_L")[R], o.get("C_L")[R]) < 1e-11
    assert abs(o.stats()["n_ch"][stage] - s.stats()["n_ch"][stage]) <= 1


# one workgroup's worth of ghosts a field and several, with parts left over
@pytest.mark.parametrize("nx,ny", [(8, 8), (33, 9), (300, 11), (16, 600)])
def test_fused_boundary_fill(lib, nx, ny):
    """After a substep the ghosts of u, v and p are what the fills of the
    single fields leave, which the other tests hold against the oracle."""
    p = params(nx, ny, pressure_solver=pvof.PV_PSOLVE_JACOBI_PCG, P_CG_ETOL=1e-8, P_CG_MAXIT=4000)
    s = pvof.Solver(p, lib)
    s.init_from_F(pvof.ic(lib, "bubbles", p, seed=3, nmin=2, nmax=3, rmin=0.02, rmax=0.04, gas_inside=1))
    s.call("Temporal_int_all_the_equations")
    got = {f: s.get(f).copy() for f in ("U", "V", "P")}
    assert all(np.abs(a).max() > 0 for a in got.values())
    for f in ("U", "V"):
        s.call("Velocity_update_boundaries", pvof.F[f], pvof.PV_VEL_TYPE_NORMAL)
    s.call("Pressure_apply_BCs", pvof.F["P"])
    for f, a in got.items():
        assert np.array_equal(s.get(f), a), f


# one tile, a row of tiles
@pytest.mark.parametrize("shape", [(1, 16, 16), (3, 16, 48)])
@pytest.mark.parametrize("px", [0, 1])
def test_network_gradient_small(lib, shape, px):
    """The smallest batches: the loss is a mean, so four copies of a batch have
    its gradient, summed over other workgroups (a power of two, so the BF16
    gradients scale without rounding); FP32 sums, 1e-5."""
    net = pvof.Network(pvof.Solver(pvof.config1_params(NXM=32, NYM=64), lib), seed=7)
    net.set_params(cnn_ref.init_params(5).astype(np.float32))
    rng = np.random.default_rng(sum(shape) + px)
    x, tgt = rng.standard_normal(shape + (3,)).astype(np.float32), rng.standard_normal(shape).astype(np.float32)
    one, four = (net.eval(np.concatenate([x] * k), np.concatenate([tgt] * k), px=px, border=3, want_grad=True)[2].astype(np.float64)
                 for k in (1, 4))
    for a, b in [(0, 896)] + [(896 + k * 9248, 896 + (k + 1) * 9248) for k in range(4)] + [(37888, 38177)]:
        assert 0 < np.linalg.norm(one[a:b] - four[a:b]) + np.linalg.norm(one[a:b])
        assert np.linalg.norm(one[a:b] - four[a:b]) < 1e-5 * np.linalg.norm(one[a:b]), a


def test_network_gradient_many_tiles(lib):
    """More tiles than rows of partials (1030 of 1024): workgroups with two
    tiles.  The loss is a mean, so the gradient of the batch is the mean of
    its halves' gradients; FP32 sums of 264000 pixels, 1e-5."""
    net = pvof.Network(pvof.Solver(pvof.config1_params(NXM=32, NYM=64), lib), seed=7)
    net.set_params(cnn_ref.init_params(6).astype(np.float32))
    rng = np.random.default_rng(9)
    x, tgt = rng.standard_normal((1030, 16, 16, 3)).astype(np.float32), rng.standard_normal((1030, 16, 16)).astype(np.float32)
    g = [net.eval(x[s], tgt[s], px=0, border=3, want_grad=True)[2].astype(np.float64)
         for s in (slice(None), slice(0, 515), slice(515, None))]
    assert np.linalg.norm(g[0] - 0.5 * (g[1] + g[2])) < 1e-5 * np.linalg.norm(g[0])
