"""Geometric multigrid on the device against the CPU oracle: the V-cycle
z = M r bit-identical to the oracle's cycle (2D and 3D, several depths and
smoother settings, one level), CG preconditioned by it and multigrid as
the solver within 2 iterations and 1e-8 of the oracle's, and the
refusals."""
import numpy as np
import pytest

from ba_amd import hflmp, mg
from oracle import oracle as O

pytestmark = pytest.mark.gpu

SMOOTH = [dict(pre_smooth=1, post_smooth=1, coarse_sweeps=8, omega=0.8, coarse_omega=0.8),
          dict(pre_smooth=2, post_smooth=3, coarse_sweeps=1, omega=0.6, coarse_omega=1.0)]


def _oracle_kw(p):
    return dict(pre=p["pre_smooth"], post=p["post_smooth"], coarse=p["coarse_sweeps"],
                omega=p["omega"], coarse_omega=p["coarse_omega"])


def _setup(ctx, dim, n, nlevels=None, params=SMOOTH[0], seed=7):
    kap = hflmp.fe_kappa(dim, n, 1.0, seed)
    E = hflmp.fe_element(1, dim, n)
    A = hflmp.fe_system(1, dim, n, kap)
    dA = hflmp.CsrMatrix(ctx, *A)
    M = mg.build_structured(ctx, dim, n, E, kap, dA, nlevels=nlevels, **params)
    sizes = mg.level_sizes(n, nlevels)
    mats = mg.coarse_cell_mats(dim, n, E, kap, sizes)
    levels = O.mg_levels(A, [mg.restriction(dim, nc) for nc in sizes[1:]],
                         [mg.prolongation(dim, nc) for nc in sizes[1:]], mats,
                         [hflmp.fe_cell_dofs(1, dim, nc) for nc in sizes[1:]],
                         [hflmp.fe_fixed(1, dim, nc) for nc in sizes[1:]])
    return A, dA, M, levels


@pytest.mark.parametrize("p", range(len(SMOOTH)))
@pytest.mark.parametrize("case", [(2, 32, None), (3, 16, None), (3, 12, None), (3, 16, 2)])
def test_vcycle_bit_exact(ctx, case, p):
    dim, n, nl = case
    print("vcycle", case, p, flush=True)
    A, dA, M, levels = _setup(ctx, dim, n, nl, SMOOTH[p])
    try:
        N = dA.nrow
        inner = np.ones(N, bool)
        inner[hflmp.fe_fixed(1, dim, n)] = False
        r = np.random.default_rng(n).uniform(-1, 1, N) * inner
        dr, dz = ctx.upload(r), ctx.zeros(N, np.float64)
        M.apply(dr, dz)
        z = dz.download()
        assert np.array_equal(z, O.mg_cycle(levels, r, **_oracle_kw(SMOOTH[p])))
        M.apply(dr, dz)     # the level buffers keep no state between cycles
        assert np.array_equal(dz.download(), z)
        M.set_structured(0, 0)   # through the stored R and P: the same cycle
        M.apply(dr, dz)
        assert np.array_equal(dz.download(), z)
        dr.free(), dz.free()
    finally:
        M.free()
        dA.free()


def test_single_level_is_damped_jacobi(ctx):
    rp, ci, v = hflmp.fe_system(1, 2, 9)
    dA = hflmp.CsrMatrix(ctx, rp, ci, v)
    M = hflmp.Multigrid(ctx, [dA], [], [], coarse_sweeps=5, coarse_omega=0.55)
    try:
        b = hflmp.fe_rhs(1, 2, 9, 2)
        db, dz = ctx.upload(b), ctx.zeros(len(b), np.float64)
        M.apply(db, dz)
        lv = [dict(A=(rp, ci, v), invd=O.invdiag(rp, ci, v))]
        assert np.array_equal(dz.download(), O.mg_cycle(lv, b, coarse=5, coarse_omega=0.55))
        db.free(), dz.free()
    finally:
        M.free()
        dA.free()


@pytest.mark.parametrize("case", [(2, 64), (3, 16), (3, 32), (3, 64)])
def test_pcg_mg_vs_oracle(ctx, case):
    dim, n = case
    print("pcg_mg", case, flush=True)
    A, dA, M, levels = _setup(ctx, dim, n)
    try:
        b = hflmp.fe_rhs(1, dim, n, 5)
        db, dx = ctx.upload(b), ctx.zeros(len(b), np.float64)
        info = M.pcg(db, dx, rtol=1e-8)
        x = dx.download()
        xo, io = O.cg_prec(A, b, lambda r: O.mg_cycle(levels, r, **_oracle_kw(SMOOTH[0])),
                           rtol=1e-8)
        assert info["status"] == 0 and io["status"] == 0
        assert abs(info["iters"] - io["iters"]) <= 2
        assert abs(info["res_init"] - io["res_init"]) <= 1e-12 * io["res_init"]
        assert np.linalg.norm(x - xo) <= 1e-8 * np.linalg.norm(xo)
        # the true residual
        res = b - O.spmv(*A, x)
        assert np.linalg.norm(res) <= 2e-8 * np.linalg.norm(b)
        _, jac = O.cg(*A, b)
        assert info["iters"] * 3 < jac["iters"]
        db.free(), dx.free()
    finally:
        M.free()
        dA.free()


@pytest.mark.parametrize("case", [(2, 32), (3, 16)])
def test_mg_solve_vs_oracle(ctx, case):
    dim, n = case
    A, dA, M, levels = _setup(ctx, dim, n)
    try:
        b = hflmp.fe_rhs(1, dim, n, 6)
        x0 = np.random.default_rng(1).uniform(-1, 1, len(b))
        x0[hflmp.fe_fixed(1, dim, n)] = 0.0
        db, dx = ctx.upload(b), ctx.upload(x0)
        info = M.solve(db, dx, rtol=1e-9, maxit=200)
        xo, io = O.mg_solve(levels, b, x0, rtol=1e-9, maxit=200, **_oracle_kw(SMOOTH[0]))
        assert info["status"] == 0 and io["status"] == 0
        assert abs(info["iters"] - io["iters"]) <= 1
        assert info["res_init"] == io["res_init"] or \
            abs(info["res_init"] - io["res_init"]) <= 1e-12 * io["res_init"]
        assert np.linalg.norm(dx.download() - xo) <= 1e-8 * np.linalg.norm(xo)
        # maxit reached: status 1 and exactly maxit cycles
        dx2 = ctx.upload(x0)
        i2 = M.solve(db, dx2, rtol=1e-30, maxit=3)
        assert i2["status"] == 1 and i2["iters"] == 3
        db.free(), dx.free(), dx2.free()
    finally:
        M.free()
        dA.free()


def test_mg_refusals(ctx):
    rp, ci, v = hflmp.fe_system(1, 2, 8)
    dA = hflmp.CsrMatrix(ctx, rp, ci, v)
    rr, rc, rv = mg.restriction(2, 4)
    pr, pc, pv = mg.prolongation(2, 4)
    R = hflmp.CsrMatrix(ctx, rr, rc, rv, ncol=81)
    P = hflmp.CsrMatrix(ctx, pr, pc, pv, ncol=25)
    Ac = hflmp.CsrMatrix(ctx, *hflmp.fe_system(1, 2, 4))
    try:
        for kw in (dict(pre_smooth=0), dict(post_smooth=-1), dict(coarse_sweeps=0),
                   dict(omega=0.0), dict(coarse_omega=-1.0)):
            with pytest.raises(hflmp.HflmpError) as e:
                hflmp.Multigrid(ctx, [dA, Ac], [R], [P], **kw)
            assert e.value.code == hflmp.EINVAL
        with pytest.raises(hflmp.HflmpError):      # R and P swapped
            hflmp.Multigrid(ctx, [dA, Ac], [P], [R])
        with pytest.raises(hflmp.HflmpError):      # coarse operator of the wrong size
            hflmp.Multigrid(ctx, [dA, dA], [R], [P])
        M = hflmp.Multigrid(ctx, [dA, Ac], [R], [P])
        try:
            for dim, nc in ((3, 8), (2, 6), (2, 3), (4, 8)):   # not this hierarchy
                with pytest.raises(hflmp.HflmpError):
                    M.set_structured(dim, nc)
            M.set_structured(2, 8)
            r = ctx.zeros(dA.nrow, np.float64)
            with pytest.raises(hflmp.HflmpError):  # z aliasing r
                M.apply(r, r)
            small = ctx.empty(16, np.uint8)
            with pytest.raises(hflmp.HflmpError):
                M.pcg(r, ctx.zeros(dA.nrow, np.float64), work=small)
            small.free(), r.free()
        finally:
            M.free()
        # the context stays usable
        z = ctx.zeros(4, np.float64)
        assert np.array_equal(z.download(), np.zeros(4))
        z.free()
    finally:
        for m in (dA, R, P, Ac):
            m.free()


def _setup_mf(ctx, dim, n, params=SMOOTH[0], seed=7):
    kap = hflmp.fe_kappa(dim, n, 1.0, seed)
    E = hflmp.fe_element(1, dim, n)
    fixed = hflmp.fe_fixed(1, dim, n)
    S = hflmp.StencilOperator(ctx, 1, dim, [n] * dim, E, kap, fixed)
    M = mg.build_structured(ctx, dim, n, E, kap, None, stencil=S, **params)
    A = hflmp.fe_system(1, dim, n, kap)
    sizes = mg.level_sizes(n)
    mats = mg.coarse_cell_mats(dim, n, E, kap, sizes)
    levels = O.mg_levels(A, [mg.restriction(dim, nc) for nc in sizes[1:]],
                         [mg.prolongation(dim, nc) for nc in sizes[1:]], mats,
                         [hflmp.fe_cell_dofs(1, dim, nc) for nc in sizes[1:]],
                         [hflmp.fe_fixed(1, dim, nc) for nc in sizes[1:]])
    del levels[0]["A"]
    levels[0]["S"] = (1, dim, [n] * dim, E, kap, fixed)
    return S, M, levels


@pytest.mark.parametrize("p", range(len(SMOOTH)))
@pytest.mark.parametrize("case", [(2, 32), (3, 16), (3, 12)])
def test_vcycle_matrix_free_bit_exact(ctx, case, p):
    dim, n = case
    print("vcycle_mf", case, p, flush=True)
    S, M, levels = _setup_mf(ctx, dim, n, SMOOTH[p])
    try:
        inner = np.ones(S.nrow, bool)
        inner[hflmp.fe_fixed(1, dim, n)] = False
        r = np.random.default_rng(n + 1).uniform(-1, 1, S.nrow) * inner
        dr, dz = ctx.upload(r), ctx.zeros(S.nrow, np.float64)
        M.apply(dr, dz)
        assert np.array_equal(dz.download(), O.mg_cycle(levels, r, **_oracle_kw(SMOOTH[p])))
        dr.free(), dz.free()
    finally:
        M.free()
        S.free()


@pytest.mark.parametrize("case", [(2, 64), (3, 32)])
def test_pcg_mg_matrix_free_vs_oracle(ctx, case):
    dim, n = case
    print("pcg_mg_mf", case, flush=True)
    S, M, levels = _setup_mf(ctx, dim, n)
    try:
        b = hflmp.fe_rhs(1, dim, n, 5)
        db, dx = ctx.upload(b), ctx.zeros(len(b), np.float64)
        info = M.pcg(db, dx, rtol=1e-8)
        x = dx.download()
        op = lambda v: O.stencil_vmadd(*levels[0]["S"], v)
        xo, io = O.cg_prec(op, b, lambda r: O.mg_cycle(levels, r, **_oracle_kw(SMOOTH[0])),
                           rtol=1e-8)
        assert info["status"] == 0 and io["status"] == 0
        assert abs(info["iters"] - io["iters"]) <= 2
        assert np.linalg.norm(x - xo) <= 1e-8 * np.linalg.norm(xo)
        assert np.linalg.norm(b - op(x)) <= 2e-8 * np.linalg.norm(b)
        # multigrid as the solver through the same hierarchy
        dx2 = ctx.zeros(len(b), np.float64)
        i2 = M.solve(db, dx2, rtol=1e-8, maxit=200)
        x2, o2 = O.mg_solve(levels, b, rtol=1e-8, maxit=200, **_oracle_kw(SMOOTH[0]))
        assert i2["status"] == 0 and abs(i2["iters"] - o2["iters"]) <= 1
        assert np.linalg.norm(dx2.download() - x2) <= 1e-8 * np.linalg.norm(x2)
        db.free(), dx.free(), dx2.free()
    finally:
        M.free()
        S.free()


def test_mg_matrix_free_refusals(ctx):
    n = 8
    kap = hflmp.fe_kappa(2, n, 1.0, 3)
    E = hflmp.fe_element(1, 2, n)
    fixed = hflmp.fe_fixed(1, 2, n)
    S32 = hflmp.StencilOperator(ctx, 1, 2, [n, n], E, kap, fixed, dtype=np.float32)
    S = hflmp.StencilOperator(ctx, 1, 2, [n, n + 2], E, np.ones(n * (n + 2)),
                              hflmp.fe_fixed(1, 2, n)[:4])
    try:
        with pytest.raises(hflmp.HflmpError) as e:     # FP32 operator
            mg.build_structured(ctx, 2, n, E, kap, None, stencil=S32)
        assert e.value.code == hflmp.EINVAL
        with pytest.raises(hflmp.HflmpError):          # node count differs from P's rows
            mg.build_structured(ctx, 2, n, E, kap, None, stencil=S)
    finally:
        S32.free()
        S.free()


@pytest.mark.parametrize("case", [(2, 32), (3, 16)])
def test_vcycle_dense_coarse_bit_exact(ctx, case):
    dim, n = case
    print("vcycle_dense", case, flush=True)
    A, dA, M, levels = _setup(ctx, dim, n, nlevels=3)
    try:
        Ac = levels[-1]["A"]
        Nc = len(Ac[0]) - 1
        import scipy.sparse as sp
        Cinv = np.linalg.inv(sp.csr_matrix((Ac[2], Ac[1], Ac[0]), shape=(Nc, Nc)).toarray())
        M.set_coarse_inverse(Cinv)
        inner = np.ones(dA.nrow, bool)
        inner[hflmp.fe_fixed(1, dim, n)] = False
        r = np.random.default_rng(2).uniform(-1, 1, dA.nrow) * inner
        dr, dz = ctx.upload(r), ctx.zeros(dA.nrow, np.float64)
        M.apply(dr, dz)
        lv = [dict(L) for L in levels]
        lv[-1]["Cinv"] = Cinv
        assert np.array_equal(dz.download(), O.mg_cycle(lv, r, **_oracle_kw(SMOOTH[0])))
        # back to the sweeps
        M.set_coarse_inverse(None)
        M.apply(dr, dz)
        assert np.array_equal(dz.download(), O.mg_cycle(levels, r, **_oracle_kw(SMOOTH[0])))
        # CG with it, built by the hierarchy builder
        b = hflmp.fe_rhs(1, dim, n, 5)
        kap = hflmp.fe_kappa(dim, n, 1.0, 7)
        M2 = mg.build_structured(ctx, dim, n, hflmp.fe_element(1, dim, n), kap, dA, nlevels=3,
                                 coarse="dense", **SMOOTH[0])
        try:
            db, dx = ctx.upload(b), ctx.zeros(len(b), np.float64)
            info = M2.pcg(db, dx, rtol=1e-8)
            xo, io = O.cg_prec(A, b, lambda v: O.mg_cycle(lv, v, **_oracle_kw(SMOOTH[0])),
                               rtol=1e-8)
            assert info["status"] == 0 and abs(info["iters"] - io["iters"]) <= 2
            assert np.linalg.norm(dx.download() - xo) <= 1e-8 * np.linalg.norm(xo)
            db.free(), dx.free()
        finally:
            M2.free()
        dr.free(), dz.free()
    finally:
        M.free()
        dA.free()


def test_dense_coarse_refusal(ctx):
    rp, ci, v = hflmp.fe_system(1, 3, 16)
    dA = hflmp.CsrMatrix(ctx, rp, ci, v)
    M = hflmp.Multigrid(ctx, [dA], [], [])
    try:
        with pytest.raises(hflmp.HflmpError) as e:   # 4913 rows > 4096
            M.set_coarse_inverse(np.eye(dA.nrow))
        assert e.value.code == hflmp.EINVAL
    finally:
        M.free()
        dA.free()


def test_single_level_jacobi_solver(ctx):
    """One level, k sweeps per residual check: the synchronous form of the
    reference's AsynchronousIterationGPU (damped, n_inner = k) on one GPU."""
    rp, ci, v = hflmp.fe_system(1, 2, 24, hflmp.fe_kappa(2, 24, 0.5, 3))
    dA = hflmp.CsrMatrix(ctx, rp, ci, v)
    M = hflmp.Multigrid(ctx, [dA], [], [], coarse_sweeps=5, coarse_omega=0.7)
    try:
        b = hflmp.fe_rhs(1, 2, 24, 8)
        db, dx = ctx.upload(b), ctx.zeros(len(b), np.float64)
        info = M.solve(db, dx, rtol=1e-6, maxit=5000)
        lv = [dict(A=(rp, ci, v), invd=O.invdiag(rp, ci, v))]
        xo, io = O.mg_solve(lv, b, rtol=1e-6, maxit=5000, coarse=5, coarse_omega=0.7)
        assert info["status"] == 0 and io["status"] == 0
        assert abs(info["iters"] - io["iters"]) <= 1
        assert np.linalg.norm(dx.download() - xo) <= 1e-8 * np.linalg.norm(xo)
        db.free(), dx.free()
    finally:
        M.free()
        dA.free()


@pytest.mark.parametrize("coarse", ["sweeps", "dense"])
@pytest.mark.parametrize("mf", [False, True])
@pytest.mark.parametrize("case", [(2, 16, None, 1, 1), (2, 64, None, 2, 1), (3, 16, 2, 1, 2),
                                  (3, 32, None, 1, 1), (3, 8, 1, 2, 1), (2, 32, 3, 3, 3)])
def test_pcg_first_step_and_dot_in_the_cycle(ctx, case, mf, coarse):
    """CG's update leaves the cycle's first step, the restriction the coarse
    level's, and the last sweep r.z: every combination of smoothing steps,
    depth, finest level and coarse solve against CG with the cycle applied
    on its own."""
    dim, n, nl, pre, post = case
    if coarse == "dense" and nl == 1:
        pytest.skip("a dense coarse solve needs two levels")
    kap = hflmp.fe_kappa(dim, n, 1.0, 9)
    E = hflmp.fe_element(1, dim, n)
    A = hflmp.fe_system(1, dim, n, kap)
    dA = hflmp.CsrMatrix(ctx, *A)
    S = hflmp.StencilOperator(ctx, 1, dim, [n] * dim, E, kap, hflmp.fe_fixed(1, dim, n)) if mf \
        else None
    M = mg.build_structured(ctx, dim, n, E, kap, None if mf else dA, nlevels=nl, stencil=S,
                            coarse=coarse, pre_smooth=pre, post_smooth=post, omega=0.7,
                            coarse_sweeps=6)
    try:
        b = hflmp.fe_rhs(1, dim, n, 5)
        db, dx = ctx.upload(b), ctx.zeros(len(b), np.float64)
        dr, dz = ctx.zeros(len(b), np.float64), ctx.zeros(len(b), np.float64)
        info = M.pcg(db, dx, rtol=1e-8, maxit=300)
        x = dx.download()

        def prec(r):
            dr.copy_from_host(r)
            M.apply(dr, dz)
            return dz.download()

        xo, io = O.cg_prec(A, b, prec, rtol=1e-8, maxit=300)
        assert info["status"] == io["status"]
        assert abs(info["iters"] - io["iters"]) <= 1
        if pre == post and info["status"] == 0:
            assert np.linalg.norm(b - O.spmv(*A, x)) <= 2e-8 * np.linalg.norm(b)
        # the same iterates to rounding while CG is well behaved
        if info["iters"] == io["iters"] and info["status"] == 0:
            assert np.linalg.norm(x - xo) <= 1e-8 * np.linalg.norm(xo)
        for a in (db, dx, dr, dz):
            a.free()
    finally:
        M.free()
        if S is not None:
            S.free()
        dA.free()
