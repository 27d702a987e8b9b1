"""Jacobi-CG of systems of a few thousand rows, whose iterations run in one
workgroup: the same x, bit for bit, the same iteration count and status as
the three-launch iteration (the solve server's solo lane runs it whatever
the size), at the edges of its slices, units and element sets and on both
sides of its limits."""
import numpy as np
import pytest

from ba_amd import hflmp
from oracle import oracle as O

pytestmark = pytest.mark.gpu
MB = 1 << 20


def banded(n, seed, far=17, wide=False):
    """A symmetric, weakly dominant system: couplings to i +- 1, i +- 2, i +-
    far (and, `wide`, to a row far away), a third of them left out."""
    rng = np.random.default_rng(seed)
    rows = [{} for _ in range(n)]
    for d in (1, 2, far) + ((n - 1 - far,) if wide else ()):
        for i in range(max(0, n - d)):
            if rng.random() < 0.67:
                w = -rng.uniform(0.1, 1.0)
                rows[i][i + d] = w
                rows[i + d][i] = w
    for i in range(n):
        rows[i][i] = sum(-w for w in rows[i].values()) + rng.uniform(0.01, 0.1)
    rp = np.concatenate([[0], np.cumsum([len(q) for q in rows])]).astype(np.int32)
    ci = np.concatenate([np.array(sorted(q), np.int32) for q in rows])
    v = np.concatenate([[q[c] for c in sorted(q)] for q in rows])
    return rp, ci, v, rng.uniform(-1, 1, n)


def single(ctx, rp, ci, v, b, flags=hflmp.SELL_COL16, rtol=1e-8, maxit=100000):
    A = hflmp.CsrMatrix(ctx, rp, ci, v)
    S = hflmp.SellMatrix(ctx, A, flags)
    invd = hflmp.invdiag(ctx, A)
    db, dx = ctx.upload(b), ctx.zeros(A.nrow, v.dtype)
    try:
        info = hflmp.pcg_jacobi_sell(ctx, S, invd, db, dx, rtol=rtol, maxit=maxit, dtol=1e300)
        return dx.download(), info
    finally:
        for a in (db, dx, invd, S, A):
            a.free()


def three_launch(ctx, rp, ci, v, b, rtol=1e-8, maxit=100000):
    sv = hflmp.Server(ctx, 256 * MB, max_active=1, chunk_iters=16, solo_min_nnz=1)
    try:
        t = sv.submit(rp, ci, v, b, rtol=rtol, maxit=maxit, precision=64)
        while sv.poll(t)["state"] != 2:
            sv.step()
        x, info = sv.take(t)
        assert sv.stats()["solo_runs"] > 0
        return x, info
    finally:
        sv.close()


@pytest.mark.parametrize("n", [20, 63, 64, 65, 255, 257, 1023, 1024, 1025, 2049, 3073, 4095, 4096,
                               4097, 6145, 8191, 8192, 8193])
def test_equals_three_launch_form(ctx, n):
    rp, ci, v, b = banded(n, n)
    x, info = single(ctx, rp, ci, v, b)
    xt, it = three_launch(ctx, rp, ci, v, b)
    assert info["status"] == 0 and it["status"] == 0
    assert info["iters"] == it["iters"] and info["res_final"] == it["res_final"]
    assert np.array_equal(x, xt)
    # int32 columns: the same iterates
    x4, i4 = single(ctx, rp, ci, v, b, flags=0)
    assert i4["iters"] == info["iters"] and np.array_equal(x4, x)


@pytest.mark.parametrize("case", [(1, 2, 62), (1, 2, 89), (1, 2, 90), (1, 3, 15), (1, 3, 19),
                                  (2, 2, 40)])
def test_fe_systems(ctx, case):
    """Matrices that fit LDS and that do not, and 3D ones on either side of
    the byte limit; iterations and solution against the CPU solve."""
    order, dim, n = case
    rp, ci, v = hflmp.fe_system(order, dim, n, hflmp.fe_kappa(dim, n, 1.0, 3))
    b = hflmp.fe_rhs(order, dim, n, 4)
    x, info = single(ctx, rp, ci, v, b)
    xt, it = three_launch(ctx, rp, ci, v, b)
    assert info["iters"] == it["iters"] and np.array_equal(x, xt)
    xo, io = O.cg(rp, ci, v, b, prec=O.PREC_JACOBI, rtol=1e-8, maxit=10000)
    assert abs(info["iters"] - io["iters"]) <= 2
    assert np.linalg.norm(x - xo) <= 1e-8 * np.linalg.norm(xo)


def test_limits_and_long_solves(ctx):
    # more iterations than one launch runs (512), and stops in between
    n = 1400
    rp = np.concatenate([[0, 2], 2 + 3 * np.arange(1, n - 1), [3 * n - 2]]).astype(np.int32)
    ci = np.concatenate([[c for c in (i - 1, i, i + 1) if 0 <= c < n] for i in range(n)])
    ci = ci.astype(np.int32)
    v = np.where(ci == np.repeat(np.arange(n), np.diff(rp)), 2.0, -1.0)
    b = np.random.default_rng(3).uniform(-1, 1, n)
    x, info = single(ctx, rp, ci, v, b)
    xt, it = three_launch(ctx, rp, ci, v, b)
    assert info["iters"] > 512 and info["status"] == 0
    assert info["iters"] == it["iters"] and np.array_equal(x, xt)
    for maxit in (1, 511, 512, 513):
        x, info = single(ctx, rp, ci, v, b, maxit=maxit)
        xt, it = three_launch(ctx, rp, ci, v, b, maxit=maxit)
        assert info["iters"] == it["iters"] == maxit and info["status"] == it["status"] == 1
        assert np.array_equal(x, xt)
    # nothing to do, and a breakdown (p.Ap = 0)
    x, info = single(ctx, rp, ci, v, np.zeros(n))
    assert info["iters"] == 0 and not x.any()
    x, info = single(ctx, np.array([0, 1, 2], np.int32), np.array([0, 1], np.int32),
                     np.array([1.0, -1.0]), np.array([1.0, 1.0]))
    assert info["status"] == 3


def test_fp32_and_mixed(ctx):
    rp, ci, v, b = banded(3000, 8)
    xo, _ = O.cg(rp, ci, v, b, prec=O.PREC_JACOBI, rtol=1e-12, maxit=10000)
    x, info = single(ctx, rp, ci, v.astype(np.float32), b.astype(np.float32), rtol=1e-4)
    # ||x - xo|| <= cond * (1e-4 + FP32 rounding); cond <= 12 / 0.01
    assert info["status"] == 0
    assert np.linalg.norm(x - xo) <= 1200 * 1.1e-4 * np.linalg.norm(xo)
    A = hflmp.CsrMatrix(ctx, rp, ci, v)
    A32 = A.astype_f32()
    S64, S32 = hflmp.SellMatrix(ctx, A, 1), hflmp.SellMatrix(ctx, A32, 1)
    invd = hflmp.invdiag(ctx, A32)
    db = ctx.upload(b)
    for flags in (0, hflmp.MP_RELIABLE):
        dx = ctx.zeros(A.nrow, np.float64)
        info = hflmp.mpcg_jacobi_sell(ctx, S64, S32, invd, db, dx, rtol=1e-10, inner_rtol=1e-2,
                                      flags=flags)
        assert info["status"] == 0
        # 1200 times the residual's 1e-10
        assert np.linalg.norm(dx.download() - xo) <= 1.3e-7 * np.linalg.norm(xo)
        dx.free()
    for a in (db, invd, S32, S64, A32.val, A):
        a.free()
