"""The SELL-64 layout's offset form: which matrices get it (the rule restated
here), and its products against the sequential CSR loop, bit for bit --
slices cut short, every remainder of offsets to a block of loads, rows that
miss entries, offsets that point outside x for other rows of the slice,
infinities and NaN where only a missing entry would read them, y += A x and
new values -- and the general form for rows it cannot hold."""
import time

import numpy as np
import pytest
import scipy.sparse as sp

from ba_amd import hflmp
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def by_offsets(nrow, ncol, offsets, keep, seed, dtype):
    """Row i has columns i + o for the offsets o that stay in the matrix,
    each with probability keep."""
    rng = np.random.default_rng(seed)
    rows = [[i + o for o in offsets if 0 <= i + o < ncol and rng.random() < keep]
            for i in range(nrow)]
    rp = np.concatenate([[0], np.cumsum([len(q) for q in rows])]).astype(np.int32)
    ci = np.array([c for q in rows for c in q], np.int32)
    return rp, ci, rng.uniform(-1, 1, len(ci)).astype(dtype)


def expected(rp, ci, ncol, vb):
    """Stored entries by the layout's rule: the offset form where its bytes
    are below 95% of the columns', for strictly ascending rows."""
    nrow = len(rp) - 1
    full = pos = 0
    fits16 = ok = True
    for s in range(0, nrow, 64):
        offs = set()
        longest = 0
        for i in range(s, min(s + 64, nrow)):
            c = ci[rp[i]:rp[i + 1]].astype(np.int64)
            longest = max(longest, len(c))
            ok = ok and bool((np.diff(c) > 0).all())
            fits16 = fits16 and (len(c) == 0 or
                                 (c.min() - s >= -32768 and c.max() - s <= 32767))
            offs.update((c - i).tolist())
        ok = ok and len(offs) <= 255
        full += 64 * longest
        pos += 64 * len(offs)
    off = ok and len(ci) > 0 and \
        pos * (vb + 12 / 64) < 0.95 * (full * (vb + (2 if fits16 else 4)) + nrow)
    return (pos if off else full), off


def check(ctx, rp, ci, v, ncol, want, hurt=False, seed=0):
    rng = np.random.default_rng(seed)
    nrow = len(rp) - 1
    entries, off = expected(rp, ci, ncol, v.itemsize)
    assert off == want
    x = rng.uniform(-1, 1, ncol).astype(v.dtype)
    if hurt:  # columns no row has: only a missing entry would read them
        free = np.setdiff1d(np.arange(ncol), ci)
        x[free] = np.resize([np.inf, -np.inf, np.nan], len(free))
    A = hflmp.CsrMatrix(ctx, rp, ci, v, ncol=ncol)
    S = hflmp.SellMatrix(ctx, A, hflmp.SELL_COL16 | hflmp.SELL_ANY_PADDING)
    try:
        assert S.info()["entries"] == entries
        dx = ctx.upload(x)
        y0 = rng.uniform(-1, 1, nrow).astype(v.dtype)
        for add in (False, True):
            dy = ctx.upload(y0)
            S.spmv(dx, dy, add=add)
            ref = O.spmv_add(rp, ci, v, x, y0.copy()) if add else O.spmv(rp, ci, v, x)
            assert np.array_equal(dy.download(), ref)
        v2 = rng.uniform(-1, 1, len(v)).astype(v.dtype)
        A2 = hflmp.CsrMatrix(ctx, rp, ci, v2, ncol=ncol)
        S.set_values(A2)
        dy = ctx.upload(y0)
        S.spmv(dx, dy)
        assert np.array_equal(dy.download(), O.spmv(rp, ci, v2, x))
        if len(ci) > 2:  # a pattern whose rows changed length is refused
            rq = rp.copy()
            rq[np.argmax(rp > 0):-1] -= 1
            A2.rp.copy_from_host(np.maximum(rq, 0))
            with pytest.raises(hflmp.HflmpError) as e:
                S.set_values(A2)
            assert e.value.code == hflmp.EFORMAT
        A2.free()
    finally:
        S.free()
        A.free()


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("noff", [1, 2, 3, 4, 5, 7, 8, 9, 11, 13, 14, 15, 16, 22, 23, 24, 27, 28, 29,
                                  30, 57])
def test_every_remainder(ctx, dtype, noff):
    offsets = sorted({(k - noff // 2) * (1 + 2 * (k % 2)) for k in range(noff)})
    rp, ci, v = by_offsets(1000 + noff, 1000 + noff, offsets, 1.0, noff, dtype)
    check(ctx, rp, ci, v, 1000 + noff, True, seed=noff)


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("nrow,ncol", [(1, 1), (63, 63), (64, 64), (65, 65), (129, 129), (300, 700),
                                       (700, 300), (257, 4000)])
def test_sizes_and_edges(ctx, dtype, nrow, ncol):
    # offsets past both ends: other rows of the slice do not have them
    offsets = [-200, -64, -1, 0, 1, 2, 63, 64, 350]
    rp, ci, v = by_offsets(nrow, ncol, offsets, 1.0, nrow + ncol, dtype)
    check(ctx, rp, ci, v, ncol, expected(rp, ci, ncol, v.itemsize)[1], hurt=True, seed=1)


@pytest.mark.parametrize("dtype,keep,want", [(np.float64, 0.95, True), (np.float64, 0.5, True),
                                             (np.float32, 0.9, True), (np.float32, 0.3, False)])
def test_missing_entries(ctx, dtype, keep, want):
    # even columns only: odd ones hold infinities and NaN
    offsets = [-90, -30, -4, -2, 0, 2, 4, 30, 90]
    n = 2000
    rp, ci, v = by_offsets(n, n, offsets, keep, 5, dtype)
    even = (np.repeat(np.arange(n), np.diff(rp)) % 2) == 0
    lens = np.where(np.arange(n) % 2 == 0, np.diff(rp), 0)
    rp2 = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    check(ctx, rp, ci, v, n, want, seed=6)
    rpe, cie, ve = rp2, ci[even], v[even]
    check(ctx, rpe, cie, ve, n, expected(rpe, cie, n, v.itemsize)[1], hurt=True, seed=7)


@pytest.mark.parametrize("dtype,extra,want", [
    (np.float64, 2, True), (np.float64, 3, False), (np.float32, 4, True), (np.float32, 5, False)])
def test_padding_limit(ctx, dtype, extra, want):
    """Even rows have 12 offsets, odd rows 12 of which `extra` are others:
    the positions grow past the columns' bytes."""
    n = 640
    a, b = list(range(-6, 6)), list(range(-6 + extra, 6 + extra))
    rows = [[i + o for o in (a if i % 2 == 0 else b) if 0 <= i + o < n] for i in range(n)]
    rp = np.concatenate([[0], np.cumsum([len(q) for q in rows])]).astype(np.int32)
    ci = np.array([c for q in rows for c in q], np.int32)
    v = np.random.default_rng(3).uniform(-1, 1, len(ci)).astype(dtype)
    check(ctx, rp, ci, v, n, want, seed=11)


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
def test_far_offsets(ctx, dtype):
    # beyond int16: the columns would be int32
    n = 70000
    rp, ci, v = by_offsets(n, n, [-40000, -1, 0, 1, 40000], 1.0, 8, dtype)
    check(ctx, rp, ci, v, n, True, seed=8)


@pytest.mark.parametrize("how", ["unsorted", "twice", "many"])
def test_rows_it_cannot_hold(ctx, how):
    n = 500
    rp, ci, v = by_offsets(n, n, [-3, -1, 0, 1, 3], 1.0, 9, np.float64)
    a = rp[100]
    if how == "unsorted":
        ci[a], ci[a + 1] = ci[a + 1], ci[a]
    elif how == "twice":
        ci[a + 1] = ci[a]
    else:  # more than 255 offsets in a slice
        rng = np.random.default_rng(1)
        rows = [np.sort(rng.choice(n, 6, replace=False)) for _ in range(n)]
        rp = (6 * np.arange(n + 1)).astype(np.int32)
        ci = np.concatenate(rows).astype(np.int32)
        v = rng.uniform(-1, 1, 6 * n)
    check(ctx, rp, ci, v, n, False, seed=10)


def test_solvers_same_bits_as_columns(ctx):
    """CG through the offset form and through int32 columns, on systems of
    each way of running the iteration."""
    for dim, n in ((2, 40), (2, 120), (3, 24), (3, 40)):
        rp, ci, v = hflmp.fe_system(1, dim, n, hflmp.fe_kappa(dim, n, 1.0, 2))
        assert expected(rp, ci, len(rp) - 1, 8)[1]
        A = hflmp.CsrMatrix(ctx, rp, ci, v)
        invd = hflmp.invdiag(ctx, A)
        db = ctx.upload(hflmp.fe_rhs(1, dim, n, 3))
        xs = []
        for flags in (0, hflmp.SELL_COL16):
            S = hflmp.SellMatrix(ctx, A, flags)
            dx = ctx.zeros(A.nrow, np.float64)
            info = hflmp.pcg_jacobi_sell(ctx, S, invd, db, dx)
            assert info["status"] == 0
            xs.append((info["iters"], dx.download()))
            S.free()
            dx.free()
        assert xs[0][0] == xs[1][0] and np.array_equal(xs[0][1], xs[1][1])
        A.free()
        invd.free()
        db.free()


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
def test_uneven_slices(ctx, dtype):
    """A few slices of about 200 offsets beside plain ones: it is all slices
    together that decide."""
    rng = np.random.default_rng(3)
    ns, plain = 40, np.arange(-4, 5)
    forms = set()
    for wild in range(0, 12):
        pick = set(rng.choice(ns, wild, replace=False).tolist())
        rows = []
        for i in range(ns * 64):  # wild: rows in threes share their offsets
            first = i + (i % 64 // 3 * 11 if i // 64 in pick else 0)
            rows.append(np.unique(np.clip(first + plain, 0, ns * 64 - 1)))
        rp = np.concatenate([[0], np.cumsum([len(q) for q in rows])]).astype(np.int32)
        ci = np.concatenate(rows).astype(np.int32)
        v = rng.uniform(-1, 1, len(ci)).astype(dtype)
        off = expected(rp, ci, ns * 64, v.itemsize)[1]
        forms.add(off)
        check(ctx, rp, ci, v, ns * 64, off, seed=wild)
    assert forms == {True, False}


@pytest.mark.parametrize("nrow", [64 * 8192 - 1, 64 * 8192, 64 * 8192 + 1, 64 * 24580])
def test_many_slices(ctx, nrow):
    """The offsets of the slices, around the slices that the scan takes a
    step (8192)."""
    lens = np.random.default_rng(nrow).integers(0, 4, nrow)
    rp = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    j = np.arange(rp[-1]) - np.repeat(rp[:-1], lens)
    ci = np.minimum(np.repeat(np.arange(nrow), lens), nrow - 4).astype(np.int32) + j.astype(np.int32)
    v = np.random.default_rng(1).uniform(-1, 1, len(ci))
    x = np.random.default_rng(2).uniform(-1, 1, nrow)
    A = hflmp.CsrMatrix(ctx, rp, ci, v)
    dx, dy = ctx.upload(x), ctx.zeros(nrow, np.float64)
    ref = O.spmv(rp, ci, v, x)
    for flags in (hflmp.SELL_ANY_PADDING, hflmp.SELL_ANY_PADDING | hflmp.SELL_COL16):
        S = hflmp.SellMatrix(ctx, A, flags)
        S.spmv(dx, dy)
        S.free()
        assert np.array_equal(dy.download(), ref)
    for a in (dx, dy, A):
        a.free()


def test_unstructured_build_keeps_its_speed(ctx):
    """Looking for shared offsets, which an unstructured matrix does not have,
    does not make its build 2.3 times that with int32 columns, which does not
    look (1.6 measured; 2.9 to 3.6 with all slices walked)."""
    rng = np.random.default_rng(0)
    rp, ci, v = hflmp.fe_system(1, 2, 300)
    n = len(rp) - 1
    p = rng.permutation(n)
    B = sp.csr_matrix((v, ci, rp), shape=(n, n))[p][:, p].tocsr()
    B.sort_indices()
    A = hflmp.CsrMatrix(ctx, B.indptr.astype(np.int32), B.indices.astype(np.int32), B.data)
    best = {}
    for flags in (0, hflmp.SELL_COL16) * 12:
        ctx.sync()
        t0 = time.perf_counter()
        S = hflmp.SellMatrix(ctx, A, flags)
        ctx.sync()
        best[flags] = min(best.get(flags, np.inf), time.perf_counter() - t0)
        S.free()
    A.free()
    assert best[hflmp.SELL_COL16] < 2.3 * best[0], best


def _solve(ctx, A, flags, invd, b, short=0, **kw):
    """x and info of Jacobi-CG over the layout; short: bytes left out of the
    workspace."""
    S = hflmp.SellMatrix(ctx, A, flags)
    need = ctx.L.hflmp_pcg_workspace_bytes(S.nrow, S.nnz, S.dtype.itemsize)
    work, db, dx = ctx.empty(need - short, np.uint8), ctx.upload(b), ctx.zeros(A.nrow, b.dtype)
    try:
        info = hflmp.pcg_jacobi_sell(ctx, S, invd, db, dx, work=work, **kw)
        return dx.download(), info["iters"], info["status"], info["res_final"]
    finally:
        for a in (work, db, dx, S):
            a.free()


def _assert_same(got, want):
    assert got[1:] == want[1:] and np.array_equal(got[0], want[0])


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("dim,n", [(2, 120), (3, 24)])
def test_two_launch_stops(ctx, dtype, dim, n):
    """More rows than one workgroup takes, so the offset form runs two launches
    an iteration: stopped at odd and even iterations by maxit (the host polls
    every 16) and by dtol, converged, started at the solution, and in a
    workspace without the second p, it leaves what three launches over int32
    columns leave."""
    rp, ci, v = hflmp.fe_system(1, dim, n, hflmp.fe_kappa(dim, n, 1.0, 2))
    assert len(rp) - 1 > 8192 and expected(rp, ci, len(rp) - 1, np.dtype(dtype).itemsize)[1]
    A = hflmp.CsrMatrix(ctx, rp, ci, v.astype(dtype))
    invd = hflmp.invdiag(ctx, A)
    b = (hflmp.fe_rhs(1, dim, n, 3) != 0).astype(dtype)  # whose residual grows at first
    rtol = 1e-8 if dtype == np.float64 else 1e-4
    runs = [(1, dict(maxit=m, rtol=0.0, dtol=1e30)) for m in (1, 2, 3, 15, 16, 17, 32, 33)]
    runs += [(2, dict(dtol=t, rtol=rtol)) for t in ((2.0, 3.0, 4.5) if dim == 2 else (1.5, 1.9))]
    runs += [(0, dict(rtol=rtol, dtol=1e30)), (0, dict(rtol=rtol, atol=1e6))]
    iters = set()
    for status, kw in runs:
        want = _solve(ctx, A, 0, invd, b, **kw)
        assert want[2] == status
        iters.add(want[1])
        _assert_same(_solve(ctx, A, hflmp.SELL_COL16, invd, b, **kw), want)
        _assert_same(_solve(ctx, A, hflmp.SELL_COL16, invd, b, short=256, **kw), want)
    assert 0 in iters and {k % 2 for k in iters} == {0, 1}
    A.free()
    invd.free()


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("block,rhs,iters", [
    ([[1]], [1], 0),                                                    # every other row -1
    ([[1, -1, -1], [-1, 1, 0], [-1, 0, 2]], [0, 2, 0], 1),
    ([[1, 0, -1], [0, 1, 0], [-1, 0, 1]], [2, -2, 0], 2),
    ([[-1, 1, 0, -1], [1, 1, -2, 1], [0, -2, 2, 0], [-1, 1, 0, 1]], [-1, 0, 2, -1], 3)])
def test_two_launch_breakdown(ctx, dtype, block, rhs, iters):
    """p.Ap = 0 at the first and at later iterations: blocks of small whole
    numbers whose steps are dyadic, so that every sum is exact in any order
    (rows hold zeros at their block's other offsets)."""
    block, m = np.array(block, dtype), len(block)
    n = 9000 // m * m
    offs = np.arange(1 - m, m) if m > 1 else np.arange(-1, 2)
    i = np.repeat(np.arange(n), len(offs))
    j = i + np.tile(offs, n)
    same = (j // m == i // m) & (j < n)
    v = np.where(same, block[i % m, j % m], 0).astype(dtype)
    if m == 1:
        v *= 1 - 2 * (i % 2)
    keep = (j >= 0) & (j < n)
    ci, v = j[keep].astype(np.int32), v[keep]
    rp = np.concatenate([[0], np.cumsum(np.bincount(i[keep], minlength=n))]).astype(np.int32)
    assert expected(rp, ci, n, v.itemsize)[1]
    A = hflmp.CsrMatrix(ctx, rp, ci, v)
    invd = hflmp.invdiag(ctx, A)
    b = np.tile(np.array(rhs, dtype), n // m)
    want = _solve(ctx, A, 0, invd, b, dtol=1e30)
    assert want[1:3] == (iters, 3)
    _assert_same(_solve(ctx, A, hflmp.SELL_COL16, invd, b, dtol=1e30), want)
    A.free()
    invd.free()


@pytest.mark.parametrize("dim,n", [(2, 120), (3, 24)])
def test_refined_solve_two_launches(ctx, dim, n):
    """The refined solve over FP32 in the offset form (two launches) and over
    int32 columns (three): the same x, corrections and inner iterations, with
    the search direction kept from inner solves of odd and even length."""
    rp, ci, v = hflmp.fe_system(1, dim, n, hflmp.fe_kappa(dim, n, 1.0, 2))
    A = hflmp.CsrMatrix(ctx, rp, ci, v)
    A32 = A.astype_f32()
    invd = hflmp.invdiag(ctx, A32)
    db = ctx.upload(hflmp.fe_rhs(1, dim, n, 3))
    S64 = hflmp.SellMatrix(ctx, A, 0)
    forms = [hflmp.SellMatrix(ctx, A32, f) for f in (0, hflmp.SELL_COL16)]
    assert expected(rp, ci, A.nrow, 4)[1]
    need = ctx.L.hflmp_mpcg_sell_workspace_bytes(A.nrow)
    first = set()
    for flags in (0, hflmp.MP_RELIABLE):
        for kw in (dict(inner_rtol=0.3), dict(inner_rtol=0.1), dict(inner_rtol=1e-2),
                   dict(inner_rtol=1e-6, inner_maxit=7), dict(inner_rtol=1e-6, inner_maxit=8)):
            got = []
            for S32, short in ((forms[0], 0), (forms[1], 0), (forms[1], 256)):
                dx, work = ctx.zeros(A.nrow, np.float64), ctx.empty(need - short, np.uint8)
                one = hflmp.mpcg_jacobi_sell(ctx, S64, S32, invd, db, dx, rtol=1e-9, max_outer=1,
                                             flags=flags, work=work, **kw)
                first.add(one["inner_iters"] % 2)
                dx.free()
                dx = ctx.zeros(A.nrow, np.float64)
                info = hflmp.mpcg_jacobi_sell(ctx, S64, S32, invd, db, dx, rtol=1e-9,
                                              max_outer=200, flags=flags, work=work, **kw)
                got.append((dx.download(), info["outer_iters"], info["inner_iters"],
                            info["status"], info["res_final"]))
                dx.free()
                work.free()
            assert got[0][1] > 1
            _assert_same(got[1], got[0])
            _assert_same(got[2], got[0])
    assert first == {0, 1}
    for a in (S64, db, invd, A32.val, A, *forms):
        a.free()


def test_new_values_keep_their_speed(ctx):
    """Refreshing the offset form's values takes no longer than refreshing
    the form with int32 columns."""
    rp, ci, v = hflmp.fe_system(1, 3, 64)
    A = hflmp.CsrMatrix(ctx, rp, ci, v)
    S = {f: hflmp.SellMatrix(ctx, A, f) for f in (0, hflmp.SELL_COL16)}
    best = {f: np.inf for f in S}
    for f in tuple(S) * 12:
        ctx.sync()
        t0 = time.perf_counter()
        S[f].set_values(A)
        ctx.sync()
        best[f] = min(best[f], time.perf_counter() - t0)
    for a in (*S.values(), A):
        a.free()
    assert best[hflmp.SELL_COL16] < best[0], best
