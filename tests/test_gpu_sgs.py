"""Symmetric Gauss-Seidel in the sequential row order (Psgauss_seidel) and
its block form (BlocksPsgauss_seidel) on the device: bit-exact against the
oracle's restatement of the CPU sweeps (which tests/test_oracle.py pins to
the dense (D + L) D^-1 (D + U) factorisations) on FE matrices, ragged block
counts, unsorted rows and FP32; then through the unchanged CG template
(Init_SymmetricGaussSeidel / the block preconditioner) against the oracle's
CG with the same preconditioner: iterations within 2, solution within
1e-8."""
import ctypes as C
import time

import numpy as np
import pytest
import scipy.sparse as sp

from ba_amd import hflmp
from oracle import oracle as O
from tests.helpers import random_csr

pytestmark = pytest.mark.gpu


def _apply(ctx, rp, ci, v, r, nb=1, host_pattern=True, inplace=False):
    A = hflmp.CsrMatrix(ctx, rp, ci, v)
    S = hflmp.Sgs(ctx, A, nb, host_pattern=(rp, ci) if host_pattern else None)
    try:
        dr = ctx.upload(r)
        if inplace:
            S.apply(dr, dr)
            return dr.download(), S.info()
        dz = ctx.empty(len(r), r.dtype)
        S.apply(dr, dz)
        return dz.download(), S.info()
    finally:
        S.destroy()


@pytest.mark.parametrize("order,dim,n", [(1, 2, 256), (1, 3, 24), (2, 2, 40)])
def test_sgs_bit_exact_fe(ctx, order, dim, n):
    rp, ci, v = hflmp.fe_system(order, dim, n, hflmp.fe_kappa(dim, n, 1.0, 7))
    r = np.random.default_rng(n).uniform(-1, 1, len(rp) - 1)
    z, info = _apply(ctx, rp, ci, v, r, host_pattern=(n % 2 == 0))
    assert np.array_equal(z, O.sgs_apply(rp, ci, v, r))
    assert info["levels_forward"] > 1 and info["launches"] >= 2


def test_sgs_bit_exact_96cube(ctx):
    # a large 3D system: most levels hold thousands of rows (one launch each)
    rp, ci, v = hflmp.fe_system(1, 3, 96)
    r = np.random.default_rng(96).uniform(-1, 1, len(rp) - 1)
    z, info = _apply(ctx, rp, ci, v, r)
    assert np.array_equal(z, O.sgs_apply(rp, ci, v, r))
    print("96^3 SGS: levels %d/%d, %d launches" % (info["levels_forward"],
                                                   info["levels_backward"], info["launches"]))


@pytest.mark.parametrize("nb", [2, 7, 64, 1000, 4225, 4300])
def test_block_sgs_bit_exact(ctx, nb):
    # 2D Q1 64^2: 4225 rows; 7 and 64 leave a longer last range, 4225 gives
    # one row per range, 4300 > nrow makes one range of all rows
    rp, ci, v = hflmp.fe_system(1, 2, 64, hflmp.fe_kappa(2, 64, 1.0, 8))
    r = np.random.default_rng(nb).uniform(-1, 1, len(rp) - 1)
    z, info = _apply(ctx, rp, ci, v, r, nb=nb)
    assert info["num_blocks"] == nb
    assert np.array_equal(z, O.block_sgs_apply(rp, ci, v, nb, r))


def test_sgs_fp32_and_in_place(ctx):
    rp, ci, v = hflmp.fe_system(1, 3, 12, hflmp.fe_kappa(3, 12, 1.0, 9))
    r = np.random.default_rng(5).uniform(-1, 1, len(rp) - 1)
    v32, r32 = v.astype(np.float32), r.astype(np.float32)
    z32, _ = _apply(ctx, rp, ci, v32, r32, nb=3)
    assert np.array_equal(z32, O.block_sgs_apply(rp, ci, v32, 3, r32))
    z, _ = _apply(ctx, rp, ci, v, r, inplace=True)
    assert np.array_equal(z, O.sgs_apply(rp, ci, v, r))


@pytest.mark.parametrize("nb", [1, 5])
def test_sgs_unsorted_rows(ctx, nb):
    """Rows in arbitrary column order: the forward sweep stops at the first
    diagonal entry and the backward one takes every upper entry, as the
    reference's loops do; the device follows the same entries."""
    n = 300
    rng = np.random.default_rng(11)
    lengths = rng.integers(1, 12, n)
    rp, ci, v = random_csr(n, n, lengths, 12)
    # every row gets its diagonal (dominant), then the row is shuffled
    rows_c, rows_v = [], []
    for i in range(n):
        c = list(ci[rp[i]:rp[i + 1]])
        w = list(v[rp[i]:rp[i + 1]])
        if i not in c:
            c.append(i)
            w.append(0.0)
        k = c.index(i)
        w[k] = 20.0 + rng.uniform()
        perm = rng.permutation(len(c))
        rows_c.append(np.array(c)[perm])
        rows_v.append(np.array(w)[perm])
    rp = np.concatenate([[0], np.cumsum([len(c) for c in rows_c])]).astype(np.int32)
    ci = np.concatenate(rows_c).astype(np.int32)
    v = np.concatenate(rows_v)
    r = rng.uniform(-1, 1, n)
    z, _ = _apply(ctx, rp, ci, v, r, nb=nb, host_pattern=False)
    assert np.array_equal(z, O.block_sgs_apply(rp, ci, v, nb, r))


@pytest.mark.parametrize("e,width,n,dtype", [
    (4, 1, 300, np.float64),        # a chain: one row a level
    (5, 64, 1000, np.float64),      # a full wave, eight entries' slots
    (8, 65, 977, np.float32),
    (9, 130, 2000, np.float64),
    (16, 512, 3000, np.float64),    # the widest level and the longest row
    (17, 40, 900, np.float64),      # one entry more: the CSR walk
    (3, 513, 3000, np.float64),     # one row more a level: the CSR walk
    (2, 100, 18432, np.float64),    # z just fits LDS
    (2, 100, 18433, np.float64),    # and no longer does
    (4, 100, 36865, np.float32),
])
def test_sgs_level_widths_and_row_lengths(ctx, e, width, n, dtype):
    """Row i is coupled to rows i -+ k width, k = 1..e: levels of `width`
    rows and up to e entries on either side, with one row in seven cut short,
    so that the level-ordered sweep meets its limits and its tails."""
    rng = np.random.default_rng(e * 1000 + width)
    rows = []
    for i in range(n):
        k = 1 if i % 7 == 3 else e
        c = [i + d * width for d in range(-k, k + 1)]
        rows.append([q for q in c if 0 <= q < n])
    rp = np.concatenate([[0], np.cumsum([len(q) for q in rows])]).astype(np.int32)
    ci = np.concatenate(rows).astype(np.int32)
    v = rng.uniform(-1, 1, len(ci)).astype(dtype)
    diag = np.repeat(np.arange(n), np.diff(rp)) == ci
    v[diag] = 40.0 + rng.uniform(0, 1, n).astype(dtype)
    r = rng.uniform(-1, 1, n).astype(dtype)
    z, _ = _apply(ctx, rp, ci, v, r)
    assert np.array_equal(z, O.sgs_apply(rp, ci, v, r))
    z, _ = _apply(ctx, rp, ci, v, r, inplace=True)
    assert np.array_equal(z, O.sgs_apply(rp, ci, v, r))


def test_sgs_refuses_missing_diagonal(ctx):
    rp, ci, v = hflmp.fe_system(1, 2, 4)
    ci = ci.copy()
    # replace row 7's diagonal entry by a second entry at another column
    k = int(rp[7]) + list(ci[rp[7]:rp[8]]).index(7)
    ci[k] = 0 if ci[rp[7]] != 0 else 1
    A = hflmp.CsrMatrix(ctx, rp, ci, v)
    with pytest.raises(hflmp.HflmpError, match="no diagonal"):
        hflmp.Sgs(ctx, A, 1, host_pattern=(rp, ci))


@pytest.mark.parametrize("prec,nb", [(hflmp.LMP_PREC_SGS, 1), (hflmp.LMP_PREC_BSGS, 6)])
def test_lmp_cg_sgs_vs_oracle(prec, nb):
    """CG<LAD> with PreconditionerBlockJacobiStand::Init_SymmetricGaussSeidel
    (or the block SGS preconditioner) against the oracle's CG with the same
    preconditioner (cg.h:165-246)."""
    rp, ci, v = hflmp.fe_system(1, 2, 48, hflmp.fe_kappa(2, 48, 1.0, 21))
    b = hflmp.fe_rhs(1, 2, 48, 22)
    x, res = hflmp.lmp_solve(rp, ci, v, b, precond=prec, sgs_blocks=nb, rtol=1e-8, maxit=2000)
    oprec = O.PREC_SGS if prec == hflmp.LMP_PREC_SGS else O.PREC_BSGS
    xo, io = O.cg(rp, ci, v, b, prec=oprec, rtol=1e-8, maxit=2000, num_blocks=nb)
    assert res["status"] == 0 and io["status"] == 0
    assert abs(res["iters"] - io["iters"]) <= 2, (res["iters"], io["iters"])
    assert np.linalg.norm(x - xo) <= 1e-8 * np.linalg.norm(xo)
    # SGS preconditions better than Jacobi on this system
    _, ij = O.cg(rp, ci, v, b, prec=O.PREC_JACOBI, rtol=1e-8, maxit=2000)
    assert io["iters"] < ij["iters"]


def _free_bytes():
    hip = C.CDLL("libamdhip64.so")
    free, total = C.c_size_t(), C.c_size_t()
    assert hip.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return free.value


def test_level_copy_is_bounded(ctx):
    """Levels of 64 rows beside one of 512, rows of two entries beside one of
    17: the level-ordered copy would be 30 times the matrix, so the sweeps run
    without it, with the same bits."""
    n = 100_000
    rows = [[i] if i < 512 else [i - 64, i] for i in range(n)]
    rows[5000] = list(range(4984, 5000)) + [5000]
    rp = np.concatenate([[0], np.cumsum([len(q) for q in rows])]).astype(np.int32)
    ci = np.concatenate(rows).astype(np.int32)
    A = sp.csr_matrix((np.ones(len(ci)), ci, rp), shape=(n, n))
    A = (A + A.T).tocsr()
    A.sort_indices()
    rp, ci = A.indptr.astype(np.int32), A.indices.astype(np.int32)
    rng = np.random.default_rng(4)
    v = np.where(np.repeat(np.arange(n), np.diff(rp)) == ci, 4.0, rng.uniform(-1, 1, len(ci)))
    r = rng.uniform(-1, 1, n)
    _apply(ctx, rp[:601], ci[:rp[600]] % 600, v[:rp[600]], r[:600])  # (kernels loaded)
    M = hflmp.CsrMatrix(ctx, rp, ci, v)
    dr, dz = ctx.upload(r), ctx.empty(n, np.float64)
    before = _free_bytes()
    S = hflmp.Sgs(ctx, M, 1, host_pattern=(rp, ci))
    held = before - _free_bytes()
    S.apply(dr, dz)
    S.destroy()
    assert np.array_equal(dz.download(), O.sgs_apply(rp, ci, v, r))
    for a in (dr, dz, M):
        a.free()
    assert held <= 2 * max(16 << 20, 4 * (12 * len(ci) + 4 * n)) + (8 << 20), held


def test_level_copy_costs_little_to_make(ctx):
    """Making the sweeps' level-ordered copies takes less than the rest of the
    analysis: the same mesh with one row of more than 16 lower and one of more
    than 16 upper entries has none."""
    rp, ci, v = hflmp.fe_system(1, 3, 24)
    n = len(rp) - 1
    far = 30 + 2 * np.arange(17)  # (through COO: stored zeros stay)
    B = sp.coo_matrix((np.append(v, np.ones(34)),
                       (np.concatenate([np.repeat(np.arange(n), np.diff(rp)), np.full(17, n - 1),
                                        np.zeros(17, int)]),
                        np.concatenate([ci, n - 1 - far, far]))), shape=(n, n)).tocsr()
    B.sort_indices()
    best = []
    for q in ((rp, ci, v), (B.indptr.astype(np.int32), B.indices.astype(np.int32), B.data)):
        M = hflmp.CsrMatrix(ctx, *q)
        t = []
        for _ in range(9):
            ctx.sync()
            t0 = time.perf_counter()
            S = hflmp.Sgs(ctx, M, 1, host_pattern=q[:2])
            t.append(time.perf_counter() - t0)
            S.destroy()
        M.free()
        best.append(min(t))
    assert best[0] < 1.9 * best[1], best


def test_host_pattern_alone_at_creation(ctx):
    """With the pattern given on the host, the device arrays need not hold it
    before the first apply."""
    rp, ci, v = hflmp.fe_system(1, 2, 40)
    r = np.random.default_rng(1).uniform(-1, 1, len(rp) - 1)
    A = hflmp.CsrMatrix(ctx, rp, ci, v)
    A.rp.copy_from_host(np.zeros_like(rp))
    A.ci.copy_from_host(np.zeros_like(ci))
    S = hflmp.Sgs(ctx, A, 1, host_pattern=(rp, ci))
    A.rp.copy_from_host(rp)
    A.ci.copy_from_host(ci)
    dr, dz = ctx.upload(r), ctx.empty(len(r), np.float64)
    S.apply(dr, dz)
    assert np.array_equal(dz.download(), O.sgs_apply(rp, ci, v, r))
    S.destroy()
    for a in (dr, dz, A):
        a.free()
