"""The work whose speed this framework is measured by, through its public
entry points (ba_amd.hflmp, ba_amd.mg): one dict per case.

Every system is a Dirichlet finite-element matrix of a structured mesh, the
kind the framework is used on: Q1 in 2D and 3D, Q2 in 2D, diffusivity 1 or
log-normal per cell, right-hand sides uniform in [-1, 1] and zero on the
boundary.  Kinds of work:

  vec       the vector operations of one iteration of a host-driven Krylov
            solver (copies, axpy, scaleadd, Jacobi apply, norm and dot
            read back by the host)
  spmv      y = A x through the SELL-64 layout or the CSR arrays
  spmm      Y = A X for a block of vectors through the block layout
  cg        Jacobi-CG to 1e-8 on the device (SELL-64, CSR or matrix-free)
  mixed     FP32-inner / FP64-refined CG to 1e-10
  batched   one CG solve for up to 64 right-hand sides
  mgcg      multigrid-preconditioned CG to 1e-8
  assemble  a cell -> dof table and cell factors to a CSR matrix
  serve     a burst of systems of uneven sizes through the solve server
  lmp       the C++ solver templates over the lmp classes, host arrays in
            and out
"""
import ctypes
import itertools

import numpy as np
import torch

from ba_amd import hflmp, mg

DEV = "cuda"
F64, F32 = "f64", "f32"
NPT = {F64: np.float64, F32: np.float32}
THT = {F64: torch.float64, F32: torch.float32}
LMP_SOLVER = {"cg": hflmp.LMP_CG, "gmres": hflmp.LMP_GMRES, "fgmres": hflmp.LMP_FGMRES,
              "bicgstab": hflmp.LMP_BICGSTAB}
LMP_PREC = {"jacobi": hflmp.LMP_PREC_JACOBI, "sgs": hflmp.LMP_PREC_SGS}

_ctx = None


def context():
    """The program's one device context."""
    global _ctx
    if _ctx is None:
        _ctx = hflmp.Context(0)
    return _ctx


def listed():
    return [
        # a host-driven solver's vector work on the 2D Q1 256^2 system: the
        # smallest calls, where launches and the wait for a scalar count
        dict(name="vec_2d256", kind="vec", n=66049, dtype=F64),
        # the product behind every solver, at the size the framework is
        # rated on, in the layout HIP_CSR_lMatrix runs
        dict(name="spmv_3d128", kind="spmv", order=1, dim=3, n=128, kappa=0, layout="sell16",
             dtype=F64),
        # many vectors at once, the product of the block solver
        dict(name="spmm_q2_512_k64", kind="spmm", order=2, dim=2, n=512, kappa=0, k=64, dtype=F64),
        # the smallest solves: one time step of a small 2D model
        dict(name="cg_2d32", kind="cg", order=1, dim=2, n=32, kappa=1, op="sell16"),
        # the ordinary small solve
        dict(name="cg_2d256", kind="cg", order=1, dim=2, n=256, kappa=0, op="sell16"),
        # the large solve
        dict(name="cg_3d128", kind="cg", order=1, dim=3, n=128, kappa=0, op="sell16"),
        # the large variable-coefficient solve in mixed precision
        dict(name="mixed_3d128", kind="mixed", dim=3, n=128, kappa=1, reliable=True),
        # 64 load cases of one structure
        dict(name="batched_q2_128_k64", kind="batched", order=2, dim=2, n=128, kappa=0, k=64,
             mode=F64),
        # the fastest way to a large solution: matrix-free multigrid CG
        dict(name="mgcg_3d128", kind="mgcg", dim=3, n=128, kappa=1, fine="stencil"),
        # a mesh coming in: pattern and values of a large 3D mesh
        dict(name="assemble_3d96", kind="assemble", order=1, dim=3, n=96, dtype=F64),
        # a burst of requests at a solve service
        dict(name="serve_32", kind="serve", count=32, nmax2=384, nmax3=40),
        # an existing C++ application on the reference's classes
        dict(name="lmp_cg_sgs_2d96", kind="lmp", dim=2, n=96, kappa=1, solver="cg",
             prec="sgs"),
    ]


def draw(rng):
    def size(lo, hi):
        return int(round(lo * (hi / lo) ** rng.random()))

    kind = rng.choice(["vec", "spmv", "spmm", "cg", "mixed", "batched", "mgcg", "assemble",
                       "serve", "lmp"])
    dim = rng.choice([2, 3])
    kappa = rng.choice([0, 1])
    if kind == "vec":
        return dict(kind=kind, n=size(289, 2200000), dtype=rng.choice([F64, F32]))
    if kind == "spmv":
        order = rng.choice([1, 2]) if dim == 2 else 1
        n = size(8, 128) if dim == 3 else size(16, 1024 // order)
        return dict(kind=kind, order=order, dim=dim, n=n, kappa=kappa,
                    layout=rng.choice(["sell16", "sell16", "sell32", "csr"]),
                    dtype=rng.choice([F64, F32]))
    if kind == "spmm":
        order = rng.choice([1, 2]) if dim == 2 else 1
        n = size(8, 48) if dim == 3 else size(16, 512 // order)
        return dict(kind=kind, order=order, dim=dim, n=n, kappa=kappa, k=rng.randint(1, 64),
                    dtype=rng.choice([F64, F32]))
    if kind == "cg":
        n = size(8, 96) if dim == 3 else size(16, 400)
        return dict(kind=kind, order=1, dim=dim, n=n, kappa=kappa,
                    op=rng.choice(["sell16", "sell16", "sell32", "csr", "stencil"]))
    if kind == "mixed":
        n = size(12, 96) if dim == 3 else size(24, 300)
        return dict(kind=kind, dim=dim, n=n, kappa=kappa, reliable=rng.choice([True, False]))
    if kind == "batched":
        return dict(kind=kind, order=rng.choice([1, 2]), dim=2, n=size(12, 96), kappa=kappa,
                    k=rng.randint(2, 64), mode=rng.choice([F64, F64, "mixed"]))
    if kind == "mgcg":
        n = rng.choice([16, 24, 32, 40, 48, 64, 80, 96]) if dim == 3 else \
            rng.choice([32, 48, 80, 96, 128, 160, 192, 256, 320, 384])
        return dict(kind=kind, dim=dim, n=n, kappa=kappa, fine=rng.choice(["stencil", "sell"]))
    if kind == "assemble":
        order = rng.choice([1, 2]) if dim == 2 else 1
        n = size(6, 80) if dim == 3 else size(12, 400)
        return dict(kind=kind, order=order, dim=dim, n=n, dtype=rng.choice([F64, F32]))
    if kind == "serve":
        return dict(kind=kind, count=rng.randint(2, 32), nmax2=size(48, 300),
                    nmax3=rng.randint(17, 36))
    solver = rng.choice(["cg", "gmres", "fgmres", "bicgstab"])
    prec = rng.choice(["jacobi", "jacobi", "sgs"])
    n = size(6, 24) if dim == 3 else size(12, 80)
    return dict(kind="lmp", dim=dim, n=n, kappa=kappa, solver=solver, prec=prec)


# ---- the finite-element systems ------------------------------------------------
def element(order, dim, h):
    """Element stiffness matrix of -div grad on a cube of edge h, local nodes
    lexicographic (x fastest)."""
    if order == 1:
        K = np.array([[1.0, -1.0], [-1.0, 1.0]]) / h
        M = np.array([[2.0, 1.0], [1.0, 2.0]]) * h / 6.0
    else:
        K = np.array([[7.0, -8.0, 1.0], [-8.0, 16.0, -8.0], [1.0, -8.0, 7.0]]) / (3.0 * h)
        M = np.array([[4.0, 2.0, -1.0], [2.0, 16.0, 2.0], [-1.0, 2.0, 4.0]]) * h / 30.0
    if dim == 2:
        return np.kron(M, K) + np.kron(K, M)
    return (np.kron(np.kron(M, M), K) + np.kron(np.kron(M, K), M) + np.kron(np.kron(K, M), M))


class Bands:
    """The system by neighbour offset, on the GPU: coef[o][i] = A[i, i + shift[o]]
    (zero where there is no entry), have[o][i] whether there is an entry;
    offsets in ascending column order."""

    def __init__(self, order, dim, n, kappa):
        p = order * n + 1
        q = order + 1
        self.N = p ** dim
        E = element(order, dim, 1.0 / n)
        shape = (p,) * dim
        loc = list(itertools.product(range(q), repeat=dim))  # (z, y, x)
        offs = sorted({tuple(b[d] - a[d] for d in range(dim)) for a in loc for b in loc})
        at = {o: k for k, o in enumerate(offs)}
        self.coef = torch.zeros((len(offs),) + shape, dtype=torch.float64, device=DEV)
        self.have = torch.zeros((len(offs),) + shape, dtype=torch.bool, device=DEV)
        kap = kappa.reshape((n,) * dim)
        for ia, a in enumerate(loc):
            sl = tuple(slice(a[d], a[d] + order * (n - 1) + 1, order) for d in range(dim))
            for ib, b in enumerate(loc):
                k = at[tuple(b[d] - a[d] for d in range(dim))]
                self.coef[(k,) + sl] += kap * float(E[ia, ib])
                self.have[(k,) + sl] = True
        edge = torch.zeros(shape, dtype=torch.bool, device=DEV)
        for d in range(dim):
            edge.select(d, 0).fill_(True)
            edge.select(d, p - 1).fill_(True)
        self.coef[:, edge] = 0.0
        mid = at[(0,) * dim]
        self.coef[mid][edge] = 1.0
        self.edge = edge.reshape(-1)
        self.coef = self.coef.reshape(len(offs), -1)
        self.have = self.have.reshape(len(offs), -1)
        self.shift = [sum(o[d] * p ** (dim - 1 - d) for d in range(dim)) for o in offs]
        self.diag = self.coef[mid]

    def csr(self, dtype=torch.float64):
        """row_ptr, col (int32) and values as tensors on the GPU."""
        m = self.have.t().contiguous()
        rp = torch.zeros(self.N + 1, dtype=torch.int32, device=DEV)
        rp[1:] = torch.cumsum(m.sum(1), 0).to(torch.int32)
        i = torch.arange(self.N, dtype=torch.int32, device=DEV)
        col = (i[:, None] + torch.tensor(self.shift, dtype=torch.int32, device=DEV)[None, :])[m]
        val = self.coef.t()[m].to(dtype)
        return rp, col, val

    def mult(self, x, dtype=None):
        """A x in 64 bits (x: N or N x k); dtype: values rounded to it first."""
        w = max(self.shift)
        xp = torch.zeros((self.N + 2 * w,) + x.shape[1:], dtype=torch.float64, device=DEV)
        xp[w:w + self.N] = x
        y = torch.zeros_like(x, dtype=torch.float64)
        for k, s in enumerate(self.shift):
            c = self.coef[k] if dtype is None else self.coef[k].to(dtype).double()
            y += (c if x.dim() == 1 else c[:, None]) * xp[w + s:w + s + self.N]
        return y


def system(c, rng, order=None):
    """Bands of a case's system."""
    n, dim = c["n"], c["dim"]
    kap = torch.ones(n ** dim, dtype=torch.float64, device=DEV)
    if c.get("kappa"):
        kap = torch.from_numpy(np.exp(rng.standard_normal(n ** dim))).to(DEV)
    return Bands(c.get("order", 1) if order is None else order, dim, n, kap), kap


def rhs(B, rng, k=0):
    """Right-hand side(s): uniform in [-1, 1], zero on the boundary."""
    b = torch.from_numpy(rng.uniform(-1.0, 1.0, (B.N, k) if k else B.N)).to(DEV)
    b[B.edge] = 0.0
    return b


def solve64(B, b, rtol=1e-13, maxit=20000):
    """Jacobi-CG in 64 bits on torch tensors (b: N or N x k), run until the
    residual stops at rtol."""
    dinv = 1.0 / B.diag if b.dim() == 1 else (1.0 / B.diag)[:, None]
    x = torch.zeros_like(b)
    r = b.clone()
    z = r * dinv
    p = z.clone()
    rz = (r * z).sum(0)
    r0 = torch.linalg.vector_norm(r, dim=0)
    for it in range(maxit):
        Ap = B.mult(p)
        alpha = rz / (p * Ap).sum(0)
        alpha = torch.where(torch.isfinite(alpha), alpha, torch.zeros_like(alpha))
        x += alpha * p
        r -= alpha * Ap
        if it % 16 == 15 and bool((torch.linalg.vector_norm(r, dim=0) <= rtol * r0).all()):
            break
        z = r * dinv
        rzn = (r * z).sum(0)
        beta = rzn / rz
        p = z + torch.where(torch.isfinite(beta), beta, torch.zeros_like(beta)) * p
        rz = rzn
    return x


# ---- what a program holds ---------------------------------------------------------
class Buf:
    """A torch tensor as the device array that ba_amd's calls take."""

    def __init__(self, t):
        self.t = t.contiguous()
        self.n = self.t.numel()
        self.dtype = np.dtype({torch.float64: np.float64, torch.float32: np.float32,
                               torch.int32: np.int32, torch.uint8: np.uint8}[t.dtype])
        self.nbytes = self.n * self.dtype.itemsize
        self.ptr = ctypes.c_void_p(self.t.data_ptr())

    def free(self):
        self.t = None


class State:
    """Handles and buffers of one case; the handles go with it."""

    def __init__(self, case):
        self.case = case
        self.owned = []

    def own(self, h):
        self.owned.append(h)
        return h

    def __del__(self):
        for h in reversed(self.owned):
            (h.close if hasattr(h, "close") else h.free)()


class DeviceResult:
    """A device array made by the framework, given to torch without a copy."""

    def __init__(self, a, n):
        self.a = a
        self.__cuda_array_interface__ = {
            "shape": (int(n),), "typestr": a.dtype.str, "data": (a.ptr.value, False), "version": 2}

    def __del__(self):
        self.a.free()


def vector(N, dtype=torch.float64):
    return Buf(torch.zeros(N, dtype=dtype, device=DEV))


def workspace(n):
    return Buf(torch.empty(max(int(n), 1), dtype=torch.uint8, device=DEV))


def zero(ctx, x):
    ctx.check(ctx.L.hflmp_fill_zero(ctx.h, x.ptr, x.nbytes), "fill_zero")


def csr_matrix(ctx, B, dtype=torch.float64):
    rp, ci, v = B.csr(dtype)
    return hflmp.csr_from_device(ctx, B.N, B.N, ci.numel(), Buf(rp), Buf(ci), Buf(v))


def cell_dofs(order, dim, n):
    """Cell -> dof table, cells and local nodes lexicographic (x fastest)."""
    p = order * n + 1
    c, l = np.arange(n), np.arange(order + 1)
    one = order * c[:, None] + l[None, :]  # cell, local
    if dim == 2:
        t = one[None, :, None, :] + p * one[:, None, :, None]
        return t.reshape(n * n, -1).astype(np.int32)
    t = (one[None, None, :, None, None, :] + p * (one[None, :, None, None, :, None]
         + p * one[:, None, None, :, None, None]))
    return t.reshape(n ** 3, -1).astype(np.int32)


def serve_sizes(c, rng):
    """70% 2D, 30% 3D, log-uniform in the cells per direction."""
    got = []
    for _ in range(c["count"]):
        dim = 2 if rng.random() < 0.7 else 3
        top = c["nmax2"] if dim == 2 else c["nmax3"]
        got.append((dim, int(round(16 * (top / 16) ** rng.random()))))
    # the same mix for every seed: the largest of each kind is there
    got[0] = (2, c["nmax2"])
    got[-1] = (3, c["nmax3"])
    return got


def serve_systems(c, seed):
    mix = np.random.default_rng(c["count"] + 1000 * c["nmax2"] + 1000000 * c["nmax3"])
    rng = np.random.default_rng(seed)
    for dim, n in serve_sizes(c, mix):
        B, _ = system(dict(n=n, dim=dim, kappa=1), rng)
        yield B, rhs(B, rng)


def lmp_options(c):
    return dict(solver=LMP_SOLVER[c["solver"]], precond=LMP_PREC[c["prec"]], rtol=1e-8,
                maxit=5000, basis=60)


def prepare(case, seed):
    s = State(case)
    ctx = s.ctx = context()
    kind = case["kind"]
    rng = np.random.default_rng(seed)
    if kind == "vec":
        dt = THT[case["dtype"]]
        n = case["n"]
        s.inp = [Buf(torch.from_numpy(rng.uniform(-1, 1, n)).to(DEV, dt)) for _ in range(4)]
        s.out = [vector(n, dt) for _ in range(3)]
        torch.cuda.synchronize()
        return s
    if kind == "serve":
        s.reqs = []
        for B, b in serve_systems(case, seed):
            s.reqs.append([t.cpu().numpy() for t in B.csr()] + [b.cpu().numpy()])
        s.server = s.own(hflmp.Server(ctx, 4 << 30, 256, 16, True, 65536, 0.1, 0))
        return s
    if kind == "assemble":
        n, dim, order = case["n"], case["dim"], case["order"]
        s.nnode = (order * n + 1) ** dim
        s.dofs = cell_dofs(order, dim, n)
        s.E = element(order, dim, 1.0 / n)
        s.factor = np.exp(rng.standard_normal(n ** dim))
        return s
    B, kap = system(case, rng)
    if kind == "lmp":
        s.A = [t.cpu().numpy() for t in B.csr()]
        s.b = rhs(B, rng).cpu().numpy()
        return s
    dt = THT[case.get("dtype", F64)]
    if kind in ("spmv", "spmm"):
        k = case.get("k", 0)
        A = csr_matrix(ctx, B, dt)
        s.x = Buf(torch.from_numpy(rng.uniform(-1, 1, (B.N, k) if k else B.N)).to(DEV, dt))
        s.y = Buf(torch.zeros_like(s.x.t))
        torch.cuda.synchronize()
        if kind == "spmm":
            s.A = A
            s.plan = s.own(hflmp.SpmmPlan(ctx, A, k))
        elif case["layout"] == "csr":
            s.A = A
        else:
            s.S = s.own(hflmp.SellMatrix(
                ctx, A, hflmp.SELL_COL16 if case["layout"] == "sell16" else 0))
        ctx.sync()
        return s
    k = case.get("k", 0)
    s.b = Buf(rhs(B, rng, k))
    s.x = Buf(torch.zeros_like(s.b.t))
    L = ctx.L
    if kind == "cg" and case["op"] == "stencil" or kind == "mgcg" and case["fine"] == "stencil":
        n, dim = case["n"], case["dim"]
        fixed = torch.nonzero(B.edge).reshape(-1).to(torch.int32).cpu().numpy()
        s.S = s.own(hflmp.StencilOperator(ctx, 1, dim, [n] * dim, element(1, dim, 1.0 / n)[None],
                                          kap.cpu().numpy(), fixed=fixed))
        A = None
    else:
        A = csr_matrix(ctx, B)
    torch.cuda.synchronize()
    if kind == "cg":
        if case["op"] == "stencil":
            s.invd = s.own(s.S.invdiag())
            s.work = workspace(L.hflmp_pcg_stencil_workspace_bytes(B.N, 8))
        else:
            s.A = A
            s.invd = s.own(hflmp.invdiag(ctx, A))
            if case["op"] != "csr":
                s.S = s.own(hflmp.SellMatrix(
                    ctx, A, hflmp.SELL_COL16 if case["op"] == "sell16" else 0))
            s.work = workspace(L.hflmp_pcg_workspace_bytes(B.N, A.nnz, 8))
    elif kind == "mixed":
        A32 = A.astype_f32()
        s.invd = s.own(hflmp.invdiag(ctx, A32))
        s.S64 = s.own(hflmp.SellMatrix(ctx, A, hflmp.SELL_COL16))
        s.S32 = s.own(hflmp.SellMatrix(ctx, A32, hflmp.SELL_COL16))
        A32.val.free()
        s.work = workspace(L.hflmp_mpcg_sell_workspace_bytes(B.N))
    elif kind == "batched":
        s.A = A
        if case["mode"] == "mixed":
            s.A32 = A.astype_f32()
            s.own(s.A32.val)
            s.invd = s.own(hflmp.invdiag(ctx, s.A32))
            s.plan = s.own(hflmp.SpmmPlan(ctx, s.A32, k))
            s.work = workspace(L.hflmp_batched_mpcg_workspace_bytes(ctx.h, B.N, k))
        else:
            s.invd = s.own(hflmp.invdiag(ctx, A))
            s.plan = s.own(hflmp.SpmmPlan(ctx, A, k))
            s.work = workspace(L.hflmp_batched_pcg_workspace_bytes(ctx.h, B.N, k, 8))
    else:
        n, dim = case["n"], case["dim"]
        s.M = s.own(mg.build_structured(
            ctx, dim, n, element(1, dim, 1.0 / n), kap.cpu().numpy(), A,
            stencil=s.S if A is None else None, min_cells=8, coarse="dense", pre_smooth=1,
            post_smooth=1, omega=0.8))
        s.work = workspace(s.M.workspace_bytes())
    ctx.sync()
    return s


def run(s):
    c, ctx = s.case, s.ctx
    kind = c["kind"]
    if kind == "vec":
        f = lambda name: getattr(ctx.L, "hflmp_%s_%s" % (name, c["dtype"]))
        n = c["n"]
        r0, ap, d, p0 = s.inp
        r, z, p = s.out
        ctx.check(f("copy")(ctx.h, n, r0.ptr, r.ptr))
        ctx.check(f("axpy")(ctx.h, n, -0.375, ap.ptr, r.ptr))
        res = hflmp.nrm2(ctx, r)
        ctx.check(f("jacobi_apply")(ctx.h, n, d.ptr, r.ptr, z.ptr))
        rz = hflmp.dot(ctx, r, z)
        ctx.check(f("copy")(ctx.h, n, p0.ptr, p.ptr))
        ctx.check(f("scaleadd")(ctx.h, n, 0.625, z.ptr, p.ptr))
        return dict(r=r.t, z=z.t, p=p.t, res=res, rz=rz)
    if kind == "spmv":
        if c["layout"] == "csr":
            hflmp.spmv(ctx, s.A, s.x, s.y)
        else:
            s.S.spmv(s.x, s.y)
        return s.y.t
    if kind == "spmm":
        s.plan.spmm(s.A, s.x, s.y, c["k"])
        return s.y.t
    if kind == "assemble":
        mesh = hflmp.FeMesh(ctx, s.nnode, s.dofs)
        try:
            rp, ci = mesh.pattern()
            val = mesh.assemble(rp, ci, E=s.E, factor=s.factor, dtype=NPT[c["dtype"]])
        finally:
            mesh.free()
        return [torch.as_tensor(DeviceResult(a, m), device=DEV)
                for a, m in ((rp, s.nnode + 1), (ci, mesh.nnz), (val, mesh.nnz))]
    if kind == "serve":
        sv = s.server
        tickets = [sv.submit(*q, rtol=1e-8, precision=0) for q in s.reqs]
        left, got = set(tickets), {}
        while left:
            if sv.step():
                for t in list(left):
                    if sv.poll(t)["state"] == 2:
                        got[t] = sv.take(t)[0]
                        left.discard(t)
        return [got[t] for t in tickets]
    if kind == "lmp":
        return hflmp.lmp_solve(*s.A, s.b, **lmp_options(c))[0]
    zero(ctx, s.x)
    if kind == "cg":
        if c["op"] == "csr":
            hflmp.pcg_jacobi(ctx, s.A, s.invd, s.b, s.x, rtol=1e-8, work=s.work)
        elif c["op"] == "stencil":
            hflmp.pcg_jacobi_stencil(ctx, s.S, s.invd, s.b, s.x, rtol=1e-8, work=s.work)
        else:
            hflmp.pcg_jacobi_sell(ctx, s.S, s.invd, s.b, s.x, rtol=1e-8, work=s.work)
    elif kind == "mixed":
        hflmp.mpcg_jacobi_sell(ctx, s.S64, s.S32, s.invd, s.b, s.x, rtol=1e-10,
                               inner_rtol=1e-2 if c["reliable"] else 1e-4,
                               flags=hflmp.MP_RELIABLE if c["reliable"] else 0, work=s.work)
    elif kind == "batched":
        if c["mode"] == "mixed":
            hflmp.batched_mpcg_jacobi(ctx, s.A, s.A32, s.invd, s.b, s.x, c["k"], rtol=1e-8,
                                      work=s.work, plan32=s.plan)
        else:
            hflmp.batched_pcg_jacobi(ctx, s.A, s.invd, s.b, s.x, c["k"], rtol=1e-8,
                                     work=s.work, plan=s.plan)
    else:
        s.M.pcg(s.b, s.x, rtol=1e-8, work=s.work)
    return s.x.t


def exact(case, seed):
    kind = case["kind"]
    rng = np.random.default_rng(seed)
    if kind == "vec":
        dt = THT[case["dtype"]]
        r0, ap, d, p0 = [torch.from_numpy(rng.uniform(-1, 1, case["n"])).to(DEV, dt).double()
                         for _ in range(4)]
        r = r0 - 0.375 * ap
        z = r * d
        return dict(r=r, z=z, p=0.625 * p0 + z, res=float(torch.linalg.vector_norm(r)),
                    rz=float((r * z).sum()))
    if kind == "serve":
        return [solve64(B, b).cpu().numpy() for B, b in serve_systems(case, seed)]
    if kind == "assemble":
        n, dim, order = case["n"], case["dim"], case["order"]
        dt = THT[case["dtype"]]
        E = torch.from_numpy(element(order, dim, 1.0 / n)).to(dt).double().to(DEV)
        f = torch.from_numpy(np.exp(rng.standard_normal(n ** dim))).to(dt).double().to(DEV)
        dofs = torch.from_numpy(cell_dofs(order, dim, n)).to(DEV).long()
        N = (order * n + 1) ** dim
        B = Bands(order, dim, n, torch.ones(n ** dim, dtype=torch.float64, device=DEV))
        rp, ci, _ = B.csr()
        key = torch.repeat_interleave(torch.arange(N, device=DEV),
                                      (rp[1:] - rp[:-1]).long()) * N + ci.long()
        val = torch.zeros(ci.numel(), dtype=torch.float64, device=DEV)
        for a in range(E.shape[0]):
            for b in range(E.shape[0]):
                at = torch.searchsorted(key, dofs[:, a] * N + dofs[:, b])
                val.index_add_(0, at, f * E[a, b])
        return [rp, ci, val]
    B, _ = system(case, rng)
    if kind in ("spmv", "spmm"):
        dt = THT[case["dtype"]]
        k = case.get("k", 0)
        x = torch.from_numpy(rng.uniform(-1, 1, (B.N, k) if k else B.N)).to(DEV, dt).double()
        return B.mult(x, dt)
    x = solve64(B, rhs(B, rng, case.get("k", 0)))
    return x.cpu().numpy() if kind == "lmp" else x


# ---- bytes and operations -----------------------------------------------------------
def sizes(order, dim, n):
    p = order * n + 1
    one = 3 * p - 2 if order == 1 else (n + 1) * 5 - 4 + n * 3  # row lengths along a line
    return p ** dim, one ** dim


def iterations(n, kappa, order=1, digits=8.0):
    """About the iterations Jacobi-CG takes on these systems."""
    return max(8, int((2.05 if not kappa else 2.45) * n * (2.5 if order == 2 else 1)
                      * digits / 8.0))


def work(case):
    kind = case["kind"]
    vb = 4 if case.get("dtype") == F32 else 8
    if kind == "vec":
        n = case["n"]
        return dict(bytes=7 * vb * n, flops=9 * n)
    if kind == "serve":
        mix = np.random.default_rng(case["count"] + 1000 * case["nmax2"]
                                    + 1000000 * case["nmax3"])
        t = dict(bytes=0, flops=0)
        for dim, n in serve_sizes(case, mix):
            w = work(dict(kind="cg", dim=dim, n=n, kappa=1))
            t = {q: t[q] + w[q] for q in t}
        return t
    order, dim, n = case.get("order", 1), case["dim"], case["n"]
    N, nnz = sizes(order, dim, n)
    k = case.get("k", 1)
    matrix = (vb + 4) * nnz + 4 * (N + 1)
    if kind in ("spmv", "spmm"):
        return dict(bytes=matrix + 2 * k * vb * N, flops=2 * k * nnz)
    if kind == "assemble":
        cells, q = n ** dim, (order + 1) ** dim
        return dict(bytes=cells * (4 * q + vb) + matrix, flops=2 * cells * q * q)
    if kind == "mgcg":
        # per cycle and iteration: two sweeps, a residual and a product on
        # the finest level and about 1/7 (3D) or 1/3 (2D) of it below
        its = 16 if case["kappa"] else 10
        below = 8.0 / 7.0 if dim == 3 else 4.0 / 3.0
        return dict(bytes=its * 8 * N * 20 * below, flops=its * below * 4 * 2 * nnz)
    # a Krylov solve: per iteration the matrix and the vectors p, Ap, x, r, D
    its = iterations(n, case["kappa"], order, 10.0 if kind == "mixed" else 8.0)
    if kind == "cg" and case.get("op") == "stencil":
        matrix = 8 * n ** dim
    if kind == "mixed":
        return dict(bytes=its * (8 * nnz + 4 * 8 * N), flops=its * (2 * nnz + 12 * N))
    return dict(bytes=its * (matrix + 8 * 8 * k * N), flops=its * k * (2 * nnz + 12 * N))


def tolerance(case):
    """Four to five times what these paths show against 64-bit solutions
    (measured over the ranges of draw()).  Products, vectors and assembled
    values differ by the rounding of their sums.  A solve that stops at a
    relative residual of 1e-8 is up to 3e-7 from the solution (7e-9 with
    multigrid; 2e-9 for the refined solve, which stops at 1e-10), and another
    order of the sums can move the iteration at which it stops."""
    kind = case["kind"]
    if kind in ("vec", "spmv", "spmm", "assemble"):
        return dict(rel=1e-6 if case["dtype"] == F32 else 1e-14)
    return dict(rel={"mixed": 1e-8, "mgcg": 4e-8}.get(kind, 1.5e-6))
