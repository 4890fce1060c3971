"""Performance cases of the assemble-and-solve path on one MI355X.

Each case is one call, or one short sequence of calls, that a program using
this package makes through its public entry points.  The kinds:

  residual  matvec + waxpby + dot on an assembled box: r = b - A x and r.r, as
            an outer loop of the user's own writes it (many small calls)
  cg        cg_solve in FP64 on an assembled box, with unit conductivity (the
            reference's problem) or one conductivity per element; the load is
            the user's own, random per free node
  mixed     cg_solve_mixed on an assembled box, restarting or keeping the
            direction across refinements
  assemble  generate_matrix_structure, assemble_FE_data, both Dirichlet passes,
            make_local_matrix, and the first product with the new matrix
  batch     Batch.solve: many boxes of uneven size in one launch, and their
            solutions copied out
  multi     cg_solve_multi: 4, 8 or 16 right-hand sides on one matrix
  grad      loss and gradient of the differentiable solve (forward CG, adjoint
            CG, element gradient) through torch.autograd
  upload    cg_solve on a matrix that the user brought: symmetric, ragged rows,
            scattered columns within a band

Sizes are elements per side.  Loads, conductivities, initial vectors, box
sizes and matrices come from the seed.
"""
import numpy as np
import torch

import minife_amd as mfe
from minife_amd import adjoint

DEV = "cuda"
F64 = torch.float64


def listed():
    return [
        # the driver's default box: the smallest call, all latency
        dict(name="residual_10", kind="residual", nx=10, ny=10, nz=10, kappa=False),
        # the plain 30^3 problem, at most 200 iterations
        dict(name="cg_30", kind="cg", nx=30, ny=30, nz=30, kappa=False, iters=200, tol=1e-10),
        # an ordinary box with uneven sides and a conductivity field
        dict(name="cg_kappa_97x71x45", kind="cg", nx=97, ny=71, nz=45, kappa=True, iters=2000, tol=1e-10),
        # an ordinary cube, the reference's 200 iterations
        dict(name="cg_100", kind="cg", nx=100, ny=100, nz=100, kappa=False, iters=200, tol=1e-10),
        # the headline problem: 300^3 elements, 200 iterations
        dict(name="cg_300", kind="cg", nx=300, ny=300, nz=300, kappa=False, iters=200, tol=1e-10),
        # mixed precision to a tight true residual, both refinement forms
        dict(name="mixed_keep_200", kind="mixed", nx=200, ny=200, nz=200, keep=True, tol=1e-11),
        dict(name="mixed_restart_64x48x40", kind="mixed", nx=64, ny=48, nz=40, keep=False, tol=1e-11),
        # a new matrix of the headline size and the first product with it
        dict(name="assemble_300", kind="assemble", nx=300, ny=300, nz=300, kappa=False),
        # 64 uneven boxes, sides 16 to 96
        dict(name="batch_64", kind="batch", count=64, lo=16, hi=96, sizes=0, tol=1e-13),
        # 16 load cases on one matrix
        dict(name="multi_128x16", kind="multi", nx=128, ny=128, nz=128, nrhs=16, tol=1e-10),
        # one step of a conductivity fit (the operator is assembled anew in each)
        dict(name="grad_128", kind="grad", nx=128, ny=128, nz=128, tol=1e-13),
        # a matrix from elsewhere
        dict(name="upload_400k", kind="upload", n=400_003, degree=4, band=1500, tol=1e-10),
    ]


def _log(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    kind = rng.choice(["residual", "cg", "cg", "mixed", "assemble", "batch", "multi", "grad", "upload"])
    top = {"residual": 300, "cg": 300, "mixed": 200, "assemble": 300, "multi": 128, "grad": 128}
    if kind == "batch":
        lo = rng.randint(8, 32)
        return dict(kind=kind, count=_log(rng, 4, 64), lo=lo, hi=rng.randint(lo + 8, 96),
                    sizes=rng.randint(1, 1 << 20), tol=1e-13)
    if kind == "upload":
        return dict(kind=kind, n=_log(rng, 2_000, 1_000_000), degree=rng.randint(2, 4),
                    band=_log(rng, 100, 5_000), tol=1e-10)
    c = dict(kind=kind)
    base = _log(rng, 10, top[kind])  # sides within a factor of about two of each other
    for side in ("nx", "ny", "nz"):
        c[side] = max(8, min(top[kind], int(round(base * (0.6 + 0.8 * rng.random())))))
    if kind in ("residual", "assemble"):
        c["kappa"] = rng.random() < 0.5
    elif kind == "cg":
        c.update(kappa=rng.random() < 0.5, iters=200, tol=1e-10)
    elif kind == "mixed":
        c.update(keep=rng.random() < 0.5, tol=1e-11)
    elif kind == "multi":
        c.update(nrhs=rng.choice([4, 8, 16]), tol=1e-10)
    else:
        c.update(tol=1e-13)
    return c


# ---- inputs (from the seed alone) ------------------------------------------


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _boxes(c):
    rng = np.random.default_rng(c["sizes"])
    return rng.integers(c["lo"], c["hi"], size=(c["count"], 3), endpoint=True).astype(np.int32)


def _nodes(c):
    return (c["nx"] + 1) * (c["ny"] + 1) * (c["nz"] + 1)


def _grid(c):
    return c["nz"] + 1, c["ny"] + 1, c["nx"] + 1


def _kappa(c, g):
    """Conductivities exp(N(0, 0.5^2)) per element."""
    return torch.exp(0.5 * torch.randn(c["nx"] * c["ny"] * c["nz"], generator=g, device=DEV, dtype=F64))


def _load(c, g, k=1):
    """Loads N(0, 1) on the free nodes, 0 on the Dirichlet faces (n x k, row-major)."""
    b = torch.zeros(*_grid(c), k, device=DEV, dtype=F64)
    b[1:-1, 1:-1, 1:-1] = torch.randn(b[1:-1, 1:-1, 1:-1].shape, generator=g, device=DEV, dtype=F64)
    return b.reshape(-1)


def _inputs(c, seed):
    """Every random input of a case, as torch tensors (or arrays), by name."""
    g, kind, d = _gen(seed), c["kind"], {}
    if kind == "batch":
        # the same boxes (as many rows) for every seed, turned and in another order
        rng = np.random.default_rng(seed)
        d["dims"] = rng.permuted(rng.permutation(_boxes(c)), axis=1)
        return d
    if kind == "upload":
        return _upload_matrix(c, seed)
    if c.get("kappa") or kind == "grad":
        d["kappa"] = _kappa(c, g)
    if kind in ("residual", "assemble"):
        d["x"] = torch.randn(_nodes(c), generator=g, device=DEV, dtype=F64)
    if kind in ("residual", "cg", "mixed"):
        d["b"] = _load(c, g)
    if kind == "multi":
        d["b"] = _load(c, g, c["nrhs"])
    if kind == "grad":
        # a smooth target between the two face values
        gz, gy, gx = _grid(c)
        a = 0.5 + torch.rand(3, generator=g, device=DEV, dtype=F64)
        z, y, x = (torch.linspace(0, 1, m, device=DEV, dtype=F64) for m in (gz, gy, gx))
        t = (x[None, None] ** a[0]) * torch.sin(np.pi * y)[None, :, None] ** a[1] * torch.sin(np.pi * z)[:, None, None] ** a[2]
        d["target"] = t.reshape(-1).contiguous()
    return d


def _upload_matrix(c, seed):
    """A diagonally dominant symmetric matrix: each row draws up to `degree`
    larger columns within `band`; CSR with ascending columns."""
    n, rng = c["n"], np.random.default_rng(seed)
    i = np.repeat(np.arange(n, dtype=np.int64), c["degree"])
    j = i + rng.integers(1, c["band"] + 1, i.shape[0])
    keep = (j < n) & (rng.random(i.shape[0]) < 0.9)
    key = np.unique(i[keep] * n + j[keep])
    i, j = key // n, key % n
    v = -rng.uniform(0.1, 1.0, i.shape[0])
    s = -(np.bincount(i, v, n) + np.bincount(j, v, n))
    rows = np.concatenate([i, j, np.arange(n)])
    cols = np.concatenate([j, i, np.arange(n)])
    vals = np.concatenate([v, v, s + rng.uniform(0.01, 0.1, n)])
    order = np.argsort(rows * n + cols, kind="stable")
    ro = np.zeros(n + 1, np.int32)
    np.cumsum(np.bincount(rows, minlength=n), out=ro[1:])
    return dict(row_offsets=ro, cols=cols[order].astype(np.int32), vals=vals[order], b=rng.standard_normal(n))


# ---- what a program has in hand --------------------------------------------


def _view(t, ctx):
    return mfe.Vector.wrap(t.data_ptr(), t.numel(), ctx, owner=t)


def prepare(case, seed):
    c, kind = case, case["kind"]
    d = _inputs(c, seed)
    s = dict(case=c, kind=kind, d=d)
    if kind == "batch":
        s["batch"] = mfe.Batch(d["dims"])
        return s
    if kind == "grad":
        d["kappa"].requires_grad_(True)
        s["dims"] = (c["nx"], c["ny"], c["nz"])
        return s
    # the block solver's program tunes its one matrix once and keeps the context
    ctx = s["ctx"] = mfe.Context(0) if kind == "multi" else mfe.default_context()
    torch.cuda.synchronize()  # the library works on its own stream
    if kind == "upload":
        s["A"] = mfe.CSRMatrix.from_host(d["row_offsets"], d["cols"], d["vals"], ctx=ctx)
        mfe.make_local_matrix(s["A"])
        s["tb"] = torch.from_numpy(d["b"]).to(DEV)
        s["tx"] = torch.zeros(c["n"], device=DEV, dtype=F64)
    elif kind == "assemble":
        s["mesh"] = mfe.simple_mesh_description([0, c["nx"], 0, c["ny"], 0, c["nz"]])
        s["tx"] = d["x"]
        s["tb"] = torch.zeros(_nodes(c), device=DEV, dtype=F64)
        s["ty"] = torch.zeros(_nodes(c), device=DEV, dtype=F64)
    else:
        kappa = _view(d["kappa"], ctx) if c.get("kappa") else None
        _, s["A"], _ = mfe.build_problem(c["nx"], c["ny"], c["nz"], ctx=ctx, kappa=kappa)
        s["tb"] = d["b"]
        s["tx"] = d["x"] if kind == "residual" else torch.zeros_like(d["b"])
    if kind == "residual":
        s["ty"], s["tr"] = (torch.zeros(_nodes(c), device=DEV, dtype=F64) for _ in range(2))
    for name in ("tb", "tx", "ty", "tr"):
        if name in s:
            s[name[1:]] = _view(s[name], ctx)
    if kind == "assemble" and c["kappa"]:
        s["kappa"] = _view(d["kappa"], ctx)
    if kind == "multi":
        mfe.spmm_tune(s["A"], c["nrhs"])
    elif "A" in s:
        mfe.spmv_plan(s["A"])
    if kind == "mixed":
        mfe.matvec_fp32(s["A"], s["b"], s["x"])  # the FP32 copy of the matrix exists too
    ctx.synchronize()
    return s


# ---- one pass ---------------------------------------------------------------


def run(s):
    c, kind = s["case"], s["kind"]
    if kind == "residual":
        mfe.matvec(s["A"], s["x"], s["y"])
        mfe.waxpby(1.0, s["b"], -1.0, s["y"], s["r"])
        return {"r": s["tr"], "rr": mfe.dot(s["r"], s["r"])}
    if kind in ("cg", "upload"):
        s["x"].fill(0.0)
        res = mfe.cg_solve(s["A"], s["b"], s["x"], max_iter=c.get("iters", 2000), tolerance=c["tol"], relative=True)
        if kind == "upload" or c["kappa"]:
            return {"x": s["tx"]}  # the last norm and the count follow the rounding there
        return {"x": s["tx"], "iters": res.num_iters, "normr": res.normr}
    if kind == "mixed":
        s["x"].fill(0.0)
        mfe.cg_solve_mixed(s["A"], s["b"], s["x"], outer_tol=c["tol"], keep_direction=c["keep"])
        return {"x": s["tx"]}
    if kind == "assemble":
        mesh = s["mesh"]
        gx, gy, gz = mesh.nodes
        A = s["A"] = mfe.CSRMatrix(s["ctx"])
        if mfe.generate_matrix_structure(mesh, A) != 0:
            raise MemoryError("generate_matrix_structure: out of device memory")
        s["b"].fill(0.0)
        mfe.assemble_FE_data(mesh, A, s["b"], kappa=s.get("kappa"))
        mfe.impose_dirichlet(0.0, A, s["b"], gx, gy, gz, mesh.bc_rows_0)
        mfe.impose_dirichlet(1.0, A, s["b"], gx, gy, gz, mesh.bc_rows_1)
        mfe.make_local_matrix(A)
        mfe.matvec(A, s["x"], s["y"])
        return {"b": s["tb"], "y": s["ty"]}
    if kind == "batch":
        B = s["batch"]
        B.solve(max_iter=5000, rel_tol=c["tol"])
        return {"x": np.concatenate([B.download(p, matrix=False)["x"] for p in range(B.nprob)])}
    if kind == "multi":
        s["x"].fill(0.0)
        res = mfe.cg_solve_multi(s["A"], s["b"], s["x"], c["nrhs"], rel_tol=c["tol"])
        return {"x": s["tx"], "iters": res.iters}
    # grad
    d = s["d"]
    u = adjoint.solve(d["kappa"], s["dims"], c["tol"])
    loss = 0.5 * torch.sum((u - d["target"]) ** 2)
    (grad,) = torch.autograd.grad(loss, d["kappa"])
    return {"u": u.detach(), "loss": loss.detach(), "grad": grad}


# ---- what a pass cannot do without -------------------------------------------


def _iterations(c):
    """About the CG iterations of a pass: they grow with the largest side."""
    if c["kind"] == "upload":
        return 100
    top = _boxes(c).max(axis=1).mean() if c["kind"] == "batch" else max(c["nx"], c["ny"], c["nz"])
    n = 2.2 * top * (1.3 if c["tol"] <= 1e-12 else 1.0)
    return min(n, c["iters"]) if "iters" in c else n


def work(case):
    """Bytes: vectors as often as an iteration must read or write them (p, r and
    x both ways, A p once each way), the matrix values once per iteration where
    they are the user's own (the 14 upper ones of a row of a symmetric box, or
    12 bytes per entry of an uploaded matrix); a unit-conductivity box's values
    repeat from row to row and are not counted."""
    c, kind = case, case["kind"]
    if kind == "batch":
        n = float(np.prod(_boxes(c).astype(np.float64) + 1, axis=1).sum())
        it = _iterations(c)
        return {"bytes": 64.0 * n * it, "flops": (54 + 10) * n * it}
    if kind == "upload":
        nnz = c["n"] * (1 + 1.8 * c["degree"])
        it = _iterations(c)
        return {"bytes": (12.0 * nnz + 64.0 * c["n"]) * it, "flops": (2 * nnz + 10 * c["n"]) * it}
    n, ne = _nodes(c), c["nx"] * c["ny"] * c["nz"]
    mat = 112.0 * n if c.get("kappa") or kind == "grad" else 0.0
    if kind == "residual":
        return {"bytes": 24.0 * n + mat, "flops": (54 + 4) * n}
    if kind == "assemble":
        # the new matrix (values, columns, row offsets, row ids), b, y; x
        return {"bytes": 12.0 * 27 * n + 8.0 * n + 24.0 * n + (8.0 * ne if c["kappa"] else 0.0),
                "flops": 4888.0 * ne + 54.0 * n}
    it = _iterations(c)
    if kind == "multi":
        return {"bytes": 64.0 * n * c["nrhs"] * it, "flops": (54 + 10) * n * c["nrhs"] * it}
    if kind == "mixed":
        return {"bytes": 32.0 * n * it, "flops": (54 + 10) * n * it}
    if kind == "grad":
        it *= 2
    return {"bytes": (64.0 * n + mat) * it, "flops": (54 + 10) * n * it}


# ---- the same results in plain 64-bit torch -----------------------------------


class _Box:
    """The box operator, matrix-free: trilinear elements with 2x2x2 Gauss
    points at +-0.577350269 (the abscissa the problem is defined with), u = 0 on
    five faces and u = 1 on x = 1."""

    def __init__(self, nx, ny, nz, kappa=None):
        self.shape = (nz + 1, ny + 1, nx + 1)
        h = np.array([1.0 / nx, 1.0 / ny, 1.0 / nz])
        corners = [(a, b, e) for e in (0, 1) for b in (0, 1) for a in (0, 1)]  # (x, y, z)
        K, F = np.zeros((8, 8)), np.zeros(8)
        g = 0.577350269
        for qx in (-g, g):
            for qy in (-g, g):
                for qz in (-g, g):
                    q = (qx, qy, qz)
                    phi = [[0.5 * (1 - q[d]), 0.5 * (1 + q[d])] for d in range(3)]
                    grad = np.zeros((8, 3))
                    for m, cn in enumerate(corners):
                        F[m] += np.prod([phi[d][cn[d]] for d in range(3)]) * h.prod() / 8
                        for d in range(3):
                            o = [phi[e][cn[e]] for e in range(3) if e != d]
                            grad[m, d] = (0.5 if cn[d] else -0.5) * o[0] * o[1] * 2 / h[d]
                    K += grad @ grad.T * h.prod() / 8
        self.K, self.F = K, F
        self.kappa = None if kappa is None else kappa.detach().reshape(nz, ny, nx)
        nzs = (nz, ny, nx)
        self.at = [tuple(slice(cn[2 - d], cn[2 - d] + nzs[d]) for d in range(3)) for cn in corners]
        free = torch.zeros(self.shape, device=DEV, dtype=F64)
        free[1:-1, 1:-1, 1:-1] = 1.0
        self.free = free

    def stiff(self, u):
        """K u without boundary conditions (trailing dimensions allowed)."""
        y = torch.zeros_like(u)
        for m in range(8):
            t = torch.zeros_like(u[self.at[0]])
            for n in range(8):
                t.add_(u[self.at[n]], alpha=float(self.K[m, n]))
            if self.kappa is not None:
                t *= self.kappa.reshape(self.kappa.shape + (1,) * (u.dim() - 3))
            y[self.at[m]] += t
        return y

    def mask(self, u):
        return self.free.reshape(self.shape + (1,) * (u.dim() - 3))

    def apply(self, u):
        f = self.mask(u)
        return f * self.stiff(f * u) + (1 - f) * u

    def rhs(self):
        """Q = 1 and the lifted u = 1 face (its edges, doubly constrained, lift 0)."""
        b = torch.zeros(self.shape, device=DEV, dtype=F64)
        for m in range(8):
            b[self.at[m]] += float(self.F[m])
        one = torch.zeros_like(b)
        one[1:-1, 1:-1, -1] = 1.0
        b = self.free * (b - self.stiff(one))
        b[:, :, -1] = 1.0
        return b


def _plain_cg(apply, b, iters, tol):
    """The textbook iteration per trailing column, and the loop test of
    cg_solve: iteration k runs while the norm at the start of the one before
    exceeds tol ||b||.  Returns x, the iterations and that norm."""
    x, r = torch.zeros_like(b), b.clone()
    rr = torch.sum(r * r)
    stop, p, k = tol * float(torch.sqrt(rr)), None, 0
    normr = float(torch.sqrt(rr))
    while k < iters and normr > stop:
        k += 1
        if k > 1:
            new = torch.sum(r * r)
            p = r + (new / rr) * p
            rr = new
            normr = float(torch.sqrt(rr))
        else:
            p = r.clone()
        Ap = apply(p)
        a = rr / torch.sum(p * Ap)
        x += a * p
        r -= a * Ap
    return x, k, normr


def exact(case, seed):
    c, kind = case, case["kind"]
    d = _inputs(c, seed)
    if kind == "batch":
        xs = []
        for nx, ny, nz in d["dims"].tolist():
            op = _Box(nx, ny, nz)
            xs.append(_plain_cg(op.apply, op.rhs(), 5000, c["tol"])[0].reshape(-1).cpu().numpy())
        return {"x": np.concatenate(xs)}
    if kind == "upload":
        A = torch.sparse_csr_tensor(torch.from_numpy(d["row_offsets"]), torch.from_numpy(d["cols"]),
                                    torch.from_numpy(d["vals"]), size=(c["n"], c["n"])).to(DEV)
        return {"x": _plain_cg(lambda p: A @ p, torch.from_numpy(d["b"]).to(DEV), 2000, c["tol"])[0]}
    op = _Box(c["nx"], c["ny"], c["nz"], d.get("kappa"))
    if kind == "residual":
        r = (d["b"].reshape(op.shape) - op.apply(d["x"].reshape(op.shape))).reshape(-1)
        return {"r": r, "rr": float(torch.sum(r * r))}
    if kind == "assemble":
        return {"b": op.rhs().reshape(-1), "y": op.apply(d["x"].reshape(op.shape)).reshape(-1)}
    if kind == "cg":
        x, _, normr = _plain_cg(op.apply, d["b"].reshape(op.shape), c["iters"], c["tol"])
        if c["kappa"]:
            return {"x": x.reshape(-1)}
        return {"x": x.reshape(-1), "iters": None, "normr": normr}
    if kind == "mixed":
        return {"x": _plain_cg(op.apply, d["b"].reshape(op.shape), 20000, 1e-13)[0].reshape(-1)}
    if kind == "multi":
        b = d["b"].reshape(*op.shape, c["nrhs"])
        xs = [_plain_cg(op.apply, b[..., k].contiguous(), 5000, c["tol"] * 1e-2)[0] for k in range(c["nrhs"])]
        return {"x": torch.stack(xs, -1).reshape(-1), "iters": None}
    # grad: u, then the adjoint solution and -lambda_e^T K_e u_e per element
    u = _plain_cg(op.apply, op.rhs(), 50000, c["tol"] * 1e-1)[0]
    g = u - d["target"].reshape(op.shape)
    loss = 0.5 * torch.sum(g * g)
    lam = _plain_cg(op.apply, op.free * g, 50000, c["tol"] * 1e-1)[0]
    ut = u * op.free
    ut[1:-1, 1:-1, -1] = u[1:-1, 1:-1, -1]
    grad = torch.zeros_like(op.kappa)
    for m in range(8):
        t = torch.zeros_like(grad)
        for n in range(8):
            t.add_(ut[op.at[n]], alpha=float(op.K[m, n]))
        grad -= lam[op.at[m]] * t
    return {"u": u.reshape(-1), "loss": loss, "grad": grad.reshape(-1)}
