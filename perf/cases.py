"""The framework's main paths as measurable cases.

Every case is one call (or one short sequence of calls) that a user's program
makes: an operator applied to a vector, a V-cycle used as a preconditioner, a
whole solve, a block solve, a differentiable solve with its backward pass, a
Galerkin product, and a hierarchy setup followed by the solve it was made for.
The matrices are the gallery's (27-point Laplacian, rotated anisotropic
9-point, 7-point finite volume with variable coefficients) and one unstructured
matrix; sizes go from the smallest the solvers are used at to the benchmark's.

A case is a dict of plain values:
  kind       op, cycle, solve, block, adjoint, galerkin or setup
  matrix     lap27 (m^3 rows), aniso (m^2), fv7 (m^3) or graph (m rows)
  m          the size
and, by kind, `op`, `prec` (32 or 64: the cycle's precision), `method`, `k`.
"""
import functools
import math

import numpy as np
import torch  # before the library is loaded: one HIP runtime in the process

import raptor_amd as ra
import raptor_amd.autograd

OMEGA = 2.0 / 3.0
RTOL = 1e-8
PREC = {64: ra.PREC_FP64, 32: ra.PREC_FP32}


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------
def listed():
    return [
        # one preconditioner application on the smallest benchmark problem:
        # launches and latency are all of it
        {"name": "cycle_aniso_100", "kind": "cycle", "matrix": "aniso", "m": 100, "prec": 64},
        # the smallest benchmark problem solved with the reference's PCG
        {"name": "pcg_aniso_100", "kind": "solve", "matrix": "aniso", "m": 100, "method": "pcg", "prec": 64},
        # y = A x with an unstructured matrix, row lengths from 1 to over a hundred
        {"name": "mult_graph_300k", "kind": "op", "matrix": "graph", "m": 300001, "op": "mult"},
        # r = b - A x with a stencil matrix outside any solver
        {"name": "residual_lap27_192", "kind": "op", "matrix": "lap27", "m": 192, "op": "residual"},
        # the FP32 preconditioner on a grid whose sizes divide nothing
        {"name": "cycle32_lap27_101", "kind": "cycle", "matrix": "lap27", "m": 101, "prec": 32},
        # an ordinary solve, everything in FP64
        {"name": "fpcg64_lap27_128", "kind": "solve", "matrix": "lap27", "m": 128, "method": "fpcg", "prec": 64},
        # the benchmark: the largest solve, FP32 cycle inside the FP64 iteration
        {"name": "fpcg32_lap27_256", "kind": "solve", "matrix": "lap27", "m": 256, "method": "fpcg", "prec": 32},
        # a training step through the solver: forward solve and adjoint backward
        {"name": "adjoint_fv7_96", "kind": "adjoint", "matrix": "fv7", "m": 96, "prec": 64},
        # many right-hand sides with one operator
        {"name": "block_aniso_1024_k32", "kind": "block", "matrix": "aniso", "m": 1024, "k": 32, "prec": 32},
        # the coarse operator P^T A P of new coefficients with an interpolation
        # that is kept, brought to the host
        {"name": "galerkin_lap27_96", "kind": "galerkin", "matrix": "lap27", "m": 96},
        # a system that is solved once: Ruge-Stuben setup from host arrays, then the solve
        {"name": "setup_lap27_128", "kind": "setup", "matrix": "lap27", "m": 128, "prec": 32},
        # the same with smoothed aggregation on variable coefficients
        {"name": "setup_fv7_96", "kind": "setup", "matrix": "fv7", "m": 96, "prec": 64},
    ]


# sizes that draw() spreads over, by kind and matrix
RANGES = {
    "op": {"lap27": (48, 192), "aniso": (320, 2048), "fv7": (48, 192), "graph": (30000, 600000)},
    "cycle": {"lap27": (16, 128), "aniso": (64, 1024), "fv7": (16, 96)},
    "solve": {"lap27": (16, 160), "aniso": (64, 1024), "fv7": (16, 96)},
    "adjoint": {"fv7": (16, 96)},
    "block": {"aniso": (64, 1024), "lap27": (16, 64)},
    "galerkin": {"lap27": (16, 96), "aniso": (64, 1024), "fv7": (16, 96)},
    "setup": {"lap27": (16, 128), "aniso": (64, 1024), "fv7": (16, 96)},
}


def draw(rng):
    kind = rng.choice(sorted(RANGES))
    matrix = rng.choice(sorted(RANGES[kind]))
    lo, hi = RANGES[kind][matrix]
    m = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    case = {"kind": kind, "matrix": matrix, "m": m}
    if kind == "op":
        case["op"] = rng.choice(["mult", "mult_T", "residual"] + ([] if matrix == "graph" else ["jacobi"]))
    if kind in ("cycle", "adjoint", "block", "setup"):
        case["prec"] = rng.choice([32, 64])
    if kind == "solve":
        case["method"] = rng.choice(["fpcg", "fpcg", "pcg"])
        case["prec"] = 64 if case["method"] == "pcg" else rng.choice([32, 64])
    if kind == "block":
        case["k"] = rng.choice([2, 3, 4, 7, 8, 12, 16, 21, 32])
    return case


# ---------------------------------------------------------------------------
# matrices
# ---------------------------------------------------------------------------
def _graph(n, seed):
    """A square unsymmetric matrix without grid structure: most columns near
    the row (as a renumbered mesh has them), a tenth anywhere, log-normal row
    lengths of mean about 17, the diagonal always there."""
    rng = np.random.default_rng(seed)
    length = np.minimum(np.exp(rng.normal(2.6, 0.6, n)).astype(np.int64) + 1, 160)
    row = np.repeat(np.arange(n, dtype=np.int64), length)
    near = np.rint(rng.laplace(0.0, 0.004 * n + 8, row.size)).astype(np.int64)
    col = (row + near) % n
    far = rng.random(row.size) < 0.1
    col[far] = rng.integers(0, n, int(far.sum()))
    key = np.unique(np.concatenate([row * n + col, np.arange(n, dtype=np.int64) * (n + 1)]))
    row, col = key // n, key % n
    rp = np.zeros(n + 1, np.int32)
    np.cumsum(np.bincount(row, minlength=n), out=rp[1:])
    val = rng.normal(0.0, 1.0, col.size)
    return rp, col.astype(np.int32), val


@functools.lru_cache(maxsize=2)
def _gallery(matrix, m):
    return ra.gallery_laplace27(m) if matrix == "lap27" else ra.gallery_aniso2d(m, 0.001, math.pi / 8)


def rescaled(M, seed):
    """D A D: the same operator with other coefficients."""
    rp, col, val = M
    s = np.random.default_rng(seed).uniform(0.8, 1.25, rp.size - 1)
    return rp, col, val * (np.repeat(s, np.diff(rp)) * s[col])


def host_matrix(case, seed):
    """(rowptr, col, val) of the case's matrix."""
    if case["matrix"] == "graph":
        return _graph(case["m"], seed)
    if case["matrix"] == "fv7":
        # a Galerkin product's interpolation is one the program kept: its
        # coefficients do not follow the seed (rescaled() makes the new ones)
        return ra.gallery_fv7(case["m"], seed=3 if case["kind"] == "galerkin" else seed)
    return _gallery(case["matrix"], case["m"])


def rows(case):
    return {"lap27": case["m"] ** 3, "fv7": case["m"] ** 3, "aniso": case["m"] ** 2, "graph": case["m"]}[case["matrix"]]


def entries(case):
    m = case["m"]
    return {"lap27": (3 * m - 2) ** 3, "aniso": (3 * m - 2) ** 2, "fv7": 7 * m ** 3 - 6 * m * m, "graph": 17 * m}[
        case["matrix"]]


@functools.lru_cache(maxsize=1)
def context():
    return ra.Context(0)


def solver(case, ctx):
    """The hierarchy each matrix is used with in the benchmark's workloads."""
    if case["matrix"] == "lap27":
        ml = ra.ParRugeStubenSolver(ctx, 0.25, ra.PMIS, ra.Extended, ra.Classical, ra.Jacobi)
    elif case["matrix"] == "aniso":
        ml = ra.ParRugeStubenSolver(ctx, 0.25, ra.CLJP, ra.ModClassical, ra.Classical, ra.Jacobi)
    else:
        ml = ra.ParSmoothedAggregationSolver(ctx, 0.08, ra.Symmetric, ra.Jacobi)
    ml.relax_weight = OMEGA
    return ml


# ---------------------------------------------------------------------------
# vectors
# ---------------------------------------------------------------------------
class _Memory:
    """A device vector as torch sees it, without a copy."""

    def __init__(self, vec, shape):
        self.vec = vec
        self.__cuda_array_interface__ = {"data": (vec.ptr.value, False), "shape": shape, "version": 2,
                                         "typestr": vec.dtype.str}


def tensor(vec, *shape):
    return torch.as_tensor(_Memory(vec, shape or (vec.n,)), device="cuda")


def vector(ctx, a):
    return ra.ParVector.from_numpy(ctx, a)


def solution(n, seed, k=None):
    """The solution a right-hand side is made from: a smooth part and noise,
    as a discretised field has them."""
    rng = np.random.default_rng(seed)
    t = np.arange(n) * (2.0 * math.pi / n)
    shape = n if k is None else (n, k)
    f, p = rng.uniform(1.0, 9.0, k), rng.uniform(0.0, 6.0, k)
    smooth = np.sin(np.multiply.outer(t, f) + p if k else f * t + p)
    return smooth + 0.3 * rng.standard_normal(shape)


def applied(A, x):
    """A x as a new host array."""
    xd, yd = vector(A.ctx, x), ra.ParVector(A.ctx, x.size)
    A.mult(xd, yd)
    return yd.numpy()


# ---------------------------------------------------------------------------
# what a program has in hand, and one pass
# ---------------------------------------------------------------------------
def prepare(case, seed):
    ctx = context()
    n = rows(case)
    rp, col, val = host_matrix(case, seed)
    st = {"case": case, "ctx": ctx}
    kind = case["kind"]
    if kind == "setup":
        # the host arrays are the input; the operator of the outer iteration is made in the pass
        A = ra.ParCSRMatrix.from_csr(ctx, rp, col, val)
        st.update(csr=(rp, col, val), b=vector(ctx, applied(A, solution(n, seed))), x=ra.ParVector(ctx, n))
        A.free()
        st["out"] = tensor(st["x"])
        return st
    A = st["A"] = ra.ParCSRMatrix.from_csr(ctx, rp, col, val)
    if kind == "op":
        rng = np.random.default_rng(seed)
        st["x"] = vector(ctx, rng.standard_normal(n))
        st["b"] = vector(ctx, rng.standard_normal(n))
        st["y"] = ra.ParVector(ctx, n)
        if case["op"] == "jacobi":
            st["tmp"] = ra.ParVector(ctx, n)
        st["out"] = tensor(st["y"])
        return st
    ml = st["ml"] = solver(case, ctx).setup(rp, col, val)
    if kind == "galerkin":
        st["P"] = ml.level(0)[1]
        st["A"] = ra.ParCSRMatrix.from_csr(ctx, *rescaled((rp, col, val), seed))
        return st
    if case.get("prec") == 32:
        ml.enable_fp32()
    if kind == "cycle":
        dt = np.float32 if case["prec"] == 32 else np.float64
        st["b"] = vector(ctx, np.random.default_rng(seed).standard_normal(n).astype(dt))
        st["x"] = ra.ParVector(ctx, n, dt)
    elif kind == "solve":
        st["b"] = vector(ctx, applied(A, solution(n, seed)))
        st["x"] = ra.ParVector(ctx, n)
    elif kind == "block":
        k = case["k"]
        X = solution(n, seed, k)
        st["B"] = vector(ctx, np.stack([applied(A, np.ascontiguousarray(X[:, c])) for c in range(k)], axis=1).ravel())
        st["X"] = ra.ParVector(ctx, n * k)
        st["out"] = tensor(st["X"], n, k)
    elif kind == "adjoint":
        b = torch.from_numpy(applied(A, solution(n, seed))).cuda()
        g = torch.from_numpy(applied(A, solution(n, seed + 1))).cuda()
        st.update(vals=torch.from_numpy(val).cuda().requires_grad_(True), b=b.requires_grad_(True), g=g)
        torch.cuda.synchronize()
    if "x" in st:
        st["out"] = tensor(st["x"])
    return st


def _solve(case, A, ml, x, b):
    x.set_const_value(0.0)
    if case.get("method") == "pcg":
        ra.PCG(A, ml, x, b, tol=RTOL)
    else:
        ra.FPCG(A, ml, x, b, rtol=RTOL, cycle_prec=PREC[case["prec"]])


def run(st):
    case, ctx = st["case"], st["ctx"]
    kind = case["kind"]
    if kind == "op":
        A, op = st["A"], case["op"]
        if op == "mult":
            A.mult(st["x"], st["y"])
        elif op == "mult_T":
            A.mult_T(st["x"], st["y"])
        elif op == "residual":
            A.residual(st["x"], st["b"], st["y"])
        else:
            # one smoothing step: from the right-hand side as the first
            # iterate, so that a pass does not depend on the one before it
            st["y"].copy(st["b"])
            A.jacobi(st["y"], st["x"], st["tmp"], 1, OMEGA)
        return st["out"]
    if kind == "cycle":
        if case["prec"] == 32:
            st["ml"].cycle_fp32(st["x"], st["b"])
        else:
            st["x"].set_const_value(0.0)
            st["ml"].cycle(st["x"], st["b"], x_is_zero=True)
        return st["out"]
    if kind == "solve":
        _solve(case, st["A"], st["ml"], st["x"], st["b"])
        return st["out"]
    if kind == "block":
        k = case["k"]
        st["X"].set_const_value(0.0)
        ra.FPCG_block(st["A"], st["ml"], st["X"], st["B"], k, rtol=RTOL, cycle_prec=PREC[case["prec"]])
        return st["out"]
    if kind == "adjoint":
        x = raptor_amd.autograd.amg_solve(st["vals"], st["b"], st["ml"], st["A"], rtol=1e-10,
                                          cycle_prec=PREC[case["prec"]])
        dvals, db = torch.autograd.grad(x, (st["vals"], st["b"]), st["g"])
        return {"x": x.detach(), "dvals": dvals, "db": db}
    if kind == "galerkin":
        C = st["A"].galerkin(st["P"])
        out = C.to_csr()
        C.free()
        return out
    if kind == "setup":
        rp, col, val = st["csr"]
        ml = solver(case, ctx).setup(rp, col, val)
        A = ra.ParCSRMatrix.from_csr(ctx, rp, col, val)
        _solve(case, A, ml, st["x"], st["b"])
        sizes, nnz, _ = ml.level_sizes()
        A.free()
        ml.free()
        # by level, zero below the coarsest (the number of levels follows the coefficients)
        return {"x": st["out"], "rows": np.pad(sizes, (0, 25 - sizes.size)), "entries": np.pad(nnz, (0, 25 - nnz.size))}
    raise ValueError(kind)


# ---------------------------------------------------------------------------
# what a pass cannot do without, and how far results may be apart
# ---------------------------------------------------------------------------
def work(case):
    n, nnz, kind = rows(case), entries(case), case["kind"]
    matrix = 12.0 * nnz + 4.0 * n
    if kind == "op":
        vectors = {"mult": 2, "mult_T": 2, "residual": 3, "jacobi": 3}[case["op"]]
        return {"bytes": matrix + 8.0 * vectors * n, "flops": 2.0 * nnz}
    # a hierarchy holds about this many times the fine matrix's entries
    # (operators and interpolations of the levels together)
    grow = {"lap27": 1.4, "aniso": 4.8, "fv7": 2.0}[case["matrix"]]
    sv = 4.0 if case.get("prec") == 32 else 8.0
    k = case.get("k", 1)
    # a cycle reads each level's operator for its residual and again for its
    # last sweep, whose input depends on all coarser levels
    cycle = {"bytes": 2.0 * grow * nnz * (sv + 4.0) + 8.0 * sv * n * k, "flops": 4.0 * grow * nnz * k}
    if kind == "cycle":
        return cycle
    if kind == "galerkin":
        # about four products per entry of A for A P and two for P^T (A P);
        # the coarse operator has about a fifth of the fine one's entries
        return {"bytes": 1.5 * matrix, "flops": 2.0 * 6.0 * nnz}
    # an iteration: a cycle, the outer product, the vectors of the update
    per = {"bytes": cycle["bytes"] + matrix + 80.0 * n * k, "flops": cycle["flops"] + (2.0 * nnz + 12.0 * n) * k}
    its = {"lap27": 10, "aniso": 36, "fv7": 25}[case["matrix"]]
    if case.get("method") == "pcg":
        its = {"lap27": 7, "aniso": 7, "fv7": 15}[case["matrix"]]
    extra = {"bytes": 0.0, "flops": 0.0}
    if kind == "adjoint":
        its = 60  # two solves to a smaller tolerance
        extra = {"bytes": 20.0 * nnz, "flops": 1.0 * nnz}
    if kind == "setup":
        extra = {"bytes": 4.0 * grow * matrix, "flops": 12.0 * nnz}
    return {"bytes": its * per["bytes"] + extra["bytes"], "flops": its * per["flops"] + extra["flops"]}


def tolerance(case):
    kind = case["kind"]
    if kind in ("op", "galerkin"):
        # one FP64 sum of products per value: 2e-16 (2-norm) from exact(),
        # which adds in another order
        return {"rel": 1e-15, "max": 2e-14}
    if kind == "cycle":
        # other roundings everywhere (the right-hand side times three, the
        # result divided by three) moved the result by 6e-16 in 64 bits and
        # by 1.9e-7 in 32, the largest entry by 3e-15 and 1.7e-6
        return {"rel": 1e-6, "max": 1e-5} if case["prec"] == 32 else {"rel": 4e-15, "max": 4e-14}
    # iterations to a residual tolerance: the same change moved the solutions
    # by up to 5e-14 with FP64 cycles and 1.6e-11 with FP32 cycles (largest
    # entry 2.4e-13 and 1.9e-10), an anisotropic problem's the most
    return {"rel": 1e-10, "max": 1e-9} if case.get("prec") == 32 else {"rel": 1e-12, "max": 1e-11}


# ---------------------------------------------------------------------------
# the same in plain 64-bit numpy / torch
# ---------------------------------------------------------------------------
def _mv(M, x):
    rp, col, val = M[0], M[1], M[2]
    out = np.zeros(rp.size - 1)
    full = rp[1:] > rp[:-1]
    if col.size:
        out[full] = np.add.reduceat(val * x[col], rp[:-1][full].astype(np.int64))
    return out


def _mv_t(M, x, n_cols):
    rp, col, val = M[0], M[1], M[2]
    return np.bincount(col, weights=val * np.repeat(x, np.diff(rp)), minlength=n_cols)


def _diag(M):
    rp, col, val = M[0], M[1], M[2]
    d = np.zeros(rp.size - 1)
    row = np.repeat(np.arange(rp.size - 1), np.diff(rp))
    on = row == col
    d[row[on]] = val[on]
    return d


def _cycle(levels, l, b):
    """One V(1,1) cycle from zero with weighted Jacobi on plain arrays."""
    A, P, nc = levels[l]
    if P is None:
        dense = np.zeros((b.size, b.size))
        dense[np.repeat(np.arange(b.size), np.diff(A[0])), A[1]] = A[2]
        return np.linalg.solve(dense.T, b)  # the reference factors the transpose
    d = _diag(A)
    x = OMEGA * b / d
    r = b - _mv(A, x)
    x = x + _mv(P, _cycle(levels, l + 1, _mv_t(P, r, nc)))
    return x + OMEGA * (b - _mv(A, x)) / d


def _product(A, B, n_cols):
    """A B, rows sorted by column, entries within 1e-16 of zero dropped."""
    (ap, ac, av), (bp, bc, bv) = [[torch.from_numpy(np.ascontiguousarray(t)).cuda() for t in M] for M in (A, B)]
    bp = bp.long()
    count = (bp[1:] - bp[:-1])[ac.long()]
    rows_ = torch.repeat_interleave(torch.arange(ap.numel() - 1, device="cuda"), (ap[1:] - ap[:-1]).long())
    entry = torch.repeat_interleave(torch.arange(ac.numel(), device="cuda"), count)
    first = torch.cumsum(count, 0) - count
    at = bp[ac.long()][entry] + torch.arange(entry.numel(), device="cuda") - first[entry]
    key = rows_[entry] * n_cols + bc[at].long()
    key, inv = torch.unique(key, return_inverse=True)
    v = torch.zeros(key.numel(), dtype=torch.float64, device="cuda").index_add_(0, inv, av[entry] * bv[at])
    keep = v.abs() > 1e-16
    key, v = key[keep], v[keep]
    n = ap.numel() - 1
    rp = torch.zeros(n + 1, dtype=torch.int64, device="cuda")
    rp[1:] = torch.cumsum(torch.bincount(key // n_cols, minlength=n), 0)
    return rp.int().cpu().numpy(), (key % n_cols).int().cpu().numpy(), v.cpu().numpy()


def _transpose(M, n_cols):
    rp, col, val = M
    row = np.repeat(np.arange(rp.size - 1, dtype=np.int32), np.diff(rp))
    order = np.argsort(col, kind="stable")
    out = np.zeros(n_cols + 1, np.int32)
    np.cumsum(np.bincount(col, minlength=n_cols), out=out[1:])
    return out, row[order], val[order]


def exact(case, seed):
    kind, n = case["kind"], rows(case)
    if kind == "op":
        M = host_matrix(case, seed)
        rng = np.random.default_rng(seed)
        x, b = rng.standard_normal(n), rng.standard_normal(n)
        if case["op"] == "mult":
            return _mv(M, x)
        if case["op"] == "mult_T":
            return _mv_t(M, x, n)
        if case["op"] == "residual":
            return b - _mv(M, x)
        return b + OMEGA * (x - _mv(M, b)) / _diag(M)
    if kind == "cycle":
        # the hierarchy is the path's input; the cycle on it is plain numpy
        ml = solver(case, context()).setup(*host_matrix(case, seed))
        levels = []
        for l in range(ml.num_levels):
            A, P = ml.level(l)
            levels.append((A.to_csr(), P.to_csr() if P else None, P.n_cols if P else 0))
        ml.free()
        b = np.random.default_rng(seed).standard_normal(n)
        if case["prec"] == 32:
            b = b.astype(np.float32).astype(np.float64)
        return _cycle(levels, 0, b)
    if kind == "galerkin":
        ml = solver(case, context()).setup(*host_matrix(case, seed))
        P = ml.level(0)[1]
        nc, P = P.n_cols, P.to_csr()
        ml.free()
        A = rescaled(host_matrix(case, seed), seed)
        rp, col, val = _product(_transpose(P, nc), _product(A, P, nc), nc)
        # the diagonal first in each row
        row = np.repeat(np.arange(nc), np.diff(rp))
        order = np.lexsort((col, col != row, row))
        return rp, col[order], val[order]
    if kind == "solve":
        return solution(n, seed)
    if kind == "block":
        return solution(n, seed, case["k"])
    if kind == "adjoint":
        rp, col, val = host_matrix(case, seed)
        x, lam = solution(n, seed), solution(n, seed + 1)
        return {"x": x, "dvals": -np.repeat(lam, np.diff(rp)) * x[col], "db": lam}
    return {"x": solution(n, seed), "rows": None, "entries": None}
