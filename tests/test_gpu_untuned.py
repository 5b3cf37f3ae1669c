"""A matrix that no tuner has seen: on both sides of the sizes between which its
entries are read through the caches (24 to 96 MB of them, 50 with a cycle
between the products), with empty rows and rows past one workgroup's products,
every operation gives the oracle's bits, and a preconditioned solve does on
either path."""
import numpy as np
import pytest

import checkers as K
import raptor_amd as ra

pytestmark = pytest.mark.gpu


def matrix(entries, seed):
    """Unsymmetric rows of 0 to 34 entries near the diagonal, two of them with
    5000; every third row without a diagonal."""
    rng = np.random.default_rng(seed)
    n = entries // 17
    length = rng.integers(0, 35, n)
    length[[3, n // 2]] = 5000
    row = np.repeat(np.arange(n, dtype=np.int64), length)
    col = (row + rng.integers(-3000, 3001, row.size)) % n
    diag = np.arange(n, dtype=np.int64)[np.arange(n) % 3 != 0]
    key = np.unique(np.concatenate([row * n + col, diag * (n + 1)]))
    row, col = key // n, key % n
    rp = np.concatenate([[0], np.cumsum(np.bincount(row, minlength=n))]).astype(np.int32)
    return K.Csr(rp, col.astype(np.int32), rng.standard_normal(col.size))


@pytest.mark.parametrize("entries", [500_000, 1_950_000, 2_200_000, 7_500_000, 8_800_000])
def test_operations_bit_exact(ctx, entries):
    A = matrix(entries, entries)
    n = A.n_rows
    D = ra.ParCSRMatrix.from_csr(ctx, A.rowptr, A.col, A.val)
    assert not D.diagonals()
    rng = np.random.default_rng(1)
    x, b = rng.standard_normal(n), rng.standard_normal(n)

    def dev(a):
        return ra.ParVector.from_numpy(ctx, a)

    y = ra.ParVector(ctx, n)
    D.mult(dev(x), y)
    assert np.array_equal(y.numpy(), K.spmv(A, x))
    D.residual(dev(x), dev(b), y)
    assert np.array_equal(y.numpy(), K.residual(A, x, b))
    t = dev(b)
    D.mult_append(dev(x), t)
    assert np.array_equal(t.numpy(), K.spmv_append(A, x, b))
    t = dev(x)
    D.jacobi(t, dev(b), ra.ParVector(ctx, n), 2, 2.0 / 3.0)
    assert np.array_equal(t.numpy(), K.jacobi(A, x, b, 2, 2.0 / 3.0))
    D.mult_T(dev(x), y)
    assert np.array_equal(y.numpy(), K.spmv_t(A, x))
    D.free()


@pytest.mark.parametrize("m", [46, 56])  # 2.5 and 4.6 million entries
def test_solve_operator_outside_and_inside(ctx, m):
    """The 27-point operator in CSR form (rows shuffled in groups of 64): its
    products before, during and after preconditioned solves."""
    rp, col, val = ra.gallery_laplace27(m)
    n = rp.size - 1
    rng = np.random.default_rng(m)
    q = np.arange(n)
    for s in range(0, n, 64):
        rng.shuffle(q[s:s + 64])
    at = np.empty(n, np.int64)
    at[q] = np.arange(n)
    row = at[np.repeat(np.arange(n), np.diff(rp))]
    order = np.lexsort((at[col], row))
    rp = np.concatenate([[0], np.cumsum(np.bincount(row, minlength=n))]).astype(np.int32)
    A = K.Csr(rp, at[col][order].astype(np.int32), val[order])
    D = ra.ParCSRMatrix.from_csr(ctx, A.rowptr, A.col, A.val)
    assert not D.diagonals()
    ml = ra.ParRugeStubenSolver(ctx, 0.25, ra.PMIS, ra.Extended, ra.Classical, ra.Jacobi)
    ml.relax_weight = 2.0 / 3.0
    ml.setup(A.rowptr, A.col, A.val)
    x, b = rng.standard_normal(n), rng.standard_normal(n)

    def product():
        y = ra.ParVector(ctx, n)
        D.mult(ra.ParVector.from_numpy(ctx, x), y)
        return y.numpy()

    want = K.spmv(A, x)
    assert np.array_equal(product(), want)
    seen = {}
    for graphs in (False, True):
        ctx.set_graphs(graphs)
        for prec in (ra.PREC_FP64, ra.PREC_FP32):
            u = ra.ParVector.from_numpy(ctx, np.zeros(n))
            ra.FPCG(D, ml, u, ra.ParVector.from_numpy(ctx, b), 1e-8, 100, prec)
            assert np.linalg.norm(K.residual(A, u.numpy(), b)) <= 1.001e-8 * np.linalg.norm(b)
            assert np.array_equal(seen.setdefault(prec, u.numpy()), u.numpy())
        ctx.set_graphs(False)
        assert np.array_equal(product(), want)
    seen = []
    for _ in range(2):  # PCG and BiCGStab: the same bits again after the scope's end
        u = ra.ParVector.from_numpy(ctx, np.zeros(n))
        ra.PCG(D, ml, u, ra.ParVector.from_numpy(ctx, b), tol=1e-8)
        v = ra.ParVector.from_numpy(ctx, np.zeros(n))
        ra.Pre_BiCGStab(D, v, ra.ParVector.from_numpy(ctx, b), ml, tol=1e-8)
        assert np.array_equal(product(), want)
        seen.append((u.numpy(), v.numpy()))
    assert np.array_equal(seen[0][0], seen[1][0]) and np.array_equal(seen[0][1], seen[1][1])
    assert np.isfinite(seen[0][0]).all() and np.isfinite(seen[0][1]).all()
    ml.free()
