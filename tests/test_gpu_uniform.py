"""Operators with one value per diagonal: the kernels that read no values give
the oracle's bits on 27- and 7-point grids whose lines are multiples of 64, 32,
16 or of none, with fewer planes than a workgroup walks and more, in ascending
order and diagonal first; one changed value turns them off and back on."""
import numpy as np
import pytest

import checkers as K
import raptor_amd as ra

pytestmark = pytest.mark.gpu


def grid(nx, ny, nz, pts, seed=1):
    """27- or 7-point operator on nx x ny x nz with one random value per offset."""
    rng = np.random.default_rng(seed)
    i, j, k = np.meshgrid(np.arange(nx), np.arange(ny), np.arange(nz), indexing="ij")
    i, j, k = [t.transpose(2, 1, 0).ravel() for t in (i, j, k)]  # x fastest
    row = np.arange(nx * ny * nz)
    rows, cols, vals = [], [], []
    for dz in (-1, 0, 1):
        for dy in (-1, 0, 1):
            for dx in (-1, 0, 1):
                if pts == 7 and abs(dx) + abs(dy) + abs(dz) > 1:
                    continue
                ok = (0 <= i + dx) & (i + dx < nx) & (0 <= j + dy) & (j + dy < ny) & (0 <= k + dz) & (k + dz < nz)
                rows.append(row[ok])
                cols.append((row + dx + nx * dy + nx * ny * dz)[ok])
                v = rng.standard_normal() + (30.0 if dx == dy == dz == 0 else 0.0)
                vals.append(np.full(int(ok.sum()), np.float64(np.float32(v)) if seed % 2 else v))
    rows, cols, vals = np.concatenate(rows), np.concatenate(cols), np.concatenate(vals)
    order = np.lexsort((cols, rows))
    rp = np.concatenate([[0], np.cumsum(np.bincount(rows, minlength=row.size))])
    return K.Csr(rp.astype(np.int32), cols[order].astype(np.int32), vals[order])


def check(ctx, D, A, seed=3):
    rng = np.random.default_rng(seed)
    n = A.n_rows
    x, b = rng.standard_normal(n), rng.standard_normal(n)
    x[::5], b[::3] = -0.0, -0.0
    y = ra.ParVector(ctx, n)

    def dev(a):
        return ra.ParVector.from_numpy(ctx, a)

    def same(got, want):
        # the sign of zero too (a NaN's sign and payload are the hardware's)
        got, want = [np.where(np.isnan(t), np.nan, t).view(np.int64) for t in (got, want)]
        assert np.array_equal(got, want)

    D.mult(dev(x), y)
    same(y.numpy(), K.spmv(A, x))
    D.residual(dev(x), dev(b), y)
    same(y.numpy(), K.residual(A, x, b))
    same_b = dev(b)
    D.mult_append(dev(x), same_b)
    same(same_b.numpy(), K.spmv_append(A, x, b))
    xj = dev(x)
    D.jacobi(xj, dev(b), ra.ParVector(ctx, n), 2, 2.0 / 3.0)
    same(xj.numpy(), K.jacobi(A, x, b, 2, 2.0 / 3.0))


@pytest.mark.parametrize("pts", [27, 7])
@pytest.mark.parametrize("dims", [(16, 16, 16), (32, 16, 17), (64, 15, 16), (65, 18, 14), (17, 19, 23), (128, 14, 13)])
@pytest.mark.parametrize("diag_first", [False, True])
def test_uniform_operator_bit_exact(ctx, dims, pts, diag_first):
    A = grid(*dims, pts, seed=sum(dims))
    if diag_first:
        A = K.move_diag(A)
    D = ra.ParCSRMatrix.from_csr(ctx, A.rowptr, A.col, A.val)
    assert D.diagonals() == pts and D.uniform()
    check(ctx, D, A)  # the rule's choice
    for mode, planes in ((0, 0), (2, 4), (2, 5), (2, 16)):
        for pp in (0, 2):
            D.set_dia_staging(pp, mode, planes)
        check(ctx, D, A)


@pytest.mark.parametrize("what", ["one value", "signed zero", "nan"])
def test_value_changes_turn_it_off_and_on(ctx, what):
    A = grid(17, 16, 18, 27, seed=8)
    D = ra.ParCSRMatrix.from_csr(ctx, A.rowptr, A.col, A.val)
    v = A.val.copy()
    off = np.flatnonzero(A.col != np.repeat(np.arange(A.n_rows), np.diff(A.rowptr)))
    if what == "signed zero":
        d = A.col - np.repeat(np.arange(A.n_rows), np.diff(A.rowptr))
        v[d == 1] = 0.0
        v[np.flatnonzero(d == 1)[-1]] = -0.0
    else:
        v[off[-1]] = np.nan if what == "nan" else np.nextafter(v[off[-1]], 9.0)
    D.set_values(ra.ParVector.from_numpy(ctx, v))
    assert not D.uniform()
    check(ctx, D, K.Csr(A.rowptr, A.col, v))
    D.set_values(ra.ParVector.from_numpy(ctx, 2.0 * A.val))
    assert D.uniform()
    check(ctx, D, K.Csr(A.rowptr, A.col, 2.0 * A.val))


@pytest.mark.parametrize("dims,pts", [((58, 58, 58), 27), ((60, 58, 58), 27), ((82, 83, 83), 7), ((84, 85, 81), 7),
                                      ((3, 700, 300), 7)])
def test_both_sides_of_the_untimed_rule(ctx, dims, pts):
    """The largest grids that the gather takes before any timing, the smallest
    that the plane march takes, and one whose tiles are a fifth full."""
    A = grid(*dims, pts, seed=5)
    D = ra.ParCSRMatrix.from_csr(ctx, A.rowptr, A.col, A.val)
    assert D.uniform() and D.dia_staging(0)[0] == -1
    check(ctx, D, A)


def test_small_operators_are_timed_against_the_gather(ctx):
    """On 20 x 20 x 20 the march takes 9 us and the gather 5: a solve's timing
    sees both."""
    A = grid(20, 20, 20, 27, seed=5)
    A.val[:] = np.where(A.col == np.repeat(np.arange(A.n_rows), np.diff(A.rowptr)), 26.5, -1.0)
    ml = ra.ParRugeStubenSolver(ctx, 0.25, ra.PMIS, ra.Extended, ra.Classical, ra.Jacobi)
    ml.relax_weight = 2.0 / 3.0
    ml.setup(A.rowptr, A.col, A.val)
    D = ra.ParCSRMatrix.from_csr(ctx, A.rowptr, A.col, A.val)
    b = ra.ParVector.from_numpy(ctx, np.random.default_rng(1).standard_normal(A.n_rows))
    ra.FPCG(D, ml, ra.ParVector.from_numpy(ctx, np.zeros(A.n_rows)), b, 1e-8, 100, ra.PREC_FP32)
    assert D.uniform() and ml.level(0)[0].uniform()
    assert D.dia_staging(2)[0] in (0, 1)
    assert ml.level(0)[0].dia_staging(1)[0] in (0, 1)
    ml.free()


@pytest.mark.parametrize("prec", [ra.PREC_FP64, ra.PREC_FP32])
@pytest.mark.parametrize("block", [False, True])
def test_replayed_solves_follow_new_values(ctx, prec, block):
    """One capture serves every constant-coefficient operator: scaled values
    between replayed solves give the eager solves' bits, and so do values that
    are not uniform and uniform ones again."""
    A = grid(65, 64, 66, 27, seed=5)  # past the size from which the march is taken
    diag = A.col == np.repeat(np.arange(A.n_rows), np.diff(A.rowptr))
    A.val[:] = np.where(diag, 26.5, -1.0)
    ml = ra.ParRugeStubenSolver(ctx, 0.25, ra.PMIS, ra.Extended, ra.Classical, ra.Jacobi)
    ml.relax_weight = 2.0 / 3.0
    ml.setup(A.rowptr, A.col, A.val)
    D = ra.ParCSRMatrix.from_csr(ctx, A.rowptr, A.col, A.val)
    n, k = A.n_rows, 2
    b = np.random.default_rng(1).standard_normal((n, k) if block else n)

    def solve(graphs):
        x = ra.ParVector.from_numpy(ctx, np.zeros(b.size))
        if block:
            ra.FPCG_block(D, ml, x, ra.ParVector.from_numpy(ctx, b.ravel()), k, 1e-8, 100, prec, graphs)
        else:
            ctx.set_graphs(graphs)
            ra.FPCG(D, ml, x, ra.ParVector.from_numpy(ctx, b), 1e-8, 100, prec)
            ctx.set_graphs(False)
        return x.numpy()

    seen = []
    for step in range(6):
        v = A.val * (1.0 + step)
        if step == 3:
            v[diag] += np.linspace(0.0, 0.1, n)
        D.set_values(ra.ParVector.from_numpy(ctx, v))
        assert D.uniform() == (step != 3)
        got = solve(True)
        assert np.array_equal(got, solve(False)), step
        x = got.reshape(n, -1)[:, 0]
        res = b.reshape(n, -1)[:, 0] - K.spmv(K.Csr(A.rowptr, A.col, v), np.ascontiguousarray(x))
        assert np.linalg.norm(res) <= 2e-8 * np.linalg.norm(b.reshape(n, -1)[:, 0])
        seen.append(got)
    assert not any(np.array_equal(seen[0], s) for s in seen[1:])
    ml.free()


def test_choices_follow_the_kind_of_values(ctx):
    """The timed kernel choice of a uniform operator and that of the same
    operator with other values are kept apart, a forced one holds for both, and
    the solve without allocations runs on a kind of values not timed yet."""
    A = grid(33, 32, 34, 27, seed=5)
    diag = A.col == np.repeat(np.arange(A.n_rows), np.diff(A.rowptr))
    A.val[:] = np.where(diag, 26.5, -1.0)
    n = A.n_rows
    other = A.val + np.where(diag, np.float64(np.float32(np.linspace(0.0, 0.5, A.val.size))), 0.0)
    ml = ra.ParRugeStubenSolver(ctx, 0.25, ra.PMIS, ra.Extended, ra.Classical, ra.Jacobi)
    ml.relax_weight = 2.0 / 3.0
    ml.setup(A.rowptr, A.col, A.val)
    D = ra.ParCSRMatrix.from_csr(ctx, A.rowptr, A.col, A.val)
    b = np.random.default_rng(1).standard_normal(n)

    def solve(f):
        x = ra.ParVector.from_numpy(ctx, np.zeros(n))
        f(D, ml, x, ra.ParVector.from_numpy(ctx, b), 1e-8, 100, ra.PREC_FP32)
        return x.numpy()

    def values(v):
        D.set_values(ra.ParVector.from_numpy(ctx, v))

    solve(ra.FPCG)
    first = D.dia_staging(2)
    assert first[0] >= 0
    values(other)
    assert not D.uniform() and D.dia_staging(2)[0] == -1
    assert D.dia_tile() == 64  # lines of 33: no narrower tile divides them
    x = solve(ra.FPCG_noalloc)
    assert np.linalg.norm(b - K.spmv(K.Csr(A.rowptr, A.col, other), x)) <= 2e-8 * np.linalg.norm(b)
    solve(ra.FPCG)
    second = D.dia_staging(2)
    assert second[0] >= 0
    values(3.0 * A.val)
    assert D.uniform() and D.dia_staging(2) == first
    assert D.dia_tile() == 16  # the fewest positions past the grid
    values(other)
    assert D.dia_staging(2) == second
    D.set_dia_staging(2, 2, 5)
    for v in (A.val, other, A.val):
        values(v)
        solve(ra.FPCG)
        assert D.dia_staging(2)[:2] == (2, 5)
    ml.free()
