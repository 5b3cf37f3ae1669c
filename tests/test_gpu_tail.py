"""The coarse tail's packed matrices and operation list at their edges: level
sizes around a slice of 64 rows, coarse systems from 1 to 64 rows (the LU's
steps of four), rows of one entry and rows past one step of eight, sweep
counts 0 to 2, each start level, both precisions -- every cycle bit for bit
the one with a launch per operation."""
import numpy as np
import pytest

import raptor_amd as ra

pytestmark = pytest.mark.gpu


def laplace_1d(n, wide=1):
    """Symmetric diagonally dominant band matrix of 2 * wide + 1 diagonals."""
    rng = np.random.default_rng(n + wide)
    d = np.zeros((n, n))
    for k in range(1, min(wide, n - 1) + 1):
        off = -rng.uniform(0.5, 1.5, n - k)
        d += np.diag(off, k) + np.diag(off, -k)
    d += np.diag(1.001 * np.abs(d).sum(axis=1) + 0.01)
    rp = np.concatenate([[0], np.cumsum((d != 0).sum(axis=1))])
    return rp.astype(np.int32), np.nonzero(d)[1].astype(np.int32), d[d != 0]


@pytest.mark.parametrize("sweeps", [0, 1, 2])
@pytest.mark.parametrize("n,wide,max_coarse", [(129, 1, 64), (130, 1, 33), (131, 9, 20), (257, 1, 1), (500, 4, 63),
                                               (1000, 17, 64), (2100, 1, 40)])
def test_tail_levels_bit_exact(ctx, n, wide, max_coarse, sweeps):
    ml = ra.ParRugeStubenSolver(ctx, 0.25, ra.PMIS, ra.Direct, ra.Classical, ra.Jacobi)
    ml.relax_weight = 2.0 / 3.0
    ml.max_coarse = max_coarse
    ml.num_smooth_sweeps = sweeps
    ml.setup(*laplace_1d(n, wide))
    ml.enable_fp32()
    _, first = ml.tail_level()
    assert first >= 1
    b = np.random.default_rng(n).standard_normal(n)
    b[::7] = 0.0  # exact zeros reach the coarse levels too
    out = {}
    for mode in [-1] + list(range(first, ml.num_levels)):
        ml.set_tail(mode)
        x = ra.ParVector.from_numpy(ctx, np.full(n, 3.0))
        ml.cycle(x, ra.ParVector.from_numpy(ctx, b), x_is_zero=True)
        x32 = ra.ParVector.from_numpy(ctx, np.full(n, 3.0, np.float32))
        ml.cycle_fp32(x32, ra.ParVector.from_numpy(ctx, b.astype(np.float32)))
        out[mode] = (x.numpy(), x32.numpy())
        assert np.isfinite(out[mode][0]).all()
    for mode in out:
        assert np.array_equal(out[mode][0], out[-1][0]), mode
        assert np.array_equal(out[mode][1], out[-1][1]), mode
    ml.free()


@pytest.mark.parametrize("first", ["cycle_fp32", "fpcg", "block"])
def test_fp32_enabled_while_tracking(ctx, first):
    """FP32 levels made while per-level timing is on have their tail as well:
    with timing off again, the cycles with every tail run, and equal the one
    without."""
    n = 1000
    M = laplace_1d(n, 17)
    ml = ra.ParRugeStubenSolver(ctx, 0.25, ra.PMIS, ra.Direct, ra.Classical, ra.Jacobi)
    ml.relax_weight = 2.0 / 3.0
    ml.setup(*M)
    A = ra.ParCSRMatrix.from_csr(ctx, *M)
    b = np.random.default_rng(n).standard_normal(n)

    def cycle():
        x = ra.ParVector(ctx, n, np.float32)
        ml.cycle_fp32(x, ra.ParVector.from_numpy(ctx, b.astype(np.float32)))
        return x.numpy()

    ml.set_track_times(True)
    if first == "cycle_fp32":
        cycle()
    elif first == "fpcg":
        ra.FPCG(A, ml, ra.ParVector.from_numpy(ctx, np.zeros(n)), ra.ParVector.from_numpy(ctx, b), 1e-8, 100,
                ra.PREC_FP32)
    else:
        X = ra.ParVector(ctx, 2 * n, np.float32)
        ra.vcycle_block(ml, X, ra.ParVector.from_numpy(ctx, np.repeat(b, 2).astype(np.float32)), 2, ra.PREC_FP32)
    ml.set_track_times(False)
    ml.set_tail(-1)
    want = cycle()
    _, start = ml.tail_level(ra.PREC_FP32)
    assert start >= 1
    for mode in [0] + list(range(start, ml.num_levels)):
        ml.set_tail(mode)
        assert np.array_equal(cycle(), want), mode
    ml.free()


def band(n, wide):
    """laplace_1d's matrix without its dense form, constant coefficients."""
    k = np.arange(-wide, wide + 1)
    col = np.arange(n)[:, None] + k
    ok = (col >= 0) & (col < n)
    val = np.where(k == 0, 2.001 * wide, -1.0) + np.zeros(col.shape)
    rp = np.concatenate([[0], np.cumsum(ok.sum(axis=1))])
    return rp.astype(np.int32), col[ok].astype(np.int32), val[ok]


@pytest.mark.parametrize("n,accepted", [(4000, True), (8190, True), (8191, True), (8192, True), (8193, False)])
def test_set_tail_by_sizes(ctx, n, accepted):
    """A start that its sizes allow is taken whether or not its packed form
    fits; the tail then starts below it, with the bits of no tail."""
    ml = ra.ParRugeStubenSolver(ctx, 0.25, ra.PMIS, ra.Direct, ra.Classical, ra.Jacobi)
    ml.relax_weight = 2.0 / 3.0
    ml.setup(*band(n, 9))
    rows, nnz, nnz_p = ml.level_sizes()
    assert rows[1] <= 2048 and nnz[1] <= 32768 and nnz_p[0] <= 65536 and rows[-1] <= 64 and ml.num_levels >= 3
    ml.enable_fp32()
    _, first = ml.tail_level()
    assert first >= 2 or n <= 8190
    b = np.random.default_rng(n).standard_normal(n)

    def cycles():
        x = ra.ParVector(ctx, n)
        ml.cycle(x, ra.ParVector.from_numpy(ctx, b), x_is_zero=True)
        x32 = ra.ParVector(ctx, n, np.float32)
        ml.cycle_fp32(x32, ra.ParVector.from_numpy(ctx, b.astype(np.float32)))
        return x.numpy(), x32.numpy()

    ml.set_tail(-1)
    want = cycles()
    if accepted:
        ml.set_tail(1)
        assert ml.tail_level()[0] == first
        got = cycles()
        assert np.array_equal(got[0], want[0]) and np.array_equal(got[1], want[1])
    else:
        with pytest.raises(ra.RamdError):
            ml.set_tail(1)
    ml.set_track_times(True)
    with pytest.raises(ra.RamdError):
        ml.set_tail(1)
    ml.set_track_times(False)
    for level in (-2, ml.num_levels):
        with pytest.raises(ra.RamdError):
            ml.set_tail(level)
    ml.free()
