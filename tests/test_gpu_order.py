"""Row order of a hierarchy's fine matrix formed on the device (rows sorted,
diagonal first): rows in any order, without a diagonal, with one stored twice,
empty, and unsorted rows up to and past the lengths at which the device changes
its sort (32 entries) and leaves it to the host (2048) give the level that the
host's ordering gives; bad columns and row pointers are refused."""
import numpy as np
import pytest

import raptor_amd as ra

pytestmark = pytest.mark.gpu


def matrix(n, longest, twice, seed):
    rng = np.random.default_rng(seed)
    rp, col, val = [0], [], []
    for i in range(n):
        if i % 97 == 5:
            c = np.array([i])  # a row with its diagonal only
        else:
            k = longest if i == n // 2 else int(rng.integers(1, 12))
            c = np.unique(np.concatenate([rng.integers(0, n, k), [i]]))[: longest]
            if i not in c:
                c[0] = i
                c = np.unique(c)
            if i % 3 != 0:
                rng.shuffle(c)
        v = rng.uniform(-1.0, 0.0, c.size)
        v[c == i] = 20.0 + longest
        if twice and i % 11 == 0:
            c, v = np.append(c, i), np.append(v, 1.0)
        col.append(c)
        val.append(v)
        rp.append(rp[-1] + c.size)
    return np.array(rp, np.int32), np.concatenate(col).astype(np.int32), np.concatenate(val)


@pytest.mark.parametrize("n,longest,twice", [(130, 20, False), (700, 512, False), (700, 513, False), (1500, 700, True),
                                             (200, 32, False), (200, 33, True), (200, 64, False), (200, 65, True)])
def test_fine_level_order(ctx, n, longest, twice):
    M = matrix(n, longest, twice, n + longest)
    got = []
    for device in (True, False):
        ml = ra.ParRugeStubenSolver(ctx, 0.25, ra.PMIS, ra.Direct, ra.Classical, ra.Jacobi)
        ml.device_setup = device
        ml.max_levels = 1
        ml.setup(*M)
        got.append(ml.level(0)[0].to_csr())
        ml.free()
    for a, b in zip(*got):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("n", [100, 30000])  # checked on the host, and on the device (from 131 thousand entries)
def test_bad_input_refused(ctx, n):
    rp, col, val = matrix(n, 10, False, 1)
    assert (col.size > 1 << 17) == (n > 100)
    for c in (-1, n, 2**31 - 1):
        bad = col.copy()
        bad[37] = c
        with pytest.raises(ra.RamdError):
            ra.ParRugeStubenSolver(ctx, 0.25, ra.PMIS, ra.Direct).setup(rp, bad, val)
        with pytest.raises(ra.RamdError):
            ra.ParCSRMatrix.from_csr(ctx, rp, bad, val)
    down = rp.copy()
    down[5], down[6] = rp[6], rp[5]
    with pytest.raises(ra.RamdError):
        ra.ParCSRMatrix.from_csr(ctx, down, col, val)
    for device in (True, False):  # refused on the host: no kernel follows such pointers
        ml = ra.ParRugeStubenSolver(ctx, 0.25, ra.PMIS, ra.Direct)
        ml.device_setup = device
        with pytest.raises(ra.RamdError, match="rowptr decreases"):
            ml.setup(down, col, val)


@pytest.mark.parametrize("order", ["shuffled", "descending"])
@pytest.mark.parametrize("length", [31, 32, 33, 63, 64, 65, 300, 2047, 2048, 2049])
@pytest.mark.parametrize("diagonals", [0, 1, 2])
def test_one_long_row_each_way(ctx, length, order, diagonals):
    """Rows of one length, repeated columns among them, with no diagonal, one
    and two: the entries in the host's stable order."""
    n = 500
    rng = np.random.default_rng(length + diagonals)
    rp, col, val = [0], [], []
    for i in range(n):
        if i % 61 == 7:
            c = rng.choice(np.delete(np.arange(n), i), length - diagonals)
            c[: length // 8] = c[length // 8: 2 * (length // 8)]  # some at least twice
            c = np.concatenate([c, np.full(diagonals, i)])
            c = rng.permutation(c) if order == "shuffled" else -np.sort(-c)
        else:
            c = np.array([i])
        col.append(c)
        val.append(rng.uniform(1.0, 2.0, c.size))
        rp.append(rp[-1] + c.size)
    M = np.array(rp, np.int32), np.concatenate(col).astype(np.int32), np.concatenate(val)
    got = []
    for device in (True, False):
        ml = ra.ParRugeStubenSolver(ctx, 0.25, ra.PMIS, ra.Direct, ra.Classical, ra.Jacobi)
        ml.device_setup = device
        ml.max_levels = 1
        ml.setup(*M)
        got.append(ml.level(0)[0].to_csr())
        ml.free()
    for a, b in zip(*got):
        assert np.array_equal(a, b)
