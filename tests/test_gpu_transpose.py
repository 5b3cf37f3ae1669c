"""The device transpose at its edges: columns of 0 to 2049 entries (in a thread's
registers up to 16, else 4, 16 and 64 lanes per column, the longest sorted on
the host) and rows that store a column twice.  A^T x adds each column's products
in ascending row order, so the bits follow the order."""
import numpy as np
import pytest

import checkers as K
import raptor_amd as ra

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,cols,avg,longest,twice", [
    (3000, 900, 3, 15, False), (3000, 900, 5, 16, False), (3000, 900, 5, 17, False), (3000, 900, 4, 9, True),
    (400, 300, 1, 1, False), (3000, 900, 3, 40, False), (3000, 900, 11, 30, True), (2000, 333, 12, 17, False), (2000, 333, 31, 64, True),
    (5000, 70, 40, 65, False), (5000, 70, 200, 600, True), (2100, 5, 1000, 2048, False), (2100, 5, 1000, 2049, False)])
def test_transpose_order_bit_exact(ctx, rows, cols, avg, longest, twice):
    rng = np.random.default_rng(rows + cols + avg)
    r, c = [], []
    for j in range(cols):
        k = longest if j == cols // 2 else int(rng.integers(0, 2 * avg + 1)) % (longest + 1)
        r.append(np.sort(rng.choice(rows, k, replace=False)))
        c.append(np.full(k, j))
    r, c = np.concatenate(r), np.concatenate(c)
    if twice:
        again = rng.choice(r.size, r.size // 10, replace=False)
        r, c = np.concatenate([r, r[again]]), np.concatenate([c, c[again]])
    order = np.lexsort((rng.random(r.size), r))  # columns of a row in any order
    r, c = r[order], c[order]
    rp = np.concatenate([[0], np.cumsum(np.bincount(r, minlength=rows))]).astype(np.int32)
    A = K.Csr(rp, c.astype(np.int32), rng.standard_normal(r.size), cols)
    D = ra.ParCSRMatrix.from_csr(ctx, A.rowptr, A.col, A.val, cols)
    x = rng.standard_normal(rows)
    y = ra.ParVector(ctx, cols)
    D.mult_T(ra.ParVector.from_numpy(ctx, x), y)
    assert np.array_equal(y.numpy(), K.spmv_t(A, x))
