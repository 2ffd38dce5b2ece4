"""CSR and COO products of blocks with short rows on either side of the sizes
up to which every row is read by a thread of its own (200,000 rows in FP64,
300,000 in FP32), against the oracle: bit for bit."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu


def ragged(n, m, rng):
    """Rows of 0 to 14 entries, 6 on average, in random column order."""
    cnt = np.minimum(rng.integers(0, 13, n), rng.integers(4, 15, n))
    xadj = np.concatenate([[0], np.cumsum(cnt)])
    cols = rng.integers(0, m, xadj[-1])
    return xadj, cols, rng.normal(size=xadj[-1])


@pytest.mark.parametrize("n,m", [(1, 3), (255, 1), (257, 5000), (60000, 7), (199999, 200001), (200001, 1000),
                                 (299999, 300000), (300001, 299999)])
def test_short_rows(gpu, n, m):
    rng = np.random.default_rng(71 + n)
    xadj, cols, vals = ragged(n, m, rng)
    if xadj[-1] == 0:
        xadj, cols, vals = np.arange(n + 1), np.zeros(n, dtype=np.int64), np.ones(n)
    A = O.CSR(xadj + 1, cols + 1, vals)
    M = gpu.Matrix.from_csr(xadj, cols, vals, ncols=m, index_base=0)
    x, y = rng.normal(size=m), rng.normal(size=n)
    np.testing.assert_array_equal(M.spmv(x), O.spmv_csr(A, x))
    np.testing.assert_array_equal(M.spmv(x, y, accumulate=True), O.spmv_csr(A, x, y.copy()))
    np.testing.assert_array_equal(M.spmv_f32(x), O.spmv_csr_f32(A, x.astype(np.float32)))
    rows = np.repeat(np.arange(n), np.diff(xadj))
    for acc in (False, True):
        got = M.spmv(x, y, fmt=gpu.FMT_COO, accumulate=acc)
        ref = O.spmv_coo(rows + 1, cols + 1, vals, 0, 0, x, y.copy() if acc else np.zeros(n))
        np.testing.assert_array_equal(got, ref)
