"""PCG on matrices of short rows with a few long ones, on either side of the
longest row (24 entries) from which those are loaded several entries at a
time: six iterations against the same recurrence in numpy, rows that end
inside a group of eight loads and tiles larger than the LDS stage among
them, for matrices whose longest row the library knows from its host arrays
and for assembled ones, where it looks it up."""
import numpy as np
import pytest
import scipy.sparse as sp

from test_gpu_keep import close, run, six_iterations

pytestmark = pytest.mark.gpu


def with_long_rows(n, longest, rng):
    """Symmetric, diagonally dominant: about 5 entries a row; every 997th row
    has about `longest` entries."""
    i = np.arange(n)
    rows, cols = [i, i], [(i + 1) % n, (i + 13) % n]
    for r in range(5, n, 997):
        k = max(longest - 5, 0)
        rows.append(np.full(k, r))
        cols.append(rng.choice(n, size=k, replace=False))
    rows, cols = np.concatenate(rows), np.concatenate(cols)
    A = sp.coo_matrix((-0.5 - rng.random(rows.size), (rows, cols)), shape=(n, n)).tocsr()
    A = A + A.T
    A.setdiag(0)
    A.eliminate_zeros()
    A = (A + sp.diags(1.0 - np.asarray(A.sum(1)).ravel())).tocsr()
    A.sort_indices()
    return A


@pytest.mark.parametrize("prec", ["fp64", "mixed"])
@pytest.mark.parametrize("n,longest", [(3001, 5), (3001, 23), (3001, 27), (30011, 33), (30011, 3000),
                                       (150001, 64), (400009, 1000), (3000017, 40)])
def test_few_long_rows(gpu, n, longest, prec):
    rng = np.random.default_rng(n + longest)
    A = with_long_rows(n, longest, rng)
    M = gpu.Matrix.from_csr(A.indptr, A.indices, A.data, index_base=0)
    M.set_jacobi()
    b = rng.normal(size=n)
    ref = six_iterations(A, M.jacobi(), b)
    x = run(gpu, M, b, gpu.FMT_CSR, prec)
    close(x, ref, prec)
    np.testing.assert_array_equal(run(gpu, M, b, gpu.FMT_COO, prec), x)
    if n < 100000:
        rows = np.repeat(np.arange(n), np.diff(A.indptr))
        p = rng.permutation(A.nnz)
        N = gpu.Matrix.from_coo_sorted(n, rows[p], A.indices[p], A.data[p], index_base=0, mode=gpu.SORT_ROW_COL)
        N.set_jacobi()
        np.testing.assert_array_equal(run(gpu, N, b, gpu.FMT_CSR, prec), x)
