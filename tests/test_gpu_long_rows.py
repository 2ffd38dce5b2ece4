"""CSR kernels of blocks with more than 7.5 entries per row on average (tiles
split by entries instead of rows): bitwise the oracle's row sums at the
edges of the 2,048-entry segments, in every kernel that walks such tiles."""
import numpy as np
import pytest

import oracle as O
from helpers import random_csr, stencil27

pytestmark = pytest.mark.gpu


def uniform(n, k, rng):
    """n rows of exactly k entries."""
    cols = np.concatenate([np.sort(rng.choice(n, size=k, replace=False)) + 1 for _ in range(n)])
    return O.CSR(np.arange(n + 1) * k + 1, cols, rng.normal(size=n * k))


def cases():
    rng = np.random.default_rng(71)
    # one row over three segments, every other row empty
    lens = np.zeros(600, dtype=np.int64)
    lens[257] = 5000
    one = O.CSR(np.concatenate([[1], 1 + np.cumsum(lens)]), np.sort(rng.choice(6000, 5000, replace=False)) + 1,
                rng.normal(size=5000))
    return [
        ("k8_one_segment", uniform(256, 8, rng), None),        # 2,048 entries: one segment to its end
        ("k16_two_segments", uniform(512, 16, rng), None),     # segments end on row ends
        ("k9_odd", uniform(257, 9, rng), None),                # 2,304 entries, then a tile of one row
        ("ragged_24", random_csr(1021, 1021, 12, rng, empty_every=5), None),
        ("long_rows", random_csr(513, 513, 9, rng, long_rows=(0, 255, 256, 512)), None),
        ("one_row", O.CSR(np.array([1, 10]), np.arange(1, 10), rng.normal(size=9)), 9),
        ("one_long_row", one, 6000),
    ]


CASES = cases()


@pytest.mark.parametrize("name,A,ncols", CASES, ids=[c[0] for c in CASES])
def test_products_bitwise(gpu, name, A, ncols):
    assert A.nnz > 7.5 * A.n
    nc = A.n if ncols is None else ncols
    M = gpu.Matrix.from_csr(A.xadj, A.cols, A.vals, ncols=nc, index_base=1)
    rng = np.random.default_rng(5)
    x, y0 = rng.normal(size=nc), rng.normal(size=A.n)
    rows = np.repeat(np.arange(1, A.n + 1), np.diff(A.xadj))
    # the row sums entry by entry, every product rounded before its add
    def ref(dt, start):
        y = start.astype(dt)
        for i, c, v in zip(rows - 1, A.cols - 1, A.vals.astype(dt)):
            y[i] = y[i] + dt(v) * x.astype(dt)[c] if dt is np.float32 else y[i] + v * x[c]
        return y
    r64 = ref(np.float64, np.zeros(A.n))
    np.testing.assert_array_equal(M.spmv(x), r64)
    np.testing.assert_array_equal(M.spmv(x, y0, accumulate=True), y0 + r64)
    np.testing.assert_array_equal(M.spmv(x, y0, fmt=gpu.FMT_COO, accumulate=True), ref(np.float64, y0))
    np.testing.assert_array_equal(M.spmv_f32(x.astype(np.float32)), O.spmv_csr_f32(A, x.astype(np.float32))
                                  if ncols is None else ref(np.float32, np.zeros(A.n)))
    if nc == A.n:
        y, dot = M.spmv_dot(x)
        np.testing.assert_array_equal(y, r64)
        assert abs(dot - np.dot(x, r64)) <= 1e-12 * np.dot(np.abs(x), np.abs(r64))


def test_gmres_product_and_residual_bitwise_across_forms(gpu):
    """The fused products of the GMRES cycle: CSR against JAD, whose product and
    dot products are separate kernels, bit for bit."""
    A = stencil27(11, 9, 10)
    b = np.random.default_rng(6).normal(size=A.shape[0])
    out = []
    for fmt in (gpu.FMT_CSR, gpu.FMT_JAD):
        M = gpu.Matrix.from_csr(A.indptr, A.indices, A.data, index_base=0)
        M.set_jacobi()
        M.to_jad()
        out.append(M.gmres(b, restart=3, iter_max=6, eps=1e-8, fmt=fmt))
    assert out[0]["iters"] == out[1]["iters"]
    np.testing.assert_array_equal(out[0]["x"], out[1]["x"])
