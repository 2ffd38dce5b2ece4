"""Device memory reused from call to call: results stay bitwise right when
blocks come back of other sizes and with other contents, with matrices
destroyed and rebuilt in between, and after the library gave everything back."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu


def test_reused_blocks_keep_results(gpu):
    rng = np.random.default_rng(51)
    shapes = [(9, 8, 7), (31, 17, 65), (64, 64, 64), (33, 17, 9), (60, 64, 66), (9, 8, 7)]
    for again in range(3):
        for k, shape in enumerate(shapes):
            A = O.gen_poisson7(*shape)
            n = int(np.prod(shape))
            M = gpu.Matrix.poisson7(*shape)
            M.set_jacobi()
            M.to_dia()
            M.to_jad()
            x = rng.normal(size=n)
            ref = O.spmv_csr(A, x)
            for fmt in (gpu.FMT_CSR, gpu.FMT_DIA, gpu.FMT_JAD):
                np.testing.assert_array_equal(M.spmv(x, fmt=fmt), ref)
            rows = np.repeat(np.arange(1, n + 1), np.diff(A.xadj))
            order = rng.permutation(rows.size)
            B = gpu.Matrix.from_coo_sorted(n, rows[order], A.cols[order], A.vals[order], mode=gpu.SORT_ROW_COL)
            M.destroy()
            np.testing.assert_array_equal(B.spmv(x), ref)
            if k % 2:
                B.destroy()
        if again == 1:
            assert gpu.lib().cel_gpu_finalize() == 0
            gpu.init()
