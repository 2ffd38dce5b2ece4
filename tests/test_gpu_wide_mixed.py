"""Mixed solves in the caller's diagonal storage on either side of the row count
from which symmetric values are read by the wide walk instead of the
two-kernel iteration: against the entry-by-entry walk, bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(95, 94, 93), (97, 96, 95), (109, 108, 107)])
def test_own_diagonals(gpu, shape):
    rng = np.random.default_rng(7)
    n = int(np.prod(shape))
    M = gpu.Matrix.diffusion7(*shape, np.exp(rng.normal(0.0, 0.5, n)))
    M.set_jacobi()
    M.to_dia()
    b = rng.normal(size=n)
    kw = dict(precision=gpu.PREC_MIXED, tol=1e-300, tol_mode=gpu.TOL_REL_B, alpha_stop=0, iter_max=40)
    ref = M.pcg(b, fmt=gpu.FMT_COO, **kw)
    for _ in range(2):
        out = M.pcg(b, fmt=gpu.FMT_DIA, **kw)
        assert (out["iters"], out["outer_iters"], out["final_norm"]) == \
            (ref["iters"], ref["outer_iters"], ref["final_norm"])
        np.testing.assert_array_equal(out["x"], ref["x"])
        # all 7 arrays below the line, 4 of them and the mask above it
        assert (out["spmv_bytes"] == 25.0 * n) == (n >= 850000)
