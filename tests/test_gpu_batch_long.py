"""Batches of matrices whose 256-row chunks hold more entries than the LDS stage,
read eight entries at a time: rows that end inside a group of eight, one row
of thousands, an odd row count, one and several right-hand sides, against
the single-system solver after a few iterations."""
import numpy as np
import pytest

from helpers import stencil27
from test_gpu_batch_paths import TOL, six
from test_gpu_deep_rows import with_long_rows

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rhs", [1, 2, 3, 9])
def test_long_rows(gpu, rhs):
    rng = np.random.default_rng(51 + rhs)
    mats = []
    for A in (stencil27(17, 16, 15), with_long_rows(3001, 2500, rng), with_long_rows(1003, 12, rng),
              stencil27(4, 4, 3)):
        M = gpu.Matrix.from_csr(A.indptr, A.indices, A.data, index_base=0)
        M.set_jacobi()
        mats.append(M)
    bs = [rng.normal(size=(rhs, m.n)) for m in mats]
    out = gpu.Batch(mats, [rhs] * len(mats)).solve([b if rhs > 1 else b[0] for b in bs], tol=1e-300,
                                                   tol_mode=gpu.TOL_REL_B, iter_max=6, x0_mode=gpu.X0_ZERO,
                                                   alpha_stop=0)
    for x, m, b in zip(out["x"], mats, bs):
        for j in (0, rhs - 1):
            ref = six(gpu, m, b[j])
            assert np.linalg.norm(np.asarray(x).reshape(rhs, -1)[j] - ref) <= TOL * np.linalg.norm(ref)
