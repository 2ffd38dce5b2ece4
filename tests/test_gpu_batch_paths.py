"""Paths of the batched solver that sizes choose, against the single-system
solver after a few iterations."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# six iterations of rounding, each within a few units of the vectors' type
TOL = 1e-12


def six(gpu, M, b):
    return M.pcg(b, tol=1e-300, tol_mode=gpu.TOL_REL_B, x0_mode=gpu.X0_ZERO, iter_max=6, alpha_stop=0)["x"]


# bytes of the vectors: below, between and above the lines (240 and 450 MB)
@pytest.mark.parametrize("rhs", [3, 8, 16])
def test_vectors_of_large_batches(gpu, rhs):
    shape = (101, 99, 103)
    rng = np.random.default_rng(41)
    M = gpu.Matrix.poisson7(*shape)
    small = gpu.Matrix.poisson7(5, 4, 3)
    for m in (M, small):
        m.set_jacobi()
    B = rng.normal(size=(rhs, M.n))
    c = rng.normal(size=small.n)
    out = gpu.Batch([small, M], [1, rhs]).solve([c, B], tol=1e-300, tol_mode=gpu.TOL_REL_B, iter_max=6,
                                                x0_mode=gpu.X0_ZERO, alpha_stop=0)
    xs = [np.asarray(x) for x in out["x"]]
    for x, m, b in [(xs[0].ravel(), small, c)] + [(xs[1].reshape(rhs, -1)[j], M, B[j]) for j in (0, rhs - 1)]:
        ref = six(gpu, m, b)
        assert np.linalg.norm(x - ref) <= TOL * np.linalg.norm(ref)
