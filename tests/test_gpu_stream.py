"""The vector kernels of large solves, which mark vectors that no kernel finds
in the cache again as read once: the same bits on either side of the sizes
that decide it.  A solve on row classes touches fewer bytes of vectors than
the entry-by-entry walk of the same matrix, so between the two sizes they
run with different marks."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# marks of the walk / of the classes: x / none, all / x, all / all
SHAPES = {"fp64": [(187, 186, 188), (219, 218, 220), (231, 229, 230)],
          "mixed": [(237, 236, 238), (275, 274, 276), (283, 282, 285)]}


@pytest.mark.parametrize("prec,shape", [(k, s) for k, v in SHAPES.items() for s in v])
def test_marks_keep_the_bits(gpu, prec, shape):
    M = gpu.Matrix.poisson7(*shape)
    M.set_jacobi()
    b = np.random.default_rng(23).random(int(np.prod(shape))) - 0.5
    kw = dict(tol=1e-300, tol_mode=gpu.TOL_REL_B, alpha_stop=0, x0_mode=gpu.X0_ONE, iter_max=33,
              precision=gpu.PREC_MIXED if prec == "mixed" else gpu.PREC_FP64)
    ref = M.pcg(b, fmt=gpu.FMT_COO, **kw)
    out = M.pcg(b, fmt=gpu.FMT_CSR, **kw)
    assert (out["status"], out["iters"], out["outer_iters"], out["final_norm"]) == \
        (ref["status"], ref["iters"], ref["outer_iters"], ref["final_norm"])
    np.testing.assert_array_equal(out["x"], ref["x"])
