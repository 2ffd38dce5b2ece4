"""Replayed solves whose chunk is an odd number of iterations: the same bits as
without a graph, where an iteration is two kernels (its direction alternates
between two buffers) and where it is three, stopping inside a chunk, at its
end and at iter_max."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(13, 11, 12), (71, 68, 67)])
@pytest.mark.parametrize("every", [1, 3, 17])
def test_odd_chunks(gpu, shape, every):
    rng = np.random.default_rng(every)
    n = int(np.prod(shape))
    M = gpu.Matrix.diffusion7(*shape, np.exp(rng.normal(0.0, 0.4, n)))
    M.set_jacobi()
    b = rng.normal(size=n)
    for prec in (gpu.PREC_FP64, gpu.PREC_MIXED):
        for tol, iter_max in ((1e-8, 1000), (1e-300, 34), (1e-300, 51)):
            kw = dict(precision=prec, tol=tol, tol_mode=gpu.TOL_REL_B, alpha_stop=0, iter_max=iter_max)
            ref = M.pcg(b, **kw)
            for _ in range(2):
                out = M.pcg(b, use_graph=1, check_every=every, **kw)
                assert (out["status"], out["iters"], out["outer_iters"], out["final_norm"]) == \
                    (ref["status"], ref["iters"], ref["outer_iters"], ref["final_norm"])
                np.testing.assert_array_equal(out["x"], ref["x"])
