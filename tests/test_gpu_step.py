"""The two-kernel PCG iteration of small systems (the update of the vectors
and the next product in one kernel) against the three-kernel one, which a
profiled solve runs: the same bits, histories, iteration and replacement
counts, in every form and precision and under iteration caps; the mixed
form's replacement residual, taken in place of a product, against the FP64
operator."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu

# one row; below, at and above one tile pair (512 rows); partial tiles; an odd
# box of several vector units; just below the FP64 line (300,000 rows)
SHAPES = [(1, 1, 1), (7, 5, 3), (16, 16, 2), (19, 27, 1), (33, 17, 9), (41, 37, 43), (71, 61, 69)]


def solve(gpu, M, b, **kw):
    """The result, or the code of the error it ends with (a one-row system
    whose residual vanishes in FP32 breaks down)."""
    try:
        return M.pcg(b, **kw)
    except gpu.CelError as e:
        return e.code


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("mixed", [False, True], ids=["fp64", "mixed"])
def test_two_kernel_iterations_are_the_three_kernel_ones(gpu, shape, mixed):
    n = int(np.prod(shape))
    rng = np.random.default_rng(91)
    M = gpu.Matrix.diffusion7(*shape, np.exp(rng.normal(0.0, 0.7, n)))
    M.set_jacobi()
    M.to_jad()
    M.to_dia()
    b = rng.normal(size=n)
    x0 = rng.normal(size=n)
    runs = [dict(tol=1e-9, tol_mode=gpu.TOL_REL_B, x0_mode=gpu.X0_ZERO, iter_max=4000, alpha_stop=0),
            dict(tol=1e-30, tol_mode=gpu.TOL_ABS, x0=x0, iter_max=7, alpha_stop=0),
            dict(tol=1e-30, tol_mode=gpu.TOL_ABS, x0_mode=gpu.X0_ONE, iter_max=0, alpha_stop=0)]
    if mixed:
        runs.append(dict(runs[0], ru_restart=1))
    for kw in runs:
        for fmt in (gpu.FMT_CSR, gpu.FMT_COO, gpu.FMT_JAD, gpu.FMT_DIA):
            kw = dict(kw, fmt=fmt, precision=gpu.PREC_MIXED if mixed else gpu.PREC_FP64, history=True)
            three = solve(gpu, M, b, profile=1, **kw)
            if isinstance(three, int):
                assert all(solve(gpu, M, b, **kw, **extra) == three
                           for extra in (dict(), dict(use_graph=1), dict(use_graph=1, check_every=5)))
                continue
            assert three["iters"] <= kw["iter_max"]
            for extra in (dict(), dict(check_every=1), dict(use_graph=1), dict(use_graph=1, check_every=5)):
                two = solve(gpu, M, b, **kw, **extra)
                assert (two["status"], two["iters"], two["outer_iters"]) == \
                    (three["status"], three["iters"], three["outer_iters"])
                np.testing.assert_array_equal(two["x"], three["x"])
                np.testing.assert_array_equal(two["hist"], three["hist"])
                assert two["final_norm"] == three["final_norm"]


def test_mixed_replacement_residual_is_the_fp64_one(gpu):
    """The reported norm of a mixed solve is that of b - A x in FP64 (to the
    rounding of the sums: 1e-12 of |b|)."""
    shape = (23, 31, 19)
    n = int(np.prod(shape))
    rng = np.random.default_rng(92)
    kappa = np.exp(rng.normal(0.0, 0.5, n))
    M = gpu.Matrix.diffusion7(*shape, kappa)
    M.set_jacobi()
    M.to_jad()
    M.to_dia()
    A = O.gen_diffusion7(*shape, kappa)
    b = rng.normal(size=n)
    for fmt in (gpu.FMT_CSR, gpu.FMT_JAD, gpu.FMT_DIA):
        for kw in (dict(), dict(ru_restart=1)):
            out = M.pcg(b, tol=1e-10, tol_mode=gpu.TOL_REL_B, x0_mode=gpu.X0_ZERO, iter_max=4000, alpha_stop=0,
                        precision=gpu.PREC_MIXED, fmt=fmt, **kw)
            assert out["status"] == 0 and out["outer_iters"] >= 3
            true = np.linalg.norm(b - O.spmv_csr(A, out["x"]))
            assert abs(out["final_norm"] - true) <= 1e-12 * np.linalg.norm(b)
