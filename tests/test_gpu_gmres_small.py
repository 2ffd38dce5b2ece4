"""GMRES columns in one launch (small systems, CSR and DIA) against the JAD
form, whose products, dot products and vector updates are launches of their
own: the same bits at the edges of the 2,048-row chunks and the 1,024-thread
blocks, for restarts up to the largest, when the first column converges, and
above the line where the forms share the separate launches."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SHAPES = [(1, 1, 1), (5, 3, 2), (32, 32, 1), (41, 25, 1), (64, 32, 1), (2049, 1, 1), (17, 11, 23), (64, 32, 3)]


def run(gpu, M, b, **kw):
    return [M.gmres(b, fmt=f, **kw) for f in (gpu.FMT_JAD, gpu.FMT_CSR, gpu.FMT_DIA)]


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("restart", [1, 2, 3, 5, 32])
def test_one_launch_columns_are_the_separate_ones(gpu, shape, restart):
    n = int(np.prod(shape))
    rng = np.random.default_rng(17)
    M = gpu.Matrix.diffusion7(*shape, np.exp(rng.normal(0.0, 0.5, n)))
    M.set_jacobi()
    M.to_jad()
    M.to_dia()
    b = rng.normal(size=n)
    for kw in (dict(eps=1e-7, iter_max=400), dict(eps=1e-30, iter_max=2), dict(eps=1e3, iter_max=5),
               dict(eps=1e-6, iter_max=3, x0=rng.normal(size=n))):
        ref, *others = run(gpu, M, b, restart=restart, **kw)
        for out in others:
            assert (out["status"], out["iters"], out["cycles"]) == (ref["status"], ref["iters"], ref["cycles"])
            np.testing.assert_array_equal(out["x"], ref["x"])
            np.testing.assert_array_equal([out["norm0"], out["final_norm"]], [ref["norm0"], ref["final_norm"]])


def test_above_the_line(gpu):
    shape = (85, 84, 86)  # 614,040 rows
    n = int(np.prod(shape))
    M = gpu.Matrix.poisson7(*shape)
    M.set_jacobi()
    M.to_jad()
    M.to_dia()
    ref, *others = run(gpu, M, np.random.default_rng(18).normal(size=n), eps=1e-9, iter_max=2)
    for out in others:
        np.testing.assert_array_equal(out["x"], ref["x"])


def test_tiny_and_huge_vectors(gpu):
    """Quotients near the ends of the exponent range: a right-hand side whose
    Krylov vectors span hundreds of orders of magnitude."""
    n = 3000
    M = gpu.Matrix.poisson7(n, 1, 1)
    M.set_jacobi()
    M.to_jad()
    M.to_dia()
    b = np.ldexp(1.0, -np.arange(n) % 900 - 50) * np.random.default_rng(19).normal(size=n)
    for scale in (1.0, 2.0 ** 500):
        outs = []
        for fmt in (gpu.FMT_JAD, gpu.FMT_CSR, gpu.FMT_DIA):
            try:
                outs.append(M.gmres(b * scale, fmt=fmt, restart=3, eps=1e-300, iter_max=3, x0_mode=gpu.X0_ZERO)["x"])
            except gpu.CelError as e:  # (norms whose squares leave the range: in every form)
                outs.append(np.array([e.code]))
        for out in outs[1:]:
            np.testing.assert_array_equal(out, outs[0])
