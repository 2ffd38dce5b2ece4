"""PCG iterations on either side of the size up to which a solve loads its
matrix so that it stays in the infinity cache: six iterations against the
same recurrence in numpy.  The bits do not depend on the side: where CSR and
DIA fall on different ones, they are compared bit for bit."""
import numpy as np
import pytest
import scipy.sparse as sp

from helpers import stencil27

pytestmark = pytest.mark.gpu

# rows x forms: the 7-point boxes keep the matrix at the first size of a pair
# in every form, and the last not in any; at the middle size CSR does not and
# DIA does.  (Fewer rows than the first size take the two-kernel iterations.)
BOXES = {"fp64": [(71, 67, 69), (136, 135, 137), (144, 143, 145)],
         "mixed": [(109, 107, 111), (163, 165, 164), (176, 175, 177)]}


def six_iterations(A, d, b):
    """x after six Jacobi-PCG iterations from 0."""
    x = np.zeros_like(b)
    r = b.copy()
    p = z = d * r
    rz = r @ z
    for _ in range(6):
        v = A @ p
        sigma = rz / (v @ p)
        x = x + sigma * p
        r = r - sigma * v
        z = d * r
        rz, old = r @ z, rz
        p = (rz / old) * p + z
    return x


def run(gpu, M, b, fmt, prec):
    return M.pcg(b, fmt=fmt, precision=gpu.PREC_MIXED if prec == "mixed" else gpu.PREC_FP64, x0_mode=gpu.X0_ZERO,
                 tol=1e-300, tol_mode=gpu.TOL_REL_B, alpha_stop=0, ru_delta=1e-30, iter_max=6)["x"]


def close(x, ref, prec):
    # six iterations of rounding, each within a few units of the vectors' type
    tol = 1e-12 if prec == "fp64" else 1e-5
    assert np.linalg.norm(x - ref) <= tol * np.linalg.norm(ref)


@pytest.mark.parametrize("prec,shape", [(k, s) for k, v in BOXES.items() for s in v])
def test_seven_point_boxes(gpu, prec, shape):
    rng = np.random.default_rng(17)
    n = int(np.prod(shape))
    M = gpu.Matrix.diffusion7(*shape, np.exp(rng.normal(0.0, 0.5, n)))
    M.set_jacobi()
    M.to_dia()
    M.to_jad()
    b = rng.normal(size=n)
    xadj, cols, vals = M.get_csr()
    A = sp.csr_matrix((vals, cols - 1, xadj - 1), shape=(n, n))
    ref = six_iterations(A, M.jacobi(), b)
    csr = run(gpu, M, b, gpu.FMT_CSR, prec)
    close(csr, ref, prec)
    np.testing.assert_array_equal(run(gpu, M, b, gpu.FMT_DIA, prec), csr)
    close(run(gpu, M, b, gpu.FMT_JAD, prec), ref, prec)


# 27-point rows: FP64 CSR keeps the matrix up to 797,000 rows, mixed CSR up to
# 1.2 million
@pytest.mark.parametrize("prec,shape", [("fp64", (41, 43, 42)), ("fp64", (94, 93, 95)),
                                        ("mixed", (41, 43, 42)), ("mixed", (109, 108, 107))])
def test_long_rows(gpu, prec, shape):
    rng = np.random.default_rng(18)
    A = stencil27(*shape)
    n = A.shape[0]
    M = gpu.Matrix.from_csr(A.indptr, A.indices, A.data, index_base=0)
    M.set_jacobi()
    M.to_dia()
    b = rng.normal(size=n)
    csr = run(gpu, M, b, gpu.FMT_CSR, prec)
    close(csr, six_iterations(A, M.jacobi(), b), prec)
    np.testing.assert_array_equal(run(gpu, M, b, gpu.FMT_DIA, prec), csr)
