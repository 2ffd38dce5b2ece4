"""Long solves on the derived forms of a block (row classes, diagonal storage;
built inside the first such solve of 800,000 rows or more) against the same
solve on the CSR arrays themselves, which the COO form walks entry by
entry: bit for bit, for matrices on either side of every rule that chooses
the form, and after the values, the Jacobi vector or the scaling change."""
import numpy as np
import pytest

from helpers import stencil27

pytestmark = pytest.mark.gpu

SHAPE = (97, 93, 91)  # 820,911 rows: an odd box, the last tile partial
N = 97 * 93 * 91


def kappa_of(kind, rng):
    x, y, z = SHAPE
    k = np.ones((z, y, x))
    if kind == "two_materials":      # a few dozen forms
        k[:, :, x // 3:] = 7.5
    elif kind == "layers":           # more than 256 forms, constant along x and y
        k *= np.exp(0.1 * np.arange(z))[:, None, None]
    elif kind == "random":
        k = np.exp(rng.normal(0.0, 0.5, k.shape))
    return k.ravel()


def same(gpu, M, b, **kw):
    """The solve in CSR (a derived form where one fits) and in DIA, where the
    matrix has it, against the entry-by-entry walk."""
    for prec in (gpu.PREC_FP64, gpu.PREC_MIXED):
        ref = M.pcg(b, fmt=gpu.FMT_COO, precision=prec, **kw)
        for fmt in (gpu.FMT_CSR,) + ((gpu.FMT_DIA,) if M.dia_info() else ()):
            out = M.pcg(b, fmt=fmt, precision=prec, **kw)
            assert (out["status"], out["iters"], out["outer_iters"], out["final_norm"]) == \
                (ref["status"], ref["iters"], ref["outer_iters"], ref["final_norm"])
            np.testing.assert_array_equal(out["x"], ref["x"])


@pytest.mark.parametrize("kind", ["poisson", "two_materials", "layers", "random"])
def test_derived_forms_keep_the_bits(gpu, kind):
    rng = np.random.default_rng(31)
    M = gpu.Matrix.poisson7(*SHAPE) if kind == "poisson" else gpu.Matrix.diffusion7(*SHAPE, kappa_of(kind, rng))
    M.set_jacobi()
    b = rng.normal(size=N)
    x0 = rng.normal(size=N)
    kw = dict(tol=1e-300, tol_mode=gpu.TOL_REL_B, alpha_stop=0, ru_delta=1e-2)
    same(gpu, M, b, x0=x0, iter_max=8, **kw)        # too short to build a form
    same(gpu, M, b, x0_mode=gpu.X0_ONE, iter_max=48, **kw)
    same(gpu, M, b, x0=x0, iter_max=8, **kw)        # on the form that is there
    M.to_dia()
    same(gpu, M, b, x0=x0, iter_max=33, use_graph=1, **kw)
    # the row-scaled matrix: values and Jacobi vector are others
    M.scale_diagonal()
    M.set_jacobi(row_scaled=True)
    same(gpu, M, b, x0=x0, iter_max=40, **kw)
    # the values of before with another Jacobi vector
    M.set_jacobi()
    same(gpu, M, b, x0=x0, iter_max=40, **kw)


def test_matrices_without_a_derived_form(gpu):
    """More than 8 diagonals; no diagonals at all; unsorted rows."""
    rng = np.random.default_rng(32)
    kw = dict(tol=1e-300, tol_mode=gpu.TOL_REL_B, alpha_stop=0, x0_mode=gpu.X0_ZERO, iter_max=40)
    A = stencil27(94, 93, 92)
    M = gpu.Matrix.from_csr(A.indptr, A.indices, A.data, index_base=0)
    M.set_jacobi()
    same(gpu, M, rng.normal(size=A.shape[0]), **kw)
    n = 800001  # a symmetric matrix of random pairs: row i and its partner
    perm = rng.permutation(n - 1)
    pair = np.empty(n, dtype=np.int64)
    pair[perm[: (n - 1) // 2]] = perm[(n - 1) // 2:]
    pair[perm[(n - 1) // 2:]] = perm[: (n - 1) // 2]
    pair[n - 1] = n - 1
    cols = np.stack([pair, np.arange(n)], axis=1)  # the diagonal last: unsorted where the partner is right of it
    vals = np.tile([-1.0, 3.0], n)
    cols[n - 1] = (n - 2, n - 1)
    vals[2 * (n - 1)] = 0.0
    for c in (np.sort(cols, axis=1), cols):
        v = np.where(c == np.arange(n)[:, None], 3.0, -1.0)
        v[n - 1] = np.where(c[n - 1] == n - 1, 3.0, 0.0)
        M = gpu.Matrix.from_csr(2 * np.arange(n + 1), c.ravel(), v.ravel(), index_base=0)
        M.set_jacobi()
        same(gpu, M, rng.normal(size=n), **kw)
