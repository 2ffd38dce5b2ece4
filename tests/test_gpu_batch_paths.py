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


# matrices in every form K1 reads (CSR arrays below 20,000 rows and off the
# diagonals, diagonals symmetric or row-scaled, row classes), one and several
# right-hand sides, tiles and chunks with a remainder: 40 iterations against
# the single-system solver
@pytest.mark.parametrize("rhs", [1, 2, 5])
@pytest.mark.parametrize("scaled", [False, True])
def test_forms_of_batched_matrices(gpu, rhs, scaled):
    rng = np.random.default_rng(43 + rhs)
    mats = [gpu.Matrix.diffusion7(nx, ny, nz, np.exp(rng.normal(0.0, 0.3, nx * ny * nz)))
            for nx, ny, nz in ((9, 8, 7), (31, 29, 33), (28, 27, 27), (400, 50, 1), (1, 1, 20001))]
    mats.append(gpu.Matrix.poisson7(97, 93, 91))
    n = 21001  # a ring: offsets 1 and n - 1, no row has all of its neighbours in reach
    i = np.arange(n)
    cols = np.sort(np.stack([(i - 1) % n, i, (i + 1) % n], 1), 1)
    mats.append(gpu.Matrix.from_csr(3 * np.arange(n + 1), cols.ravel(),
                                    np.where(cols == i[:, None], 3.0, -1.0).ravel(), index_base=0))
    for m in mats:
        m.set_jacobi()
        if scaled:
            m.scale_diagonal()
            m.set_jacobi(row_scaled=True)
    bs = [rng.normal(size=(rhs, m.n)) for m in mats]
    kw = dict(tol=1e-300, tol_mode=gpu.TOL_REL_B, iter_max=40, x0_mode=gpu.X0_ZERO, alpha_stop=0)
    batch = gpu.Batch(mats, [rhs] * len(mats))
    for _ in range(2):  # building the forms, and on the built ones
        out = batch.solve([b if rhs > 1 else b[0] for b in bs], **kw)
        for x, m, b in zip(out["x"], mats, bs):
            for j in (0, rhs - 1):
                ref = m.pcg(b[j], fmt=gpu.FMT_COO, **kw)["x"]
                # 40 iterations of rounding, amplified by at most the condition of a few hundred
                assert np.linalg.norm(np.asarray(x).reshape(rhs, -1)[j] - ref) <= 1e-9 * np.linalg.norm(ref)
