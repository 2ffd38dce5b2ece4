"""FP64 solves on long rows in a narrow band, whose product gathers from a copy
of the band's columns in LDS, on either side of the rule (120,000 rows, a band of
3,582), against a handle whose band is too wide because of one far pair of
entries that are zero, bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def mesh(n, band, far, rng):
    """Symmetric, dominant diagonal, about 13 entries per row within `band`
    (which it attains), row-sorted; far: a zero pair (0, n - 1) besides."""
    i = np.repeat(np.arange(n, dtype=np.int64), 6)
    j = i + 1 + rng.integers(0, band, i.size)
    key = np.unique(np.concatenate([(i * n + j)[j < n], [band]]))  # (0, band)
    i, j = key // n, key % n
    w = rng.integers(1, 9, i.size) / 8.0
    if far:
        i, j, w = np.append(i, 0), np.append(j, n - 1), np.append(w, 0.0)
    d = np.full(n, 0.5)
    np.add.at(d, i, w)
    np.add.at(d, j, w)
    a = np.arange(n)
    r, c, v = np.concatenate([i, j, a]), np.concatenate([j, i, a]), np.concatenate([-w, -w, d])
    o = np.argsort(r * n + c)
    return np.concatenate([[0], np.cumsum(np.bincount(r, minlength=n))]), c[o], v[o]


@pytest.mark.parametrize("n,band", [(119999, 900), (120000, 900), (120001, 3582), (130817, 3583), (200193, 40),
                                    (262144, 3580)])
def test_band_in_lds_keeps_the_bits(gpu, n, band):
    rng = np.random.default_rng(n + band)
    b, x0 = rng.normal(size=n), rng.normal(size=n)
    kw = dict(tol=1e-300, tol_mode=gpu.TOL_REL_B, alpha_stop=0, iter_max=33, x0=x0)
    outs = []
    for far in (False, True):
        A = mesh(n, band, far, np.random.default_rng(7))
        M = gpu.Matrix.from_csr(*A, index_base=0)
        M.set_jacobi()
        for fmt in (gpu.FMT_CSR, gpu.FMT_COO):
            outs.append(M.pcg(b, fmt=fmt, **kw))
            outs.append(M.pcg(b, fmt=fmt, use_graph=1, **kw))
    for out in outs[1:]:
        assert (out["status"], out["iters"], out["final_norm"]) == \
            (outs[0]["status"], outs[0]["iters"], outs[0]["final_norm"])
        np.testing.assert_array_equal(out["x"], outs[0]["x"])
