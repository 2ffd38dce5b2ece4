"""Products with several consecutive rows per lane (row classes and diagonal
storage of long solves): solves against the entry-by-entry walk, bit for
bit, on matrices of 1 to 8 diagonals with near, far and one-sided offsets,
row counts on either side of the lanes', waves' and groups' sizes, and
values that are constant (classes) or not, symmetric or not."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

BASE = 1563 * 512  # 800,256 rows: whole groups of two 256-row tiles


def banded(n, offsets, values, rng):
    """CSR arrays of the matrix on `offsets` (0 among them, its values the
    largest), entry (i, i + o) absent where it leaves the matrix and, off the
    diagonal, in every 29th row."""
    i = np.arange(n, dtype=np.int64)
    cols, vals, keep = [], [], []
    for o in sorted(offsets):
        on = (i + o >= 0) & (i + o < n)
        if o:
            on &= np.minimum(i, i + o) % 29 != 7  # the same pairs on both sides
        v = np.full(n, 20.0 if o == 0 else -1.0)
        if values != "constant" and o:
            w = 0.5 + rng.random(n)
            if values == "symmetric":  # one weight per pair
                w = 0.5 + ((np.minimum(i, i + o) * 2654435761 + abs(o) * 40503) % 65536) / 65536.0
            v = -w
        if values != "constant" and not o:
            v = 20.0 + rng.random(n)
        cols.append(i + o)
        vals.append(v)
        keep.append(on)
    keep = np.stack(keep, 1)
    xadj = np.concatenate([[0], np.cumsum(keep.sum(1))])
    return xadj, np.stack(cols, 1)[keep], np.stack(vals, 1)[keep]


@pytest.mark.parametrize("values", ["constant", "symmetric", "general"])
@pytest.mark.parametrize("n,offsets", [
    (BASE, (0,)),
    (BASE + 1, (-1, 0, 1)),
    (BASE + 2, (-733, -1, 0, 1, 733)),
    (BASE - 1, (-8101, -89, -1, 0, 1, 89, 8101)),
    (BASE + 255, (-8100, -90, -1, 0, 1, 2, 90, 8100)),
    (BASE + 257, (0, 1, 3, 4000)),
    (BASE + 3, (-5000, -2, 0)),
    (BASE + 129, (-500000, -1, 0, 1, 500000)),
])
def test_wide_rows_keep_the_bits(gpu, n, offsets, values):
    rng = np.random.default_rng(n + len(offsets))
    xadj, cols, vals = banded(n, offsets, values, rng)
    M = gpu.Matrix.from_csr(xadj, cols, vals, index_base=0)
    M.set_jacobi()
    b, x0 = rng.normal(size=n), rng.normal(size=n)
    kw = dict(tol=1e-300, tol_mode=gpu.TOL_REL_B, alpha_stop=0, iter_max=33, x0=x0)
    refs = {p: M.pcg(b, fmt=gpu.FMT_COO, precision=p, **kw) for p in (gpu.PREC_FP64, gpu.PREC_MIXED)}
    for fmt in (gpu.FMT_CSR, gpu.FMT_DIA):
        if fmt == gpu.FMT_DIA:
            M.to_dia()
        for p, ref in refs.items():
            out = M.pcg(b, fmt=fmt, precision=p, **kw)
            assert (out["status"], out["iters"], out["final_norm"]) == (ref["status"], ref["iters"], ref["final_norm"])
            np.testing.assert_array_equal(out["x"], ref["x"])
