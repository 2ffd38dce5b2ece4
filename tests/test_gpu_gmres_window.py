"""GMRES of small systems in the DIA form, whose product takes the inner
diagonals from LDS where they lie within 1,024 of the main one, and in CSR,
against the JAD form (separate kernels): bit for bit, for offsets on either
side of that line, one to eight diagonals, chunks with a remainder, and
column counts on either side of the ones whose algebra runs in registers."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def banded(n, offsets, rng):
    i = np.arange(n, dtype=np.int64)
    cols = np.stack([i + o for o in offsets], 1)
    vals = np.stack([np.full(n, 3.0 * len(offsets)) if o == 0 else -0.5 - rng.random(n) for o in offsets], 1)
    keep = (cols >= 0) & (cols < n) & ((i[:, None] % 31 != 5) | (np.asarray(offsets) == 0))
    return np.concatenate([[0], np.cumsum(keep.sum(1))]), cols[keep], vals[keep]


@pytest.mark.parametrize("m", [1, 3, 4, 6])
@pytest.mark.parametrize("n,offsets", [
    (7, (0,)),
    (1, (0,)),
    (2049, (-1, 0, 1)),
    (5000, (0, 3)),
    (6145, (-2048, -1024, -1, 0, 1, 1024, 2048)),
    (6143, (-2050, -1025, -1, 0, 1, 1025, 2050)),
    (4097, (-3000, -1024, -2, -1, 0, 1, 2, 1024)),
    (70001, (-9001, -97, -1, 0, 1, 97, 9001)),
])
def test_forms_agree(gpu, n, offsets, m):
    rng = np.random.default_rng(61 + n)
    xadj, cols, vals = banded(n, offsets, rng)
    M = gpu.Matrix.from_csr(xadj, cols, vals, index_base=0)
    M.set_jacobi()
    M.to_jad()
    M.to_dia()
    b = rng.normal(size=n)
    for eps, iters in ((1e-300, 3), (1e-6 * np.linalg.norm(b), 50)):
        outs = []
        for fmt in (gpu.FMT_JAD, gpu.FMT_DIA, gpu.FMT_CSR):
            try:
                o = M.gmres(b, fmt=fmt, restart=m, eps=eps, iter_max=iters)
                outs.append(((o["status"], o["iters"], o["cycles"], o["final_norm"]), o["x"]))
            except gpu.CelError as e:  # (an exact solution in fewer columns: in every form)
                outs.append(((e.code,), np.zeros(0)))
        for key, x in outs[1:]:
            assert key == outs[0][0]
            np.testing.assert_array_equal(x, outs[0][1])
