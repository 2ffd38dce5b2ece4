"""Solves from several host threads at once, a matrix handle each (products of
different forms and sizes, derived forms and kept memory among them): the
results of the same solves one after another."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_a_handle_per_thread(gpu):
    shapes = [(13, 12, 11), (40, 41, 39), (71, 70, 69), (97, 93, 91)]

    def work(i, out):
        rng = np.random.default_rng(i)
        s = shapes[i % len(shapes)]
        n = int(np.prod(s))
        M = gpu.Matrix.diffusion7(*s, np.exp(rng.normal(0.0, 0.4, n)))
        M.set_jacobi()
        M.to_dia()
        b = rng.normal(size=n)
        res = []
        for fmt in (gpu.FMT_CSR, gpu.FMT_DIA):
            for prec in (gpu.PREC_FP64, gpu.PREC_MIXED):
                r = M.pcg(b, fmt=fmt, precision=prec, tol=1e-8, tol_mode=gpu.TOL_REL_B, alpha_stop=0)
                res.append((r["iters"], r["x"]))
            res.append((0, M.spmv(b, fmt=fmt)))
        out[i] = res

    alone, together = {}, {}
    for i in range(6):
        work(i, alone)
    threads = [threading.Thread(target=work, args=(i, together)) for i in range(6)]
    for t in threads:
        t.start()
    for t in threads:
        t.join(timeout=100)
    assert sorted(together) == list(range(6))
    for i in range(6):
        for (ka, xa), (kb, xb) in zip(alone[i], together[i]):
            assert ka == kb
            np.testing.assert_array_equal(xa, xb)
