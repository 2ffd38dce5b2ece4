"""A batch whose systems stop at different times, so that their blocks are dealt
again to those still running: every solve on a handle gives the same bits, the
first one, which builds the derived forms on the way, too."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("chunk", [0, 1, 3, 8])
def test_first_and_later_solves(gpu, chunk):
    rng = np.random.default_rng(61)
    mats = [gpu.Matrix.diffusion7(*s, np.exp(rng.normal(0.0, 0.4, int(np.prod(s)))))
            for s in ((8, 9, 10), (28, 29, 27), (40, 41, 42), (61, 60, 59))]
    for m in mats:
        m.set_jacobi()
    ks = [1, 3, 1, 2]
    bs = [rng.normal(size=(k, m.n)) if k > 1 else rng.normal(size=m.n) for m, k in zip(mats, ks)]
    outs = []
    batch = gpu.Batch(mats, ks)
    if chunk:
        batch.set_config(batch.info()["grid"] or 512, chunk=chunk)
    for _ in range(3):
        outs.append(batch.solve(bs, tol=1e-9, alpha_stop=0))
    iters = [l["iters"] for l in outs[0]["lanes"]]
    assert max(iters) > min(iters) + 16
    for out in outs[1:]:
        assert [l["iters"] for l in out["lanes"]] == iters
        for x, y in zip(out["x"], outs[0]["x"]):
            np.testing.assert_array_equal(x, y)
