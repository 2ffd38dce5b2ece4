"""Why a block has no DIA form: the same reason every time, unsorted rows before
too many diagonals, with their number."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def block(n, offsets, unsorted):
    i = np.arange(n)
    rows = [[o + r for o in sorted(offsets) if 0 <= o + r < n] for r in i]
    for r in unsorted:
        rows[r] = rows[r][::-1]
    xadj = np.concatenate([[0], np.cumsum([len(r) for r in rows])])
    return xadj, np.concatenate(rows)


@pytest.mark.parametrize("n,offsets,unsorted,reason", [
    (5000, range(-16, 17), (), "33 diagonals: more than the DIA form holds (32)"),
    (5000, [0] + list(range(-4999, 5000, 100)), (), "101 diagonals: more"),
    (40000, list(range(-20, 21)), (39990,), "not strictly ascending"),
    (40000, list(range(-20, 21)), (0,), "not strictly ascending"),
    (5000, (-1, 0, 1), (2500,), "not strictly ascending"),
])
def test_the_reason_does_not_depend_on_timing(gpu, n, offsets, unsorted, reason):
    xadj, cols = block(n, offsets, unsorted)
    M = gpu.Matrix.from_csr(xadj, cols, np.ones(cols.size), index_base=0)
    for _ in range(3):
        with pytest.raises(gpu.CelError) as e:
            M.to_dia()
        assert reason in str(e.value)
