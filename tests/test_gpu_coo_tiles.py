"""Ordering of entries whose rows average more than the 8 entries at which 256
row groups fill the LDS tile of 2,048: groups that divide the tile, that do
not, and groups longer than the tile among them."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lengths", [
    (9,), (12, 0, 31), (32,), (31, 32, 1),
    (32, 32, 2048, 5), (2047, 1, 2049, 1), (20,) * 60 + (5000,), (33, 8),
])
@pytest.mark.parametrize("nrows", [255, 256, 1027])
def test_order_of_long_rows(gpu, nrows, lengths):
    rng = np.random.default_rng(91 + nrows)
    rows = np.repeat(np.arange(nrows), [lengths[i % len(lengths)] for i in range(nrows)])
    cols = rng.integers(0, 57, rows.size)  # repeated columns
    vals = np.arange(rows.size) + 0.5      # the order they came in
    p = rng.permutation(rows.size)
    rows, cols = rows[p], cols[p]
    order = np.lexsort((np.arange(rows.size), cols, rows))
    _, r, c, v = gpu.coo_sort(nrows, rows, cols, vals, ncols=57, index_base=0, mode=gpu.SORT_ROW_COL)
    np.testing.assert_array_equal(r, rows[order])
    np.testing.assert_array_equal(c, cols[order])
    np.testing.assert_array_equal(v, vals[order])
