"""Ordering by (row, column) on either side of the row count up to which every
row is a group (twice the entries): empty rows, rows of every kind of group
(up to 32, up to 4,096 and more entries), repeated columns, and an index out
of range, after which the caller's arrays are untouched."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nrows,lengths", [
    (1, (1,)),
    (2, (1,)),
    (3, (1,)),
    (4000, (7, 0, 1, 33, 0, 5)),
    (60, (0, 31, 32, 33, 4096, 0)),
    (60, (0, 3, 4097, 0, 9000, 40)),
    (12000, (4097, 31, 2)),
])
def test_order_by_row_and_column(gpu, nrows, lengths):
    rng = np.random.default_rng(81 + nrows)
    count = np.zeros(nrows, dtype=np.int64)
    at = np.sort(rng.choice(nrows, size=min(nrows, 4 * len(lengths)), replace=False))
    count[at] = [lengths[i % len(lengths)] for i in range(at.size)]
    if count.sum() == 0:
        count[0] = 1
    rows = np.repeat(np.arange(nrows), count)
    cols = rng.integers(0, 97, rows.size)  # repeated columns in the longer rows
    vals = np.arange(rows.size) + 0.5      # the order they came in
    p = rng.permutation(rows.size)
    rows, cols = rows[p], cols[p]
    order = np.lexsort((np.arange(rows.size), cols, rows))
    _, r, c, v = gpu.coo_sort(nrows, rows, cols, vals, ncols=97, index_base=0, mode=gpu.SORT_ROW_COL)
    np.testing.assert_array_equal(r, rows[order])
    np.testing.assert_array_equal(c, cols[order])
    np.testing.assert_array_equal(v, vals[order])


@pytest.mark.parametrize("nrows", [50, 5000])
def test_bad_index_leaves_the_arrays(gpu, nrows):
    rng = np.random.default_rng(82)
    rows, cols = rng.integers(0, nrows, 1000), rng.integers(0, 40, 1000)
    rows[417] = nrows
    arrays = [gpu.DeviceArray.from_host(a) for a in
              (rows.astype(np.int32), cols.astype(np.int32), rng.normal(size=1000))]
    before = [a.to_host() for a in arrays]
    rc = gpu.lib().cel_gpu_coo_sort(nrows, 40, 1000, *(a.ptr for a in arrays), 0, 0, 0, gpu.SORT_ROW_COL,
                                    gpu.MEM_DEVICE)
    assert rc == gpu.ERR_BAD_MATRIX
    for a, b in zip(arrays, before):
        np.testing.assert_array_equal(a.to_host(), b)
