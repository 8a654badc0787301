"""Dense matrices keep the values they were given, around the sizes where the
host copy takes large pages (4 MiB) and several threads (8 MiB on, up to eight
shares of 4 MiB, the last one ragged)."""
import numpy as np
import pytest

import device_lib as D


@pytest.mark.parametrize("rows,cols", [
    (1, 1), (1, (1 << 20) - 1), (1 << 20, 1), ((1 << 20) + 1, 1), ((1 << 21) - 1, 1), (1 << 21, 1), (700001, 3),
    (131071, 73)])
@pytest.mark.parametrize("form", ["float32", "strided", "float64", "missing"])
def test_dense_values_survive(xgb, rows, cols, form):
    n = rows * cols
    values = np.arange(n, dtype=np.float32).reshape(rows, cols)  # below 2^24: all distinct
    given, missing = values, np.nan
    if form == "strided":
        wide = np.full((rows, cols + 1), np.nan, np.float32)
        wide[:, :cols] = values
        given = wide[:, :cols]
    elif form == "float64":
        given = values.astype(np.float64)
    elif form == "missing":
        missing = float(n - 1)
    got = xgb.DMatrix(given, missing=missing).get_data()
    want = values.reshape(-1)[:-1] if form == "missing" else values.reshape(-1)
    assert got.shape == values.shape
    np.testing.assert_array_equal(got.data, want)
    np.testing.assert_array_equal(got.indices, np.tile(np.arange(cols), rows)[:len(want)])


def test_empty_matrix(xgb):
    assert xgb.DMatrix(np.empty((0, 4), np.float32)).num_row() == 0


# Uploads from 8 MiB on go through pinned chunks of 2 MiB, filled by six threads
# with two chunks each: below, at and past the limit, ragged last chunks, and
# several turns of every chunk.
@pytest.mark.gpu
@pytest.mark.parametrize("nbytes", [
    (8 << 20) - 1, 8 << 20, (8 << 20) + 1, (12 << 20) + 4097, (24 << 20) + 2, (26 << 20) - 3, (70 << 20) + 5])
def test_large_uploads(nbytes):
    rng = np.random.default_rng(nbytes)
    for _ in range(2):
        host = rng.integers(0, 256, nbytes, dtype=np.uint8)
        dev = D.Device.of(host)
        host_after = host.copy()
        host[:] = 0  # the copy is complete when the call returns
        np.testing.assert_array_equal(dev.read(np.uint8, nbytes), host_after)


@pytest.mark.parametrize("rows,cols", [(1, 1), (7, 1), (1, 9), (13, 5), (1000, 17)])
@pytest.mark.parametrize("dtype", ["float16", "float32", "float64", "int8", "uint16", "int32", "int64", "bool"])
def test_layouts_and_types_keep_their_values(xgb, rows, cols, dtype):
    """Every order and stride of every element type, 1-dimensional labels among
    them."""
    rng = np.random.default_rng(rows * 31 + cols)
    plain = rng.integers(0, 2 if dtype == "bool" else 100, size=(rows, cols)).astype(dtype)
    wide = np.zeros((2 * rows, 3 * cols), dtype)
    wide[::2, ::3] = plain
    want = plain.astype(np.float32)
    for given in (plain, np.asfortranarray(plain), wide[::2, ::3], plain[::-1, ::-1][::-1, ::-1], wide[::2, ::3][::-1][::-1]):
        got = xgb.DMatrix(given).get_data()
        np.testing.assert_array_equal(got.toarray(), want)
    reverse = xgb.DMatrix(plain[::-1, ::-1]).get_data()
    np.testing.assert_array_equal(reverse.toarray(), want[::-1, ::-1])
    labelled = xgb.DMatrix(plain, label=wide[::2, 0])
    np.testing.assert_array_equal(labelled.get_label(), want[:, 0])


@pytest.mark.parametrize("kind", ["csr", "csc", "coo"])
def test_sparse_offsets_and_columns_past_2_24(xgb, kind):
    """Offsets and indices that binary32 does not hold."""
    import scipy.sparse as sp
    n = (1 << 24) + 1
    if kind == "csr":
        # Row 0 is column 0's .. 2^24's, row 1 one entry behind them.
        m = sp.csr_matrix((np.ones(n + 1, np.float32), np.append(np.arange(n), n).astype(np.int64),
                           np.array([0, n, n + 1], np.int64)), shape=(2, n + 2))
    elif kind == "csc":
        m = sp.csc_matrix((np.ones(n + 1, np.float32), np.append(np.arange(n), n).astype(np.int64),
                           np.array([0, n, n + 1], np.int64)), shape=(n + 2, 2))
    else:
        m = sp.coo_matrix((np.array([3.0, 4.0], np.float32), (np.array([n, 5]), np.array([1, n]))), shape=(n + 2, n + 2))
    got = xgb.DMatrix(m).get_data()
    want = m.tocsr()
    assert got.shape == want.shape
    np.testing.assert_array_equal(got.indptr, want.indptr)
    np.testing.assert_array_equal(got.indices, want.indices)
    np.testing.assert_array_equal(got.data, want.data)
