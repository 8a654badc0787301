"""Bin codes against a count of the cuts at or below each value: both code
widths, every layout with its column-major copy, row counts and tiles whose
codes leave in whole words and those that do not, tiles that hold padding
features only, and one cut to 4,096 a feature."""
import ctypes

import numpy as np
import pytest

import device_lib as D

pytestmark = pytest.mark.gpu


def _codes(X, cuts, counts, missing):
    out = np.full(X.shape, missing, np.int64)
    for f in range(X.shape[1]):
        v = X[:, f]
        ok = ~np.isnan(v)
        if counts[f]:
            out[ok, f] = np.minimum(np.searchsorted(cuts[f, :counts[f]], v[ok], side="right"), counts[f] - 1)
    return out


@pytest.mark.parametrize("rows", [1, 127, 128, 4100, 4101, 70002])
@pytest.mark.parametrize("cols,stride", [(1, 2), (3, 255), (21, 256), (70, 256), (19, 1000), (5, 4096), (130, 1)])
@pytest.mark.parametrize("bin_bytes,G,group_major", [
    (1, 1, False), (1, 1, True), (1, 2, True), (1, 4, False), (1, 16, True), (2, 1, True), (2, 2, True),
    (2, 16, False), (2, 8, True)])
def test_codes_match_cut_counts(rows, cols, stride, bin_bytes, G, group_major):
    rng = np.random.default_rng(rows * 131 + cols)
    if bin_bytes == 1:
        stride = min(stride, 255)
    counts = rng.integers(1, stride + 1, cols).astype(np.uint32)
    counts[0] = stride
    cuts = np.full((cols, stride), 7.5, np.float32)  # past a feature's cuts lie other values
    for f in range(cols):
        cuts[f, :counts[f]] = np.sort(rng.normal(size=counts[f])).astype(np.float32)
    X = rng.normal(size=(rows, cols)).astype(np.float32)
    on = rng.random(X.shape) < 0.2  # on a cut: counted
    X[on] = np.take_along_axis(cuts.T, rng.integers(0, 1 << 30, (rows, cols)) % counts, axis=0)[on]
    X[rng.random(X.shape) < 0.1] = np.nan
    X[rng.random(X.shape) < 0.02] = np.inf
    X[rng.random(X.shape) < 0.02] = -np.inf
    m, dbins, bins, missing = D.quantize_bins(X, cuts, counts, stride, bin_bytes, G, group_major=group_major)
    want = _codes(X, cuts, counts, 0xFF if bin_bytes == 1 else 0xFFFF)
    np.testing.assert_array_equal(bins[:, :cols], want)
    assert missing == bool(np.isnan(X).any())
    # The column-major copy, the buffer after it untouched.
    dtype = np.uint8 if bin_bytes == 1 else np.uint16
    dX, dcuts, dcounts, flag = D.Device.of(X), D.Device.of(cuts), D.Device.of(counts), D.Device(4)
    columns = D.Device.of(np.full(rows * cols + 64, 0x5A, dtype))
    D.check(D.lib().mgb_quantize_bins_columns(dX.ptr, dcuts.ptr, dcounts.ptr, ctypes.byref(m), dbins.ptr, columns.ptr,
                                              flag.ptr))
    got = columns.read(dtype, rows * cols + 64)
    np.testing.assert_array_equal(got[:rows * cols].reshape(cols, rows).T, want)
    assert (got[rows * cols:] == 0x5A).all()


@pytest.mark.parametrize("count", [1, 63, 255, 256, 2047, 2049, 300001, 5000003])
def test_missing_scan(count):
    X = np.ones(count, np.float32)
    for at in (None, 0, count // 2, count - 1):
        if at is not None:
            X[:] = 1
            X[at] = np.nan
        dX, flag = D.Device.of(X), D.Device(4)
        D.check(D.lib().mgb_any_missing(dX.ptr, ctypes.c_uint64(count), flag.ptr))
        assert flag.read(np.uint32, 1)[0] == (0 if at is None else 1)
