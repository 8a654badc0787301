"""Scratch of exact contributions (mgb_shap_scratch_bytes, the plan that
mgb_predict_shap allocates by): at most 256 MB whatever the rows, the features
and the leaves, and enough for a tile's keys and one partial; host arithmetic,
no device."""
import ctypes

import pytest

import device_lib as D


def _scratch(rows, features, leaves, elements=8):
    p = D.MgbShap(rows=rows, cols=features, leaves=leaves, elements=elements, trees=1, features=features)
    D.lib().mgb_shap_scratch_bytes.restype = ctypes.c_size_t
    return D.lib().mgb_shap_scratch_bytes(ctypes.byref(p))


@pytest.mark.parametrize("rows", [1, 63, 64, 65, 700, 5000, 1_000_000, 2**32 - 1])
@pytest.mark.parametrize("features", [0, 1, 32, 64, 65, 199, 200, 299, 300, 700, 2000, 16_000, 20_000, 100_000, 174_000,
                                      350_000, 524_286])
def test_scratch_is_bounded(rows, features):
    tile = (features + 1) * 64 * 4
    blocks = (256 << 20) // tile
    walk = blocks < 64 and (rows + 63) // 64 > 6 * blocks
    for leaves in (0, 1, 100, 25_600, 6_553_600, 2**32 - 1):
        got = _scratch(rows, features, leaves)
        if walk:
            assert got == 0
        else:
            assert 2 * tile <= got <= 256 << 20, (rows, features, leaves, got)


def test_no_plan_past_the_bound():
    """One partial beside the keys no longer fits: the caller walks the tree
    records instead (mgb_predict_contribs)."""
    for features in (524_288, 1 << 24, 2**32 - 1):
        assert _scratch(64, features, 1000) == 0
    assert _scratch(0, 10, 10) == 0
