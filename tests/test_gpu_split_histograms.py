"""Small matrices' levels, whose split items build their own histograms from
the column-major codes, against the histogram launches (which a matrix without
the column copy, hip_partition_columns=0, takes at every level): the same
trees and margins bit for bit, over row counts around the limits, both code
widths, every bin count's item shape, unit and weighted Hessians, sampling,
missing values and constraints."""
import json

import numpy as np
import pytest

import workloads as W

pytestmark = pytest.mark.gpu


def _both(xgb, X, y, params, rounds, weight=None):
    out = []
    for columns in (1, 0):
        d = xgb.DMatrix(X, label=y, weight=weight)
        bst = xgb.train(dict(params, hip_partition_columns=columns), d, rounds)
        trees = json.loads(bst.save_raw("json"))["learner"]["gradient_booster"]["model"]["trees"]
        out.append((trees, bst.predict(d, output_margin=True)))
    assert out[0][0] == out[1][0]
    np.testing.assert_array_equal(out[0][1], out[1][1])
    return out[0][0]


@pytest.mark.parametrize("rows,cols,depth,max_bin", [
    (2, 1, 2, 16), (65, 3, 4, 2), (257, 17, 6, 256), (5003, 20, 6, 256), (4099, 70, 8, 256), (3000, 9, 10, 64),
    (2500, 5, 5, 300), (6000, 12, 7, 1024), (6000, 3, 4, 4096), (5000, 3, 12, 4096), (33000, 8, 3, 256),
    (65536, 6, 4, 255), (65537, 6, 4, 255)])
@pytest.mark.parametrize("missing", [False, True])
def test_same_trees_as_histogram_launches(xgb, rows, cols, depth, max_bin, missing):
    X, y = W.config1(rows=rows, cols=cols) if missing else W.config0(rows=rows, cols=cols)
    trees = _both(xgb, X, y, {"max_depth": depth, "max_bin": max_bin, "eta": 0.5}, 3)
    if rows > 1000:
        assert max(len(t["left_children"]) for t in trees) > 2 * depth


@pytest.mark.parametrize("extra", [
    {"objective": "binary:logistic"}, {"subsample": 0.6, "colsample_bytree": 0.5, "seed": 3},
    {"objective": "binary:logistic", "subsample": 0.5, "scale_pos_weight": 3.0},
    {"monotone_constraints": "(1,-1,0,1)"}, {"reg_alpha": 0.5, "max_delta_step": 0.7},
    {"hip_stable_partition": 1}, {"hip_histogram_features": 2, "hip_bin_layout": "group"}])
def test_same_trees_over_options(xgb, extra):
    X, y = W.config1(rows=7001, cols=11)
    if "logistic" in extra.get("objective", ""):
        y = (y > 0).astype(np.float32)
    params = {"max_depth": 6, "max_bin": 128, **extra}
    _both(xgb, X, y, params, 4)
    _both(xgb, X, y, params, 4, weight=np.random.default_rng(1).uniform(0, 2, 7001).astype(np.float32))


@pytest.mark.parametrize("rows,share", [(70000, 0.9), (80000, 0.9), (150000, 1.0), (600000, 0.95)])
def test_csr_row_tiles_train_the_same_trees(xgb, rows, share):
    """CSR row tiles are work units only: the default, which grows with a
    column's entries (64 rows up to 65,536, 512 from 262,145 on), and given ones
    train the same trees."""
    import scipy.sparse as sp
    rng = np.random.default_rng(rows)
    dense = rng.normal(size=(rows, 3)).astype(np.float32)
    dense[rng.random(dense.shape) > share] = 0
    y = (dense[:, 0] * dense[:, 1] + 0.2 * rng.normal(size=rows)).astype(np.float32)
    d = xgb.DMatrix(sp.csr_matrix(dense), label=y)
    params = {"max_depth": 5, "max_bin": 64, "eta": 0.5}
    models = []
    for extra in ({}, {"hip_histogram_rows": 64}, {"hip_histogram_rows": 512}):
        bst = xgb.train({**params, **extra}, d, 2)
        models.append(json.loads(bst.save_raw("json"))["learner"]["gradient_booster"]["model"]["trees"])
    assert models[0] == models[1] == models[2]


@pytest.mark.parametrize("rows,cols", [(40960, 5), (40961, 5), (49153, 47), (49153, 48)])
def test_same_trees_of_few_columns(xgb, rows, cols):
    X, y = W.config1(rows=rows, cols=cols)
    _both(xgb, X, y, {"max_depth": 5, "max_bin": 200}, 2)
    _both(xgb, X, (y > 0).astype(np.float32), {"max_depth": 5, "max_bin": 200, "objective": "binary:logistic"}, 2)
