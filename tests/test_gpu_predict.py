"""Margin prediction over packed trees against a plain numpy walk of the
model (value < threshold goes left, NaN and absent entries follow
default_left; binary32 sums in tree order): bit-identical at the edges of the
row tiles, for rows too wide for LDS, trees larger than the staged buffer,
models whose children are not neighbours, and models the packed form does not
hold."""
import json

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _random_tree(rng, cols, depth, shuffle):
    left, right, feat, cond, dleft, level = [-1], [-1], [0], [0.0], [0], [0]
    k = 0
    while k < len(left):
        if level[k] < depth and (level[k] == 0 or rng.random() < 0.93):
            left[k], right[k] = len(left), len(left) + 1
            feat[k], dleft[k] = int(rng.integers(cols)), int(rng.integers(2))
            cond[k] = float(np.float32(rng.normal()))
            for lst, v in ((left, -1), (right, -1), (feat, 0), (cond, 0.0), (dleft, 0), (level, level[k] + 1)):
                lst.extend([v, v])
        else:
            cond[k] = float(np.float32(rng.normal() * 0.1))
        k += 1
    n = len(left)
    ids = np.arange(n)
    if shuffle and n > 1:  # a preorder-like numbering: children are not neighbours
        ids[1:] = 1 + rng.permutation(n - 1)
    out = {key: [0] * n for key in ("left_children", "right_children", "split_indices", "split_conditions",
                                    "default_left", "parents", "loss_changes", "sum_hessian", "base_weights")}
    out["parents"][0] = 2147483647
    for i in range(n):
        k = int(ids[i])
        out["left_children"][k] = int(ids[left[i]]) if left[i] >= 0 else -1
        out["right_children"][k] = int(ids[right[i]]) if left[i] >= 0 else -1
        out["split_indices"][k], out["split_conditions"][k] = feat[i], cond[i]
        out["default_left"][k] = dleft[i]
        if left[i] >= 0:
            out["parents"][int(ids[left[i]])] = out["parents"][int(ids[right[i]])] = k
    return out


def _booster(xgb, trees, cols, objective="reg:squarederror"):
    model = {"version": [3, 5, 0], "learner": {
        "attributes": {}, "feature_names": [], "feature_types": [],
        "learner_model_param": {"base_score": "0.25", "num_class": "0", "num_feature": str(cols), "num_target": "1"},
        "objective": {"name": objective},
        "gradient_booster": {"name": "gbtree", "model": {"trees": trees, "tree_info": [0] * len(trees)}}}}
    return xgb.Booster(model_file=bytearray(json.dumps(model).encode()))


def _margins(trees, X, base):
    out = np.broadcast_to(np.asarray(base, np.float32), (len(X),)).copy()
    rows = np.arange(len(X))
    for t in trees:
        left, right = np.array(t["left_children"]), np.array(t["right_children"])
        feat, cond = np.array(t["split_indices"]), np.array(t["split_conditions"], np.float32)
        dleft = np.array(t["default_left"])
        at = np.zeros(len(X), np.int64)
        while np.any(left[at] >= 0):
            v = X[rows, feat[at]]
            go = np.where(np.isnan(v), dleft[at] != 0, v < cond[at])
            at = np.where(left[at] < 0, at, np.where(go, left[at], right[at]))
        out = out + cond[at]
    return out


def _values(rng, rows, cols, missing):
    X = rng.normal(size=(rows, cols)).astype(np.float32)
    X[rng.random(X.shape) < missing] = np.nan
    return X


@pytest.mark.parametrize("rows,cols,trees,depth,shuffle", [
    (1, 1, 1, 1, False), (3, 7, 130, 4, True), (64, 32, 65, 6, False), (12287, 5, 3, 3, False),
    (12288, 31, 9, 5, True), (12289, 64, 70, 8, False), (16384 + 63, 32, 33, 6, False),
    (70000, 9, 5, 4, False), (81921, 64, 7, 8, False), (13000, 200, 11, 5, False), (12500, 520, 6, 6, False),
    (12300, 1200, 5, 5, False), (12400, 4, 1100, 2, False), (13000, 6, 2, 13, False), (300, 6, 2, 12, False),
    (150000, 2, 1, 2, False)])
def test_margins_equal_plain_walk(xgb, rows, cols, trees, depth, shuffle):
    rng = np.random.default_rng(rows * 31 + cols)
    forest = [_random_tree(rng, cols, depth, shuffle) for _ in range(trees)]
    X = _values(rng, rows, cols, 0.1)
    bst = _booster(xgb, forest, cols)
    expect = _margins(forest, X, 0.25)
    np.testing.assert_array_equal(bst.predict(xgb.DMatrix(X), output_margin=True), expect)
    np.testing.assert_array_equal(bst.inplace_predict(X), expect)
    base = rng.normal(size=rows).astype(np.float32)
    np.testing.assert_array_equal(bst.predict(xgb.DMatrix(X, base_margin=base)), _margins(forest, X, base))
    if trees > 2:
        np.testing.assert_array_equal(bst.predict(xgb.DMatrix(X), iteration_range=(1, trees - 1)),
                                      _margins(forest[1:trees - 1], X, 0.25))


@pytest.mark.parametrize("rows,cols,trees,depth,share", [
    (1, 40, 3, 3, 0.2), (6143, 33, 70, 5, 0.3), (6144, 31, 12, 5, 1.0), (13001, 2000, 20, 6, 0.01),
    (20000, 64, 9, 8, 0.5), (12500, 30000, 4, 5, 0.002), (300, 33000, 3, 4, 0.01)])
def test_csr_margins_equal_plain_walk(xgb, rows, cols, trees, depth, share):
    """Rows of very uneven length, some empty; 33,000 features are past the
    packed form."""
    import scipy.sparse as sp
    rng = np.random.default_rng(rows + cols)
    used = rng.integers(0, cols, size=min(cols, 60))  # the columns the trees look at
    forest = [_random_tree(rng, len(used), depth, False) for _ in range(trees)]
    for t in forest:
        t["split_indices"] = [int(used[f]) for f in t["split_indices"]]
    nnz = np.minimum(rng.poisson(share * cols, size=rows), cols)
    nnz[0] = 0
    nnz[rows // 2] = min(cols, 4000)
    indptr = np.concatenate([[0], np.cumsum(nnz)])
    indices = np.concatenate([np.sort(rng.choice(cols, size=n, replace=False)) for n in nnz]).astype(np.int32)
    values = rng.normal(size=indptr[-1]).astype(np.float32)
    values[rng.random(len(values)) < 0.05] = np.nan
    csr = sp.csr_matrix((values, indices, indptr), shape=(rows, cols))
    small = np.full((rows, len(used)), np.nan, np.float32)
    position = {int(c): j for j, c in enumerate(used)}
    row_of = np.repeat(np.arange(rows), nnz)
    keep = np.isin(indices, used)
    small[row_of[keep], [position[int(c)] for c in indices[keep]]] = values[keep]
    plain = [dict(t, split_indices=[position[f] if l >= 0 else 0 for f, l in
                                    zip(t["split_indices"], t["left_children"])]) for t in forest]
    bst = _booster(xgb, forest, cols)
    np.testing.assert_array_equal(bst.predict(xgb.DMatrix(csr)), _margins(plain, small, 0.25))
    np.testing.assert_array_equal(bst.inplace_predict(csr), _margins(plain, small, 0.25))


def test_trees_added_and_replaced_are_predicted(xgb):
    """A booster that predicted keeps its packed trees: later rounds join
    them, and a loaded model takes their place."""
    rng = np.random.default_rng(3)
    X = _values(rng, 5000, 8, 0.1)
    y = np.nan_to_num(X[:, 0] - X[:, 1]).astype(np.float32)
    d, other = xgb.DMatrix(X, label=y), xgb.DMatrix(X[::-1].copy())
    params = {"max_depth": 5, "max_bin": 64}
    bst = xgb.train(params, d, 2)
    for rounds in (3, 9, 30):
        bst = xgb.train(params, d, rounds - bst.num_boosted_rounds(), xgb_model=bst)
        np.testing.assert_array_equal(bst.predict(other)[::-1], bst.predict(d))
    growing = xgb.Booster(params, [d])
    for r in range(6):
        growing.update(d, r)
        np.testing.assert_array_equal(growing.predict(other)[::-1], growing.predict(d))
    forest = [_random_tree(rng, 8, 4, False) for _ in range(3)]
    growing.load_model(_booster(xgb, forest, 8).save_raw())
    np.testing.assert_array_equal(growing.predict(other), _margins(forest, X[::-1], 0.25))


@pytest.mark.parametrize("rows", [7, 13000])
def test_logistic_output_is_the_sigmoid_of_the_margin(xgb, rows):
    rng = np.random.default_rng(rows)
    forest = [_random_tree(rng, 12, 5, False) for _ in range(20)]
    X = _values(rng, rows, 12, 0.2)
    bst = _booster(xgb, forest, 12, "binary:logistic")
    margin = bst.predict(xgb.DMatrix(X), output_margin=True)
    # Rounding of e^x, two sums and a division: a few units of 2^-24.
    np.testing.assert_allclose(bst.predict(xgb.DMatrix(X)), 1.0 / (1.0 + np.exp(-margin.astype(np.float64))),
                               rtol=4e-7, atol=0)


def _special_values(rng, forest, X):
    """Leaves of +0 and -0 at every depth (the leaves nearest the root among
    them) and thresholds at zeros, infinities and the rows' own values."""
    special = [0.0, -0.0, np.inf, -np.inf]
    flat = X[~np.isnan(X)]
    for t in forest:
        for k, left in enumerate(t["left_children"]):
            u = rng.random()
            if left < 0:
                t["split_conditions"][k] = 0.0 if u < 0.5 else -0.0 if u < 0.6 else t["split_conditions"][k]
            elif u < 0.5:
                t["split_conditions"][k] = float(special[rng.integers(4)] if u < 0.2 or not len(flat) else rng.choice(flat))
    X[rng.random(X.shape) < 0.1] = 0.0
    X[rng.random(X.shape) < 0.1] = -0.0
    X[rng.random(X.shape) < 0.05] = np.inf
    X[rng.random(X.shape) < 0.05] = -np.inf


def _stump(value):
    return {"left_children": [-1], "right_children": [-1], "split_indices": [0], "split_conditions": [value],
            "default_left": [0], "parents": [2147483647], "loss_changes": [0], "sum_hessian": [0], "base_weights": [0]}


def _same_bits(got, expect):
    np.testing.assert_array_equal(np.asarray(got, np.float32).view(np.uint32), expect.view(np.uint32))


@pytest.mark.parametrize("rows,cols,trees,depth,shuffle", [
    (1, 1, 1, 1, False), (16, 9, 130, 5, True), (300, 6, 3, 12, False), (12287, 31, 20, 6, True),
    (12289, 31, 20, 6, False), (20000, 64, 70, 8, False), (13000, 6, 2, 13, False), (12300, 1200, 5, 5, False)])
def test_leaves_of_zero_hold_the_walk(xgb, rows, cols, trees, depth, shuffle):
    """Single leaves of +0 before, between and after deeper trees, +0 and -0
    leaves above the deepest level, thresholds equal to the values compared."""
    rng = np.random.default_rng(rows * 7 + cols)
    forest = [_random_tree(rng, cols, depth if t % 3 == 0 else int(rng.integers(1, depth + 1)), shuffle)
              for t in range(trees)]
    X = _values(rng, rows, cols, 0.1)
    _special_values(rng, forest, X)
    forest = [_stump(0.0), *forest[:1], _stump(0.0), *forest[1:], _stump(-0.0), _stump(0.0)]
    bst = _booster(xgb, forest, cols)
    loaded = json.loads(bst.save_raw("json"))["learner"]["gradient_booster"]["model"]["trees"]
    expect = _margins(loaded, X, 0.25)
    _same_bits(bst.predict(xgb.DMatrix(X)), expect)
    _same_bits(bst.inplace_predict(X), expect)
    base = rng.normal(size=rows).astype(np.float32)
    base[::2] = -0.0
    _same_bits(bst.predict(xgb.DMatrix(X, base_margin=base)), _margins(loaded, X, base))
    _same_bits(bst.predict(xgb.DMatrix(X), iteration_range=(0, 1)), _margins(loaded[:1], X, 0.25))
    _same_bits(bst.predict(xgb.DMatrix(X), iteration_range=(2, len(loaded))), _margins(loaded[2:], X, 0.25))
    _same_bits(_booster(xgb, [_stump(0.0)], cols).predict(xgb.DMatrix(X)), np.full(rows, 0.25, np.float32))


@pytest.mark.parametrize("rows,cols,trees,depth", [(5, 40, 9, 4), (6145, 33, 70, 6), (13000, 2000, 20, 7)])
def test_leaves_of_zero_hold_the_walk_csr(xgb, rows, cols, trees, depth):
    import scipy.sparse as sp
    rng = np.random.default_rng(rows + cols)
    used = np.sort(rng.choice(cols, size=min(cols, 50), replace=False))
    forest = [_random_tree(rng, len(used), 1 + t % depth, False) for t in range(trees)]
    small = _values(rng, rows, len(used), 0.6)
    _special_values(rng, forest, small)
    forest = [_stump(0.0), *forest, _stump(0.0)]
    r, c = np.nonzero(~np.isnan(small))
    csr = sp.csr_matrix((small[r, c], (r, used[c])), shape=(rows, cols))
    wide = [dict(t, split_indices=[int(used[f]) for f in t["split_indices"]]) for t in forest]
    bst = _booster(xgb, wide, cols)
    loaded = json.loads(bst.save_raw("json"))["learner"]["gradient_booster"]["model"]["trees"]
    plain = [dict(t, split_conditions=l["split_conditions"]) for t, l in zip(forest, loaded)]
    expect = _margins(plain, small, 0.25)
    _same_bits(bst.predict(xgb.DMatrix(csr)), expect)
    _same_bits(bst.inplace_predict(csr), expect)


@pytest.mark.parametrize("rows", [700, 13000])
def test_fits_with_leaves_of_zero(xgb, rows):
    """A learning rate that reaches 0, rows without weight and gradients of 0
    leave +0 and -0 leaves; a new matrix of the training rows gets the training
    margins."""
    rng = np.random.default_rng(rows)
    X = _values(rng, rows, 6, 0.1)
    y = (np.nan_to_num(X[:, 0]) * np.nan_to_num(X[:, 1])).astype(np.float32)
    weight = (np.nan_to_num(X[:, 2]) > 0).astype(np.float32)
    params = {"max_depth": 5, "max_bin": 32, "eta": 0.4, "min_child_weight": 0, "lambda": 0}
    schedule = xgb.callback.LearningRateScheduler(lambda r: 0.4 if r < 3 else 0.0)

    def nothing(margin, dtrain):
        return np.zeros(rows, np.float32), np.ones(rows, np.float32)

    fits = [xgb.train(params, xgb.DMatrix(X, label=y), 6, callbacks=[schedule]),
            xgb.train(params, xgb.DMatrix(X, label=y, weight=weight), 4),
            xgb.train(params, xgb.DMatrix(X, label=y), 3, obj=nothing)]
    for bst in fits:
        trees = json.loads(bst.save_raw("json"))["learner"]["gradient_booster"]["model"]["trees"]
        base = float(json.loads(bst.save_raw("json"))["learner"]["learner_model_param"]["base_score"].strip("[]"))
        expect = _margins(trees, X, base)
        np.testing.assert_array_equal(bst.predict(xgb.DMatrix(X), output_margin=True), expect)
        np.testing.assert_array_equal(bst.inplace_predict(X), expect)
    zeros = json.loads(fits[0].save_raw("json"))["learner"]["gradient_booster"]["model"]["trees"][-1]
    assert any(l < 0 and v == 0 for l, v in zip(zeros["left_children"], zeros["split_conditions"]))


def _chain(rng, cols, depth):
    """A tree whose every right child is split again, `depth` levels down."""
    n = 2 * depth + 1
    inner = [0] + [2 * d for d in range(1, depth)]
    left, right = [-1] * n, [-1] * n
    for d, k in enumerate(inner):
        left[k], right[k] = 2 * d + 1, 2 * d + 2
    cond = [float(np.float32(-1.0 - rng.random())) if left[k] >= 0 else float(np.float32(rng.normal())) for k in range(n)]
    parents = [2147483647] + [0] * (n - 1)
    for k in inner:
        parents[left[k]] = parents[right[k]] = k
    return {"left_children": left, "right_children": right, "split_indices": [int(f) for f in rng.integers(cols, size=n)],
            "split_conditions": cond, "default_left": [0] * n, "parents": parents, "loss_changes": [0] * n,
            "sum_hessian": [0] * n, "base_weights": [0] * n}


@pytest.mark.parametrize("rows,cols,trees,depth,chain", [
    (1, 5, 1, 8, 0), (63, 5, 1, 9, 0), (65, 9, 2, 4, 0), (12289, 9, 1, 6, 0), (49151, 120, 2, 4, 0), (49152, 120, 2, 4, 0),
    (50000, 120, 3, 3, 0), (50000, 1200, 12, 6, 0), (50000, 1200, 13, 6, 0), (13000, 6, 30, 3, 150), (300, 6, 30, 3, 150),
    (32769, 6, 3, 3, 500), (12300, 6, 1, 3, 3000)])
def test_margins_where_rows_take_few_or_uneven_steps(xgb, rows, cols, trees, depth, chain):
    """Both sides of the limits of the row-a-lane kernel: few steps a row, wide
    rows of some steps, one tree much deeper than the others."""
    import scipy.sparse as sp
    rng = np.random.default_rng(rows + cols + trees)
    forest = [_random_tree(rng, cols, depth, False) for _ in range(trees)]
    if chain:
        forest.insert(1, _chain(rng, cols, chain))
    X = _values(rng, rows, cols, 0.15)
    _special_values(rng, forest[:1] if chain else forest, X)
    bst = _booster(xgb, forest, cols)
    base = rng.normal(size=rows).astype(np.float32)
    expect = _margins(forest, X, base)
    _same_bits(bst.predict(xgb.DMatrix(X, base_margin=base)), expect)
    keep = np.arange(rows) if cols <= 120 else np.arange(7000)
    r, c = np.nonzero(~np.isnan(X[keep]))
    csr = sp.csr_matrix((X[r, c], (r, c)), shape=(len(keep), cols))
    _same_bits(bst.predict(xgb.DMatrix(csr, base_margin=base[keep])), expect[keep])
    _same_bits(bst.predict(xgb.DMatrix(X), iteration_range=(0, 1)), _margins(forest[:1], X, 0.25))
    logistic = _booster(xgb, forest, cols, "binary:logistic")
    margin = logistic.predict(xgb.DMatrix(X), output_margin=True).astype(np.float64)
    np.testing.assert_allclose(logistic.predict(xgb.DMatrix(X)), 1.0 / (1.0 + np.exp(-margin)), rtol=4e-7, atol=0)
