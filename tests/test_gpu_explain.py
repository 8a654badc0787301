"""Leaf indices, feature contributions and their interactions on the GPU
(reference src/learner.cpp:455-560, prediction types 2 to 6), checked against
references computed here from the saved model JSON:

- leaf ids: a plain walk of every tree (value < threshold goes left, NaN
  follows default_left);
- approximate contributions: each split's feature credited with the change
  of the cover-weighted node mean along the row's path, in binary64;
- exact contributions: Shapley values by their definition, over every subset
  of the features, with the path-dependent value function TreeSHAP computes
  (a tree's expectation where the subset fixes a feature the walk follows the
  row, elsewhere the children are weighted by their cover), in binary64;
- exact interactions: the Shapley interaction index by its definition, and on
  the diagonal each feature's value less its interactions; approximate ones
  carry the approximate contributions on the diagonal.

The kernels compute in binary32, so contributions compare within 2e-5 of the
margin's scale; leaf ids are exact.  Local accuracy (contributions plus bias
equal the margin prediction) is checked on every case."""
import json
import math
from itertools import combinations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


class _Tree:
    def __init__(self, t):
        self.left = np.array(t["left_children"], dtype=np.int64)
        self.right = np.array(t["right_children"], dtype=np.int64)
        self.feature = np.array(t["split_indices"], dtype=np.int64)
        self.cond = np.array(t["split_conditions"], dtype=np.float32)
        self.dleft = np.array(t["default_left"], dtype=bool)
        self.cover = np.array(t["sum_hessian"], dtype=np.float64)
        self.mean = np.zeros(len(self.left))
        for k in range(len(self.left) - 1, -1, -1):
            l, r = self.left[k], self.right[k]
            self.mean[k] = (float(self.cond[k]) if l < 0 else
                            (self.mean[l] * self.cover[l] + self.mean[r] * self.cover[r]) / self.cover[k])

    def child(self, k, x):
        v = x[self.feature[k]]
        go_left = self.dleft[k] if np.isnan(v) else v < self.cond[k]
        return self.left[k] if go_left else self.right[k]

    def leaf(self, x):
        k = 0
        while self.left[k] >= 0:
            k = self.child(k, x)
        return k

    def expect(self, x, subset, k=0):
        """E[tree | the features in `subset` fixed at x], path-dependent."""
        if self.left[k] < 0:
            return float(self.cond[k])
        if self.feature[k] in subset:
            return self.expect(x, subset, self.child(k, x))
        l, r = self.left[k], self.right[k]
        return (self.cover[l] * self.expect(x, subset, l) + self.cover[r] * self.expect(x, subset, r)) / self.cover[k]


def _trees(bst):
    model = json.loads(bytes(bst.save_raw("json")))
    return [_Tree(t) for t in model["learner"]["gradient_booster"]["model"]["trees"]]


def _shapley(trees, x, cols):
    phi = np.zeros(cols)
    for f in range(cols):
        others = [g for g in range(cols) if g != f]
        for size in range(cols):
            w = math.factorial(size) * math.factorial(cols - size - 1) / math.factorial(cols)
            for s in combinations(others, size):
                s = set(s)
                phi[f] += w * sum(t.expect(x, s | {f}) - t.expect(x, s) for t in trees)
    return phi


def _interactions(trees, x, cols):
    """SHAP interaction values by their definition: off the diagonal the
    Shapley interaction index over every subset of the other features, on it
    the feature's Shapley value less its interactions."""
    def f(s):
        return sum(t.expect(x, s) for t in trees)
    phi = _shapley(trees, x, cols)
    m = np.zeros((cols + 1, cols + 1))
    for i in range(cols):
        for j in range(cols):
            if i == j:
                continue
            others = [g for g in range(cols) if g not in (i, j)]
            for size in range(cols - 1):
                w = math.factorial(size) * math.factorial(cols - size - 2) / (2 * math.factorial(cols - 1))
                for s in combinations(others, size):
                    s = set(s)
                    m[i, j] += w * (f(s | {i, j}) - f(s | {i}) - f(s | {j}) + f(s))
        m[i, i] = phi[i] - sum(m[i, j] for j in range(cols) if j != i)
    return m


def _saabas(trees, x, cols):
    phi = np.zeros(cols + 1)
    for t in trees:
        k = 0
        phi[cols] += t.mean[0]
        while t.left[k] >= 0:
            nxt = t.child(k, x)
            phi[t.feature[k]] += t.mean[nxt] - t.mean[k]
            k = nxt
    return phi


def _data(rows=60, cols=5, seed=7, missing=0.15):
    rng = np.random.default_rng(seed)
    X = rng.normal(size=(rows, cols)).astype(np.float32)
    y = (X[:, 0] * 1.5 - X[:, 1] + 0.5 * X[:, 2] * X[:, 3] + 0.1 * rng.normal(size=rows)).astype(np.float32)
    X[rng.random(X.shape) < missing] = np.nan
    return X, y


@pytest.mark.parametrize("objective", ["reg:squarederror", "binary:logistic"])
def test_leaf_and_contributions_match_definitions(xgb, objective):
    X, y = _data()
    if objective == "binary:logistic":
        y = (y > 0).astype(np.float32)
    d = xgb.DMatrix(X, label=y)
    bst = xgb.train({"objective": objective, "max_depth": 3, "max_bin": 32, "eta": 0.5}, d, 4)
    trees = _trees(bst)
    margin = bst.predict(d, output_margin=True).astype(np.float64)
    scale = max(1.0, float(np.abs(margin).max()))

    leaf = bst.predict(d, pred_leaf=True)
    assert leaf.shape == (len(X), 4) and leaf.dtype == np.float32
    expect = np.array([[t.leaf(x) for t in trees] for x in X], dtype=np.float32)
    np.testing.assert_array_equal(leaf, expect)

    approx = bst.predict(d, pred_contribs=True, approx_contribs=True).astype(np.float64)
    assert approx.shape == (len(X), X.shape[1] + 1)
    base = margin - np.array([sum(float(t.cond[t.leaf(x)]) for t in trees) for x in X])
    for i, x in enumerate(X):
        ref = _saabas(trees, x, X.shape[1])
        ref[-1] += base[i]
        np.testing.assert_allclose(approx[i], ref, rtol=0, atol=2e-5 * scale)
    np.testing.assert_allclose(approx.sum(axis=1), margin, rtol=0, atol=2e-5 * scale)

    exact = bst.predict(d, pred_contribs=True).astype(np.float64)
    assert exact.shape == (len(X), X.shape[1] + 1)
    for i, x in enumerate(X[:20]):
        phi = _shapley(trees, x, X.shape[1])
        np.testing.assert_allclose(exact[i, :-1], phi, rtol=0, atol=2e-5 * scale)
        np.testing.assert_allclose(exact[i, -1], base[i] + sum(t.mean[0] for t in trees), rtol=0, atol=2e-5 * scale)
    np.testing.assert_allclose(exact.sum(axis=1), margin, rtol=0, atol=2e-5 * scale)


def test_contributions_csr_equal_dense_and_follow_base_margin(xgb):
    import scipy.sparse as sp
    X, y = _data(rows=80, cols=6, seed=11, missing=0.3)
    bst = xgb.train({"max_depth": 4, "max_bin": 64, "eta": 0.3}, xgb.DMatrix(X, label=y), 5)
    rows, cols = np.nonzero(~np.isnan(X))
    csr = sp.csr_matrix((X[rows, cols], (rows, cols)), shape=X.shape)
    dense, sparse = xgb.DMatrix(X), xgb.DMatrix(csr)
    for kw in ({"pred_leaf": True}, {"pred_contribs": True}, {"pred_contribs": True, "approx_contribs": True}):
        np.testing.assert_array_equal(bst.predict(dense, **kw), bst.predict(sparse, **kw))
    offset = np.linspace(-1.0, 1.0, len(X)).astype(np.float32)
    shifted = xgb.DMatrix(X, base_margin=offset)
    plain = bst.predict(dense, pred_contribs=True)
    moved = bst.predict(shifted, pred_contribs=True)
    np.testing.assert_array_equal(moved[:, :-1], plain[:, :-1])
    base = float(plain[0, -1]) - sum(t.mean[0] for t in _trees(bst))
    np.testing.assert_allclose(moved[:, -1] - plain[:, -1], offset - base, rtol=0, atol=1e-5)
    np.testing.assert_allclose(moved.sum(axis=1), bst.predict(shifted, output_margin=True), rtol=0, atol=1e-4)


def test_deep_trees_are_locally_accurate_and_shaped(xgb):
    X, y = _data(rows=300, cols=6, seed=3, missing=0.05)
    d = xgb.DMatrix(X, label=y)
    bst = xgb.train({"max_depth": 9, "max_bin": 128, "eta": 0.3}, d, 6)
    margin = bst.predict(d, output_margin=True)
    exact = bst.predict(d, pred_contribs=True)
    np.testing.assert_allclose(exact.sum(axis=1), margin, rtol=0, atol=1e-4 * max(1.0, np.abs(margin).max()))
    trees = _trees(bst)
    for x, row in zip(X[:2], exact[:2]):
        np.testing.assert_allclose(row[:-1], _shapley(trees, x, X.shape[1]), rtol=0, atol=1e-4)
    # Rounds [0, 3) only.
    part = bst.predict(d, pred_contribs=True, iteration_range=(0, 3))
    np.testing.assert_allclose(part.sum(axis=1), bst.predict(d, output_margin=True, iteration_range=(0, 3)),
                               rtol=0, atol=1e-4)
    assert bst.predict(d, pred_leaf=True, strict_shape=True).shape == (len(X), 6, 1, 1)
    assert bst.predict(d, pred_contribs=True, strict_shape=True).shape == (len(X), 1, X.shape[1] + 1)
    assert bst.predict(d, pred_leaf=True, iteration_range=(0, 2)).shape == (len(X), 2)


def test_interactions_match_definitions(xgb):
    X, y = _data(rows=40, cols=5, seed=5)
    d = xgb.DMatrix(X, label=y)
    bst = xgb.train({"max_depth": 3, "max_bin": 32, "eta": 0.5}, d, 3)
    trees = _trees(bst)
    margin = bst.predict(d, output_margin=True).astype(np.float64)
    scale = max(1.0, float(np.abs(margin).max()))
    exact = bst.predict(d, pred_interactions=True).astype(np.float64)
    assert exact.shape == (len(X), 6, 6)
    contribs = bst.predict(d, pred_contribs=True).astype(np.float64)
    for i, x in enumerate(X[:12]):
        ref = _interactions(trees, x, 5)
        np.testing.assert_allclose(exact[i, :5, :5], ref[:5, :5], rtol=0, atol=2e-5 * scale)
    np.testing.assert_allclose(exact[:, :5, :5].sum(axis=2), contribs[:, :5], rtol=0, atol=2e-5 * scale)
    np.testing.assert_allclose(exact[:, 5, 5], contribs[:, 5], rtol=0, atol=1e-6 * scale)
    np.testing.assert_array_equal(exact[:, 5, :5], 0.0)
    np.testing.assert_array_equal(exact[:, :5, 5], 0.0)
    np.testing.assert_allclose(exact.sum(axis=(1, 2)), margin, rtol=0, atol=2e-5 * scale)
    approx = bst.predict(d, pred_interactions=True, approx_contribs=True)
    saabas = bst.predict(d, pred_contribs=True, approx_contribs=True)
    assert approx.shape == (len(X), 6, 6)
    np.testing.assert_array_equal(np.diagonal(approx, axis1=1, axis2=2), saabas)
    off = approx.copy()
    off[:, np.arange(6), np.arange(6)] = 0.0
    np.testing.assert_array_equal(off, 0.0)
    assert bst.predict(d, pred_interactions=True, strict_shape=True).shape == (len(X), 1, 6, 6)


def test_nonzero_start_and_two_types_are_refused(xgb):
    X, y = _data(rows=40, cols=4)
    d = xgb.DMatrix(X, label=y)
    bst = xgb.train({"max_depth": 2}, d, 3)
    assert bst.predict(d, pred_leaf=True, iteration_range=(0, 1)).shape == (len(X),)
    with pytest.raises(xgb.XGBoostError, match="only iteration end"):
        bst.predict(d, pred_contribs=True, iteration_range=(1, 3))
    with pytest.raises(ValueError, match="One type of prediction"):
        bst.predict(d, pred_leaf=True, pred_contribs=True)


def test_interpret_shap_values_split_the_bias(xgb):
    X, y = _data(rows=50, cols=4, seed=9)
    model = xgb.XGBRegressor(n_estimators=4, max_depth=3, max_bin=32)
    model.fit(X, y)
    values, bias = xgb.interpret.shap_values(model, X)
    contribs = model.get_booster().predict(xgb.DMatrix(X), pred_contribs=True)
    np.testing.assert_array_equal(values, contribs[:, :-1])
    np.testing.assert_array_equal(bias, contribs[:, -1])
    with pytest.raises(NotImplementedError):
        xgb.interpret.shap_values(model, X, X_background=X)
    with pytest.raises(ValueError):
        xgb.interpret.shap_values(model.get_booster(), xgb.DMatrix(X), missing=0.0)


def test_empty_matrix_and_untrained_model(xgb):
    X, y = _data(rows=30, cols=4)
    d = xgb.DMatrix(X, label=y)
    fresh = xgb.Booster({"max_depth": 2}, [d])
    contribs = fresh.predict(d, pred_contribs=True)
    assert contribs.shape == (30, 5)
    np.testing.assert_array_equal(contribs[:, :4], 0.0)
    np.testing.assert_allclose(contribs[:, 4], fresh.predict(d, output_margin=True), rtol=0, atol=1e-6)
    assert fresh.predict(d, pred_leaf=True).shape == (30, 0)
    bst = xgb.train({"max_depth": 2}, d, 2)
    empty = xgb.DMatrix(np.zeros((0, 4), dtype=np.float32))
    assert bst.predict(empty, pred_contribs=True).shape == (0, 5)
    assert bst.predict(empty, pred_interactions=True).shape == (0, 5, 5)
    assert bst.predict(empty, pred_leaf=True).size == 0


def test_estimator_apply_returns_leaf_ids(xgb):
    X, y = _data(rows=50, cols=4, seed=13)
    model = xgb.XGBRegressor(n_estimators=3, max_depth=3, max_bin=32)
    model.fit(X, y)
    leaves = model.apply(X)
    assert leaves.shape == (50, 3)
    np.testing.assert_array_equal(leaves, model.get_booster().predict(xgb.DMatrix(X), pred_leaf=True))
    trees = _trees(model.get_booster())
    np.testing.assert_array_equal(leaves, np.array([[t.leaf(x) for t in trees] for x in X], dtype=np.float32))


def test_classifier_apply(xgb):
    X, y = _data(rows=40, cols=4, seed=17)
    model = xgb.XGBClassifier(n_estimators=2, max_depth=2, max_bin=16)
    model.fit(X, (y > 0).astype(np.int64))
    np.testing.assert_array_equal(model.apply(X), model.get_booster().predict(xgb.DMatrix(X), pred_leaf=True))


def _tree_shap(t, x, cols):
    """A tree's exact contributions to row x in binary64, by TreeSHAP's own
    recursion (Lundberg, Erion and Lee 2018, Algorithm 2) over path weights."""
    phi = np.zeros(cols)

    def extend(path, z, o, f):
        path = [list(e) for e in path] + [[f, z, o, 1.0 if not path else 0.0]]
        n = len(path) - 1
        for i in range(n - 1, -1, -1):
            path[i + 1][3] += o * path[i][3] * (i + 1) / (n + 1)
            path[i][3] = z * path[i][3] * (n - i) / (n + 1)
        return path

    def unwind(path, k):
        path = [list(e) for e in path]
        n, z, o = len(path) - 1, path[k][1], path[k][2]
        nxt = path[n][3]
        for i in range(n - 1, -1, -1):
            if o != 0:
                kept = path[i][3]
                path[i][3] = nxt * (n + 1) / ((i + 1) * o)
                nxt = kept - path[i][3] * z * (n - i) / (n + 1)
            else:
                path[i][3] = path[i][3] * (n + 1) / (z * (n - i))
        for i in range(k, n):
            path[i][:3] = path[i + 1][:3]
        return path[:-1]

    def visit(k, path, z, o, f):
        path = extend(path, z, o, f)
        if t.left[k] < 0:
            for i in range(1, len(path)):
                w = sum(e[3] for e in unwind(path, i))
                phi[path[i][0]] += w * (path[i][2] - path[i][1]) * float(t.cond[k])
            return
        hot = t.child(k, x)
        cold = t.left[k] + t.right[k] - hot
        in_z, in_o = 1.0, 1.0
        for i in range(1, len(path)):
            if path[i][0] == t.feature[k]:
                in_z, in_o = path[i][1], path[i][2]
                path = unwind(path, i)
                break
        visit(hot, path, in_z * t.cover[hot] / t.cover[k], in_o, t.feature[k])
        visit(cold, path, in_z * t.cover[cold] / t.cover[k], 0.0, t.feature[k])

    visit(0, [], 1.0, 1.0, -1)
    return phi


@pytest.mark.parametrize("rows,cols,depth,rounds", [
    (1, 3, 1, 1), (63, 2, 3, 4), (65, 9, 5, 3), (200, 40, 7, 3), (130, 90, 8, 2), (64, 200, 6, 2), (300, 7, 11, 1),
    (257, 5, 13, 1), (900, 6, 16, 1), (70, 700, 4, 3), (3000, 4, 2, 9)])
def test_contributions_over_path_lengths_and_widths(xgb, rows, cols, depth, rounds):
    """Path tables of every element count, sums in LDS and (700 features) in
    memory, rows on both sides of a 64-row tile; absent entries as NaN, in a
    dense and a CSR matrix.  Binary32 sums of products against binary64: the
    error grows with the terms added, within 2e-5 of the margins' scale."""
    import scipy.sparse as sp
    rng = np.random.default_rng(rows + cols + depth)
    train = rng.normal(size=(2000, cols)).astype(np.float32)
    y = (rng.normal(size=2000) + train[:, 0] * train[:, -1] + train[:, cols // 2]).astype(np.float32)
    train[rng.random(train.shape) < 0.1] = np.nan
    bst = xgb.train({"max_depth": depth, "max_bin": 64, "eta": 0.5, "min_child_weight": 1, "lambda": 0.1},
                    xgb.DMatrix(train, label=y), rounds)
    X = rng.normal(size=(rows, cols)).astype(np.float32)
    X[rng.random(X.shape) < 0.2] = np.nan
    d = xgb.DMatrix(X)
    exact = bst.predict(d, pred_contribs=True).astype(np.float64)
    margin = bst.predict(d, output_margin=True).astype(np.float64)
    scale = max(1.0, np.abs(margin).max())
    np.testing.assert_allclose(exact.sum(axis=1), margin, rtol=0, atol=2e-5 * scale)
    trees = _trees(bst)
    picked = sorted({0, min(rows - 1, 63), min(rows - 1, 64), rows - 1})[:3 if depth < 11 else 1]
    for i in picked:
        ref = sum(_tree_shap(t, X[i], cols) for t in trees)
        np.testing.assert_allclose(exact[i, :-1], ref, rtol=0, atol=2e-5 * scale)
    r, c = np.nonzero(~np.isnan(X))
    csr = sp.csr_matrix((X[r, c], (r, c)), shape=X.shape)
    np.testing.assert_array_equal(bst.predict(xgb.DMatrix(csr), pred_contribs=True), exact.astype(np.float32))
    # A shorter range of rounds, then the whole model again.
    if rounds > 1:
        part = bst.predict(d, pred_contribs=True, iteration_range=(0, 1))
        np.testing.assert_allclose(part.sum(axis=1), bst.predict(d, output_margin=True, iteration_range=(0, 1)),
                                   rtol=0, atol=2e-5 * scale)
        np.testing.assert_array_equal(bst.predict(d, pred_contribs=True), exact.astype(np.float32))


def _covered_forest(xgb, rng, cols, trees, depth, features=None):
    """Boosted-looking trees with covers, split features among `features`
    (default: all), loaded as a model; and the trees."""
    features = np.arange(cols) if features is None else features
    out = []
    for _ in range(trees):
        t = {key: [] for key in ("left_children", "right_children", "split_indices", "split_conditions", "default_left",
                                 "parents", "sum_hessian")}

        def add(parent, cover):
            for key, v in (("left_children", -1), ("right_children", -1), ("split_indices", 0),
                           ("split_conditions", float(np.float32(rng.normal() * 0.1))), ("default_left", 0),
                           ("parents", parent), ("sum_hessian", float(cover))):
                t[key].append(v)
            return len(t["left_children"]) - 1

        level = {add(2147483647, 4096): 0}
        k = 0
        while k < len(t["left_children"]):
            cover = t["sum_hessian"][k]
            if level[k] < depth and cover >= 2 and (level[k] == 0 or rng.random() < 0.97):
                a = int(rng.integers(1, cover))
                t["split_indices"][k] = int(rng.choice(features))
                t["split_conditions"][k] = float(np.float32(rng.normal()))
                t["default_left"][k] = int(rng.integers(2))
                t["left_children"][k] = add(k, a)
                t["right_children"][k] = add(k, cover - a)
                level[t["left_children"][k]] = level[t["right_children"][k]] = level[k] + 1
            k += 1
        t["loss_changes"] = t["base_weights"] = [0] * len(t["left_children"])
        out.append(t)
    model = {"version": [3, 5, 0], "learner": {
        "attributes": {}, "feature_names": [], "feature_types": [],
        "learner_model_param": {"base_score": "0.25", "num_class": "0", "num_feature": str(cols), "num_target": "1"},
        "objective": {"name": "reg:squarederror"},
        "gradient_booster": {"name": "gbtree", "model": {"trees": out, "tree_info": [0] * trees}}}}
    return xgb.Booster(model_file=bytearray(json.dumps(model).encode())), out


@pytest.mark.parametrize("rows,cols,trees,depth,some", [
    (1, 65, 9, 5, False), (130, 65, 2, 2, False), (65, 290, 30, 4, False), (1, 2000, 60, 8, False),
    (130, 2000, 12, 6, False), (3, 100_000, 40, 7, False), (200, 40_000, 3, 3, True), (64, 5000, 20, 6, True)])
def test_contributions_of_wide_rows(xgb, rows, cols, trees, depth, some):
    """Tables over the features that some split names, more rows than a tile,
    columns that no split names (their contributions are 0); exact values of a
    few rows in binary64, and the sums of all against the margins."""
    import scipy.sparse as sp
    rng = np.random.default_rng(rows + cols)
    features = np.sort(rng.choice(cols, size=25, replace=False)) if some else None
    if some:
        features[-1] = cols - 1
    bst, forest = _covered_forest(xgb, rng, cols, trees, depth, features)
    used = sorted({f for t in forest for f, l in zip(t["split_indices"], t["left_children"]) if l >= 0})
    X = np.full((rows, cols), np.nan, np.float32)
    keep = rng.random((rows, len(used))) < 0.6
    X[:, used] = np.where(keep, rng.normal(size=keep.shape).astype(np.float32), np.nan)
    extra = rng.integers(0, cols, size=rows)
    X[np.arange(rows), extra] = 1.0
    d = xgb.DMatrix(X) if cols <= 5000 else None
    r, c = np.nonzero(~np.isnan(X))
    csr = xgb.DMatrix(sp.csr_matrix((X[r, c], (r, c)), shape=X.shape))
    got = bst.predict(csr, pred_contribs=True)
    if d is not None:
        np.testing.assert_array_equal(bst.predict(d, pred_contribs=True), got)
    margin = bst.predict(csr, output_margin=True).astype(np.float64)
    scale = max(1.0, np.abs(margin).max())
    np.testing.assert_allclose(got.astype(np.float64).sum(axis=1), margin, rtol=0, atol=2e-5 * scale)
    assert not got[:, np.setdiff1d(np.arange(cols), used)].any()
    plain = [_Tree(t) for t in forest]
    for i in sorted({0, rows - 1}):
        ref = sum(_tree_shap(t, X[i], cols) for t in plain)
        np.testing.assert_allclose(got[i, :-1], ref, rtol=0, atol=2e-5 * scale)


@pytest.mark.parametrize("rows,cols,trees,depth", [(1, 3, 1, 1), (70, 12, 6, 5), (130, 300, 5, 7), (9, 5, 3, 16)])
def test_contributions_by_table_and_by_walk(xgb, rows, cols, trees, depth):
    """mgb_predict_contribs, which walks the tree records where the table or its
    scratch would outgrow their bounds, agrees with the table."""
    import ctypes

    import device_lib as D
    rng = np.random.default_rng(rows * 3 + cols)
    bst, forest = _covered_forest(xgb, rng, cols, trees, depth)
    X = rng.normal(size=(rows, cols)).astype(np.float32)
    X[rng.random(X.shape) < 0.2] = np.nan
    nodes, means, offsets = [], [], [0]
    for t in forest:
        n = np.zeros(len(t["left_children"]), D.TREE_NODE)
        for key, source in (("left", "left_children"), ("right", "right_children"), ("feature", "split_indices"),
                            ("threshold", "split_conditions"), ("leaf", "split_conditions"), ("cover", "sum_hessian"),
                            ("default_left", "default_left")):
            n[key] = t[source]
        nodes.append(n)
        means.append(_Tree(t).mean.astype(np.float32))
        offsets.append(offsets[-1] + len(n))
    dX, dn, dm = D.Device.of(X), D.Device.of(np.concatenate(nodes)), D.Device.of(np.concatenate(means))
    do, out = D.Device.of(np.array(offsets, np.uint32)), D.Device(rows * (cols + 1) * 4)
    D.check(D.lib().mgb_predict_contribs(dX.ptr, None, None, ctypes.c_uint32(rows), ctypes.c_uint32(cols), dn.ptr, dm.ptr,
                                         do.ptr, ctypes.c_uint32(trees), ctypes.c_uint32(depth), ctypes.c_uint32(0),
                                         ctypes.c_uint32(0), None, ctypes.c_float(0.25), out.ptr))
    walk = out.read(np.float32, rows * (cols + 1)).reshape(rows, cols + 1)
    table = bst.predict(xgb.DMatrix(X), pred_contribs=True)
    scale = max(1.0, np.abs(table.astype(np.float64).sum(axis=1)).max())
    np.testing.assert_allclose(walk, table, rtol=0, atol=4e-5 * scale)
