"""Performance cases of the hist engine: fits, predictions and feature
contributions as a user's program asks for them through `import xgboost`.

Each case is a dict of plain values; `kind` names the call:

- fit: `xgb.train` on a DMatrix the program holds, then the margins of the
  training rows (dense matrices; `missing` is the share of NaN entries);
- fit_csr: the same on a CSR matrix (absent entries missing), binary:logistic;
- fit_eval: binary:logistic `xgb.train` with a validation matrix scored by AUC
  and logloss after every round;
- fit_arrays: from numpy arrays to a first model: QuantileDMatrix, a few
  rounds, the quantile cuts and the margins;
- predict: `Booster.predict` on a DMatrix the program holds;
- predict_inplace: `Booster.inplace_predict` of a numpy array (a request);
- predict_csr: `Booster.predict` on a CSR matrix;
- contribs: `Booster.predict(pred_contribs=True)`, exact TreeSHAP.

Models to predict with are drawn from the seed and loaded as model JSON.
"""
import json
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "xgboost-metal_amd", "python"))
import xgboost as xgb  # noqa: E402

DEVICE = "cuda" if torch.cuda.is_available() else "cpu"


def _fit(name, rows, cols, depth, rounds, max_bin=256, missing=0.0, objective="reg:squarederror", sample=1.0):
    return {"name": name, "kind": "fit", "rows": rows, "cols": cols, "depth": depth, "rounds": rounds,
            "max_bin": max_bin, "missing": missing, "objective": objective, "sample": sample}


def listed():
    return [
        # A table of a few thousand rows: every launch is short.
        _fit("fit_5k_x20", 5003, 20, 6, 50),
        # 100,000 x 32 with 15% of the entries missing, 100 rounds.
        _fit("fit_100k_x32_missing", 100000, 32, 6, 100, missing=0.15),
        # The headline workload: 262,144 x 64, depth 8, 256 bins, 100 rounds.
        _fit("fit_262k_x64", 262144, 64, 8, 100),
        # Wide bins (16-bit codes), row and column sampling, logistic loss: the
        # 10M x 128 workload's parameters on 1.5M rows.
        _fit("fit_1500k_x128_bins1024", 1500000, 128, 10, 10, max_bin=1024, objective="binary:logistic", sample=0.8),
        # Sparse classification, 2,000 columns with 20 stored entries a row.
        {"name": "fit_csr_1m_x2000", "kind": "fit_csr", "rows": 1000000, "cols": 2000, "nnz": 20, "depth": 8,
         "rounds": 10, "max_bin": 256},
        # Training watched on a validation set every round, as with early stopping.
        {"name": "fit_eval_100k_x32", "kind": "fit_eval", "rows": 100000, "valid": 25000, "cols": 32, "depth": 6,
         "rounds": 50},
        # From numpy arrays to a first model: sketch, bin matrix, a few rounds.
        {"name": "fit_arrays_262k_x64", "kind": "fit_arrays", "rows": 262144, "cols": 64, "depth": 8, "rounds": 5,
         "max_bin": 256, "missing": 0.0},
        # One request of a service: a handful of rows, answered at once.
        {"name": "predict_inplace_16_x32", "kind": "predict_inplace", "rows": 16, "cols": 32, "trees": 100,
         "depth": 6, "missing": 0.0, "objective": "binary:logistic"},
        # A held-out set with missing values, an odd row count.
        {"name": "predict_100k_x32_missing", "kind": "predict", "rows": 100003, "cols": 32, "trees": 100, "depth": 6,
         "missing": 0.15, "objective": "reg:squarederror"},
        # Batch scoring of a million rows with the headline model's shape.
        {"name": "predict_1m_x64", "kind": "predict", "rows": 1000000, "cols": 64, "trees": 100, "depth": 8,
         "missing": 0.0, "objective": "binary:logistic"},
        # Batch scoring of sparse rows.
        {"name": "predict_csr_200k_x2000", "kind": "predict_csr", "rows": 200000, "cols": 2000, "nnz": 20,
         "trees": 100, "depth": 8, "objective": "binary:logistic"},
        # Explaining a sample of the rows: exact contributions.
        {"name": "contribs_5k_x32", "kind": "contribs", "rows": 5000, "cols": 32, "trees": 100, "depth": 6,
         "missing": 0.15},
    ]


def _log_int(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choice(["fit", "fit", "fit", "fit_csr", "fit_eval", "fit_arrays", "predict", "predict",
                       "predict_inplace", "predict_csr", "contribs"])
    if kind == "fit":
        rows, cols = _log_int(rng, 2000, 300000), _log_int(rng, 6, 64)
        return {"kind": kind, "rows": rows, "cols": cols, "depth": rng.randint(4, 8), "rounds": rng.randint(10, 60),
                "max_bin": rng.choice([64, 255, 256, 256, 1024]), "missing": rng.choice([0.0, 0.05, 0.15]),
                "objective": rng.choice(["reg:squarederror", "binary:logistic"]),
                "sample": rng.choice([1.0, 1.0, 0.8])}
    if kind == "fit_csr":
        return {"kind": kind, "rows": _log_int(rng, 20000, 500000), "cols": _log_int(rng, 200, 3000),
                "nnz": rng.randint(8, 24), "depth": rng.randint(5, 8), "rounds": rng.randint(4, 10), "max_bin": 256}
    if kind == "fit_eval":
        rows = _log_int(rng, 5000, 100000)
        return {"kind": kind, "rows": rows, "valid": rows // 4 + 1, "cols": rng.randint(8, 32),
                "depth": rng.randint(4, 7), "rounds": rng.randint(10, 50)}
    if kind == "fit_arrays":
        return {"kind": kind, "rows": _log_int(rng, 5000, 262144), "cols": rng.randint(8, 64),
                "depth": rng.randint(4, 8), "rounds": rng.randint(1, 5), "max_bin": rng.choice([64, 256]),
                "missing": rng.choice([0.0, 0.1])}
    shape = {"trees": rng.randint(20, 100), "depth": rng.randint(3, 8)}
    if kind == "predict":
        return {"kind": kind, "rows": _log_int(rng, 1000, 800000), "cols": _log_int(rng, 8, 100), **shape,
                "missing": rng.choice([0.0, 0.15]),
                "objective": rng.choice(["reg:squarederror", "binary:logistic"])}
    if kind == "predict_inplace":
        return {"kind": kind, "rows": _log_int(rng, 1, 2000), "cols": _log_int(rng, 8, 100), **shape,
                "missing": rng.choice([0.0, 0.15]),
                "objective": rng.choice(["reg:squarederror", "binary:logistic"])}
    if kind == "predict_csr":
        return {"kind": kind, "rows": _log_int(rng, 1000, 200000), "cols": _log_int(rng, 200, 3000),
                "nnz": rng.randint(8, 24), **shape, "objective": "binary:logistic"}
    return {"kind": "contribs", "rows": _log_int(rng, 50, 5000), "cols": _log_int(rng, 8, 48),
            "trees": rng.randint(10, 60), "depth": rng.randint(3, 6), "missing": rng.choice([0.0, 0.15])}


# ---- inputs -------------------------------------------------------------------
def _generator(seed):
    g = torch.Generator(device=DEVICE)
    g.manual_seed(seed)
    return g


def _dense(case, seed, rows=None):
    """X (float32, NaN missing) on the device, and the margin its labels follow.

    Narrow bins: N(0,1) columns.  Wide bins: half N(0,1), a quarter uniform, a
    quarter whole numbers 0..999."""
    rows, cols = rows or case["rows"], case["cols"]
    g = _generator(seed)
    X = torch.randn(rows, cols, generator=g, device=DEVICE)
    if case.get("max_bin", 256) >= 1024:
        u = cols // 2
        q = u + cols // 4
        X[:, u:q] = torch.rand(rows, q - u, generator=g, device=DEVICE)
        X[:, q:] = torch.randint(0, 1000, (rows, cols - q), generator=g, device=DEVICE).float()
    used = min(cols, 16) if case.get("objective") == "binary:logistic" and cols > 64 else cols
    w = torch.randn(cols, generator=g, device=DEVICE)
    s = X[:, :used] @ w[:used] + 0.5 * torch.sin(X[:, 0] * X[:, 1])
    noise = torch.randn(rows, generator=g, device=DEVICE)
    if case.get("missing", 0.0) > 0:
        X[torch.rand(rows, cols, generator=g, device=DEVICE) < case["missing"]] = float("nan")
    return X, s, noise, g


def _labels(objective, s, noise, g):
    if objective == "binary:logistic":
        p = torch.sigmoid(s + 0.3 * noise)
        return (torch.rand(p.shape, generator=g, device=DEVICE) < p).float().cpu().numpy()
    return (s + 0.1 * noise).cpu().numpy()


def _csr(case, seed):
    """`nnz` stored lognormal values a row, one in each of nnz equal ranges of
    the columns, so that a row's columns are distinct and rising."""
    import scipy.sparse
    rows, cols, nnz = case["rows"], case["cols"], case["nnz"]
    g = _generator(seed)
    edges = torch.linspace(0, cols, nnz + 1, device=DEVICE).long()
    width = (edges[1:] - edges[:-1]).float()
    idx = edges[:-1] + torch.minimum((torch.rand(rows, nnz, generator=g, device=DEVICE) * width).long(),
                                     width.long() - 1)
    val = torch.exp(torch.randn(rows, nnz, generator=g, device=DEVICE))
    w = torch.randn(cols, generator=g, device=DEVICE) * 0.5
    w[torch.rand(cols, generator=g, device=DEVICE) > 0.1] = 0
    s = (val * w[idx]).sum(1)
    y = _labels("binary:logistic", s, torch.zeros(rows, device=DEVICE), g)
    indptr = np.arange(0, (rows + 1) * nnz, nnz, dtype=np.int64)
    m = scipy.sparse.csr_matrix((val.reshape(-1).cpu().numpy(), idx.reshape(-1).int().cpu().numpy(), indptr),
                                shape=(rows, cols))
    return m, y


def _forest(case, seed):
    """Trees such as boosting leaves: nearly full, some nodes that stop early,
    split features favouring some, thresholds at the features' quantiles, every
    node's cover split by the share of rows that its test sends left."""
    rng = np.random.default_rng(seed + 1000003)
    cols, depth = case["cols"], case["depth"]
    sparse = case["kind"] == "predict_csr"
    weight = 1.0 / (1.0 + np.arange(cols)) ** 0.5
    weight = rng.permutation(weight / weight.sum())
    present = case["nnz"] / cols if sparse else 1.0 - case["missing"]
    trees = []
    for _ in range(case["trees"]):
        left, right, parent, feature, cond, dleft, cover, level = [-1], [-1], [2147483647], [0], [0.0], [0], [1e6], [0]
        k = 0
        while k < len(left):
            d = level[k]
            if d < depth and cover[k] >= 40 and (d == 0 or rng.random() > 0.03):
                q = 0.15 + 0.7 * rng.random()
                f = int(rng.choice(cols, p=weight)) if d < 3 else int(rng.integers(cols))
                z = math.sqrt(2.0) * _erfinv(2 * q - 1)
                go = int(rng.random() < 0.5)
                share = present * q + (1.0 - present) * go
                a = min(max(round(cover[k] * share), 1), cover[k] - 1)
                left[k], right[k] = len(left), len(left) + 1
                feature[k], dleft[k] = f, go
                cond[k] = float(np.float32(math.exp(z) if sparse else z))
                for c in (a, cover[k] - a):
                    left.append(-1)
                    right.append(-1)
                    parent.append(k)
                    feature.append(0)
                    cond.append(0.0)
                    dleft.append(0)
                    cover.append(float(c))
                    level.append(d + 1)
            else:
                cond[k] = float(np.float32(0.05 * rng.standard_normal()))
            k += 1
        trees.append({"left": left, "right": right, "parent": parent, "feature": feature, "cond": cond,
                      "dleft": dleft, "cover": cover})
    return trees


def _erfinv(x):
    return float(torch.erfinv(torch.tensor(x, dtype=torch.float64)))


def _model_json(case, trees):
    out = []
    for i, t in enumerate(trees):
        n = len(t["left"])
        zero = [0] * n
        out.append({"id": i, "left_children": t["left"], "right_children": t["right"], "parents": t["parent"],
                    "split_indices": t["feature"], "split_conditions": t["cond"], "default_left": t["dleft"],
                    "sum_hessian": t["cover"], "loss_changes": zero, "base_weights": zero, "split_type": zero,
                    "categories": [], "categories_nodes": [], "categories_segments": [], "categories_sizes": [],
                    "tree_param": {"num_deleted": "0", "num_feature": str(case["cols"]), "num_nodes": str(n),
                                   "size_leaf_vector": "1"}})
    return json.dumps({"version": [3, 5, 0], "learner": {
        "attributes": {}, "feature_names": [], "feature_types": [],
        "learner_model_param": {"base_score": "0.5", "num_class": "0", "num_feature": str(case["cols"]),
                                "num_target": "1", "boost_from_average": "1"},
        "objective": {"name": case.get("objective", "reg:squarederror"), "reg_loss_param": {"scale_pos_weight": "1"}},
        "gradient_booster": {"name": "gbtree", "model": {
            "gbtree_model_param": {"num_parallel_tree": "1", "num_trees": str(len(trees))},
            "iteration_indptr": list(range(len(trees) + 1)), "tree_info": [0] * len(trees), "trees": out}}}}).encode()


def _params(case):
    p = {"objective": case.get("objective", "binary:logistic"), "tree_method": "hist", "max_depth": case["depth"],
         "max_bin": case.get("max_bin", 256), "eta": 0.3, "lambda": 1, "seed": 7}
    if p["objective"] == "binary:logistic":
        p["eta"] = 0.1
    if case.get("sample", 1.0) < 1.0:
        p["subsample"] = p["colsample_bytree"] = case["sample"]
    return p


def prepare(case, seed):
    kind = case["kind"]
    state = {"case": case}
    if kind in ("fit", "fit_arrays"):
        X, s, noise, g = _dense(case, seed)
        y, X = _labels(case.get("objective"), s, noise, g), X.cpu().numpy()
        if kind == "fit_arrays":
            state.update(X=X, y=y)
        else:
            state["dtrain"] = xgb.DMatrix(X, label=y).to_device()
    elif kind == "fit_csr":
        m, y = _csr(case, seed)
        state["dtrain"] = xgb.DMatrix(m, label=y).to_device()
    elif kind == "fit_eval":
        n, v = case["rows"], case["valid"]
        X, s, noise, g = _dense(case, seed, n + v)
        y, X = _labels("binary:logistic", s, noise, g), X.cpu().numpy()
        state["dtrain"] = xgb.DMatrix(X[:n], label=y[:n]).to_device()
        state["dvalid"] = xgb.DMatrix(X[n:], label=y[n:]).to_device()
    else:
        state["booster"] = xgb.Booster(model_file=bytearray(_model_json(case, _forest(case, seed))))
        if kind == "predict_csr":
            state["data"] = xgb.DMatrix(_csr(case, seed)[0]).to_device()
        else:
            X = _dense(case, seed)[0].cpu().numpy()
            state["data"] = X if kind == "predict_inplace" else xgb.DMatrix(X).to_device()
    return state


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind in ("fit", "fit_csr"):
        booster = xgb.train(_params(case), state["dtrain"], case["rounds"], verbose_eval=False)
        return {"margin": booster.predict(state["dtrain"], output_margin=True)}
    if kind == "fit_eval":
        history = {}
        booster = xgb.train(dict(_params(case), eval_metric=["auc", "logloss"]), state["dtrain"], case["rounds"],
                            evals=[(state["dvalid"], "valid")], evals_result=history, verbose_eval=False)
        return {"margin": booster.predict(state["dvalid"], output_margin=True),
                "auc": np.array(history["valid"]["auc"]), "logloss": np.array(history["valid"]["logloss"])}
    if kind == "fit_arrays":
        dtrain = xgb.QuantileDMatrix(state["X"], label=state["y"], max_bin=case["max_bin"])
        booster = xgb.train(_params(dict(case, objective="reg:squarederror")), dtrain, case["rounds"],
                            verbose_eval=False)
        indptr, cuts = dtrain.get_quantile_cut()
        return {"margin": booster.predict(dtrain, output_margin=True), "cut_ptr": indptr, "cuts": cuts}
    if kind == "predict_inplace":
        return state["booster"].inplace_predict(state["data"])
    if kind == "contribs":
        return state["booster"].predict(state["data"], pred_contribs=True)
    return state["booster"].predict(state["data"])


def work(case):
    kind, cols = case["kind"], case["cols"]
    if kind in ("fit", "fit_arrays", "fit_eval", "fit_csr"):
        # Per round: the codes of every row at the root and of half the rows
        # (the smaller children) at each deeper level, two sums a code; each
        # row's id, gradient pair and margin once a level.
        rows, depth, rounds = case["rows"], case["depth"], case["rounds"]
        entries = case.get("nnz", cols)
        code = (2 if case.get("max_bin", 256) > 256 else 1) + (4 if kind == "fit_csr" else 0)
        built = rows * (1 + 0.5 * (depth - 1)) * case.get("sample", 1.0)
        size = rounds * (built * entries * code + rows * depth * 16) + rows * 8
        flops = rounds * 2 * built * entries
        if kind == "fit_arrays":
            size += rows * cols * 4
        if kind == "fit_eval":
            size += rounds * case["valid"] * 12 + case["valid"] * cols * 4
            flops += rounds * case["valid"] * depth
        return {"bytes": size, "flops": flops}
    entries = case["nnz"] * 2 if kind == "predict_csr" else cols
    rows, trees, depth = case["rows"], case["trees"], case["depth"]
    model = trees * (2 << depth) * 8
    if kind == "contribs":
        return {"bytes": rows * (2 * cols + 1) * 4 + model, "flops": rows * trees * (2 << depth) * depth}
    return {"bytes": rows * (entries + 1) * 4 + model, "flops": rows * trees * depth}


def tolerance(case):
    kind = case["kind"]
    if kind in ("fit", "fit_csr", "fit_arrays"):
        # Histograms are exact integer sums and every later step is pinned bit
        # for bit: the same trees, margins and bytes.
        return "exact"
    if kind == "fit_eval":
        return {"rel": 1e-6, "max": 1e-5}  # logarithms and 32-bit sums of the metrics
    if kind == "contribs":
        return {"rel": 2e-6, "max": 1e-4}  # 32-bit sums of products over every path of every tree
    return {"rel": 1e-6, "max": 1e-5}  # a 32-bit sum of one leaf a tree


# ---- 64-bit references ----------------------------------------------------------
def _columns(trees, cols, device):
    n = max(len(t["left"]) for t in trees)
    pad = {"left": -1, "feature": 0, "cond": 0.0, "dleft": 0, "right": -1}
    kinds = {"cond": torch.float32}
    return {key: torch.tensor([t[key] + [fill] * (n - len(t[key])) for t in trees],
                              dtype=kinds.get(key, torch.int64), device=device) for key, fill in pad.items()}


def _dense_values(case, seed):
    if case["kind"] != "predict_csr":
        return _dense(case, seed)[0]
    m = _csr(case, seed)[0]
    X = torch.full((case["rows"], case["cols"]), float("nan"), device=DEVICE)
    r = torch.arange(case["rows"], device=DEVICE).repeat_interleave(case["nnz"])
    X[r, torch.from_numpy(m.indices.astype(np.int64)).to(DEVICE)] = torch.from_numpy(m.data).to(DEVICE)
    return X


def _exact_margin(case, seed):
    X = _dense_values(case, seed)
    trees = _forest(case, seed)
    c = _columns(trees, case["cols"], DEVICE)
    base = 0.0 if case["objective"] == "binary:logistic" else 0.5
    margin = torch.full((len(X),), base, dtype=torch.float64, device=DEVICE)
    rows = torch.arange(len(X), device=DEVICE)
    for t in range(len(trees)):
        at = torch.zeros(len(X), dtype=torch.int64, device=DEVICE)
        for _ in range(case["depth"]):
            v = X[rows, c["feature"][t][at]]
            go = torch.where(torch.isnan(v), c["dleft"][t][at] != 0, v < c["cond"][t][at])
            nxt = torch.where(go, c["left"][t][at], c["right"][t][at])
            at = torch.where(c["left"][t][at] < 0, at, nxt)
        margin += c["cond"][t][at].double()
    return torch.sigmoid(margin) if case["objective"] == "binary:logistic" else margin


def _exact_contribs(case, seed):
    """Shapley values of every leaf's path, in closed form: the weight of a
    subset of the path's other features is a Beta integral, so feature i's
    share of a leaf is v (o_i - z_i) times the integral over t in [0, 1] of
    the product over j != i of (o_j t + z_j (1 - t)), o the row's pass flags
    and z the shares of the cover; Gauss-Legendre nodes integrate the
    polynomial exactly."""
    X = _dense(case, seed)[0]
    rows, cols, depth = len(X), case["cols"], case["depth"]
    nodes, weights = np.polynomial.legendre.leggauss((depth + 1) // 2 + 1)
    ts, ws = (nodes + 1) / 2, weights / 2
    phi = torch.zeros(rows, cols + 1, dtype=torch.float64, device=DEVICE)
    phi[:, cols] = 0.5
    for t in _forest(case, seed):
        paths = []  # per leaf: value, [(feature, share, [(node, goes left)])]
        stack = [(0, [])]
        while stack:
            k, path = stack.pop()
            if t["left"][k] < 0:
                merged = {}
                for node, left in path:
                    child = t["left"][node] if left else t["right"][node]
                    e = merged.setdefault(t["feature"][node], [1.0, []])
                    e[0] *= t["cover"][child] / t["cover"][node]
                    e[1].append((node, left))
                paths.append((t["cond"][k], t["cover"][k] / t["cover"][0], merged))
            else:
                stack += [(t["left"][k], path + [(k, True)]), (t["right"][k], path + [(k, False)])]
        n = len(t["left"])
        f = torch.tensor(t["feature"], device=DEVICE)
        v = X[:, f]
        go = torch.where(torch.isnan(v), torch.tensor(t["dleft"], device=DEVICE) != 0,
                         v < torch.tensor(t["cond"], dtype=torch.float32, device=DEVICE))
        flags = torch.cat([~go, go, torch.ones(rows, 1, dtype=torch.bool, device=DEVICE)], 1)  # node, n + node, true
        L, M = len(paths), depth
        test = np.full((L, M, depth), 2 * n)
        z, real = np.ones((L, M)), np.zeros((L, M), bool)
        feat = np.full((L, M), cols)
        value = np.array([p[0] for p in paths])
        for i, (_, _, merged) in enumerate(paths):
            for j, (ff, (share, tests)) in enumerate(merged.items()):
                z[i, j], feat[i, j], real[i, j] = share, ff, True
                for q, (node, left) in enumerate(tests):
                    test[i, j, q] = node + (n if left else 0)
        o = flags[:, torch.from_numpy(test.reshape(-1)).to(DEVICE)].view(rows, L, M, depth).all(3).double()
        zt, rt = torch.from_numpy(z).to(DEVICE), torch.from_numpy(real).to(DEVICE)
        total = torch.zeros(rows, L, M, dtype=torch.float64, device=DEVICE)
        for tq, wq in zip(ts, ws):
            factor = torch.where(rt, o * tq + zt * (1 - tq), 1.0)
            total += wq * factor.prod(2, keepdim=True) / factor
        share = total * (o - zt) * torch.from_numpy(value).to(DEVICE)[None, :, None]
        share = torch.where(rt, share, 0.0).reshape(rows, L * M)
        phi.index_add_(1, torch.from_numpy(feat.reshape(-1)).to(DEVICE), share)
        phi[:, cols] += float(sum(p[0] * p[1] for p in paths))
    return phi


def exact(case, seed):
    if case["kind"] in ("predict", "predict_inplace", "predict_csr"):
        return _exact_margin(case, seed)
    if case["kind"] == "contribs":
        return _exact_contribs(case, seed)
    return None  # a fit's discrete decisions follow the 32-bit margins
