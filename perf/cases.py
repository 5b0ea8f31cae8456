"""The work a user of this package has it do, as cases that can be timed.

Five kinds of work, each through the package's public entry points:

  train     a booster grown from nothing over a matrix that is already prepared (DMatrix kept:
            parameter searches, cross-validation, one matrix and many boosters): `train`, the trees
            and the training predictions read back.  Resident 8-bit and 16-bit bins, missing values,
            wide matrices, soft-max, the exact method, bins streamed from host memory.
  fit       from numpy arrays to a fitted estimator and its predictions: the data matrix is built,
            quantised and trained on, optionally with an evaluation set scored every round.
  predict   rows that have just arrived through a model that is kept: a data matrix is built from
            them and predicted on.
  eval      prediction on a matrix that is kept (an evaluation set, looked at again and again).
  hist_sum  histogram sums of node segments for bins and gradients that live on the GPU.

Inputs are made on the GPU from the seed and handed over as the entry points take them.
"""
import math

import numpy as np
import torch

import arboretum_amd as arb

# A drawn case grows at most this many rows x features x trees (under half of the largest listed one:
# wide and deep trees cost more per update), and its matrix holds at most this many bytes.
MOST_UPDATES = 6_000_000_000
MOST_CELLS = 10_500_000 * 28


def _train(name, rows, features, trees, depth, bins, objective, **more):
    case = {"name": name, "kind": "train", "rows": rows, "features": features, "trees": trees, "depth": depth,
            "bins": bins, "objective": objective, "classes": 1, "missing": 0.0, "matrix": "floats",
            "double_precision": True}
    case.update(more)
    return case


def listed():
    return [
        # Serving: a handful of rows arrive and are scored by a model of a hundred trees.  The
        # smallest call; latency is all there is.
        {"name": "predict_64", "kind": "predict", "rows": 64, "features": 28, "trees": 100, "depth": 6, "classes": 1,
         "missing": 0.0},
        # Batch scoring of a million fresh rows by 200 trees of depth 8, some values missing.
        {"name": "predict_1m", "kind": "predict", "rows": 1_000_003, "features": 28, "trees": 200, "depth": 8,
         "classes": 1, "missing": 0.02},
        # The regression configuration of the benchmark (10,000 rows, ten trees), from numpy arrays
        # to predictions: what most first scripts do.
        {"name": "fit_10k", "kind": "fit", "rows": 10_000, "features": 28, "trees": 10, "depth": 6, "bins": 256,
         "objective": 0, "missing": 0.0, "eval_rows": 0, "column_share": 1.0},
        # An estimator fitted with an evaluation set scored after every round (early stopping), the
        # estimators' own defaults for columns and bins.
        {"name": "fit_eval_200k", "kind": "fit", "rows": 200_000, "features": 50, "trees": 40, "depth": 6, "bins": 255,
         "objective": 0, "missing": 0.0, "eval_rows": 50_000, "column_share": 0.8},
        # The headline of the benchmark: 10.5 M rows, logistic, 256 bins, max_depth 8.
        _train("train_10m", 10_500_000, 28, 50, 8, 256, 1),
        # An ordinary table with gaps, sizes that divide nothing: 256 value bins and the bin of the
        # missing values (257 ids), squared error.
        _train("train_300k_missing", 300_007, 29, 100, 6, 256, 0, missing=0.05, double_precision=False),
        # Wide and sparse-ish: 200 features of 64 bins and 30 % missing values, max_depth 10.
        _train("train_wide", 1_500_000, 200, 20, 10, 64, 0, missing=0.3, matrix="bins"),
        # Ten classes, ten trees a round.
        _train("train_softmax", 1_000_000, 100, 50, 6, 256, 4, classes=10, matrix="bins"),
        # Bins of 16 bits: more than 256 thresholds per feature.
        _train("train_16bit", 500_000, 20, 50, 6, 1000, 1, matrix="floats"),
        # Bins that stay in host memory and are streamed block by block at every level.
        _train("train_streamed", 2_000_000, 128, 2, 8, 256, 1, matrix="streamed"),
        # The exact method on continuous columns.
        _train("train_exact", 400_000, 20, 20, 6, 0, 1, matrix="exact"),
        # Histogram sums of the sixteen nodes of a level, smaller siblings only.
        {"name": "hist_sum_4m", "kind": "hist_sum", "rows": 4_000_000, "features": 28, "nodes": 16, "hess": True,
         "trick": True, "alloc": True},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["train", "train", "train", "fit", "predict", "eval", "hist_sum"])
    if kind in ("predict", "eval"):
        features = _log(rng, 4, 100)
        lo, hi, cells = (1, 1_000_003, 28_000_000) if kind == "predict" else (10_000, 2_000_000, 56_000_000)
        return {"kind": kind, "rows": min(_log(rng, lo, hi), cells // features), "features": features,
                "trees": _log(rng, 10, 200), "depth": rng.randint(4, 8), "classes": rng.choice([1, 1, 3]),
                "missing": rng.choice([0.0, 0.02])}
    if kind == "fit":
        rows = _log(rng, 1_000, 200_000)
        return {"kind": kind, "rows": rows, "features": _log(rng, 4, 50), "trees": _log(rng, 5, 40),
                "depth": rng.randint(3, 8), "bins": rng.choice([64, 255, 256]), "objective": rng.choice([0, 1]),
                "missing": rng.choice([0.0, 0.05]), "eval_rows": rng.choice([0, rows // 4 + 1]),
                "column_share": rng.choice([0.8, 1.0])}
    if kind == "hist_sum":
        rows, features, nodes = _log(rng, 50_000, 6_000_000), _log(rng, 4, 64), rng.choice([1, 2, 8, 32])
        hess = rng.choice([True, False])
        # what the call without allocations has room for (its header): 32 MB of slabs, two spare per node
        items = min(1024, (32 << 20) // ((features + 15) // 16 * (128 << 10 if hess else 64 << 10)))
        small = rows <= (items - 2 * nodes - 2) * 60_000
        return {"kind": kind, "rows": rows, "features": features, "nodes": nodes, "hess": hess,
                "trick": nodes > 1 and rng.choice([True, False]), "alloc": not small or rng.choice([True, False])}
    matrix = rng.choice(["floats", "floats", "bins", "bins", "streamed", "exact"])
    objective = rng.choice([0, 1, 1, 4]) if matrix in ("floats", "bins") else 1
    lo, hi, flo, fhi = {"floats": (5_000, 4_000_000, 4, 60), "bins": (5_000, 6_000_000, 4, 200),
                        "streamed": (200_000, 2_000_000, 20, 128), "exact": (10_000, 400_000, 4, 20)}[matrix]
    features = _log(rng, flo, fhi)
    # (a matrix of floats is four times the bytes of one of bin ids)
    rows = min(_log(rng, lo, hi), MOST_CELLS // (features * (4 if matrix == "floats" else 1)))
    trees = {"streamed": rng.randint(1, 2), "exact": rng.randint(5, 20)}.get(matrix, _log(rng, 10, 100))
    classes = 1
    if objective == 4:
        classes = rng.randint(3, 8)
        trees = max(1, trees // (2 * classes)) * classes
    trees = max(1, min(trees, MOST_UPDATES // (rows * features)) // classes) * classes
    bins = rng.choice([32, 64, 255, 256]) if matrix != "floats" else rng.choice([64, 255, 256, 1000])
    depth = rng.randint(4, 8) if matrix in ("exact", "streamed") else rng.randint(4, 10)
    case = _train("", rows, features, trees, depth, 0 if matrix == "exact" else bins, objective, classes=classes,
                  matrix=matrix, missing=0.0 if matrix == "exact" else rng.choice([0.0, 0.05, 0.3]),
                  double_precision=rng.choice([True, False]))
    del case["name"]
    return case


def _signal(X, gen):
    """The benchmark's score: eight products of three stumps, plus noise."""
    rows, features = X.shape
    score = torch.zeros(rows, device="cuda")
    for _ in range(8):
        prod = torch.ones(rows, dtype=torch.bool, device="cuda")
        for _ in range(3):
            f = int(torch.randint(0, features, (1,), generator=gen, device="cuda"))
            column = X[:, f].float()
            t = torch.quantile(column[:100_000], 0.3 + 0.4 * float(torch.rand(1, generator=gen, device="cuda")))
            prod &= column > t
        score += prod
    return score + 0.5 * torch.randn(rows, generator=gen, device="cuda")


def _targets(X, gen, objective, classes):
    """(y, labels) of the objective, on the host."""
    score = _signal(X, gen)
    rows = X.shape[0]
    if classes > 1:
        other = torch.stack([torch.roll(score, k) if k else score for k in range(classes)])
        other += torch.stack([X[:, k % X.shape[1]].float() * (k + 1) / classes for k in range(classes)])
        return None, torch.argmax(other, dim=0).to(torch.uint8).cpu().numpy()
    if objective == 1:
        p = torch.sigmoid(score - score.mean() + 0.12)
        return (torch.rand(rows, generator=gen, device="cuda") < p).float().cpu().numpy(), None
    return score.cpu().numpy(), None


def _floats(rows, features, gen, missing):
    """N(0, 1) columns, the last quarter log-normal, `missing` of the values NaN."""
    X = torch.randn(rows, features, generator=gen, device="cuda")
    X[:, features - features // 4:] = X[:, features - features // 4:].exp()
    full = X
    if missing > 0:
        full = X.clone()
        X[torch.rand(rows, features, generator=gen, device="cuda") < missing] = float("nan")
    return X, full


def _bin_ids(rows, features, gen, bins, missing):
    """Half the columns uniform over the bins, half piled up in the low ones; missing values in a bin of their own."""
    top = min(bins, 256 if missing == 0 else 255)
    X = torch.randint(0, top, (rows, features), generator=gen, device="cuda", dtype=torch.uint8)
    half = features // 2
    u = torch.rand(rows, features - half, generator=gen, device="cuda")
    X[:, half:] = (u * u * u * top).to(torch.uint8)
    del u
    full = X
    if missing > 0:
        full = X.clone()
        X[torch.rand(rows, features, generator=gen, device="cuda") < missing] = top
    return X, full


def _config(case):
    config = {"objective": case["objective"], "method": 0 if case["matrix"] == "exact" else 1,
              "internals": {"hist_size": max(case["bins"], 1), "double_precision": case["double_precision"],
                            "use_hist_subtraction_trick": True, "upload_features": case["matrix"] != "streamed"},
              "tree": {"max_depth": case["depth"], "eta": 0.1, "lambda": 1.0, "min_child_weight": 1.0,
                       "min_leaf_size": 1, "colsample_bytree": 1.0, "colsample_bylevel": 1.0}}
    if case["classes"] > 1:
        config["tree"]["labels_count"] = case["classes"]
    if case["matrix"] == "streamed":
        # nothing stays in device memory: the case of a matrix much larger than it
        config["internals"]["stream_resident_bytes"] = 0
        config["internals"]["stream_block_rows"] = 1 << 19
    return config


def _host(X):
    return X.cpu().numpy()


def _prepare_train(case, gen):
    if case["matrix"] in ("bins", "streamed"):
        X, full = _bin_ids(case["rows"], case["features"], gen, case["bins"], case["missing"])
    else:
        X, full = _floats(case["rows"], case["features"], gen, case["missing"])
    y, labels = _targets(full, gen, case["objective"], case["classes"])
    quantized = case["matrix"] in ("bins", "streamed")
    data = arb.DMatrix(_host(X), y=y, labels=labels, quantized=quantized)
    del X, full
    config = _config(case)
    if case["matrix"] in ("floats", "bins"):
        data.quantize(case["bins"])
    else:
        arb.train(config, data, 1).synchronize()  # the first booster has the matrix laid out
    return {"kind": "train", "config": config, "data": data, "rounds": case["trees"] // case["classes"]}


def _prepare_fit(case, gen):
    rows = case["rows"] + case["eval_rows"]
    X, full = _floats(rows, case["features"], gen, case["missing"])
    y, _ = _targets(full, gen, case["objective"], 1)
    X = _host(X)
    n = case["rows"]
    return {"kind": "fit", "case": case, "X": X[:n], "y": y[:n], "eval_X": X[n:], "eval_y": y[n:]}


def _prepare_predict(case, gen):
    # the model: grown on a table of the same columns
    fit_rows = 20_000
    X, full = _floats(fit_rows + case["rows"], case["features"], gen, case["missing"])
    y, labels = _targets(full[:fit_rows], gen, 1 if case["classes"] == 1 else 4, case["classes"])
    config = {"objective": 1 if case["classes"] == 1 else 4, "method": 1,
              "internals": {"hist_size": 255, "double_precision": True},
              "tree": {"max_depth": case["depth"], "eta": 0.1, "lambda": 1.0, "min_child_weight": 0.1}}
    if case["classes"] > 1:
        config["tree"]["labels_count"] = case["classes"]
    rounds = max(1, case["trees"] // case["classes"])
    X = _host(X)
    model = arb.train(config, arb.DMatrix(X[:fit_rows], y=y, labels=labels), rounds)
    model.synchronize()
    fresh = np.ascontiguousarray(X[fit_rows:])
    if case["kind"] == "eval":
        return {"kind": "eval", "model": model, "data": arb.DMatrix(fresh)}
    return {"kind": "predict", "model": model, "X": fresh}


def _prepare_hist_sum(case, gen):
    rows, features, nodes = case["rows"], case["features"], case["nodes"]
    quads = (features + 3) // 4
    stride = (rows + 63) // 64 * 64
    bins = torch.randint(0, 256, (quads, stride, 4), generator=gen, device="cuda", dtype=torch.uint8)
    if features % 4:
        bins[-1, :, features % 4:] = 0
    g = torch.rand(rows, generator=gen, device="cuda") * 2 - 1
    h = torch.rand(rows, generator=gen, device="cuda") * 0.25 if case["hess"] else None
    cuts = torch.randint(0, rows + 1, (nodes - 1,), generator=gen, device="cuda").sort().values
    ends = torch.tensor([0, rows], device="cuda")
    node_size = torch.cat([ends[:1], cuts, ends[1:]]).to(torch.int32)

    def cells(n):
        return (torch.zeros(n, 4 * quads, 256, dtype=torch.int64, device="cuda"),
                torch.zeros(n, 4 * quads, 256, dtype=torch.int64, device="cuda") if case["hess"] else None,
                torch.zeros(n, 4 * quads, 256, dtype=torch.int32, device="cuda"))

    state = {"kind": "hist_sum", "bins": bins, "stride": stride, "g": g, "h": h, "node_size": node_size,
             "out": cells(nodes), "parents": (None, None, None), "rows": rows, "features": features, "nodes": nodes,
             "trick": case["trick"], "alloc": case["alloc"]}
    if case["trick"]:
        parents = dict(state, out=cells(nodes // 2), node_size=node_size[::2].contiguous(), nodes=nodes // 2,
                       trick=False, alloc=True)
        torch.cuda.synchronize()
        run(parents)
        state["parents"] = parents["out"]
    return state


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    make = {"train": _prepare_train, "fit": _prepare_fit, "predict": _prepare_predict, "eval": _prepare_predict,
            "hist_sum": _prepare_hist_sum}[case["kind"]]
    return make(case, gen)


def _trees(model):
    trees = [model.tree(t) for t in range(model.num_trees())]
    return {key: np.stack([t[key] for t in trees]) for key in trees[0]}


def _run_train(state):
    model = arb.train(state["config"], state["data"], state["rounds"])
    return {"trees": _trees(model), "y_hat": model.train_yhat()}


def _run_fit(state):
    case = state["case"]
    make = arb.ArboretumRegression if case["objective"] == 0 else arb.ArboretumClassifier
    estimator = make(max_depth=case["depth"], learning_rate=0.1, n_estimators=case["trees"], verbosity=0,
                     hist_size=case["bins"], colsample_bytree=case["column_share"], l1=0.0)
    if case["eval_rows"] == 0:
        estimator.fit(state["X"], state["y"])
        return estimator.predict(state["X"])
    scores = []

    def squared_error(y, p):
        scores.append(float(np.mean((y - p) ** 2)))
        return scores[-1]

    estimator.fit(state["X"], state["y"], eval_set=state["eval_X"], eval_labels=state["eval_y"],
                  early_stopping_rounds=case["trees"], eval_metric=squared_error)
    return {"scores": np.array(scores), "predictions": estimator.predict(state["eval_X"])}


def _run_hist_sum(state):
    address = [None if t is None else t.data_ptr() for t in
               (*state["out"], state["g"], state["h"], state["node_size"], state["bins"], *state["parents"])]
    call = arb.hist_sum if state["alloc"] else arb.hist_sum_no_alloc
    call(*address[:7], state["stride"], state["rows"], state["features"], state["nodes"], 30, 32,
         use_trick=state["trick"], parent_g=address[7], parent_h=address[8], parent_c=address[9])
    return [t for t in state["out"] if t is not None]


def run(state):
    kind = state["kind"]
    if kind == "train":
        return _run_train(state)
    if kind == "fit":
        return _run_fit(state)
    if kind == "predict":
        return state["model"].predict(arb.DMatrix(state["X"]))
    if kind == "eval":
        return state["model"].predict(state["data"])
    return _run_hist_sum(state)


def work(case):
    rows, features = case["rows"], case["features"]
    if case["kind"] == "hist_sum":
        nodes, cell = case["nodes"], 20 if case["hess"] else 12
        cells = nodes * features * 256 * cell
        return {"bytes": rows * (features + (8 if case["hess"] else 4)) + cells * (1.5 if case["trick"] else 1),
                "flops": rows * features * (2 if case["hess"] else 1)}
    if case["kind"] in ("predict", "eval"):
        nodes = case["trees"] * (8 * (2 ** case["depth"] - 1) + 4 * 2 ** case["depth"])
        return {"bytes": rows * (4 * features + 4 * case["classes"]) + nodes,
                "flops": rows * case["trees"] * (case["depth"] + 1)}
    # training: a tree reads the bins and the target once and updates the prediction; its gradients
    # are known only when the tree before it is done
    if case["kind"] == "fit":
        read, trees = rows * features * 4 + case["eval_rows"] * features * 4, case["trees"]
        width = 1
    else:
        read, trees = 0, case["trees"]
        width = 4 if case["matrix"] == "exact" else 2 if case["bins"] > 256 else 1
    return {"bytes": read + trees * rows * (features * width + 12), "flops": trees * rows * features * 2}


def tolerance(case):
    # integers: histogram cells, split features and bins.  Gains, leaf weights and predictions are
    # 32-bit sums.
    return "exact" if case["kind"] == "hist_sum" else {"rel": 1e-5}
