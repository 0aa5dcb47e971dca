"""The work that users of this package have it do, as cases that can be timed: whole calls of `fit`, `predict` and
`predict_leaf_idx`, from the matrices or tables that a program holds in host memory to the trees or values it gets back.

A case is a dict of plain values.  "do" is "fit", "predict" or "leaf_idx"; "form" is how the features are held:

  matrix_c  a numpy matrix in numpy's own order (rows one after the other), what most programs build
  matrix_f  a numpy matrix in column order, as a DataFrame of one type hands it out and as a Julia matrix lies
  table     a dict of columns: real ones, whole-number ones and Bool ones (the Tables interface)

Sizes and learners' settings are the benchmark's configurations (cfg1 to cfg5 in bench.py) where a case names one, the learners'
defaults or ordinary values elsewhere."""
import importlib.util
import math
import os
import sys

import numpy as np
import torch

TRAIN_ROWS = 20_000  # rows the model of a prediction case is fitted on


def _package():
    """This repository's package: its folder's name is no module name, so it is loaded from its path, as bench.py does."""
    name = "evotrees_jl_amd"
    if name in sys.modules:
        return sys.modules[name]
    folder = os.path.join(os.getcwd(), "evotrees.jl_amd")
    spec = importlib.util.spec_from_file_location(name, os.path.join(folder, "__init__.py"), submodule_search_locations=[folder])
    module = importlib.util.module_from_spec(spec)
    sys.modules[name] = module
    spec.loader.exec_module(module)
    return module


def _fit(name, loss, rows, feats, **more):
    case = dict(name=name, do="fit", loss=loss, rows=rows, feats=feats, form="matrix_c", dtype="float64", nbins=64, depth=6, rounds=200, eta=0.1,
                rowsample=1.0, colsample=1.0, tree_type="binary", eval_rows=0, weights=False, classes=0)
    case.update(more)
    return case


def _use(name, do, loss, rows, feats, **more):
    case = dict(name=name, do=do, loss=loss, rows=rows, feats=feats, form="matrix_c", dtype="float64", nbins=64, depth=6, rounds=100, classes=0)
    case.update(more)
    return case


def listed():
    return [
        # one row scored by a service that keeps the model: the smallest call there is, the learners' default model size
        _use("predict_one_row", "predict", "mse", 1, 20),
        # a request of a few thousand rows against a boosted classifier (cfg4's features, bins and depth)
        _use("predict_batch", "predict", "logloss", 4_001, 28, nbins=128, depth=8, rounds=200),
        # a nightly scoring job in single precision (cfg2's features)
        _use("predict_500k", "predict", "mse", 500_000, 100, dtype="float32", rounds=200),
        # class probabilities of a multi-class model over an odd number of rows
        _use("predict_classes", "predict", "mlogloss", 200_003, 54, dtype="float32", classes=7),
        # leaf ids as features of another model
        _use("leaf_idx", "leaf_idx", "mse", 100_000, 20),
        # the smallest fits: a few thousand rows, the learners' defaults (a fold of a cross-validation, a test)
        _fit("fit_small", "mse", 2_000, 10, rounds=100),
        # cfg1, with the eval set that early stopping needs
        _fit("fit_cfg1_eval", "mse", 100_000, 10, eval_rows=25_000),
        # cfg2: rows and columns sampled, single-precision matrix
        _fit("fit_cfg2", "mse", 1_000_000, 100, dtype="float32", rowsample=0.5, colsample=0.5),
        # cfg4: a classifier on many rows, deeper trees and more bins, with an eval set
        _fit("fit_cfg4_eval", "logloss", 1_000_000, 28, form="matrix_f", nbins=128, depth=8, eta=0.05, rowsample=0.8, eval_rows=100_000),
        # cfg5's learner and features on an odd number of rows, oblivious trees, two outputs
        _fit("fit_mle_oblivious", "gaussian_mle", 500_009, 50, depth=7, tree_type="oblivious", rounds=100),
        # a weighted multi-class model on a table whose columns are real, whole-number and Bool
        _fit("fit_classes_table", "mlogloss", 60_013, 30, form="table", weights=True, classes=7, rounds=50),
        # cfg3, the headline configuration, whole: 200 rounds of depth 11 on 10M x 100
        _fit("fit_cfg3", "mse", 10_000_000, 100, form="matrix_f", depth=11),
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """A case of the same kinds with its sizes anywhere between the listed ones: up to 60 million cells and 300 trees of depth 9."""
    do = rng.choice(["fit", "fit", "fit", "fit", "predict", "predict", "predict", "leaf_idx"])
    loss = rng.choice(["mse", "mse", "logloss", "gaussian_mle", "mlogloss"])
    feats = _log_uniform(rng, 5, 120)
    classes = rng.randint(3, 9) if loss == "mlogloss" else 0
    case = dict(do=do, loss=loss, feats=feats, form=rng.choice(["matrix_c", "matrix_c", "matrix_f", "table"]), dtype=rng.choice(["float32", "float64"]),
                nbins=rng.choice([32, 64, 64, 128, 255]), depth=rng.randint(4, 9), classes=classes)
    table = case["form"] == "table"
    if do == "fit":
        cells = 4_000_000 if table or loss == "mlogloss" else 40_000_000
        rows = _log_uniform(rng, 1_000, min(1_000_000, cells // feats))
        case.update(rows=rows, rounds=_log_uniform(rng, 20, 60 if loss == "mlogloss" else 200), eta=rng.choice([0.05, 0.1, 0.3]),
                    rowsample=rng.choice([1.0, 1.0, 0.8, 0.5]), colsample=rng.choice([1.0, 1.0, 0.5]),
                    tree_type=rng.choice(["binary", "binary", "binary", "oblivious"]), eval_rows=rng.choice([0, 0, rows // 4]), weights=rng.choice([False, False, True]))
    elif do == "predict":
        case.update(rows=_log_uniform(rng, 1, min(1_000_000, (4_000_000 if table else 60_000_000) // feats)), rounds=_log_uniform(rng, 20, 300))
    else:
        case.update(rows=_log_uniform(rng, 1, min(200_000, 4_000_000 // feats)), rounds=_log_uniform(rng, 20, 200))
    return case


def _features(case, rows, gen):
    """(feats, rows) on the GPU, of the case's type: what the configurations of bench.py draw for the loss; in a table every third column
    holds whole numbers and every fifth truth values."""
    kind = torch.float32 if case["dtype"] == "float32" else torch.float64
    x = torch.empty((case["feats"], rows), dtype=kind, device="cuda")
    for j in range(case["feats"]):
        if case["form"] == "table" and j % 5 == 4:
            x[j] = (torch.rand(rows, generator=gen, device="cuda") < 0.3).to(kind)
        elif case["form"] == "table" and j % 3 == 2:
            x[j] = torch.randint(0, 40 * (1 + j % 7), (rows,), generator=gen, device="cuda").to(kind)
        elif case["loss"] in ("logloss", "mlogloss"):
            x[j].normal_(generator=gen)
        elif case["loss"] == "gaussian_mle":
            x[j].uniform_(-1, 1, generator=gen)
        else:
            x[j].uniform_(0, 1, generator=gen)
    return x


def _target(case, x, law, gen):
    """The target of every row, on the GPU: a signal of the loss's own kind, with noise.  `law` seeds its coefficients: the same for the
    training and the eval rows."""
    feats, rows = x.shape
    kind = x.dtype
    law = torch.Generator(device="cuda").manual_seed(law)

    def noise():
        return torch.randn(rows, generator=gen, device="cuda", dtype=kind)

    if case["loss"] == "mse" and feats == 100 and case.get("depth") == 11:  # cfg3: the target is noise
        return torch.rand(rows, generator=gen, device="cuda", dtype=kind)
    used = min(10, feats)
    coef = torch.randn((max(1, case["classes"]), used), generator=law, device="cuda", dtype=kind)
    z = x[:used] if case["form"] != "table" else (x[:used] - x[:used].mean(1, keepdim=True)) / (x[:used].std(1, keepdim=True) + 1e-9)
    if case["loss"] == "mse":
        return (coef[0, :, None] * z).sum(0) + 0.1 * noise()
    if case["loss"] == "logloss":
        s = 0.5 * (coef[0, :, None] * z).sum(0) + 0.5 * z[0] * z[1]
        return (torch.rand(rows, generator=gen, device="cuda", dtype=kind) < torch.sigmoid(s)).to(kind)
    if case["loss"] == "gaussian_mle":
        return torch.sin(3 * z[0]) + z[1] + torch.exp(0.5 * z[2]) * noise()
    best, y = None, torch.zeros(rows, dtype=torch.int64, device="cuda")
    for k in range(case["classes"]):
        s = (coef[k, :, None] * z).sum(0) + noise()
        if best is None:
            best = s
        else:
            y[s > best] = k
            best = torch.maximum(best, s)
    y[: case["classes"]] = torch.arange(case["classes"], device="cuda")[:rows]  # no class is without a row
    return y


def _host(case, x):
    """(feats, rows) on the GPU -> the matrix or the columns a program holds."""
    if case["form"] == "matrix_c":
        return x.T.contiguous().cpu().numpy()
    if case["form"] == "matrix_f":
        return x.cpu().numpy().T
    cols = {}
    for j, col in enumerate(x.cpu().numpy()):
        if j % 5 == 4:
            col = col > 0.5
        elif j % 3 == 2:
            col = col.astype(np.int64)
        cols["x%d" % (j + 1)] = np.ascontiguousarray(col)
    return cols


def _learner(pkg, case):
    args = dict(loss=case["loss"], nbins=case["nbins"], max_depth=case["depth"], nrounds=case["rounds"], eta=case.get("eta", 0.1),
                rowsample=case.get("rowsample", 1.0), colsample=case.get("colsample", 1.0), tree_type=case.get("tree_type", "binary"))
    kind = {"gaussian_mle": pkg.EvoTreeMLE, "mlogloss": pkg.EvoTreeClassifier}.get(case["loss"], pkg.EvoTreeRegressor)
    return kind(**args)


def _data(case, rows, law, gen):
    x = _features(case, rows, gen)
    y = _target(case, x, law, gen).cpu().numpy()
    return _host(case, x), y


def prepare(case, seed):
    pkg = _package()
    law = 2 * seed + 1
    gen = torch.Generator(device="cuda").manual_seed(2 * seed)
    config = _learner(pkg, case)
    table = case["form"] == "table"
    if case["do"] != "fit":  # a fitted model, kept by the program, and new rows
        x, y = _data(case, TRAIN_ROWS, law, gen)
        if table:
            model = pkg.fit(config, dict(x, y=y), target_name="y", verbosity=0)
        else:
            model = pkg.fit(config, x_train=x, y_train=y, verbosity=0)
        return dict(do=case["do"], pkg=pkg, model=model, x=_host(case, _features(case, case["rows"], gen)))
    x, y = _data(case, case["rows"], law, gen)
    w = (0.5 + torch.rand(case["rows"], generator=gen, device="cuda")).cpu().numpy() if case["weights"] else None
    xe, ye = _data(case, case["eval_rows"], law, gen) if case["eval_rows"] else (None, None)
    if not table:
        return dict(do="fit", pkg=pkg, config=config, args=dict(x_train=x, y_train=y, w_train=w, x_eval=xe, y_eval=ye, verbosity=0))
    args = dict(dtrain=dict(x, y=y), target_name="y", verbosity=0)
    if w is not None:
        args["dtrain"]["w"] = w
        args["weight_name"] = "w"
    if xe is not None:
        args["deval"] = dict(xe, y=ye)
        if w is not None:
            args["deval"]["w"] = np.ones(case["eval_rows"], np.float32)
    return dict(do="fit", pkg=pkg, config=config, args=args)


def run(state):
    pkg = state["pkg"]
    if state["do"] == "predict":
        return pkg.predict(state["model"], state["x"])
    if state["do"] == "leaf_idx":
        return pkg.predict_leaf_idx(state["model"], state["x"])
    m = pkg.fit(state["config"], **state["args"])
    out = {"bias": m.trees[0].pred}
    for field in ("feat", "cond_bin", "split", "w", "gain", "pred"):  # the whole model: every array of every tree
        out[field] = np.stack([getattr(t, field) for t in m.trees[1:]])
    if m.info["logger"] is not None:
        out["metric"] = np.asarray(m.info["logger"]["metrics"])
    return out


def _outputs(case):
    return case["classes"] if case["loss"] == "mlogloss" else 2 if case["loss"] == "gaussian_mle" else 1


def work(case):
    """A prediction reads the features and the model and writes its values; a fit reads its data once, and every round reads each sampled bin
    once (a byte) and each row's target and prediction, writes the prediction, and returns a tree.  Operations: a comparison for
    each level of each tree walked; an addition for each gradient row of each sampled bin."""
    rows, feats, rounds, size = case["rows"], case["feats"], case["rounds"], 4 if case["dtype"] == "float32" else 8
    if case["form"] == "table":  # a column in three holds Int64, one in five Bool
        size = 8
    outs, nodes = _outputs(case), (1 << case["depth"]) - 1
    if case["do"] != "fit":
        back = rows * 4 * (outs if case["do"] == "predict" else rounds + 1)
        return {"bytes": rows * feats * size + rounds * nodes * (4 + 4 * outs) + back, "flops": rows * rounds * (case["depth"] - 1)}
    kept, used, more = rows * case["rowsample"], math.ceil(feats * case["colsample"]), case["eval_rows"]
    once = (rows + more) * (feats * size + size)
    each = kept * used + rows * (4 + 8 * outs) + nodes * (18 + 4 * outs) + more * (case["depth"] - 1 + 4 + 8 * outs)
    return {"bytes": once + rounds * each, "flops": rounds * (kept * used * (2 * outs + 1) + more * (case["depth"] - 1))}


def tolerance(case):
    """Features, bins and leaf ids are whole numbers and stay the same; values, gains and metrics are 32-bit results."""
    return "exact" if case["do"] == "leaf_idx" else {"rel": 1e-5}
