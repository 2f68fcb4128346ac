"""Performance cases: the work a user has this library do, through its public
entry points.

Kinds of case:

- ``fit``: one complete training run (edges, binning, every tree, the model's
  readback), then the predictions of a held-out set and the model's feature
  importances, which is what a training program takes from it.  ``source`` says
  where the features are: ``host`` (``macboost_train``) or ``device``
  (``mbk_fit`` on features already in GPU memory).
- ``predict``: batch prediction of a trained model, of host rows
  (``macboost_predict``) or of rows and a forest in GPU memory
  (``mbk_predict_forest``).
- ``contrib``: TreeSHAP contributions of a trained model, of host rows
  (``macboost_predict_contrib``) or of rows in GPU memory (``mbk_treeshap``).

Data is synthetic: Friedman #1 (uniform features, the first five informative)
or "skewed" columns (normal, exponential and product columns, the shape of
collider data), optionally with categorical columns and missing entries.
"""
import ctypes
import json
import math
import os
import tempfile

import numpy as np
import torch

import macboost_amd as mb

# The shape of a case's model and data, and what a field is when a case does
# not name it.
_DEFAULTS = {
    "source": "host", "data": "friedman", "objective": "regression", "classes": 1,
    "bins": 256, "trees": 100, "depth": 6, "leaves": 0, "rate": 0.1, "cats": 0,
    "missing": 0.0, "weights": False, "goss": False, "subsample": 1.0, "valid": 0,
    "held": 20000,
}


def _full(case):
    return {**_DEFAULTS, **case}


def listed():
    return [
        # Interactive use: a model of a few hundred rows, every launch and
        # host-side step visible.
        {"name": "fit_tiny", "kind": "fit", "rows": 1000, "cols": 10, "objective": "binary",
         "bins": 64, "trees": 20, "depth": 4, "held": 200},
        # The 20k x 100 regression at 64 bins from host memory, the size most
        # tabular data sets have.
        {"name": "fit_20k", "kind": "fit", "rows": 20000, "cols": 100, "bins": 64},
        # Multiclass with sample weights on sizes that are multiples of nothing.
        {"name": "fit_multiclass_odd", "kind": "fit", "rows": 99991, "cols": 37,
         "objective": "multiclass", "classes": 5, "bins": 128, "trees": 20, "depth": 5,
         "weights": True},
        # 1M x 100 with 20 categorical columns and 20% missing entries, scored
        # on a 200k-row validation set after every tree.
        {"name": "fit_mixed_1m", "kind": "fit", "rows": 1000000, "cols": 100, "cats": 20,
         "missing": 0.2, "valid": 200000},
        # Deep trees, leaf renewal (absolute error) and bagging on odd sizes.
        {"name": "fit_deep_odd", "kind": "fit", "rows": 500009, "cols": 53, "objective": "mae",
         "bins": 255, "trees": 50, "depth": 9, "subsample": 0.8, "source": "device"},
        # Best-first growth with 63 leaves.
        {"name": "fit_leafwise_2m", "kind": "fit", "rows": 2000000, "cols": 100, "leaves": 63,
         "source": "device"},
        # 10M x 28 binary classification with gradient-based sampling.
        {"name": "fit_goss_10m", "kind": "fit", "rows": 10000000, "cols": 28, "data": "skewed",
         "objective": "binary", "goss": True, "source": "device"},
        # The largest: 10M x 100 regression, 100 level-wise trees of depth 6.
        {"name": "fit_10m", "kind": "fit", "rows": 10000000, "cols": 100, "source": "device"},
        # Serving: one small request against a 100-tree model.
        {"name": "predict_1k", "kind": "predict", "rows": 1003, "cols": 100},
        # Batch inference of 500k rows through 100 trees.
        {"name": "predict_500k", "kind": "predict", "rows": 500000, "cols": 100},
        # TreeSHAP of 200k rows through 100 trees of depth 6.
        {"name": "contrib_200k", "kind": "contrib", "rows": 200000, "cols": 100},
        # TreeSHAP of a deeper model with categorical and missing values, rows
        # resident on the GPU, odd sizes.
        {"name": "contrib_deep_odd", "kind": "contrib", "rows": 20011, "cols": 41, "cats": 5,
         "missing": 0.1, "trees": 50, "depth": 8, "source": "device"},
    ]


def _spread(rng, lo, hi):
    """An integer of [lo, hi], uniform in its logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    case = {"kind": rng.choice(["fit", "fit", "fit", "predict", "contrib"])}
    case["cols"] = _spread(rng, 5, 200)
    case["depth"] = rng.choice([3, 4, 5, 6, 6, 7, 8, 9])
    case["bins"] = rng.choice([32, 64, 128, 255, 256, 256])
    case["data"] = rng.choice(["friedman", "skewed"])
    case["cats"] = rng.choice([0, 0, rng.randint(1, max(1, case["cols"] // 4))])
    case["cats"] = min(case["cats"], case["cols"] - 5)
    case["missing"] = rng.choice([0.0, 0.0, 0.1, 0.3])
    case["source"] = rng.choice(["host", "device"])
    case["trees"] = rng.randint(10, 100)
    if case["kind"] == "fit":
        case["objective"] = rng.choice(["regression", "regression", "binary", "multiclass", "mae",
                                        "huber", "quantile", "poisson", "tweedie"])
        if case["objective"] == "multiclass":
            case["classes"] = rng.randint(3, 6)
            case["trees"] = max(5, case["trees"] // case["classes"])
        most = 20_000_000 if case["source"] == "host" else 500_000_000
        top = max(1000, min(10_000_000, most // case["cols"]))
        if case["depth"] > 7 or case["objective"] in ("multiclass", "mae", "quantile"):
            top = max(1000, min(top, 50_000_000 // case["cols"]))
        case["rows"] = _spread(rng, 500, top)
        case["held"] = _spread(rng, 100, 20000)
        if rng.random() < 0.3 and case["depth"] <= 8:
            case["leaves"] = rng.randint(4, min(63, 2 ** case["depth"]))
        case["weights"] = rng.random() < 0.25
        sampling = rng.random()
        if sampling < 0.2 and case["objective"] != "multiclass":
            case["goss"] = True
        elif sampling < 0.35:
            case["subsample"] = rng.choice([0.5, 0.8])
        if rng.random() < 0.2:
            case["valid"] = max(100, case["rows"] // 5)
    elif case["kind"] == "predict":
        case["rows"] = _spread(rng, 1, min(1_000_000, 50_000_000 // case["cols"]))
    else:
        per_row = case["trees"] * 2 ** case["depth"]
        case["rows"] = _spread(rng, 1, min(200_000, 1_000_000_000 // per_row))
    return case


# ---- data -----------------------------------------------------------------

def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _features(c, rows, gen):
    """Feature-major [cols][rows] float32 on the GPU, and the noise-free score."""
    x = torch.empty((c["cols"], rows), device="cuda")
    if c["data"] == "friedman":
        x.uniform_(generator=gen)
        score = (10 * torch.sin(math.pi * x[0] * x[1]) + 20 * (x[2] - 0.5) ** 2
                 + 10 * x[3] + 5 * x[4])
    else:
        for f in range(c["cols"]):
            if f % 4 == 3 and f >= 5:                # derived column
                torch.mul(x[f - 3], x[f - 2], out=x[f])
            elif f % 3 == 2:
                x[f].exponential_(generator=gen)
            else:
                x[f].normal_(generator=gen)
        score = (torch.where(x[0] > 0.2, x[1], -x[1]) + torch.sqrt(x[2]) * (x[3] > 0)
                 + 0.5 * x[4].clamp(-2, 2))
    return x, score


def _categories(c, x, score, gen):
    """The last c["cats"] columns become integer categories, each with an
    offset of its own in the score."""
    most = min(64, c["bins"] - 2)
    for j in range(c["cats"]):
        f = c["cols"] - c["cats"] + j
        card = 2 + (7 * j + 3 * c["cols"]) % (most - 1)
        offsets = torch.randn(card, generator=torch.Generator().manual_seed(17 + j)).cuda()
        codes = torch.randint(card, (x.shape[1],), generator=gen, device="cuda")
        x[f] = codes.float()
        score += offsets[codes]


def _labels(c, score, gen):
    noise = torch.empty_like(score).normal_(generator=gen)
    objective = c["objective"]
    if objective == "binary":
        z = (score - score.mean()) / score.std().clamp_min(1e-6)
        return (2 * z + noise > 0).float()
    if objective in ("poisson", "tweedie"):
        z = (score - score.mean()) / score.std().clamp_min(1e-6)
        return torch.poisson(torch.exp(0.5 * z), generator=gen)
    if objective == "multiclass":
        z = (score - score.mean()) / score.std().clamp_min(1e-6) + 0.3 * noise
        return (torch.special.ndtr(z / 1.05) * c["classes"]).floor().clamp(0, c["classes"] - 1)
    return score + noise


def _data(c, rows, gen):
    """(x on the GPU, y on the host) of `rows` new rows."""
    x, score = _features(c, rows, gen)
    if c["cats"]:
        _categories(c, x, score, gen)
    y = _labels(c, score, gen).cpu().numpy()
    if c["missing"]:
        for f in range(c["cols"] - c["cats"]):
            x[f].masked_fill_(torch.rand(rows, generator=gen, device="cuda") < c["missing"],
                              float("nan"))
    return x, y


def _config(c):
    config = {"num_trees": c["trees"], "max_depth": c["depth"], "num_bins": c["bins"],
              "learning_rate": c["rate"], "objective": c["objective"]}
    if c["objective"] == "multiclass":
        config["num_class"] = c["classes"]
    if c["leaves"]:
        config["num_leaves"] = c["leaves"]
    if c["goss"]:
        config.update(goss=True, goss_top_rate=0.2, goss_other_rate=0.1)
    if c["subsample"] < 1.0:
        config["subsample"] = c["subsample"]
    if c["cats"]:
        config["categorical_features"] = list(range(c["cols"] - c["cats"], c["cols"]))
    if c["objective"] == "quantile":
        config["alpha"] = 0.7
    if c["objective"] == "huber":
        config["alpha"] = 1.0
    return config


# ---- a trained model and its flat arrays ----------------------------------

_MODEL_ROWS = 100_000


def _model(c, gen):
    x, y = _data(c, _MODEL_ROWS, gen)
    return mb.train(_config(c), x.cpu().numpy(), y, feature_major=True)


def _forest(handle):
    """The model file's trees as flat arrays [trees][nodes]."""
    with tempfile.TemporaryDirectory() as folder:
        path = os.path.join(folder, "model.json")
        mb.save(handle, path)
        with open(path) as f:
            model = json.load(f)
    trees = model["trees"]
    nodes = max(len(t["feature"]) for t in trees)
    shape = (len(trees), nodes)
    forest = {"feature": np.full(shape, -1, np.int32), "threshold": np.zeros(shape, np.float32),
              "flags": np.zeros(shape, np.uint8), "leaf": np.zeros(shape, np.float32),
              "cover": np.zeros(shape, np.float32), "mask": np.zeros(shape + (8,), np.uint32)}
    for i, t in enumerate(trees):
        n = len(t["feature"])
        for key in ("feature", "threshold", "flags", "leaf", "cover"):
            forest[key][i, :n] = np.array(t[key])
        if t["catMask"]:
            forest["mask"][i, :n] = np.array(t["catMask"], np.uint32).reshape(n, 8)
    forest["has_mask"] = any(len(t["catMask"]) for t in trees)
    forest["base"] = float(np.float32(model["baseScore"]))
    forest["bins"] = model["numBins"]
    return forest


# ---- prepare and run ------------------------------------------------------

def prepare(case, seed):
    c = _full(case)
    gen = _generator(seed)
    state = {"case": c, "config": _config(c)}
    if c["kind"] == "fit":
        x, state["y"] = _data(c, c["rows"], gen)
        state["w"] = None
        if c["weights"]:
            w = torch.rand(c["rows"], generator=gen, device="cuda") + 0.5
            state["w"] = w.cpu().numpy()
        held, _ = _data(c, c["held"], gen)
        state["held"] = held.cpu().numpy()
        state["eval"] = None
        if c["valid"]:
            xv, yv = _data(c, c["valid"], gen)
            state["eval"] = (xv.cpu().numpy().T, yv)
        if c["source"] == "device":
            state["x"] = x
            state["context"] = mb.Context()
        else:
            state["x"] = x.cpu().numpy()
    else:
        state["model"] = _model(c, gen)
        x, _ = _data(c, c["rows"], gen)
        if c["source"] == "device":
            state["x"] = x
            state["forest"] = f = _forest(state["model"])
            state["context"] = mb.Context()
            state["device"] = {k: torch.from_numpy(f[k].view(np.int32) if k == "mask" else f[k]).cuda()
                               for k in ("feature", "threshold", "flags", "leaf", "mask")}
            width = c["cols"] + 1 if c["kind"] == "contrib" else 1
            state["out"] = torch.empty((c["rows"], width), device="cuda")
        else:
            state["x"] = x.cpu().numpy()
    torch.cuda.synchronize()
    return state


def _pointer(a):
    return a.ctypes.data_as(ctypes.c_void_p)


def _run_fit(s):
    c = s["case"]
    if c["source"] == "device":
        model = s["context"].fit(s["config"], s["x"].data_ptr(), c["rows"], c["cols"], s["y"],
                                 sample_weight=s["w"], eval_set=s["eval"])
    else:
        model = mb.train(s["config"], s["x"], s["y"], eval_set=s["eval"], sample_weight=s["w"],
                         feature_major=True)
    return {"held": mb.predict(model, s["held"], feature_major=True),
            "gain": mb.feature_importance(model, "gain"),
            "splits": mb.feature_importance(model, "split"),
            "eval": mb.eval_history(model)}


def run(state):
    s, c = state, state["case"]
    if c["kind"] == "fit":
        return _run_fit(s)
    if c["source"] == "host":
        f = mb.predict if c["kind"] == "predict" else mb.predict_contrib
        return f(s["model"], s["x"], feature_major=True)
    f, d, out = s["forest"], s["device"], s["out"]
    trees, nodes = f["feature"].shape
    if c["kind"] == "predict":
        s["context"].call("mbk_predict_forest", d["feature"].data_ptr(), d["threshold"].data_ptr(),
                          d["flags"].data_ptr(), d["leaf"].data_ptr(),
                          d["mask"].data_ptr() if f["has_mask"] else None, trees, nodes,
                          s["x"].data_ptr(), c["rows"], f["bins"] - 1, f["base"], out.data_ptr())
    else:
        s["context"].call("mbk_treeshap", _pointer(f["feature"]), _pointer(f["threshold"]),
                          _pointer(f["flags"]), _pointer(f["leaf"]), _pointer(f["cover"]),
                          _pointer(f["mask"]) if f["has_mask"] else None, trees, nodes, f["base"],
                          f["bins"] - 1, s["x"].data_ptr(), c["rows"], c["cols"], out.data_ptr())
    return out


# ---- what a pass cannot do without ----------------------------------------

def work(case):
    c = _full(case)
    n, f = c["rows"], c["cols"]
    if c["kind"] == "fit":
        # X and the labels once; the bins written; then per tree every row's
        # bins and gradient word once for the root, a quarter of the rows per
        # deeper level (the smaller children: half the rows where splits are
        # even, fewer where they are not), and prediction, label and new
        # prediction of every row.  Sampled trees see their share of the rows.
        kept = 0.3 if c["goss"] else c["subsample"]
        trees = c["trees"] * c["classes"]
        visits = trees * n * kept * (1 + 0.25 * (c["depth"] - 1))
        return {"bytes": n * (5 * f + 4) + visits * (f + 4) + trees * n * 12
                + 4 * c["valid"] * f + 4 * c["held"] * (f + 1),
                "flops": 2 * visits * f}
    flops = n * c["trees"] * c["depth"]
    if c["kind"] == "contrib":
        # every path of a tree: one test and one addition per split
        flops *= 2 * 2 ** c["depth"]
        return {"bytes": 4 * n * (2 * f + 1), "flops": flops}
    return {"bytes": 4 * n * (f + 1), "flops": flops}


def tolerance(case):
    # Training sums whole numbers and picks splits by a stated order, and a
    # prediction adds its leaves in tree order: both are the same to the bit.
    # Contributions are summed in 64 bits and rounded once to 32: measured 1e-8
    # to 3e-8 from the 64-bit values (2-norm).
    return {"rel": 1e-7} if case["kind"] == "contrib" else "exact"


# ---- the same values in 64 bits -------------------------------------------

def _goes_left(f, t, n, x):
    """Which rows of the GPU matrix x take node n's left child in tree t."""
    v = x[int(f["feature"][t, n])]
    flags = int(f["flags"][t, n])
    if flags & 2:
        bins = f["bins"] - 1
        code = torch.round(v)
        code = torch.where(torch.isfinite(v) & (code >= 0) & (code < bins), code,
                           torch.full_like(code, bins)).long()
        words = torch.from_numpy(f["mask"][t, n].astype(np.int64)).cuda()
        return (words[code >> 5] >> (code & 31)) & 1 == 1
    left = v <= float(f["threshold"][t, n])
    return torch.where(torch.isnan(v), torch.full_like(left, bool(flags & 1)), left)


def _leaves(f, t):
    """Tree t's leaves as (leaf, [(node, takes the left child)] from the root)."""
    found, todo = [], [(0, [])]
    while todo:
        n, path = todo.pop()
        if f["feature"][t, n] < 0:
            found.append((n, path))
        else:
            todo += [(2 * n + 1, path + [(n, True)]), (2 * n + 2, path + [(n, False)])]
    return found


def _exact_predict(f, x):
    out = torch.full((x.shape[1],), f["base"], dtype=torch.float64, device="cuda")
    for t in range(f["feature"].shape[0]):
        inside = {0: torch.ones(x.shape[1], dtype=torch.bool, device="cuda")}
        for n in range(f["feature"].shape[1]):
            here = inside.pop(n, None)
            if here is None:
                continue
            if f["feature"][t, n] < 0:
                out += here * float(f["leaf"][t, n])
            else:
                left = _goes_left(f, t, n, x)
                inside[2 * n + 1], inside[2 * n + 2] = here & left, here & ~left
    return out


def _shapley_tables(zero):
    """zero [P][U], the unfollowed share of each feature of P paths, to
    [P][2^U][U]: per pattern of followed features, each feature's Shapley value
    of the path's product game."""
    paths, u = zero.shape
    one = ((torch.arange(1 << u, device="cuda")[:, None] >> torch.arange(u, device="cuda")) & 1
           ).double()
    table = torch.empty((paths, 1 << u, u), dtype=torch.float64, device="cuda")
    weight = torch.tensor([math.factorial(k) * math.factorial(u - 1 - k) / math.factorial(u)
                           for k in range(u)], dtype=torch.float64, device="cuda")
    for i in range(u):
        poly = torch.zeros((paths, 1 << u, u), dtype=torch.float64, device="cuda")
        poly[:, :, 0] = 1.0                            # by size of the coalition
        for j in range(u):
            if j != i:
                grown = poly * zero[:, None, j:j + 1]
                grown[:, :, 1:] += poly[:, :, :-1] * one[None, :, j:j + 1]
                poly = grown
        table[:, :, i] = (poly * weight).sum(2) * (one[:, i] - zero[:, i:i + 1])
    return table


def _exact_contrib(f, x):
    cols, rows = x.shape
    phi = torch.zeros((cols + 1, rows), dtype=torch.float64, device="cuda")
    phi[cols] = f["base"]
    for t in range(f["feature"].shape[0]):
        left = {n: _goes_left(f, t, n, x) for n in range(f["feature"].shape[1])
                if f["feature"][t, n] >= 0}
        paths = {}                                     # by number of features
        for leaf, path in _leaves(f, t):
            value = float(f["leaf"][t, leaf])
            phi[cols] += value * float(f["cover"][t, leaf]) / float(f["cover"][t, 0])
            feats, zero, follow = [], [], []
            for n, goes in path:
                share = (float(f["cover"][t, 2 * n + 1 if goes else 2 * n + 2])
                         / float(f["cover"][t, n]))
                feature = int(f["feature"][t, n])
                if feature not in feats:
                    feats.append(feature)
                    zero.append(1.0)
                    follow.append([])
                zero[feats.index(feature)] *= share
                follow[feats.index(feature)].append(left[n] if goes else ~left[n])
            paths.setdefault(len(feats), []).append((value, feats, zero, follow))
        for u, group in paths.items():
            if u == 0:
                continue
            tables = _shapley_tables(torch.tensor([p[2] for p in group], dtype=torch.float64,
                                                  device="cuda"))
            for (value, feats, _, follow), table in zip(group, tables):
                pattern = torch.zeros(rows, dtype=torch.long, device="cuda")
                for k, taken in enumerate(follow):
                    every = taken[0]
                    for other in taken[1:]:
                        every = every & other
                    pattern |= every.long() << k
                phi[feats] += value * table[pattern].T
    return phi.T.contiguous()


def exact(case, seed):
    c = _full(case)
    if c["kind"] == "fit":
        return None                                    # a fit's splits are whole-number work
    state = prepare(case, seed)
    f = state["forest"] if "forest" in state else _forest(state["model"])
    x = state["x"] if c["source"] == "device" else torch.from_numpy(state["x"]).cuda()
    if c["kind"] == "contrib":
        out = _exact_contrib(f, x)
        return out
    out = _exact_predict(f, x)
    return out.reshape(-1, 1) if c["source"] == "device" else out
