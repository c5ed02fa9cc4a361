"""Timed cases of this library: what a program that trains, scores or steps
gradient-boosted trees with it calls, from the smallest matrix to the largest.

Kinds of case (``kind``):

fit        new data to a saved model: a matrix from device arrays, labels, a
           booster, its rounds, the model JSON -- what the trainer process does
           for every plan.
rounds     boosting rounds on a matrix the program keeps (hyperparameter
           search, custom objectives with caller gradients).
predict    scoring rows with a loaded model (values, probabilities).
histogram  one histogram pass over all rows of a resident matrix.
level      one level of a tree driven through the operators: gathered
           histograms of the smaller children, siblings by subtraction, split
           evaluation, partition.
cuts       quantile cuts and uint8 bins of a raw matrix.
gradients  softmax / logistic / squared gradients and their quantiser.

All results are exact by definition: sums are integers, trees follow from
integer sums with fixed tie rules, and the float steps are IEEE operations in
a fixed order, so two correct builds agree bit for bit.
"""
import json
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "decision-programs_amd"))

import dpgbdt  # noqa: E402
from dpgbdt import ops  # noqa: E402

DEVICE = "cuda:0"


# ---------------------------------------------------------------------------
# Cases
# ---------------------------------------------------------------------------
def listed():
    return [
        # A small table (10k rows), the whole fit: launch and host latency count.
        fit("fit_10k_binary", 10_000, 8, "uniform", "binary:logistic", 6, 10),
        # The ordinary fit: a million rows of continuous features, logistic.
        fit("fit_1m_binary", 1_000_000, 28, "normal", "binary:logistic", 8, 20, eta=0.1),
        # Mostly missing wide data, squared error, 64 bins, deep trees.
        fit("fit_2m_sparse", 2_000_000, 1000, "normal", "reg:squarederror", 10, 5, missing=0.95,
            max_bin=64),
        # Ten classes of pixel rows on a kept matrix: ten trees a round.
        rounds("rounds_60k_softprob", 60_000, 784, "pixels", "multi:softprob", 6, 10, classes=10),
        # Ten million rows on a kept matrix, the program's own gradients.
        rounds("rounds_10m_custom", 10_000_000, 128, "mixed", "caller", 8, 5),
        # Online scoring: a handful of rows, latency.
        predict("predict_64", 64, 28, 1, 100, 8, 0.0),
        # Scoring a validation set with a binary model, some values missing.
        predict("predict_1m_binary", 1_000_000, 28, 1, 100, 8, 0.05),
        # Probabilities of a ten-class model (50 rounds) for its 60k rows.
        predict("predict_60k_softprob", 60_000, 784, 10, 50, 6, 0.0),
        # The root histogram of ten million rows, a quarter of the features small integers.
        {"name": "histogram_10m", "kind": "histogram", "rows": 10_000_000, "features": 128,
         "bins": 256, "small": 32},
        # One level of 32 nodes of an odd-sized matrix, operator by operator.
        {"name": "level_700k", "kind": "level", "rows": 700_001, "features": 100, "bins": 256,
         "pairs": 16},
        # Cuts and bins of a raw matrix with missing values.
        {"name": "cuts_1m_missing", "kind": "cuts", "rows": 999_983, "features": 100,
         "data": "mixed", "missing": 0.2, "max_bin": 255},
        # A ten-class objective step over a million rows.
        {"name": "gradients_1m_softprob", "kind": "gradients", "rows": 1_000_000,
         "objective": ops_objective("multi:softprob"), "classes": 10},
    ]


def draw(rng):
    def log(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["fit", "fit", "rounds", "predict", "predict", "histogram", "level", "cuts",
                       "gradients"])
    if kind in ("fit", "rounds"):
        f = log(4, 300)
        n = min(log(2_000, 3_000_000), 200_000_000 // f)
        objective = rng.choice(["binary:logistic", "reg:squarederror", "multi:softprob"] if
                               kind == "fit" else ["binary:logistic", "multi:softprob", "caller"])
        classes = rng.randint(3, 12) if objective == "multi:softprob" else 1
        depth = rng.randint(4, 9)
        make = fit if kind == "fit" else rounds
        case = make(None, n, f, rng.choice(["uniform", "normal", "mixed", "pixels"]), objective,
                    depth, rng.randint(2, 12) if classes == 1 else rng.randint(1, 4),
                    eta=rng.choice([0.1, 0.3]), classes=classes,
                    missing=rng.choice([0.0, 0.0, 0.1, 0.9]),
                    max_bin=rng.choice([32, 64, 128, 255, 256]))
    elif kind == "predict":
        classes = rng.choice([1, 1, rng.randint(3, 12)])
        f = log(4, 800)
        n = min(log(1, 2_000_000), 100_000_000 // f)
        case = predict(None, n, f, classes, log(10, 300) if classes == 1 else log(5, 60),
                       rng.randint(4, 10), rng.choice([0.0, 0.1]))
        while case["rows"] * case["rounds"] * classes > 200_000_000:
            case["rows"] //= 2
    elif kind == "histogram":
        f = log(8, 300)
        case = {"name": None, "kind": kind, "rows": min(log(20_000, 10_000_000), 600_000_000 // f),
                "features": f, "bins": rng.choice([32, 64, 255, 256]),
                "small": rng.choice([0, 0, f // 3])}
    elif kind == "level":
        f = log(8, 300)
        case = {"name": None, "kind": kind, "rows": min(log(5_000, 4_000_000), 200_000_000 // f),
                "features": f, "bins": rng.choice([32, 64, 255, 256]),
                "pairs": rng.choice([1, 2, 5, 16, 64])}
    elif kind == "cuts":
        f = log(4, 400)
        case = {"name": None, "kind": kind, "rows": min(log(1_000, 5_000_000), 200_000_000 // f),
                "features": f, "data": rng.choice(["uniform", "normal", "mixed", "pixels"]),
                "missing": rng.choice([0.0, 0.0, 0.2, 0.9]),
                "max_bin": rng.choice([16, 64, 200, 255])}
    else:
        objective = rng.choice(["binary:logistic", "reg:squarederror", "multi:softprob"])
        classes = rng.randint(3, 12) if objective == "multi:softprob" else 1
        case = {"name": None, "kind": kind, "rows": log(5_000, 8_000_000) // classes + 1,
                "objective": ops_objective(objective), "classes": classes}
    case.pop("name")
    return case


def fit(name, rows, features, data, objective, depth, n_rounds, eta=0.3, classes=1, missing=0.0,
        max_bin=256):
    return {"name": name, "kind": "fit", "rows": rows, "features": features, "data": data,
            "missing": missing, "objective": objective, "classes": classes, "depth": depth,
            "rounds": n_rounds, "eta": eta, "max_bin": max_bin}


def rounds(name, *args, **kwargs):
    return {**fit(name, *args, **kwargs), "kind": "rounds"}


def predict(name, rows, features, classes, n_rounds, depth, missing):
    return {"name": name, "kind": "predict", "rows": rows, "features": features,
            "classes": classes, "rounds": n_rounds, "depth": depth, "missing": missing}


def ops_objective(name):
    return {"binary:logistic": 0, "multi:softprob": 1, "reg:squarederror": 2}[name]


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------
def generator(seed):
    g = torch.Generator(device=DEVICE)
    g.manual_seed(seed)
    return g


def matrix(rows, features, data, missing, gen):
    """float32 [rows, features]; NaN with probability `missing`.  Made in blocks of rows, so
    that the largest matrices need no temporaries of their own size."""
    x = torch.empty((rows, features), dtype=torch.float32, device=DEVICE)
    step = max(1, (1 << 27) // features)
    for a in range(0, rows, step):
        part = x[a:a + step]
        if data == "uniform":
            part.uniform_(generator=gen)
        elif data == "pixels":  # mostly zero, else 1..255
            part.uniform_(-1020.0, 255.0, generator=gen)
            part.ceil_().clamp_(min=0.0)
        else:
            part.normal_(generator=gen)
            if data == "mixed":  # half normal, a quarter lognormal, a quarter U{0..15}
                a1, a2 = features // 2, features - features // 4
                part[:, a1:a2].exp_()
                part[:, a2:].uniform_(0.0, 16.0, generator=gen).floor_().clamp_(max=15.0)
        if missing:
            lost = torch.empty_like(part).uniform_(generator=gen) < missing
            part.masked_fill_(lost, float("nan"))
    return x


def score(x, classes, gen):
    """A signal the features carry: a sparse linear part plus pairwise products."""
    f = x.shape[1]
    pick = torch.randint(0, f, (classes, 6), generator=gen, device=DEVICE)
    w = torch.randn((classes, 6), generator=gen, device=DEVICE)
    out = torch.empty((x.shape[0], classes), device=DEVICE)
    for k in range(classes):
        part = x[:, pick[k]].nan_to_num()
        part = part / (part.abs().mean(dim=0, keepdim=True) + 1e-3)
        out[:, k] = part @ w[k] + part[:, 0] * part[:, 1]
    return out


def training_data(case, seed):
    gen = generator(seed)
    x = matrix(case["rows"], case["features"], case["data"], case["missing"], gen)
    s = score(x, case["classes"], gen)
    noise = torch.randn(s.shape, generator=gen, device=DEVICE)
    if case["objective"] == "multi:softprob":
        y = (s + noise).argmax(dim=1).float()
    elif case["objective"] == "binary:logistic":
        y = (s + noise > 0).float()[:, 0]
    else:
        y = (s + 0.1 * noise)[:, 0]
    return x, y.contiguous()


def parameters(case):
    p = {"objective": "reg:squarederror" if case["objective"] == "caller" else case["objective"],
         "tree_method": "hist", "device": "cuda:0", "max_depth": case["depth"],
         "eta": case["eta"], "lambda": 1.0, "min_child_weight": 1.0, "max_bin": case["max_bin"]}
    if case["classes"] > 1:
        p["num_class"] = case["classes"]
    return p


def forest(case, seed):
    """A random model: trees that split every node of the first three levels and six in seven
    below, thresholds at the features' values, leaves of boosted size.  Node arrays per tree."""
    rng = np.random.default_rng(seed)
    trees = []
    for _ in range(case["rounds"] * case["classes"]):
        left, level, feature, cond, default = [-1], [0], [0], [0.0], [0]
        i = 0
        while i < len(left):
            if level[i] < case["depth"] and (level[i] < 3 or rng.random() < 6.0 / 7.0):
                left[i] = len(left)
                feature[i] = int(rng.integers(case["features"]))
                cond[i] = float(np.float32(rng.normal()))
                default[i] = int(rng.integers(2))
                for _ in range(2):
                    left.append(-1)
                    level.append(level[i] + 1)
                    feature.append(0)
                    cond.append(0.0)
                    default.append(0)
            else:
                cond[i] = float(np.float32(0.1 * rng.normal()))
            i += 1
        trees.append((left, feature, cond, default))
    return trees


def model_json(case, trees):
    classes, objective = case["classes"], "binary:logistic"
    if classes > 1:
        objective = "multi:softprob"
    nodes = []
    for t, (left, feature, cond, default) in enumerate(trees):
        right = [v + 1 if v >= 0 else -1 for v in left]
        nodes.append({"id": t, "left_children": left, "right_children": right,
                      "split_indices": feature, "split_conditions": cond,
                      "default_left": default})
    model = {"gbtree_model_param": {"num_parallel_tree": "1", "num_trees": str(len(trees))},
             "iteration_indptr": list(range(0, len(trees) + 1, classes)),
             "tree_info": [t % classes for t in range(len(trees))], "trees": nodes}
    base = json.dumps([0.5 if classes == 1 else 0.0] * classes)
    return json.dumps({"learner": {
        "attributes": {}, "feature_names": [], "feature_types": [],
        "gradient_booster": {"model": model, "name": "gbtree"},
        "learner_model_param": {"base_score": base, "num_class": str(classes if classes > 1 else 0),
                                "num_feature": str(case["features"]), "num_target": "1"},
        "objective": {"name": objective}}, "version": [3, 4, 1]})


def fixed_point(x):
    """The quantiser's rule: q = rint(x * 2^e), e = 30 - the frexp exponent of max|x|."""
    e = 30 - math.frexp(float(x.abs().max()))[1]
    return torch.round(x.double() * 2.0 ** e).to(torch.int32), e


def gradient_pairs(n, gen):
    g = torch.randn(n, generator=gen, device=DEVICE)
    h = torch.rand(n, generator=gen, device=DEVICE) * 0.24 + 0.01
    (qg, eg), (qh, eh) = fixed_point(g), fixed_point(h)
    return torch.stack([qg, qh], dim=1).contiguous(), eg, eh


def binned(case, gen):
    """Resident bins of quantile-cut features (each bin as likely as the others); the last
    `small` features take 16 values.  -> layout, tile-major bins, bins per feature."""
    n, f = case["rows"], case["features"]
    n_bins = np.full(f, case["bins"], dtype=np.int32)
    if case.get("small"):
        n_bins[f - case["small"]:] = 16
    lay = ops.layout(n, f, 0, -1)
    ops.layout_pair_tiles(lay, np.concatenate([[0], np.cumsum(n_bins)]))
    bins = torch.zeros(ops.layout_bytes(lay), dtype=torch.uint8, device=DEVICE)
    tiles = bins[:lay.n_tiles * n * 16].view(lay.n_tiles, n, 16)
    for t in range(lay.n_tiles):
        width = min(16, f - 16 * t)
        for top in sorted(set(n_bins[16 * t:16 * t + width].tolist())):
            at = [j for j in range(width) if n_bins[16 * t + j] == top]
            tiles[t][:, at[0]:at[-1] + 1] = torch.randint(
                0, top, (n, at[-1] + 1 - at[0]), generator=gen, device=DEVICE, dtype=torch.uint8)
    ops.join_tiles(bins, lay)
    return lay, bins, n_bins


def prepare(case, seed):
    kind = case["kind"]
    state = {"case": case}
    if kind == "fit":
        state["x"], state["y"] = training_data(case, seed)
    elif kind == "rounds":
        x, y = training_data(case, seed)
        d = dpgbdt.DMatrix(x, y)
        state["matrix"] = d
        if case["objective"] == "caller":
            gen = generator(seed + 1)
            state["grad"] = torch.randn((case["rows"], 1), generator=gen, device=DEVICE)
            state["hess"] = torch.rand((case["rows"], 1), generator=gen, device=DEVICE) * 0.24 + 0.01
        train(state, d, 1)  # an earlier model of the search: the matrix is quantised
    elif kind == "predict":
        state["x"] = matrix(case["rows"], case["features"], "normal", case["missing"],
                            generator(seed))
        state["model"] = dpgbdt.Booster.from_buffer(model_json(case, forest(case, seed)))
    elif kind == "histogram":
        gen = generator(seed)
        state["layout"], state["bins"], n_bins = binned(case, gen)
        state["stride"] = int(n_bins.max())
        state["gpair"] = gradient_pairs(case["rows"], gen)[0]
        state["ws"] = ops.Workspace()
    elif kind == "level":
        prepare_level(state, case, seed)
    elif kind == "cuts":
        state["x"] = matrix(case["rows"], case["features"], case["data"], case["missing"],
                            generator(seed))
        state["ws"] = ops.Workspace()
        state["layout"] = ops.layout(case["rows"], case["features"], 0,
                                     255 if case["missing"] else -1)
    else:
        gen = generator(seed)
        n, k = case["rows"], case["classes"]
        state["margin"] = 2.0 * torch.randn((n, k), generator=gen, device=DEVICE)
        if case["objective"] == 2:
            state["label"] = torch.randn(n, generator=gen, device=DEVICE)
        else:
            state["label"] = torch.randint(0, max(k, 2), (n,), generator=gen,
                                           device=DEVICE).float()
        state["ws"] = ops.Workspace()
    return state


def prepare_level(state, case, seed):
    """A level of 2 * pairs nodes: random row lists, the parents' histograms."""
    gen, rng = generator(seed), np.random.default_rng(seed)
    n, pairs = case["rows"], case["pairs"]
    lay, bins, n_bins = binned(case, gen)
    gpair, eg, eh = gradient_pairs(n, gen)
    order = torch.randperm(n, generator=gen, device=DEVICE)
    edges = np.concatenate([[0], np.cumsum(rng.dirichlet(np.ones(pairs) * 2.0) * n)])
    edges = np.clip(np.round(edges).astype(np.int64), 0, n)
    edges[-1] = n
    small, other, parents = [], [], []
    for i in range(pairs):
        a, b = int(edges[i]), int(edges[i + 1])
        cut = a + int(round((b - a) * rng.uniform(0.1, 0.9)))
        halves = sorted([(a, cut), (cut, b)], key=lambda s: s[1] - s[0])
        small.append(halves[0])
        other.append(halves[1])
        parents.append((a, b))
    total = torch.cat([torch.zeros((1, 2), dtype=torch.int64, device=DEVICE),
                       gpair[order].to(torch.int64).cumsum(dim=0)])

    def sums(segments):
        at = torch.tensor(segments, device=DEVICE)
        return (total[at[:, 1]] - total[at[:, 0]]).contiguous()

    # Rows of one node ascend, as a stable partition leaves them.
    for a, b in small + other:
        order[a:b] = order[a:b].sort().values
    ridx = order.to(torch.int32)
    ws = ops.Workspace()
    stride = int(n_bins.max())
    state.update(layout=lay, bins=bins, gpair=gpair, exps=(eg, eh), ridx=ridx, small=small,
                 other=other, small_sums=sums(small), other_sums=sums(other), ws=ws,
                 stride=stride, n_bins=torch.from_numpy(n_bins).to(DEVICE),
                 parents=ops.hist_build(ws, bins, lay, gpair, parents, stride, ridx=ridx),
                 param=ops.train_param(max_depth=8))


# ---------------------------------------------------------------------------
# One pass
# ---------------------------------------------------------------------------
def train(state, d, n_rounds):
    bst = dpgbdt.Booster(parameters(state["case"]), [d])
    for r in range(n_rounds):
        if state["case"]["objective"] == "caller":
            bst.boost(d, r, state["grad"], state["hess"])
        else:
            bst.update(d, r)
    return bst


def text(case, model):
    """The model's bytes in a buffer sized for the largest model of the case (spaces after it)."""
    raw = np.frombuffer(model.encode(), dtype=np.uint8)
    nodes = case["rounds"] * case["classes"] * 2 ** (case["depth"] + 1)
    out = np.full(4096 + 128 * nodes, ord(" "), dtype=np.uint8)
    out[:raw.size] = raw
    return out


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "fit":
        d = dpgbdt.DMatrix(state["x"], state["y"])
        return text(case, train(state, d, case["rounds"]).save_raw())
    if kind == "rounds":
        bst = train(state, state["matrix"], case["rounds"])
        if case["classes"] > 1:  # the next step of a search scores the training rows
            return bst.margins(case["rows"], case["classes"])
        return text(case, bst.save_raw())
    if kind == "predict":
        return state["model"].predict(state["x"])
    if kind == "histogram":
        return ops.hist_build(state["ws"], state["bins"], state["layout"], state["gpair"],
                              [(0, case["rows"])], state["stride"])
    if kind == "level":
        ws, bins, lay, ridx = state["ws"], state["bins"], state["layout"], state["ridx"]
        built = ops.hist_build(ws, bins, lay, state["gpair"], state["small"], state["stride"],
                               ridx=ridx)
        sibling = ops.hist_subtract(state["parents"], built)
        splits = [ops.evaluate_splits(ws, h, state["n_bins"], s, *state["exps"], state["param"])
                  for h, s in ((built, state["small_sums"]), (sibling, state["other_sums"]))]
        splits = torch.cat(splits)
        rows, left = ops.partition(ws, bins, lay, ridx, state["small"] + state["other"], splits)
        return [built, sibling, splits, rows, left]
    if kind == "cuts":
        ptr, cuts, mins, _ = ops.sketch_cuts(state["ws"], state["x"], case["max_bin"])
        return [ptr, cuts, mins, ops.bin_values(state["x"], state["layout"], ptr, cuts)]
    grad, hess = ops.objective_gradients(case["objective"], state["margin"], state["label"],
                                         case["classes"])
    return [grad, hess, *ops.quantise(state["ws"], grad, hess)]


# ---------------------------------------------------------------------------
# What a pass cannot do without
# ---------------------------------------------------------------------------
def work(case):
    kind = case["kind"]
    n, k = case["rows"], case["classes"] if "classes" in case else 1
    f = case.get("features", 1)
    if kind in ("fit", "rounds"):
        # A tree: every row's bins once at the root and half the rows on each level below
        # (two adds per element), the partition's row id and split byte per level, the
        # gradients and margins once.
        present = f * (1.0 - case["missing"])
        levels = 0.5 * (case["depth"] - 1) + 1.0
        trees = k * case["rounds"]
        size = trees * n * (levels * (present + 8.0) + 9.0 * case["depth"] + 16.0)
        if kind == "fit":  # the raw values in, the bins out
            size += 4.0 * n * f + n * present
        return {"bytes": size, "flops": 2.0 * trees * levels * n * present}
    if kind == "predict":
        # every value once, the outputs, the forest (16 B a node); a compare per level
        nodes = case["rounds"] * k * 2.0 ** case["depth"]
        return {"bytes": 4.0 * n * (f + k) + 16.0 * nodes,
                "flops": float(n) * case["rounds"] * k * case["depth"]}
    if kind == "histogram":
        return {"bytes": float(n) * (f + 8) + 16.0 * f * case["bins"], "flops": 2.0 * n * f}
    if kind == "level":
        # a quarter of the rows gathered, three histogram sets, the partition's rows
        cells = 16.0 * case["pairs"] * f * case["bins"]
        return {"bytes": 0.25 * n * (f + 12) + 3.0 * cells + 9.0 * n,
                "flops": 0.5 * n * f + 40.0 * case["pairs"] * f * case["bins"]}
    if kind == "cuts":
        return {"bytes": 5.0 * n * f, "flops": 8.0 * n * f}
    return {"bytes": n * (k * 20.0 + 4.0), "flops": 20.0 * n * k}


def tolerance(case):
    # Integer sums, fixed tie rules and IEEE float steps in a fixed order: bit for bit.
    return "exact"


# ---------------------------------------------------------------------------
# The same in 64 bits
# ---------------------------------------------------------------------------
def exact(case, seed):
    kind = case["kind"]
    if kind == "predict":
        return exact_predict(case, seed)
    if kind == "cuts":
        return exact_cuts(case, seed)
    if kind == "gradients":
        return exact_gradients(case, seed)
    # fit, rounds: a model follows from integer sums of gradients in fixed point (and is
    # text); histogram, level: integers and split records.  They are compared as they are.
    return None


def exact_predict(case, seed):
    x = matrix(case["rows"], case["features"], "normal", case["missing"], generator(seed))
    k = case["classes"]
    margin = torch.zeros((case["rows"], k), dtype=torch.float64, device=DEVICE)
    at = torch.arange(case["rows"], device=DEVICE)
    for t, (left, feature, cond, default) in enumerate(forest(case, seed)):
        left = torch.tensor(left, device=DEVICE)
        feature = torch.tensor(feature, device=DEVICE)
        cond = torch.tensor(cond, dtype=torch.float32, device=DEVICE)
        default = torch.tensor(default, device=DEVICE).bool()
        node = torch.zeros(case["rows"], dtype=torch.int64, device=DEVICE)
        for _ in range(case["depth"]):
            v = x[at, feature[node]]
            goes_left = torch.where(v.isnan(), default[node], v < cond[node])
            down = left[node] + (~goes_left).long()
            node = torch.where(left[node] >= 0, down, node)
        margin[:, t % k] += cond[node].double()
    return torch.sigmoid(margin) if k == 1 else torch.softmax(margin, dim=1)


def exact_cuts(case, seed):
    x = matrix(case["rows"], case["features"], case["data"], case["missing"], generator(seed))
    most, cuts, mins = case["max_bin"], [], []
    for f in range(case["features"]):
        v = x[:, f]
        v = (v[~v.isnan()] + 0.0).sort().values
        if v.numel() == 0:
            cuts.append(torch.tensor([1e-5], dtype=torch.float64, device=DEVICE))
            mins.append(0.0)
            continue
        u = torch.unique_consecutive(v)
        if u.numel() <= most:
            inner = u[1:]
        else:
            at = torch.arange(1, most, device=DEVICE) * v.numel() // most
            inner = torch.unique_consecutive(v[at])
            inner = inner[inner > u[0]]
        last = v[-1].double()
        cuts.append(torch.cat([inner.double(), (last + (last.abs() + 1e-5)).reshape(1)]))
        mins.append(float(v[0]))
    return [None, torch.cat(cuts), torch.tensor(mins, dtype=torch.float64), None]


def exact_gradients(case, seed):
    state = prepare(case, seed)
    m, y = state["margin"].double(), state["label"].double()
    if case["objective"] == 0:
        p = torch.sigmoid(m)
        return [p - y[:, None], (p * (1.0 - p)).clamp(min=1e-16), None, None, None]
    if case["objective"] == 2:
        return [m - y[:, None], torch.ones_like(m), None, None, None]
    p = torch.softmax(m, dim=1)
    hot = torch.nn.functional.one_hot(y.long(), case["classes"]).double()
    return [p - hot, (2.0 * p * (1.0 - p)).clamp(min=1e-16), None, None, None]
