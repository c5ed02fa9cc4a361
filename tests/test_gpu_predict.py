"""Prediction of random forests against a plain numpy walk, bit for bit, where the kernels
change course: a row per thread or a tree per thread, nodes and rows in LDS or not, packed
or general nodes, large trees, several outputs, missing values, infinities, row strides."""
import json

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _forest(rng, trees, depth, features, full):
    """Node arrays (left, feature, cond, default) per tree; `full` of the inner nodes split."""
    out = []
    for _ in range(trees):
        left, level, i = [-1], [0], 0
        while i < len(left):
            if level[i] < depth and rng.random() < full:
                left[i] = len(left)
                left += [-1, -1]
                level += [level[i] + 1] * 2
            i += 1
        n = len(left)
        leaf = np.array(left) < 0
        cond = np.where(leaf, rng.normal(size=n) * 0.1, rng.normal(size=n)).astype(np.float32)
        cond[~leaf & (rng.random(n) < 0.1)] = 0.0  # zeros and the smallest numbers meet below
        out.append((np.array(left, dtype=np.int64), np.where(leaf, 0, rng.integers(0, features, n)),
                    cond, np.where(leaf, 0, rng.integers(0, 2, n))))
    return out


def _model(forest, features, classes, objective=None):
    trees = [{"left_children": left.tolist(),
              "right_children": np.where(left < 0, -1, left + 1).tolist(),
              "split_indices": feature.tolist(),
              "split_conditions": [float(c) for c in cond], "default_left": default.tolist()}
             for left, feature, cond, default in forest]
    objective = objective or ("reg:squarederror" if classes == 1 else "multi:softprob")
    return json.dumps({"learner": {
        "gradient_booster": {"model": {
            "iteration_indptr": list(range(0, len(trees) + 1, classes)),
            "tree_info": [t % classes for t in range(len(trees))], "trees": trees}},
        "learner_model_param": {"base_score": json.dumps([0.25] * classes),
                                "num_class": str(classes if classes > 1 else 0),
                                "num_feature": str(features)},
        "objective": {"name": objective}}})


def _margins(forest, x, classes):
    m = np.full((x.shape[0], classes), 0.25, dtype=np.float32)
    rows = np.arange(x.shape[0])
    for t, (left, feature, cond, default) in enumerate(forest):
        node = np.zeros(x.shape[0], dtype=np.int64)
        while (left[node] >= 0).any():
            v = x[rows, feature[node]]
            with np.errstate(invalid="ignore"):
                goes_left = np.where(np.isnan(v), default[node] == 1, v < cond[node])
            node = np.where(left[node] >= 0, left[node] + np.where(goes_left, 0, 1), node)
        m[:, t % classes] = m[:, t % classes] + cond[node]
    return m


@pytest.mark.parametrize("rows,features,trees,depth,full,classes", [
    (1, 1, 1, 0, 1.0, 1),            # one leaf
    (64, 28, 100, 8, 0.9, 1),        # a tree per thread
    (33, 5, 300, 3, 1.0, 3),         # many small trees, several outputs
    (5000, 28, 40, 8, 1.0, 1),       # between the two
    (70001, 30, 9, 6, 0.95, 1),      # a row per thread, 256 rows a workgroup
    (140000, 60, 6, 5, 1.0, 2),      # 512 rows
    (270001, 9, 37, 7, 0.97, 1),     # 1,024 rows, several batches
    (70000, 20, 5, 13, 1.0, 1),      # trees beyond a batch (16,383 nodes)
    (9000, 784, 120, 6, 1.0, 10),    # wide rows, nodes and rows in LDS
    (700, 9, 3, 4, 1.0, 11),         # outputs spread over a row's lanes, several passes
    (300, 12, 2, 3, 1.0, 65),        # more outputs than are spread
    (2000, 5000, 100, 7, 1.0, 1),    # rows too wide for many in LDS
    (2000, 5000, 12, 7, 1.0, 1),     # rows not worth staging
    (20000, 9, 40, 5, 1.0, 1),       # more threads to stage the rows than to walk them
    (40, 17000, 3, 4, 1.0, 1),       # features beyond the packed nodes
    (300, 7, 2, 17, 0.995, 1),       # trees beyond the packed nodes
    (50, 60000, 1, 2, 1.0, 1),       # small forests, general nodes
    (9000, 17000, 2, 3, 1.0, 1),
    (8192, 28, 11, 3, 1.0, 1),       # small forests: quads, a pair and a single tree
    (8193, 28, 7, 6, 0.9, 1),
    (8192, 28, 12, 3, 1.0, 1),       # and the first that is not one
    (66000, 120, 2, 6, 1.0, 3),      # against rows in LDS
    (66000, 20, 4, 4, 1.0, 1),
    (66000, 20, 5, 4, 1.0, 1),
    (100000, 130, 3, 6, 1.0, 1),     # a pair one by one
    (99999, 130, 16, 4, 1.0, 1),     # the longest chain that is direct
    (5000000, 3, 1, 3, 1.0, 1),      # more rows than the grid has threads
])
def test_margins_match_a_numpy_walk(dp, device, rows, features, trees, depth, full, classes):
    import torch

    rng = np.random.default_rng(rows + features)
    forest = _forest(rng, trees * classes, depth, features, full)
    bst = dp.Booster.from_buffer(_model(forest, features, classes))
    x = rng.normal(size=(rows, features)).astype(np.float32)
    tiny = rng.random(x.shape) < 0.02
    x[tiny] = rng.choice(np.float32([0.0, -0.0, 1e-45, -1e-45, 1e-39]), tiny.sum())
    for missing in (False, True):
        if missing:
            x[rng.random(x.shape) < 0.1] = np.nan
            x[rng.random(x.shape) < 0.01] = np.inf
            x[rng.random(x.shape) < 0.01] = -np.inf
        got = bst.predict(torch.as_tensor(x, device=device), margin=True).cpu().numpy()
        np.testing.assert_array_equal(got.view(np.uint32),
                                      _margins(forest, x, classes).view(np.uint32))
    # a sentinel for missing values
    y = np.where(np.isnan(x), np.float32(-999.0), x)
    got = bst.predict(torch.as_tensor(y, device=device), margin=True, missing=-999.0)
    np.testing.assert_array_equal(got.cpu().numpy().view(np.uint32),
                                  _margins(forest, x, classes).view(np.uint32))


@pytest.mark.parametrize("rows,classes,rounds,depth", [
    (1, 3, 3, 4), (2049, 10, 3, 4), (77, 64, 3, 4), (77, 65, 3, 4),
    (300, 3, 1, 2),      # a small forest
    (70001, 3, 12, 4)])  # a row per thread in LDS
def test_outputs_of_the_margins(dp, device, rows, classes, rounds, depth):
    """Probabilities and class ids follow from the margins: each operation of the softmax rounds
    once (2^-24), a sum of K positive terms at most K times, the exponential within 2 ulp."""
    import torch

    rng = np.random.default_rng(rows * classes)
    forest = _forest(rng, rounds * classes, depth, 6, 0.9)
    x = torch.as_tensor(rng.normal(size=(rows, 6)).astype(np.float32), device=device)
    margins = _margins(forest, x.cpu().numpy(), classes)
    p = np.exp(margins.astype(np.float64) - margins.max(axis=1, keepdims=True))
    p /= p.sum(axis=1, keepdims=True)
    bst = dp.Booster.from_buffer(_model(forest, 6, classes))
    np.testing.assert_allclose(bst.predict(x).cpu().numpy().reshape(rows, classes), p,
                               rtol=(classes + 8) * 2.0 ** -23)
    bst = dp.Booster.from_buffer(_model(forest, 6, classes, "multi:softmax"))
    np.testing.assert_array_equal(bst.predict(x).cpu().numpy().reshape(rows),
                                  margins.argmax(axis=1).astype(np.float32))


def _pruned(forest, rng):
    """A fifth of the inner nodes become leaves: the nodes below them stay, unreached."""
    out = []
    for left, feature, cond, default in forest:
        cut = (left >= 0) & (rng.random(len(left)) < 0.2)
        out.append((np.where(cut, -1, left), np.where(cut, 0, feature), cond,
                    np.where(cut, 0, default)))
    return out


def _shared(forest):
    """In each tree two inner nodes name one pair, missing values going opposite ways."""
    out = []
    for left, feature, cond, default in forest:
        left, default = left.copy(), default.copy()
        a, b = np.flatnonzero(left >= 0)[1:3]
        left[a] = left[b]
        default[a], default[b] = 0, 1
        out.append((left, feature, cond, default))
    return out


@pytest.mark.parametrize("rows,trees", [(300, 30), (70001, 30), (1000, 1)])
@pytest.mark.parametrize("shape", ["pruned", "shared"])
def test_nodes_without_or_with_two_parents(dp, device, rows, trees, shape):
    """Pruned models keep nodes that no parent names; nothing forbids two parents of a pair."""
    import torch

    rng = np.random.default_rng(rows + trees)
    forest = _forest(rng, trees, 5, 9, 1.0)
    forest = _pruned(forest, rng) if shape == "pruned" else _shared(forest)
    # a root leaf before two unreached leaves, and before an unreached inner node
    for tail in ([-1, -1, -1], [-1, 2, -1, -1]) if shape == "pruned" else ():
        n = len(tail)
        forest.append((np.array(tail), np.zeros(n, dtype=np.int64),
                       np.arange(n, dtype=np.float32) + 10, np.zeros(n, dtype=np.int64)))
    bst = dp.Booster.from_buffer(_model(forest, 9, 1))
    x = rng.normal(size=(rows, 9)).astype(np.float32)
    x[rng.random(x.shape) < 0.2] = np.nan
    got = bst.predict(torch.as_tensor(x, device=device), margin=True).cpu().numpy()
    np.testing.assert_array_equal(got.view(np.uint32), _margins(forest, x, 1).view(np.uint32))


@pytest.mark.parametrize("rows,trees", [(500, 3), (500, 60), (70001, 60)])
def test_logistic_outputs_of_the_margins(dp, device, rows, trees):
    """1 / (1 + exp(-margin)) in each kernel: three roundings and an exponential within 2 ulp."""
    import torch

    rng = np.random.default_rng(rows + trees)
    forest = _forest(rng, trees, 4, 6, 0.9)
    x = torch.as_tensor(rng.normal(size=(rows, 6)).astype(np.float32), device=device)
    bst = dp.Booster.from_buffer(_model(forest, 6, 1, "binary:logistic"))
    m = bst.predict(x, margin=True).cpu().numpy().astype(np.float64).reshape(rows)
    np.testing.assert_allclose(bst.predict(x).cpu().numpy().reshape(rows), 1 / (1 + np.exp(-m)),
                               rtol=8 * 2.0 ** -24)


SPECIALS = np.float32([np.inf, -np.inf, 3.4028235e38, -3.4028235e38, 1e-45, -1e-45, 0.0, -0.0,
                       1.1754944e-38, -1.1754944e-38, 1.0])


@pytest.mark.parametrize("rows,trees", [(300, 2), (300, 40), (70001, 40)])
@pytest.mark.parametrize("general", ["none", "infinity", "nan"])
def test_thresholds_at_the_ends_of_the_floats(dp, device, rows, trees, general):
    """Packed, missing-right nodes compare -x with the float above -t.  A threshold of -inf with
    missing values right, or of NaN, takes the general nodes."""
    import torch

    rng = np.random.default_rng(rows + trees)
    forest = _forest(rng, trees, 5, 7, 1.0)
    for left, _, cond, default in forest:
        inner = left >= 0
        cond[inner] = rng.choice(SPECIALS, inner.sum())
        if general == "nan":
            cond[inner & (rng.random(len(left)) < 0.2)] = np.nan
        elif general == "none":
            default[inner & (cond == -np.inf)] = 1
    bst = dp.Booster.from_buffer(_model(forest, 7, 1))
    x = rng.choice(np.append(SPECIALS, np.float32([np.nan, 2.0, -2.0])), (rows, 7))
    x = x.astype(np.float32)
    got = bst.predict(torch.as_tensor(x, device=device), margin=True).cpu().numpy()
    np.testing.assert_array_equal(got.view(np.uint32), _margins(forest, x, 1).view(np.uint32))


@pytest.mark.parametrize("splits,rows", [(2047, 40), (32767, 40)])
def test_a_tree_as_deep_as_packed_nodes_count(dp, device, splits, rows):
    import torch

    n = 2 * splits + 1
    inner = np.arange(n) % 2 == 0
    inner[-1] = False
    left = np.where(inner, np.arange(n) + 1, -1)
    cond = np.where(inner, np.arange(n) / n, np.arange(n) % 100).astype(np.float32)
    forest = [(left, np.where(inner, np.arange(n) % 3, 0), cond, (np.arange(n) // 2) % 2)]
    rng = np.random.default_rng(splits)
    x = np.repeat(rng.random((rows, 1)), 3, axis=1).astype(np.float32)
    x[0], x[1, 1] = 2.0, np.nan
    got = dp.Booster.from_buffer(_model(forest, 3, 1)).predict(
        torch.as_tensor(x, device=device), margin=True).cpu().numpy()
    np.testing.assert_array_equal(got.view(np.uint32), _margins(forest, x, 1).view(np.uint32))


@pytest.mark.parametrize("rows,features,trees,depth", [
    (300, 9, 2, 3),        # a small forest
    (5000, 28, 40, 6),     # rows in LDS, several trees at a time
    (2000, 5000, 12, 7),   # not worth that
    (70001, 20, 40, 6)])   # a row per thread in LDS
def test_rows_with_gaps_between_them(dp, device, rows, features, trees, depth):
    import ctypes
    import torch

    rng = np.random.default_rng(rows)
    forest = _forest(rng, trees, depth, features, 0.9)
    bst = dp.Booster.from_buffer(_model(forest, features, 1))
    wide = rng.normal(size=(rows, features + 3)).astype(np.float32)
    dev = torch.as_tensor(wide, device=device)
    shape, dim = ctypes.POINTER(ctypes.c_uint64)(), ctypes.c_uint64()
    out = ctypes.POINTER(ctypes.c_float)()
    a = json.dumps({"data": [dev.data_ptr(), True], "shape": [rows, features], "version": 3,
                    "strides": [4 * (features + 3), 4], "typestr": "<f4", "stream": 1})
    cfg = json.dumps({"type": 1, "training": False, "iteration_begin": 0, "iteration_end": 0,
                      "strict_shape": True, "cache_id": 0, "missing": float("nan")})
    dp.check(dp.load().XGBoosterPredictFromCudaArray(
        bst.handle, a.encode(), cfg.encode(), None, ctypes.byref(shape), ctypes.byref(dim),
        ctypes.byref(out)))
    got = torch.empty((rows, 1), device=device)
    dp._hip_memcpy()(ctypes.c_void_p(got.data_ptr()),
                     ctypes.c_void_p(ctypes.addressof(out.contents)), rows * 4)
    np.testing.assert_array_equal(got.cpu().numpy().view(np.uint32),
                                  _margins(forest, wide[:, :features], 1).view(np.uint32))
