"""Quantile cuts and bins against the oracle at the sizes and value patterns where the bucket
passes change course: the row counts around the in-LDS sort and the sample, features
whose distinct values are few, rare, repeated or adjacent, and missing values."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _columns(n, rng):
    """Named value patterns, each float32 [n]."""
    normal = rng.normal(size=n)
    rare = rng.random(n) < 0.002
    atom = np.where(rng.random(n) < 0.6, 1.5, normal)
    missing = np.where(rng.random(n) < 0.999, np.nan, normal)
    few = np.where(rng.random(n) < 0.97, np.nan, rng.integers(0, 9, n))
    zero = np.where(rng.random(n) < 0.5, 0.0, -0.0)
    edge = np.float32(1.0) + np.float32(2.0 ** -23) * rng.integers(0, 300, n).astype(np.float32)
    wide = np.exp(30.0 * normal)
    inf = np.where(rng.random(n) < 0.01, np.inf, np.where(rng.random(n) < 0.01, -np.inf, normal))
    columns = {
        "normal": normal, "constant": np.full(n, -3.25), "none": np.full(n, np.nan),
        "int16": rng.integers(0, 16, n), "int256": rng.integers(0, 256, n),
        "int257": rng.integers(0, 257, n),
        # few common values and a few hundred rare ones: unseen or seen once in the sample
        "rare200": np.where(rare, rng.integers(0, 200, n), 1000.0),
        "rare400": np.where(rare, rng.integers(0, 400, n), rng.integers(1000, 1003, n)),
        "atom": atom, "missing": missing, "few": few, "zero": zero, "adjacent": edge,
        "wide": wide, "inf": inf, "denormal": normal * 1e-41, "sorted": np.arange(n) - n // 2,
    }
    return {k: np.asarray(v, dtype=np.float32) for k, v in columns.items()}


@pytest.mark.parametrize("n,max_bin", [(1, 256), (2, 2), (257, 256), (8192, 255), (8193, 256),
                                       (16384, 64), (16385, 256), (16385, 2), (60001, 255),
                                       (300007, 256), (300007, 17)])
def test_cuts_match_the_oracle(dp, oracle, ws, device, n, max_bin):
    import torch
    from dpgbdt import ops

    columns = _columns(n, np.random.default_rng(n + max_bin))
    x = np.ascontiguousarray(np.stack(list(columns.values()), axis=1))
    for width in (x.shape[1], 1):  # 17 features: a ragged second tile; one feature alone
        part = np.ascontiguousarray(x[:, :width])
        ptr, cuts, mins, missing = ops.sketch_cuts(ws, torch.as_tensor(part, device=device),
                                                   max_bin)
        o_ptr, o_cuts, o_mins = oracle.compute_cuts(part, max_bin)
        for f, name in enumerate(list(columns)[:width]):
            got, want = cuts[ptr[f]:ptr[f + 1]], o_cuts[o_ptr[f]:o_ptr[f + 1]]
            np.testing.assert_array_equal(got.view(np.uint32), want.view(np.uint32), err_msg=name)
        np.testing.assert_array_equal(mins.view(np.uint32), o_mins.view(np.uint32))
        if max_bin <= 255:  # byte 255 marks a missing value
            lay = ops.layout(n, width, 0, 255)
            bins = ops.bin_values(torch.as_tensor(part, device=device), lay, ptr, cuts)
            np.testing.assert_array_equal(ops.from_tiles(bins.cpu().numpy(), lay),
                                          oracle.bin_matrix(part, o_ptr, o_cuts, 255))
        assert missing == bool(np.isnan(part).any())


@pytest.mark.parametrize("rows,features", [(1, 1), (3, 5), (256, 16), (256, 17), (241, 1003),
                                           (250, 4000), (255, 4113)])
@pytest.mark.parametrize("missing", [-999.0, np.inf, -np.inf])
def test_matrices_are_copied_whole(dp, device, rows, features, missing):
    """With at most 256 rows the cuts are the distinct values above the smallest: the copy is
    checked value by value, from aligned rows (128-bit loads) and others; infinities other than
    the value that stands for missing are refused wherever they stand."""
    import torch

    missing = np.float32(missing)
    refused = -np.inf if missing > 0 else np.inf
    rng = np.random.default_rng(rows * features)
    x = rng.normal(size=(rows, features)).astype(np.float32)
    x[rng.random(x.shape) < 0.1] = missing
    want = []
    for f in range(features):
        u = np.unique(x[:, f][x[:, f] != missing])
        top = u[-1] if u.size else np.float32(0.0)
        want.append(np.append(u[1:], top + (np.abs(top) + np.float32(1e-5))))
    want = np.concatenate(want).astype(np.float32)
    flat = torch.zeros(rows * features + 1, device=device)
    views = [torch.empty((rows, features), device=device), flat[1:].view(rows, features)]
    for v in views:
        v.copy_(torch.as_tensor(x))
        d = dp.DMatrix(v, torch.arange(rows, device=device).float(), missing=float(missing))
        dp.Booster({"objective": "reg:squarederror", "tree_method": "hist", "device": "cuda:0",
                    "max_depth": 1, "max_bin": 256}, [d]).update(d, 0)
        np.testing.assert_array_equal(d.cuts(256)[1], want)
        for at in {0, rows * features // 2, rows * features - 1}:
            v[at // features, at % features] = refused
            with pytest.raises(Exception, match="inf"):
                dp.DMatrix(v, missing=float(missing))
            v.copy_(torch.as_tensor(x))


@pytest.mark.parametrize("rows,features", [(64, (1 << 20) + 17), (40, (1 << 25) + 5)])
def test_bins_of_very_wide_matrices(dp, device, rows, features):
    """More features than a lane's 32-bit offset reaches, and than the widest matrices of
    practice; one cut at 0 and the last one."""
    import torch
    from dpgbdt import ops

    x = torch.randn((rows, features), device=device,
                    generator=torch.Generator(device).manual_seed(features))
    x[1, features - 1] = float("nan")
    lay = ops.layout(rows, features, 0, 255)
    ptr = np.arange(features + 1, dtype=np.int32) * 2
    bins = ops.bin_values(x, lay, ptr, np.tile(np.float32([0.0, 9.0]), features))
    tiles = bins.view(lay.n_tiles, rows, 16)
    want = torch.where(torch.isnan(x), 255, (x >= 0).to(torch.uint8)).to(torch.uint8)
    pad = torch.zeros((rows, lay.n_tiles * 16 - features), dtype=torch.uint8, device=device)
    want = torch.cat([want, pad], dim=1).view(rows, lay.n_tiles, 16)
    assert torch.equal(tiles, want.transpose(0, 1))


@pytest.mark.parametrize("n", [1, 255, 257, 3000, 530001])
@pytest.mark.parametrize("features", [1, 5, 8, 9])
def test_bins_of_narrow_matrices(dp, oracle, ws, device, n, features):
    """A thread per row up to 8 features, more threads than rows and fewer (2,048 workgroups)."""
    import torch
    from dpgbdt import ops

    rng = np.random.default_rng(n + features)
    x = rng.normal(size=(n, features)).astype(np.float32)
    x[:, -1] = rng.integers(-2, 2, n)
    x[rng.random(x.shape) < 0.05] = np.nan
    x[rng.random(x.shape) < 0.05] = -0.0
    for max_bin in (2, 16, 17, 255):
        ptr, cuts, _ = oracle.compute_cuts(x, max_bin)
        y = x.copy()
        y[rng.random(x.shape) < 0.05] *= 100.0  # above the last cut
        lay = ops.layout(n, features, 0, 255)
        bins = ops.bin_values(torch.as_tensor(y, device=device), lay, ptr, cuts)
        np.testing.assert_array_equal(ops.from_tiles(bins.cpu().numpy(), lay),
                                      oracle.bin_matrix(y, ptr, cuts, 255))
        tile = bins.view(-1, n, 16)[-1].cpu().numpy()
        assert not tile[:, (features - 1) % 16 + 1:].any()  # the tile's padding


@pytest.mark.parametrize("features", [1, 8, 9])
@pytest.mark.parametrize("max_bin", [200, 256])
def test_training_on_narrow_matrices_with_missing_values(dp, oracle, device, features, max_bin):
    """The column copies made with the bins: bytes, and 16-bit symbols for 256 bins."""
    import torch
    from test_gpu_booster import _compare, _train_both

    rng = np.random.default_rng(features + max_bin)
    n = 5000
    x = rng.normal(size=(n, features)).astype(np.float32)
    x[rng.random(x.shape) < 0.1] = np.nan
    y = (rng.random(n) < 0.5).astype(np.float32)
    bst, _, o_trees, o_margin, pos, _ = _train_both(
        dp, oracle, device, 0, n, features, 0, 1, {"max_depth": 5, "eta": 0.3}, 2, 0,
        max_bin=max_bin, values_labels=(torch.as_tensor(x, device=device),
                                        torch.as_tensor(y, device=device)))
    _compare(bst, o_trees, o_margin, pos, n, 1)


def test_cuts_of_more_features_than_a_block(dp, ws, device):
    """65,536 features make a block: each feature's cuts are those it has among 48 (one block)."""
    import torch
    from dpgbdt import ops

    n, base, features, max_bin = 16500, 48, (1 << 16) + 40, 16
    rng = np.random.default_rng(1)
    x = rng.normal(size=(n, base)).astype(np.float32)
    x[:, 1] = rng.integers(0, 9, n)
    x[:, 2] = np.nan
    x[rng.random(x.shape) < 0.05] = np.nan
    part = torch.as_tensor(x, device=device)
    ptr, cuts, mins, missing = ops.sketch_cuts(ws, part, max_bin)
    wide = part.repeat(1, features // base + 1)[:, :features].contiguous()
    w_ptr, w_cuts, w_mins, w_missing = ops.sketch_cuts(ws, wide, max_bin)
    of = np.arange(features) % base
    np.testing.assert_array_equal(np.diff(w_ptr), np.diff(ptr)[of])
    np.testing.assert_array_equal(w_mins.view(np.uint32), mins.view(np.uint32)[of])
    want = np.concatenate([cuts[ptr[f]:ptr[f + 1]] for f in of])
    np.testing.assert_array_equal(w_cuts.view(np.uint32), want.view(np.uint32))
    assert missing and w_missing


@pytest.mark.parametrize("rows,features", [(200, 7), (4000, 300), (70000, 20)])
def test_matrices_with_gaps_between_rows(dp, device, rows, features):
    """A matrix read from every row of a wider array trains what its copy trains."""
    import ctypes
    import json
    import torch

    rng = np.random.default_rng(rows)
    wide = torch.as_tensor(rng.normal(size=(rows, features + 5)).astype(np.float32), device=device)
    y = (wide[:, 0] > 0).float()
    view = wide[:, :features]
    d = dp.DMatrix.__new__(dp.DMatrix)
    d.handle = ctypes.c_void_p()
    a = json.dumps({"data": [view.data_ptr(), True], "shape": [rows, features], "version": 3,
                    "strides": [4 * (features + 5), 4], "typestr": "<f4", "stream": 1})
    dp.check(dp.load().XGDMatrixCreateFromCudaArrayInterface(a.encode(), b'{"missing": NaN}',
                                                             ctypes.byref(d.handle)))
    dp.check(dp.load().XGDMatrixSetInfoFromInterface(d.handle, b"label",
                                                     dp.array_interface(y).encode()))
    models = []
    for m in (d, dp.DMatrix(view.contiguous(), y)):
        bst = dp.Booster({"objective": "binary:logistic", "max_depth": 4, "dp_autotune": 0}, [m])
        bst.update(m, 0)
        bst.update(m, 1)
        models.append(bst.save_raw())
    assert models[0] == models[1]
