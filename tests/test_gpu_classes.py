"""Multi-output gradients and their quantiser against the oracle where their row tiles and
class lanes change: class counts around the workgroup's width, rows around a tile."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,k", [(1, 2), (3, 256), (255, 3), (257, 10), (1000, 64), (999, 65),
                                 (70001, 7), (2100, 255), (2100, 256), (300, 257), (300, 300),
                                 # the quantisers and maxima passes change over
                                 (500000, 2), (499999, 2), (833333, 3), (833334, 3),
                                 (250000, 10), (249999, 10), (39063, 64), (62500, 128),
                                 (62499, 128), (124100, 65), (6000, 200)])
def test_softprob_and_quantiser_match_the_oracle(dp, oracle, ws, device, n, k):
    import torch
    from dpgbdt import ops

    rng = np.random.default_rng(n * 1000 + k)
    margin = (rng.normal(size=(n, k)) * 3).astype(np.float32)
    label = rng.integers(0, k, n).astype(np.float32)
    g, h = ops.objective_gradients(1, torch.as_tensor(margin, device=device),
                                   torch.as_tensor(label, device=device), k)
    og, oh = oracle.gradients(1, margin, label, k)
    np.testing.assert_array_equal(g.cpu().numpy().view(np.uint32), og.view(np.uint32))
    np.testing.assert_array_equal(h.cpu().numpy().view(np.uint32), oh.view(np.uint32))
    exps, gpair, sums = (t.cpu().numpy() for t in ops.quantise(ws, g, h))
    for c, (eg, eh, qg, qh) in enumerate(oracle.quantise(og, oh)):
        assert (exps[c, 0], exps[c, 1]) == (eg, eh)
        np.testing.assert_array_equal(gpair[c, :, 0], qg)
        np.testing.assert_array_equal(gpair[c, :, 1], qh)
        assert sums[c, 0] == qg.astype(np.int64).sum()
        assert sums[c, 1] == qh.astype(np.int64).sum()


@pytest.mark.parametrize("k", [2, 10, 257])
def test_rounds_add_leaf_values_in_the_gradients(dp, oracle, device, k):
    """Margins after rounds whose leaf values ride in the next round's gradient kernel equal
    the model's own predictions."""
    import torch

    rng = np.random.default_rng(k)
    n = 1500
    x = torch.as_tensor(rng.normal(size=(n, 5)).astype(np.float32), device=device)
    y = torch.as_tensor(rng.integers(0, k, n).astype(np.float32), device=device)
    d = dp.DMatrix(x, y)
    bst = dp.Booster({"objective": "multi:softprob", "num_class": k, "max_depth": 3}, [d])
    for r in range(3):
        bst.update(d, r)
    np.testing.assert_array_equal(bst.margins(n, k).view(np.uint32),
                                  bst.predict(x, margin=True).cpu().numpy().view(np.uint32))


@pytest.mark.parametrize("n,k", [(250000, 10), (3000, 10), (3000, 3), (400, 130)])
def test_row_samples_of_several_outputs(dp, oracle, device, n, k):
    """Sampled rows' maxima and pairs, a draw per output, in each quantiser."""
    import torch
    from test_gpu_booster import _compare, _train_both

    rng = np.random.default_rng(n + k)
    x = torch.as_tensor(rng.integers(0, 20, (n, 3)).astype(np.float32), device=device)
    y = torch.as_tensor(rng.integers(0, k, n).astype(np.float32), device=device)
    bst, _, o_trees, o_margin, pos, _ = _train_both(
        dp, oracle, device, 0, n, 3, 1, k, {"max_depth": 2, "eta": 0.3}, 2, 0,
        values_labels=(x, y), sample={"seed": 5, "subsample": 0.7})
    _compare(bst, o_trees, o_margin, pos, n, k)
