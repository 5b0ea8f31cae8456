"""The two forms of the fused pass on either side of the line between them (items of one chunk of rows per wave, up to
about 520,000 rows), for one and several LDS histograms, packed and plain gradients, ids of 256; and the lists of the
exact method with more work items than a workgroup adds up."""
import numpy as np
import pytest

from test_gpu_parity import make_data

pytestmark = pytest.mark.gpu


def _same(arb, oracle, X, y, cfg, trees):
    ob = oracle.Booster(X, y=y, config=cfg)
    ob.grow(trees)
    g = arb.train(cfg, arb.DMatrix(X, y=y), trees)
    for t in range(trees):
        to, tg = ob.tree(t), g.tree(t)
        for key in ("fid", "quantized", "gain", "weights"):
            assert np.array_equal(to[key], tg[key], equal_nan=True), (key, t)
    assert np.array_equal(ob.leaf(), g.leaves())
    assert np.array_equal(ob.yhat(), g.train_yhat())


@pytest.mark.parametrize("n", [1, 65, 2047, 260097, 520193, 600003])
@pytest.mark.parametrize("F,objective,bins,nan_frac", [(3, 1, 64, 0.0), (13, 0, 256, 0.1), (29, 1, 256, 0.1), (28, 0, 255, 0.0),
                                                       (36, 1, 255, 0.0)])
def test_either_side_of_the_line(oracle, n, F, objective, bins, nan_frac):
    import arboretum_amd as arb
    X, y = make_data(n, F, objective, seed=n + F, nan_frac=nan_frac)
    cfg = {"objective": objective, "method": 1, "internals": {"hist_size": bins, "double_precision": True},
           "tree": {"max_depth": 4, "eta": 0.3, "lambda": 1.0, "min_child_weight": 1.0}}
    _same(arb, oracle, X, y, cfg, 2)


@pytest.mark.parametrize("n", [1, 66, 5000, 1_048_577, 1_060_003])
@pytest.mark.parametrize("F,bins,objective,nan_frac", [(5, 700, 1, 0.1), (19, 3000, 0, 0.0), (51, 255, 1, 0.0), (49, 256, 0, 0.1)])
def test_stand_alone_partitions(oracle, n, F, bins, objective, nan_frac):
    # 16-bit ids (one and two groups of words) and rows in place, on either side of a chunk of rows per wave
    import arboretum_amd as arb
    X, y = make_data(n, F, objective, seed=n + F, nan_frac=nan_frac)
    cfg = {"objective": objective, "method": 1, "internals": {"hist_size": bins, "double_precision": True},
           "tree": {"max_depth": 4, "eta": 0.3, "lambda": 1.0, "min_child_weight": 1.0}}
    _same(arb, oracle, X, y, cfg, 2)


@pytest.mark.parametrize("n,objective,extra", [(1_100_001, 1, {}), (1_100_001, 0, {"lambda": 0.0, "min_child_weight": 30.0}),
                                               (20_000, 1, {"lambda": 0.0, "min_child_weight": 0.0}),
                                               (20_000, 1, {"alpha": 0.7}), (20_000, 0, {"max_leaf_weight": 0.05})])
def test_exact_lists_of_many_items_and_limits_on_leaves(oracle, n, objective, extra):
    import arboretum_amd as arb
    X, y = make_data(n, 4, objective, seed=n)
    tree = {"max_depth": 4, "eta": 0.3, "lambda": 1.0, "min_child_weight": 1.0}
    tree.update(extra)
    cfg = {"objective": objective, "method": 0, "internals": {"double_precision": n > 100_000, "exact_sort": 1}, "tree": tree}
    _same(arb, oracle, X, y, cfg, 2)
