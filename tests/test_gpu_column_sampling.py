"""Column masks are made and copied for several trees at a time: trees beyond the first batches
against the checker."""
import numpy as np
import pytest

from test_gpu_parity import make_data

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("F,depth,trees,method", [(9, 3, 30, 1), (9, 2, 30, 0), (40, 4, 27, 1), (1024, 5, 12, 1)])
def test_masks_of_many_trees(oracle, F, depth, trees, method):
    import arboretum_amd as arb
    X, y = make_data(700, F, 1, seed=F)
    cfg = {"objective": 1, "method": method, "internals": {"hist_size": 16, "double_precision": True, "seed": 3, "exact_sort": 1},
           "tree": {"max_depth": depth, "eta": 0.2, "lambda": 1.0, "colsample_bytree": 0.7, "colsample_bylevel": 0.6}}
    ob = oracle.Booster(X, y=y, config=cfg)
    ob.grow(trees)
    g = arb.train(cfg, arb.DMatrix(X, y=y), trees)
    for t in range(trees):
        assert np.array_equal(ob.tree(t)["fid"], g.tree(t)["fid"]), t
        assert np.array_equal(ob.tree(t)["quantized"], g.tree(t)["quantized"]), t
    assert np.array_equal(ob.yhat(), g.train_yhat())
