"""Partitions of more work items than two rounds of the chip hold select no splits themselves: trees and leaves of
a matrix just above that line (its levels of few nodes are otherwise selected by the partition) against the oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("objective", [0, 1])
def test_partition_without_selection(oracle, objective):
    import arboretum_amd as arb
    n, F = 1024 * 16384 + 50_001, 2     # 256 compute units, two workgroups each, 16384 rows an item
    rng = np.random.default_rng(objective)
    X = rng.integers(0, 400, size=(n, F)).astype(np.float32)   # 400 values: bins of 16 bits
    s = (X[:, 0] > 130).astype(np.float32) + (X[:, 1] % 7 > 3) + 0.25 * rng.standard_normal(n, dtype=np.float32)
    y = s if objective == 0 else (s > 1).astype(np.float32)
    cfg = {"objective": objective, "method": 1, "internals": {"hist_size": 500, "double_precision": True},
           "tree": {"max_depth": 3, "eta": 0.3, "lambda": 1.0}}
    data = arb.DMatrix(X, y=y)
    ob = oracle.Booster(X, y=y, config=cfg)
    g = arb.Garden(cfg, data)
    for t in range(2):
        g.grow_tree()
        ob.grow(1)
        to, tg = ob.tree(t), g.tree(t)
        for key in ("fid", "quantized", "gain", "weights"):
            assert np.array_equal(to[key], tg[key]), (key, t)
        assert np.array_equal(ob.leaf(), g.leaves())
    assert np.array_equal(ob.yhat(), g.train_yhat())
