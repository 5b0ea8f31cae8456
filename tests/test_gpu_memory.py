"""Device memory that boosters hold and leave behind."""
import gc

import numpy as np
import pytest

from hipmem import free_device_bytes
from test_gpu_parity import make_data

pytestmark = pytest.mark.gpu
MB = 1 << 20


@pytest.fixture(scope="module")
def arb():
    import arboretum_amd
    if arboretum_amd.device_count() < 1:
        pytest.fail("no HIP device")
    return arboretum_amd


def _config(depth, bins=64, **tree):
    return {"objective": 1, "method": 1, "internals": {"hist_size": bins, "double_precision": True},
            "tree": dict({"max_depth": depth, "eta": 0.3, "lambda": 1.0}, **tree)}


def test_release_memory(arb):
    X, y = make_data(600000, 28, 1, seed=4)
    def use():
        data = arb.DMatrix(X, y=y)
        g = arb.train(_config(5), data, 2)
        return g.predict(data)
    first = use()                        # (code objects and the runtime's own memory)
    gc.collect()
    arb.release_memory()
    before = free_device_bytes()
    data = arb.DMatrix(X, y=y)
    g = arb.train(_config(5), data, 2)
    assert free_device_bytes() < before - 100 * MB
    arb.release_memory()                 # takes nothing that is in use
    assert np.array_equal(g.predict(data), first)
    del g, data
    gc.collect()
    assert free_device_bytes() < before - 100 * MB
    arb.release_memory()
    assert free_device_bytes() > before - 16 * MB
    assert np.array_equal(use(), first)


def _softmax_bytes(arb, F, depth, column_share):
    """Device memory of a soft-max booster of four classes over F features of 256 bins."""
    n, K = 3000, 4
    rng = np.random.default_rng(F)
    X = rng.integers(0, 256, size=(n, F), dtype=np.uint8)
    labels = ((X[:, 0] > 100).astype(np.uint8) + 2 * (X[:, F - 1] > 60)).astype(np.uint8)
    cfg = _config(depth, bins=256, labels_count=K, colsample_bytree=column_share)
    cfg["objective"] = 4
    data = arb.DMatrix(X, labels=labels, quantized=True)
    data.quantize(256)
    arb.train(dict(cfg, tree=dict(cfg["tree"], max_depth=1)), data, 1).synchronize()   # (records of the rows)
    gc.collect()
    arb.release_memory()
    before = free_device_bytes()
    g = arb.Garden(cfg, data)
    g.labels_count = K
    g.grow_tree()
    g.synchronize()
    return before - free_device_bytes()


# lanes beside the first take 8 GB at most together: two more of 3 GB, one more of 6 GB, none of 10 GB
@pytest.mark.parametrize("F,others", [(200, 2), (400, 1), (640, 0)])
def test_lanes_of_a_wide_deep_softmax_are_bounded(arb, F, others):
    one = _softmax_bytes(arb, F, 10, 1.0 - 0.5 / F)   # sampled columns: one lane
    used = _softmax_bytes(arb, F, 10, 1.0)
    assert used - one < 8 * 1024 * MB
    assert abs(used - (1 + others) * one) < 0.1 * one, (used, one)
