"""Device memory that boosters hold and leave behind."""
import ctypes
import gc

import numpy as np
import pytest

from hipmem import free_device_bytes, hip
from test_gpu_parity import make_data
from test_gpu_predict import _random_model, both_ways

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
    # (the matrix alone is 17 MB of bins and 67 MB of floats; the runtime takes memory of its own, 16 MB at a time)
    assert free_device_bytes() > before - 48 * MB
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


class Held:
    """Device memory held back, so that `leave` bytes are free."""

    def __init__(self, leave):
        self.blocks = []
        while free_device_bytes() > leave + MB:
            p = ctypes.c_void_p()
            want = min(free_device_bytes() - leave, 8 << 30)
            if hip().hipMalloc(ctypes.byref(p), want) != 0:
                break
            self.blocks.append(p.value)

    def release(self):
        for p in self.blocks:
            hip().hipFree(p)
        self.blocks = []


@pytest.fixture
def held():
    made = []

    def hold(leave):
        gc.collect()
        import arboretum_amd
        arboretum_amd.release_memory()
        made.append(Held(leave))
        return made[-1]
    yield hold
    for h in made:
        h.release()


def test_no_memory_for_another_lane(arb, oracle, held):
    # 200 features, max_depth 10: 3 GB for a lane; there is room for one
    n, F, K = 3000, 200, 4
    rng = np.random.default_rng(5)
    X = rng.integers(0, 256, size=(n, F), dtype=np.uint8)
    labels = ((X[:, 0] > 100).astype(np.uint8) + 2 * (X[:, F - 1] > 60)).astype(np.uint8)
    cfg = _config(10, bins=256, labels_count=K)
    cfg["objective"] = 4
    data = arb.DMatrix(X, labels=labels, quantized=True)

    def grow():
        g = arb.Garden(cfg, data)
        g.labels_count = K
        for _ in range(2):
            g.grow_tree()
        return g
    free = grow()
    hold = held(4608 * MB)
    assert hold.blocks and free_device_bytes() < 5000 * MB
    tight = grow()
    arb.release_memory()
    assert 512 * MB < free_device_bytes() < 2560 * MB   # one lane, and none left half made
    for t in range(2 * K):
        a, b = free.tree(t), tight.tree(t)
        for key in ("fid", "quantized", "gain", "weights"):
            assert np.array_equal(a[key], b[key], equal_nan=True), (key, t)
    assert np.array_equal(free.train_yhat(), tight.train_yhat())


def test_no_memory_for_the_rows(arb, held):
    # the rows stay on the host and are walked through a block
    n, F = 500_000, 600
    rng = np.random.default_rng(6)
    X = np.tile(rng.standard_normal((5000, F), dtype=np.float32), (n // 5000, 1))
    X[np.arange(n), rng.integers(0, F, n)] = 3.0
    g = arb.load(_random_model(rng, [6, 3, 9, 5], F, fid_max=F))
    held(1100 * MB)
    before = free_device_bytes()
    data = arb.DMatrix(X)                       # 1.2 GB
    assert free_device_bytes() > before - 300 * MB
    both_ways(g, data)
    g.append_last_tree(data)


def test_rows_beyond_what_a_matrix_may_keep_on_the_device(arb):
    # 8.6 GB of floats: quantised and walked piece by piece from the host
    n, F = 2_000_000, 1080
    rng = np.random.default_rng(8)
    tile = rng.standard_normal((2000, F), dtype=np.float32)
    tile[:, 500] = np.round(tile[:, 500])
    X = np.tile(tile, (n // 2000, 1))
    some = [0, 3, 500, F - 1]
    X[:, some] += 0.001 * rng.standard_normal((n, len(some)), dtype=np.float32)
    y = (X[:, 0] + X[:, F - 1] + 0.3 * rng.standard_normal(n, dtype=np.float32) > 0).astype(np.float32)
    before = free_device_bytes()
    data = arb.DMatrix(X, y=y)
    assert free_device_bytes() > before - 1024 * MB
    few = arb.DMatrix(X[:, some], y=y)
    g = arb.train(_config(3, bins=100), data, 2)
    few.quantize(100)
    for k, f in enumerate(some):
        a, b = data.thresholds(f, 100), few.thresholds(k, 100)
        assert a[1] == b[1] and np.array_equal(a[0], b[0]), f
    # (training walks the bins and prediction the floats: they differ where a value equals a threshold)
    p = both_ways(g, data)
    trained = 1.0 / (1.0 + np.exp(-g.train_yhat().astype(np.float64)))
    assert (np.abs(p - trained) > 1e-6).mean() < 1e-3
    assert ((p > 0.5) == (y > 0.5)).mean() > 0.6
