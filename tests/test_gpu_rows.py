"""Rows of a matrix on the device: quantiser and tree walks at the edges of their tiles, for matrices kept
in pinned memory, on the device and (built before this process used the GPU) on the host."""
import subprocess
import sys

import numpy as np
import pytest

from test_gpu_parity import make_data
from test_gpu_predict import _random_model, both_ways

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def arb():
    import arboretum_amd
    if arboretum_amd.device_count() < 1:
        pytest.fail("no HIP device: the GPU tests need an MI355X")
    return arboretum_amd


# rows: a wave, a workgroup of 64 ... 1024 rows and one more; features: a tile of values in the LDS
# beside the trees, less rows because of it, none (600: more than 64 rows' worth)
@pytest.mark.parametrize("n,F", [(1, 1), (63, 5), (64, 33), (65, 300), (1025, 600), (16385, 28), (40961, 100),
                                 (262145, 3), (262144, 36), (262300, 70)])
@pytest.mark.parametrize("depths", [[6] * 9, [3, 9, 2, 9, 9, 9, 9, 5] * 4])
def test_walks_at_tile_edges(arb, n, F, depths):
    rng = np.random.default_rng(n + F)
    g = arb.load(_random_model(rng, depths, F, fid_max=F))
    X = rng.standard_normal(size=(n, F), dtype=np.float32)
    X[::7, 0] = np.nan
    both_ways(g, arb.DMatrix(X))


# the most features of which 64 rows have their values in the LDS, and one more: read from memory row by row
@pytest.mark.parametrize("F", [467, 468])
@pytest.mark.parametrize("n", [64, 16449])
def test_walks_at_the_widest_tile(arb, n, F):
    rng = np.random.default_rng(n + F)
    g = arb.load(_random_model(rng, [7] * 30 + [4, 9], F, fid_max=F))
    both_ways(g, arb.DMatrix(rng.standard_normal((n, F), dtype=np.float32)))


@pytest.mark.parametrize("n", [1000, 70000])
def test_many_trees_of_several_labels(arb, n):
    # several chunks of trees, the labels changing inside and between them; the model is laid out again
    # when trees are added and when fewer are asked for
    X, _ = make_data(n, 6, 1, seed=3)
    labels = (np.abs(X[:, 0]) * 2).astype(np.uint8) % 3
    cfg = {"objective": 4, "method": 1, "internals": {"hist_size": 32},
           "tree": {"max_depth": 7, "eta": 0.3, "lambda": 1.0, "labels_count": 3}}
    data = arb.DMatrix(X, labels=labels)
    g = arb.train(cfg, data, 15)
    both_ways(g, data)
    both_ways(g, data, 1)
    both_ways(g, data, 20)
    g.grow_tree()
    both_ways(g, data)


# tiles of 4096 keys, 64 rows and 32 features of the transposition
@pytest.mark.parametrize("n,F,hist_size", [(1, 1, 16), (2, 3, 16), (63, 33, 255), (4095, 2, 64), (4097, 66, 255),
                                           (8193, 5, 700), (70001, 30, 256)])
@pytest.mark.parametrize("nan_frac", [0.0, 0.3])
def test_thresholds_and_bins(arb, oracle, n, F, hist_size, nan_frac):
    X, y = make_data(n, F, 1, seed=n, nan_frac=nan_frac)
    X[:, 0] *= np.where(np.arange(n) % 3 == 0, -0.0, 1.0).astype(np.float32)   # zeros of both signs
    cfg = {"objective": 1, "method": 1, "internals": {"hist_size": hist_size}, "tree": {"max_depth": 2}}
    data = arb.DMatrix(X, y=y)
    data.quantize(hist_size)
    ob = oracle.Booster(X, y=y, config=cfg)
    got = data.bins()
    assert np.array_equal(got, ob.bins().astype(got.dtype))
    for f in range(F):
        t0, s0 = ob.thresholds(f)
        t1, s1 = data.thresholds(f, hist_size)
        assert s0 == s1 and np.array_equal(t0, t1), f


def test_matrix_built_before_the_gpu_is_used(arb):
    # the first matrices of a process stay on the host and reach the device with the first booster
    code = """
import numpy as np, arboretum_amd as arb
rng = np.random.default_rng(1)
X = rng.standard_normal((50000, 9), dtype=np.float32)
y = (X[:, 0] > X[:, 3]).astype(np.float32)
cfg = {"objective": 1, "method": 1, "internals": {"hist_size": 64, "double_precision": True}, "tree": {"max_depth": 4}}
first, other = arb.DMatrix(X, y=y), arb.DMatrix(X[::-1])
g = arb.train(cfg, first, 3)
h = arb.train(cfg, arb.DMatrix(X, y=y), 3)
assert np.array_equal(g.train_yhat(), h.train_yhat())
assert np.array_equal(g.predict(other), h.predict(arb.DMatrix(X[::-1])))
"""
    subprocess.run([sys.executable, "-c", code], check=True, timeout=100)
