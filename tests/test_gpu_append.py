"""Predictions of an evaluation matrix advanced tree by tree (AAppendLastTree): on the GPU and on the host
the same bits, also where the matrix carries the predictions of a booster with another number of classes."""
import numpy as np
import pytest

from test_gpu_blocks import to_block
from test_gpu_parity import make_data
from test_gpu_predict import _random_model, both_ways

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def arb():
    import arboretum_amd
    if arboretum_amd.device_count() < 1:
        pytest.fail("no HIP device")
    return arboretum_amd


def _boosters(arb, n, F):
    X, y = make_data(n, F, 0, seed=n)
    labels = ((X[:, 0] > 0) + (X[:, 1] > 0.5)).astype(np.uint8)
    base = {"method": 1, "internals": {"hist_size": 32, "double_precision": True}}
    three = dict(base, objective=4, tree={"max_depth": 4, "eta": 0.3, "labels_count": 3})
    one = dict(base, objective=0, tree={"max_depth": 3, "eta": 0.3})
    return arb.train(three, arb.DMatrix(X, labels=labels), 2), arb.train(one, arb.DMatrix(X, y=y), 2)


def _raw(arb, linear, data, classes):
    """All predictions the matrix carries (the linear objective returns them as they are)."""
    out = np.empty(classes * data.rows, np.float32)
    assert arb.core._LIB.AGetYInto(linear.handle, data.handle, out.ctypes.data, out.size) is None
    return out


# (rows beyond 2^20 / 3 floats: the predictions of three classes leave the memory of one class's far behind)
@pytest.mark.parametrize("n", [7, 5000, 400001])
@pytest.mark.parametrize("first", ["three", "one"])
def test_boosters_of_other_numbers_of_classes(arb, n, first):
    three, one = _boosters(arb, 3000, 6)
    X, _ = make_data(n, 6, 0, seed=2)
    got = []
    for on_device in (True, False):
        data = arb.DMatrix(X)
        for g in (three, one):
            g.predict_on_device(on_device)
        order = (three, one) if first == "three" else (one, three)
        seen = []
        for g in (*order, order[1]):
            g.append_last_tree(data)
            seen.append(_raw(arb, one, data, 3 if first == "three" else 1))
        got.append(seen)
    for a, b in zip(*got):
        assert np.array_equal(a, b)
    # the booster that came second advances the classes both have, and nothing else
    assert not np.array_equal(got[0][0][:n], got[0][1][:n])
    assert np.array_equal(got[0][0][n:], got[0][2][n:])


def _appended(arb, g, data, classes, times=2):
    for _ in range(times):
        g.append_last_tree(data)
    linear = arb.Garden({"objective": 0})
    linear.predict_on_device()   # (makes its handle)
    return _raw(arb, linear, data, classes)


def _both(arb, g, make, classes):
    """Appended on the GPU and on the host: the same bits."""
    got = []
    for on_device in (True, False):
        g.predict_on_device(on_device)
        got.append(_appended(arb, g, make(), classes))
    g.predict_on_device(True)
    assert np.array_equal(*got)
    return got[0]


# the host walks what the GPU does not take: matrices without dense columns, bin ids of which one row is
# larger than a staging block (4 MB)
def test_matrix_without_dense_columns(arb):
    _, one = _boosters(arb, 3000, 6)
    categories = np.zeros((500, 2), np.uint32)
    out = _both(arb, one, lambda: arb.DMatrix(np.empty((500, 0), np.float32), data_category=categories), 1)
    assert np.isfinite(out).all() and np.unique(out).size == 1 and out[0] != 0.5


def test_rows_larger_than_a_staging_block(arb):
    F = (4 << 20) + 5
    rng = np.random.default_rng(1)
    bins = rng.integers(0, 256, size=(3, F), dtype=np.uint8)
    g = arb.load(_random_model(rng, [4, 3, 5], F, fid_max=F))
    _both(arb, g, lambda: arb.DMatrix(bins, quantized=True), 1)
    both_ways(g, arb.DMatrix(bins, quantized=True))


# sums of more than 128 MB come back in ranges of rows, of whole blocks where the bins are in blocks
@pytest.mark.parametrize("kind", ["floats", "bins", "blocks"])
def test_ranges_of_rows(arb, kind):
    K, n, F, block = 40, 900001, 5, 1 << 18
    rng = np.random.default_rng(7)
    small = rng.integers(0, 16, size=(4000, F), dtype=np.uint8)
    cfg = {"objective": 4, "method": 1, "internals": {"hist_size": 16}, "tree": {"max_depth": 3, "eta": 0.3, "labels_count": K}}
    labels = ((small[:, 0].astype(int) * 16 + small[:, 1]) % K).astype(np.uint8)
    g = arb.train(cfg, arb.DMatrix(small, labels=labels, quantized=True), 1)
    bins = rng.integers(0, 16, size=(n, F), dtype=np.uint8)
    held = [to_block(bins[r:r + block], block) for r in range(0, n, block)]
    make = {"floats": lambda: arb.DMatrix(bins.astype(np.float32)), "bins": lambda: arb.DMatrix(bins, quantized=True),
            "blocks": lambda: arb.DMatrix.from_blocks([b.ptr for b in held], block, n, F)}[kind]
    out = _both(arb, g, make, K).reshape(K, n)
    assert all(np.unique(out[k]).size > 1 for k in (0, 17, K - 1))
