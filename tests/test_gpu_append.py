"""Predictions of an evaluation matrix advanced tree by tree (AAppendLastTree): on the GPU and on the host
the same bits, also where the matrix carries the predictions of a booster with another number of classes."""
import numpy as np
import pytest

from test_gpu_parity import make_data

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
