"""Work memory, streams and threads that outlive a booster: a booster that runs on what others have
left behind grows the checker's trees, from several host threads as well."""
import threading

import numpy as np
import pytest

from test_gpu_parity import make_data

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def arb():
    import arboretum_amd
    if arboretum_amd.device_count() < 1:
        pytest.fail("no HIP device: the GPU tests need an MI355X")
    return arboretum_amd


# (rows, features, objective, hist_size, depth, NaN share, method): shapes that take each other's blocks
SHAPES = [(3000, 9, 1, 64, 4, 0.0, 1), (2900, 40, 0, 32, 5, 0.1, 1), (3100, 12, 0, 300, 3, 0.0, 1),
          (700, 5, 1, 16, 4, 0.0, 0), (3000, 70, 1, 255, 5, 0.0, 1)]


def _problem(k):
    n, F, objective, bins, depth, nan, method = SHAPES[k]
    X, y = make_data(n, F, objective, seed=50 + k, nan_frac=nan)
    cfg = {"objective": objective, "method": method,
           "internals": {"hist_size": bins, "double_precision": True, "exact_sort": 1},
           "tree": {"max_depth": depth, "eta": 0.3, "lambda": 1.0, "min_child_weight": 0.0}}
    return X, y, cfg


def _trees(arb, X, y, cfg):
    g = arb.train(cfg, arb.DMatrix(X, y=y), 3)
    return [g.tree(t) for t in range(3)], g.train_yhat()


def _check(ob, got):
    trees, yhat = got
    for t, tree in enumerate(trees):
        want = ob.tree(t)
        for key in ("fid", "quantized", "gain", "weights"):
            assert np.array_equal(want[key], tree[key], equal_nan=True), (key, t)
    assert np.array_equal(ob.yhat(), yhat)


@pytest.fixture(scope="module")
def wanted(oracle):
    out = []
    for k in range(len(SHAPES)):
        X, y, cfg = _problem(k)
        ob = oracle.Booster(X, y=y, config=cfg)
        ob.grow(3)
        out.append(ob)
    return out


def test_boosters_one_after_the_other(arb, wanted):
    for k in (0, 1, 2, 3, 4, 3, 2, 1, 0, 4, 0):
        _check(wanted[k], _trees(arb, *_problem(k)))


def test_boosters_of_several_threads(arb, wanted):
    got = [None] * (2 * len(SHAPES))

    def work(i):
        got[i] = _trees(arb, *_problem(i % len(SHAPES)))
    threads = [threading.Thread(target=work, args=(i,)) for i in range(len(got))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for i, g in enumerate(got):
        _check(wanted[i % len(SHAPES)], g)


def test_new_target_leaves_a_running_booster_alone(arb, oracle):
    import ctypes
    X, y, cfg = _problem(0)
    data = arb.DMatrix(X, y=y)
    g = arb.Garden(cfg, data)
    g.grow_tree()
    other = np.ascontiguousarray(1 - y, dtype=np.float32)
    lib = arb.core._LIB
    assert lib.ASetY(data.handle, other.ctypes.data_as(ctypes.POINTER(ctypes.c_float))) is None
    h = arb.Garden(cfg, data)   # takes blocks the old target's copy would have gone back to
    h.grow_tree()
    g.grow_tree()
    for booster, target in ((g, y), (h, other)):
        ob = oracle.Booster(X, y=target, config=cfg)
        ob.grow(booster.num_trees())
        for t in range(booster.num_trees()):
            assert np.array_equal(ob.tree(t)["fid"], booster.tree(t)["fid"])
            assert np.array_equal(ob.tree(t)["weights"], booster.tree(t)["weights"])


def test_threads_predict_on_one_booster(arb):
    # the first of them fetches the trees from the GPU, and each has its own sums
    X, y, cfg = _problem(4)
    rng = np.random.default_rng(9)
    rows = [rng.standard_normal((200 * (k + 1) + k, X.shape[1]), dtype=np.float32) for k in range(6)]
    train = arb.DMatrix(X, y=y)
    want = None
    for _ in range(6):
        g = arb.train(cfg, train, 3)
        got = [None] * len(rows)
        start = threading.Barrier(len(rows))

        def work(k):
            data = arb.DMatrix(rows[k])
            start.wait()
            for _ in range(4):
                got[k] = g.predict(data)
        threads = [threading.Thread(target=work, args=(k,)) for k in range(len(rows))]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
        if want is None:
            g.predict_on_device(False)
            want = [g.predict(arb.DMatrix(r)) for r in rows]
        assert all(np.array_equal(a, b) for a, b in zip(got, want))
